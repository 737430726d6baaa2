"""k_scales at the upper end of their type: bf16 rows of magnitude 1e34 have scales of 8e31, whose product with the constant that the folded
dequantisation subtracts (kScoreBias in csrc/intfa_device.h) is past the largest fp32 number, and a caller may bring infinite ones.  The same
values as 32-bit scales, which are converted and multiplied, give the same bits, whichever kernel runs."""
import pytest
import torch

import int_flashattention_amd as M
from many_heads import repetitions

pytestmark = pytest.mark.gpu
DEV = "cuda"
INF = float("inf")


def same(a, b):
    """Equal bits, or NaN on both sides."""
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


# (16-bit scales of the general kernels; D 256: past 256 query blocks of 128 rows, several per workgroup)
KERNELS = [("full", 64, 300, 333, False, None, 1), ("full", 64, 300, 300, True, None, 1), ("full", 64, 130, 700, True, None, 2), ("full", 64, 130, 129, False, 64, 1),
           ("full", 64, 300, 300, True, 128, 1), ("full", 64, 130, 192, False, None, 1), ("full", 128, 130, 384, False, None, 1), ("full", 128, 300, 333, False, None, 1), ("full", 128, 300, 300, True, None, 1), ("full", 128, 90, 257, False, None, 1),
           ("full", 128, 300, 700, True, None, 2), ("full", 128, 300, 300, True, 128, 1), ("full", 256, 130, 200, False, None, 1),
           ("full", 256, 200, 200, True, None, 1), ("half", 128, 200, 333, False, None, 1), ("half", 128, 257, 257, True, None, 1), ("half", 64, 300, 300, False, None, 1)]


@pytest.mark.parametrize("variant,D,Nq,Nk,causal,v_block,splits", KERNELS)
@pytest.mark.parametrize("kind,dtype", [("one", torch.bfloat16), ("some", torch.bfloat16), ("all", torch.bfloat16), ("infinite", torch.bfloat16),
                                        ("infinite", torch.float16), ("infinite_hidden_sign", torch.bfloat16), ("infinite_hidden_sign", torch.float16),
                                        ("infinite_zeros", torch.bfloat16), ("infinite_zeros", torch.float16)])
def test_large_scales(variant, D, Nq, Nk, causal, v_block, splits, kind, dtype):
    H = -(-(repetitions(1, 1, Nq, rows=128) + 1) // 8) * 8
    g = torch.Generator(device=DEV).manual_seed(D + Nk)
    q8, k8 = (torch.randint(-127, 128, (1, H, n, D), generator=g, device=DEV, dtype=torch.int32).to(torch.int8) for n in (Nq, Nk))
    v = torch.randn((1, H, Nk, D), generator=g, device=DEV).to(dtype)
    qs, ks = (torch.rand((1, H, n), generator=g, device=DEV).mul(2e-3).to(dtype) for n in (Nq, Nk))
    if kind == "one":                        # one key of one head; the other workgroups have none
        ks[:, H // 2, Nk - 1] = 3e31
        qs.mul_(1e-35)
    elif kind == "some":                     # small q_scales: scores of ordinary size and tiny ones
        ks[:, :, 1::3], ks[:, :, 5::7], ks[:, :, 2::50] = 3e31, 7e31, 1.9e31
        qs.mul_(1e-35)
    elif kind == "all":
        ks.mul_(1e37).clamp_(min=1e32)
        qs.mul_(1e-40 if D == 64 else 1e-39)
    elif kind == "infinite":
        ks[:, :, 3::50] = INF
    elif kind == "infinite_zeros":           # no score is a number: of any key, of the first ones
        k8[:, ::2] = 0
        k8[:, 1::2, :2 * Nk // 3] = 0
        ks[:] = INF
    else:                                    # sums of one sign: the scores are -infinity, the keys weigh nothing
        q8.abs_().clamp_(min=1)
        k8[:, :, 3::50] = -1
        ks[:, :, 3::50] = INF
    def run(qs, ks):
        if variant == "half":
            return M.attention_int8(q8, k8, v, qs, ks, causal, 1.0, return_lse=True, num_splits=splits)
        return M.attention_full_int8(q8, k8, v8, qs, ks, vs, causal, 1.0, out_dtype=dtype, v_scale_block=v_block, return_lse=True, num_splits=splits)
    if variant == "full":
        v8, vs = M.quant_perblock_channel(v, v_block) if v_block else M.quant_pertensor(v)
        vs = vs.float()
    (a, la), (b, lb) = run(qs, ks), run(qs.float(), ks.float())
    torch.cuda.synchronize()
    assert same(a, b) and same(la, lb)
    if kind in ("one", "some", "infinite_hidden_sign"):
        assert bool(torch.isfinite(la).all()) and bool(torch.isfinite(a).all())
    if kind == "infinite":
        assert not torch.isfinite(la).all()


def test_scales_of_the_quantiser():
    """Rows of magnitude 1e34 through the quantiser, whose keys weigh by their scores: against the oracle's definition in 64 bits."""
    D, Nq, Nk = 128, 128, 256
    H = repetitions(1, 1, Nq, rows=128) + 1
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn((1, H, n, D), generator=g, device=DEV) for n in (Nq, Nk, Nk))
    k[:, :, ::2] *= 1e34
    k[:, :, 1::2] *= 3e33
    (q8, qs), (k8, ks), (v8, vs) = M.quant_pertoken((q * 1e-34).bfloat16()), M.quant_pertoken(k.bfloat16()), M.quant_pertensor(v.bfloat16())
    assert ks.float().max().item() > 6e31
    sm = D ** -0.5
    out = M.attention_full_int8(q8, k8, v8, qs, ks, vs, False, sm, out_dtype=torch.float16)
    S = (q8[0, :8].double() @ k8[0, :8].double().transpose(1, 2).contiguous()) * qs[0, :8].double()[..., None] * ks[0, :8].double()[:, None, :] * sm
    p = (S - S.max(-1, keepdim=True).values).exp()
    V = v8[0, :8].double() * vs.double().reshape(-1)[:8, None, None]
    want = p @ V / p.sum(-1, keepdim=True)
    # P is rounded to steps of 1/127, evenly distributed errors of 1 / (127 sqrt 12) each, independent of V: six standard deviations of their sum, and fp16
    tol = 6 * V.square().sum(1, keepdim=True).sqrt() / (127 * 12 ** 0.5) / p.sum(-1, keepdim=True) + 2e-3
    assert bool(((out[0, :8].double() - want).abs() <= tol).all())
    assert (want.abs() > 4 * tol).float().mean().item() > 0.2       # (the tolerance would show keys that are missing)
