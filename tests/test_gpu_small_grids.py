"""A problem of few workgroups runs the kernel whose waves share the keys of a block, a larger one the kernel whose waves have 32
query rows each: an output must not depend on which, so one (batch, head) pair computed alone equals, bit for bit, the same pair
among so many others that the general kernel takes the call."""
import pytest
import torch

import int_flashattention_amd as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


# lengths: a part of a block, a whole one, one row past a 32-row and a 128-row query block, several blocks; more and fewer keys
# than queries; a bottom-right offset that is no multiple of a block
@pytest.mark.parametrize("Nq,Nk", [(65, 65), (128, 128), (129, 129), (257, 257), (500, 500), (200, 331), (300, 200)])
@pytest.mark.parametrize("variant,D,p_round", [("full", 128, "reference"), ("full", 128, "rne"), ("full", 64, "reference"), ("full", 256, "reference"),
                                               ("half", 64, None), ("fp", 64, None), ("half", 256, None), ("fp", 256, None)])
@pytest.mark.parametrize("causal", [False, True])
def test_output_does_not_depend_on_the_number_of_heads(variant, D, p_round, Nq, Nk, causal):
    dt = torch.bfloat16 if Nq % 2 else torch.float16
    g = torch.Generator(device=DEV).manual_seed(Nq + Nk + D)
    q, k, v = (torch.randn((1, 2, n, D), generator=g, device=DEV).to(dt) for n in (Nq, Nk, Nk))
    k[:, :, Nk // 2:] *= 3                          # the running maximum rises late: the frame of P moves
    sm = D ** -0.5
    many = 2 * 256 // ((Nq + 31) // 32) // 2 + 1    # repetitions of the two heads: past two workgroups of 32 rows per compute unit
    rep = lambda *ts: [t.repeat(1, many, *([1] * (t.dim() - 2))) for t in ts]
    if variant == "fp":
        call = lambda *a: M.attention(*a, causal, sm, return_lse=True)
        args = (q, k, v)
    else:
        (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        if variant == "half":
            call = lambda *a: M.attention_int8(*a, causal, sm, return_lse=True)
            args = (q8, k8, v, qs, ks)
        else:
            v8, vs = M.quant_pertensor(v)
            call = lambda *a: M.attention_full_int8(*a, causal, sm, out_dtype=dt, p_round=p_round, return_lse=True)
            args = (q8, k8, v8, qs, ks, vs)
    few, few_lse = call(*args)
    lots, lots_lse = call(*rep(*args))
    torch.cuda.synchronize()
    assert torch.equal(few, lots[:, -2:]) and torch.equal(few, lots[:, :2])
    assert torch.equal(few_lse, lots_lse[:, -2:])


# head_dim 64 of the 16-bit P V has a third kernel between the two; block counts 8 and 9 (even and odd), one hidden key, many
@pytest.mark.parametrize("N", [512, 513, 575, 640])
@pytest.mark.parametrize("variant", ["half", "fp"])
@pytest.mark.parametrize("causal", [False, True])
def test_output_does_not_depend_on_the_waves_per_simd(variant, N, causal):
    g = torch.Generator(device=DEV).manual_seed(N)
    q, k, v = (torch.randn((1, 2, N, 64), generator=g, device=DEV).half() for _ in range(3))
    k[:, :, N // 2:] *= 3
    if variant == "fp":
        call = lambda *a: M.attention(*a, causal, 0.125, return_lse=True)
        args = (q, k, v)
    else:
        (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        call = lambda *a: M.attention_int8(*a, causal, 0.125, return_lse=True)
        args = (q8, k8, v, qs, ks)
    outs = [call(*(t.repeat(1, heads // 2, *([1] * (t.dim() - 2))) for t in args)) for heads in (2, 48, 130)]   # 520 or more workgroups last
    torch.cuda.synchronize()
    for out, lse in outs[1:]:
        assert torch.equal(outs[0][0], out[:, -2:]) and torch.equal(outs[0][1], lse[:, -2:])
