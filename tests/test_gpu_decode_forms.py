"""The decode-shaped kernels (csrc/intfa_fwd_decode_wide.h) at the edges of their steps, frames and row tiles: key counts around a 16-key
tile, a frame and a step, rows around a 16-row tile and a 32-row block, against the oracle; and their forms (half steps past one workgroup per
compute unit, one row tile per workgroup in small grids), which a batch element meets by the number of heads beside it and which must give
the same bits."""
import pytest
import torch

import intfa_oracle as O
import int_flashattention_amd as M
from test_gpu_parity import MAX_ABS, assert_same_rounding, max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def problem(variant, H, Nq, Nk, D, seed):
    g = torch.Generator().manual_seed(seed)
    dt = torch.bfloat16 if seed % 2 else torch.float16
    q, k, v = (torch.randn((1, H, n, D), generator=g).to(dt) for n in (Nq, Nk, Nk))
    k[:, :, Nk // 2:] *= 2                               # the running maximum rises on the way: the frames differ
    if variant == "fp":
        return (q, k, v)
    (q8, qs), (k8, ks) = O.quant_pertoken(q), O.quant_pertoken(k)
    if variant == "half":
        return (q8, k8, v, qs, ks)
    v8, vs = O.quant_pertensor(v)
    return (q8, k8, v8, qs, ks, vs)


def run(variant, args, causal, sm, dt, **kw):
    args = [t.to(DEV) for t in args]
    if variant == "full":
        return M.attention_full_int8(*args, causal, sm, out_dtype=dt, return_lse=True, **kw)
    return (M.attention if variant == "fp" else M.attention_int8)(*args, causal, sm, return_lse=True, **kw)


def exact(args, variant, causal, sm):
    """Attention in float64 on the dequantised operands."""
    if variant == "fp":
        q, k, v = (t.double() for t in args)
    else:
        q, k = args[0].double() * args[3].double()[..., None], args[1].double() * args[4].double()[..., None]
        v = args[2].double() * (args[5].double()[..., None, None] if variant == "full" else 1.0)
    s = q @ k.transpose(-1, -2) * sm
    Nq, Nk = s.shape[-2:]
    if causal:
        s = s.masked_fill(torch.arange(Nk)[None, :] > torch.arange(Nq)[:, None] + (Nk - Nq), float("-inf"))
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1) * 1.4426950408889634


def oracle(args, causal, sm, D):
    """Full-int8 with the kernel's frames; the oracle has no mask for unequal lengths, and a causal row is a row of a shorter cache."""
    q8, k8, v8, qs, ks, vs = args
    Nq, Nk = q8.shape[2], k8.shape[2]
    rows = [(slice(None), Nk)] if not causal else [(slice(i, i + 1), i + Nk - Nq + 1) for i in range(Nq)]
    return torch.cat([O.attention_full_int8(q8[:, :, r], k8[:, :, :n], v8[:, :, :n], qs[:, :, r], ks[:, :, :n], vs, False, sm,
                                            block_n=M.block_n("full", D)) for r, n in rows], 2)


# Full-int8 against the oracle: the same frames and roundings but for the last place of exp2, which moves a P8 that lies on a boundary by one
# step: 1 / 127 of the row's largest v at most where that key is a row's only one, one of many keys elsewhere (the bounds of
# test_gpu_parity.py).  The 16-bit variants against float64: P and the output are rounded to 11 (bf16: 8) bits, half an ulp is 2^-12 (2^-9)
# each: 1e-3 and 8e-3 of the norm hold the sum of both.
@pytest.mark.parametrize("Nk", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 400, 513])
@pytest.mark.parametrize("variant,D", [(v, d) for v in ("full", "half", "fp") for d in (64, 128, 256)])
def test_key_counts_around_tiles_frames_and_steps(variant, D, Nk):
    for Nq, causal in ((1, False), (15, True), (17, False), (33, True)):
        if causal and Nk < Nq:
            continue
        args = problem(variant, 2, Nq, Nk, D, Nk + Nq)
        dt = args[2].dtype if variant != "full" else torch.float16
        out, lse = run(variant, args, causal, D ** -0.5, dt)
        want, want_lse = exact(args, variant, causal, D ** -0.5)
        assert (lse.double().cpu() - want_lse).abs().max().item() <= 1e-3, (Nq, causal)
        if variant != "full":
            assert (out.double().cpu() - want).norm() / want.norm() <= (1e-3 if dt == torch.float16 else 8e-3), (Nq, causal)
            continue
        ref = oracle(args, causal, D ** -0.5, D)
        assert max_abs(out, ref) <= MAX_ABS
        if Nk >= 64 and not causal:
            assert_same_rounding(out, ref)


# few heads: one row tile per workgroup, steps of two 128-key blocks; 300 heads: two row tiles and (head_dim 128) steps of one block
@pytest.mark.parametrize("Nq,Nk,causal,splits", [(1, 700, False, 1), (16, 385, True, 1), (17, 640, True, 1), (20, 300, False, 1), (40, 1029, True, 3), (33, 390, False, 1), (5, 2000, False, 5)])
@pytest.mark.parametrize("variant,D", [(v, d) for v in ("full", "half", "fp") for d in (64, 128, 256)])
def test_the_forms_give_the_same_bits(variant, D, Nq, Nk, causal, splits):
    args = problem(variant, 2, Nq, Nk, D, Nq + Nk)
    dt = args[2].dtype if variant != "full" else torch.float16
    few = run(variant, args, causal, D ** -0.5, dt, num_splits=splits)
    many = run(variant, [t.repeat(1, 150, *([1] * (t.dim() - 2))) for t in args], causal, D ** -0.5, dt, num_splits=splits)
    torch.cuda.synchronize()
    for a, b in zip(few, many):
        assert torch.equal(a, b[:, :2]) and torch.equal(a, b[:, -2:])
