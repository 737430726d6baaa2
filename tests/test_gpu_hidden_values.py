"""What lies behind the causal mask must not be seen: a V row (or the scale row of a V block) that is not finite, as the padding behind a
prompt may hold, leaves the rows alone whose keys end before it.  The kernels multiply P = 0 with the hidden keys of a 32-key sub-tile
(of a key block, for the scales) that some row of a 32-row group does see, and with no others; the eight-wave kernels of head_dim 256 do so for
the 64-key blocks that a 128-row group sees."""
import pytest
import torch

import int_flashattention_amd as M
from many_heads import repetitions

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAN = float("nan")


def inputs(variant, H, Nq, Nk, D, dt, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q, k, v = (torch.randn((1, H, n, D), generator=g, device=DEV).to(dt) for n in (Nq, Nk, Nk))
    if variant == "fp":
        return q, k, v
    (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
    return q8, k8, v, qs, ks


def call(variant, args, v, sm, **kw):
    if variant == "fp":
        return M.attention(args[0], args[1], v, True, sm, **kw)
    return M.attention_int8(args[0], args[1], v, args[3], args[4], True, sm, **kw)


# One head (times reps) per hidden position: about twenty at 300 keys, forty at 600.  Head_dim 128 is the pipelined kernel from 65 rows on;
# head_dim 64 the decode-shaped kernel up to 512 workgroups of 32 rows (N 320), the pipelined one (N 600), the one with three waves per SIMD
# past 512 workgroups of 128 rows (N 600, three times the heads); head_dim 256 the decode-shaped and the eight-wave kernel.  More keys than
# queries by a part of a sub-tile, by one and by two blocks; split passes
@pytest.mark.parametrize("variant", ["half", "fp"])
@pytest.mark.parametrize("D,reps,Nq,Nk,splits", [
    (128, 1, 300, 300, 1), (128, 1, 384, 384, 1), (128, 1, 129, 200, 1), (128, 1, 260, 324, 1), (128, 1, 256, 384, 1), (128, 1, 330, 330, 3),
    (64, 1, 320, 320, 1), (64, 1, 200, 271, 1), (64, 1, 256, 320, 1), (64, 1, 64, 100, 2),
    (64, 1, 600, 600, 1), (64, 1, 576, 640, 1), (64, 1, 600, 600, 2), (64, 3, 600, 600, 1), (256, 1, 300, 300, 1), (256, 2, 300, 300, 1),
    (64, 1, 64, 612, 1), (128, 1, 64, 612, 1), (256, 1, 64, 612, 1),
])
def test_non_finite_values_behind_the_mask_reach_no_row_before_them(variant, D, reps, Nq, Nk, splits):
    off, sm, dt = Nk - Nq, D ** -0.5, torch.bfloat16 if Nq % 2 else torch.float16
    # one hidden position per head: edges of sub-tiles and blocks, and keys in between
    at = sorted({t for s in range(0, Nk, 64) for t in (s, s + 31, s + 32, s + 63) if off < t < Nk} | {Nk - 1})
    H = len(at) * reps
    args = inputs(variant, H, Nq, Nk, D, dt, Nq + Nk + D)
    v = args[2]
    clean = call(variant, args, v, sm, num_splits=splits)
    bad = v.clone()
    for h in range(H):
        bad[0, h, at[h % len(at)]] = NAN if h % 2 else float("inf")
    got = call(variant, args, bad, sm, num_splits=splits)
    torch.cuda.synchronize()
    rows = torch.arange(Nq)
    for h in range(H):
        t = at[h % len(at)]
        if D == 256 and Nq > 64:
            safe = (rows // 128 * 128 + 127 + off) // 64 < t // 64
        else:
            safe = (rows // 32 * 32 + 31 + off) // 32 < t // 32
        sees = rows + off >= t
        o, c = got[0, h].cpu(), clean[0, h].cpu()
        assert torch.equal(o[safe], c[safe]), (t, rows[safe][(o[safe] != c[safe]).any(-1)])
        assert not torch.isfinite(o[sees]).any(), t
        assert safe.any() or t <= off + 190


# The scales of a V block behind the mask; head_dim 64 and 256 take two blocks per step in the decode-shaped kernel (reps 1), the other grids
# run the general kernels
@pytest.mark.parametrize("D,reps,Nq,Nk,vsb", [
    (64, 1, 320, 320, 64), (64, 1, 200, 456, 128), (64, 1, 60, 450, 64), (64, 16, 320, 320, 64), (128, 1, 400, 400, 128), (128, 16, 400, 400, 128),
    (256, 1, 256, 320, 64), (256, 1, 300, 300, 64), (256, 16, 256, 320, 64),
])
def test_non_finite_v_scales_behind_the_mask_reach_no_row_before_them(D, reps, Nq, Nk, vsb):
    off, sm = Nk - Nq, D ** -0.5
    first = [s for s in range(vsb, Nk, vsb) if s > off]
    H = len(first) * reps
    q8, k8, v, qs, ks = inputs("half", H, Nq, Nk, D, torch.float16, D + Nq)
    v8, vs = M.quant_perblock_channel(v, vsb)
    run = lambda s: M.attention_full_int8(q8, k8, v8, qs, ks, s, True, sm, v_scale_block=vsb)
    clean = run(vs)
    bad = vs.clone()
    for h in range(H):
        bad[0, h, first[h % len(first)] // vsb] = NAN
    got = run(bad)
    torch.cuda.synchronize()
    rows = torch.arange(Nq)
    group = 128 if D == 256 else 32
    for h in range(H):
        s = first[h % len(first)]
        safe = rows // group * group + group - 1 + off < s
        o, c = got[0, h].cpu(), clean[0, h].cpu()
        assert torch.equal(o[safe], c[safe]), (s, rows[safe][(o[safe] != c[safe]).any(-1)])
        assert not torch.isfinite(o[rows + off >= s]).any(), s


# an odd number of 64-key blocks per entry: the second block of the last step (head_dim 128: the second scale row of the last block) is past
# the entry's length
@pytest.mark.parametrize("D,Nq", [(64, 1), (64, 100), (256, 1), (256, 100), (128, 1), (128, 100)])
def test_scale_rows_past_an_entrys_length_are_not_used(D, Nq):
    lens, Nk, vsb = [64, 180], 384, 64
    g = torch.Generator(device=DEV).manual_seed(D + Nq)
    q, k, v = (torch.randn((2, 2, n, D), generator=g, device=DEV).half() for n in (Nq, Nk, Nk))
    (q8, qs), (k8, ks), (v8, vs) = M.quant_pertoken(q), M.quant_pertoken(k), M.quant_perblock_channel(v, vsb)
    run = lambda s: M.attention_full_int8(q8, k8, v8, qs, ks, s, False, D ** -0.5, v_scale_block=vsb,
                                          seqlens_k=torch.tensor(lens, dtype=torch.int32, device=DEV))
    clean = run(vs)
    bad = vs.clone()
    for b, n in enumerate(lens):
        bad[b, :, -(-n // vsb):] = NAN
    got = run(bad)
    torch.cuda.synchronize()
    assert torch.equal(got, clean) and torch.isfinite(got).all()


# Hidden keys of a row whose scores are all zero: a query row of zeros has the scale zero, sm_scale may be zero.  Every key that the row sees
# weighs the same: the output is the mean of its values.  reps: the decode-shaped and the general kernels; ragged ends and the causal diagonal
@pytest.mark.parametrize("variant", ["full", "half", "fp"])
@pytest.mark.parametrize("D,reps,Nq,Nk,splits", [(64, 1, 100, 100, 1), (64, 150, 100, 100, 1), (64, 20, 600, 600, 1), (64, 1, 5, 300, 3),
                                                 (128, 1, 100, 100, 1), (128, 150, 100, 231, 1), (128, 2, 300, 300, 2), (128, 1, 5, 300, 3),
                                                 (256, 1, 100, 100, 1), (256, 80, 100, 100, 1)])
@pytest.mark.parametrize("causal", [False, True])
def test_hidden_keys_of_a_row_without_scores(variant, D, reps, Nq, Nk, splits, causal):
    g = torch.Generator(device=DEV).manual_seed(D + Nq)
    q, k, v = (torch.randn((1, reps, n, D), generator=g, device=DEV).half() for n in (Nq, Nk, Nk))
    zero = [0, Nq // 2, Nq - 1]
    q[:, :, zero] = 0
    def run(sm):
        if variant == "fp":
            return M.attention(q, k, v, causal, sm, num_splits=splits)
        (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        if variant == "half":
            return M.attention_int8(q8, k8, v, qs, ks, causal, sm, num_splits=splits)
        v8, vs = M.quant_pertensor(v)
        return M.attention_full_int8(q8, k8, v8, qs, ks, vs, causal, sm, num_splits=splits)
    some, flat = run(D ** -0.5), run(0.0)
    torch.cuda.synchronize()
    assert torch.isfinite(some).all()
    # P is the same for every key: only V's int8 rounding (full) and the 16-bit output are left
    tol = 2e-3 + (v.abs().max().item() / 127 / 2 if variant == "full" else 0)
    for rows, out in ((zero, some), (range(0, Nq, 7), flat)):
        for r in rows:
            n = r + 1 + Nk - Nq if causal else Nk
            assert (out[0, :, r].float() - v[0, :, :n].float().mean(1)).abs().max().item() <= tol, (r, n)


# A score that is not a number, of a key that rows do see: they are NaN, also the row that sees no other key (the first one) and rows of a cache
# with one ragged block in which every key is like that.  The first key of every head; grids past the decode-shaped kernels
@pytest.mark.parametrize("variant,D,v_block", [("full", 64, None), ("full", 64, 64), ("full", 128, None), ("full", 128, 128), ("full", 128, 64), ("half", 128, None),
                                               ("fp", 128, None)])
@pytest.mark.parametrize("scale_dtype", [torch.float16, torch.float32])
def test_visible_scores_that_are_not_numbers(variant, D, v_block, scale_dtype):
    for Nq, Nk, causal in ((200, 200, True), (600, 600, True), (200, 45, False)):
        H = repetitions(1, 1, Nq)
        q, k, v = (torch.randn((1, H, n, D), generator=torch.Generator(device=DEV).manual_seed(n + i), device=DEV).half() for i, n in enumerate((Nq, Nk, Nk)))
        bad = slice(0, 1) if causal else slice(None)
        if variant == "fp":
            k[:, :, bad, 3] = NAN
            out, lse = M.attention(q, k, v, causal, 0.1, return_lse=True)
        else:
            (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
            ks[:, :, bad] = NAN
            qs, ks = qs.to(scale_dtype), ks.to(scale_dtype)
            if variant == "half":
                out, lse = M.attention_int8(q8, k8, v, qs, ks, causal, 0.1, return_lse=True)
            else:
                v8, vs = M.quant_perblock_channel(v, v_block) if v_block else M.quant_pertensor(v)
                vs = vs if v_block else vs.to(scale_dtype)
                out, lse = M.attention_full_int8(q8, k8, v8, qs, ks, vs, causal, 0.1, return_lse=True, v_scale_block=v_block)
        torch.cuda.synchronize()
        assert bool(lse.isnan().all()) and bool(out.isnan().all()), (Nq, Nk, causal, int((~lse.isnan()).sum()))
