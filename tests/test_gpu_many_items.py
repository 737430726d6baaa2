"""Full-int8 launches at head_dim 256 of more query blocks than compute units: a workgroup then takes several of them, and requests the next one's operands
under the last key blocks of the one before (launch_resident in csrc/intfa_launch.h).  Each batch entry alone is a launch of single blocks, which the
other tests compare with the oracle: same bits.  (Which launches take several: test_gpu_routes.py.)"""
import pytest
import torch

import int_flashattention_amd as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 256


def inputs(B, H, Hkv, Nq, Nk, dt, scales, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    # (query rows of a wider buffer: rows that are not back to back)
    wide = lambda x: torch.cat([x, x], dim=-1)[..., D:]
    q = torch.randn((B, H, Nq, D), generator=g, device=DEV).to(dt)
    k, v = (torch.randn((B, Hkv, Nk, D), generator=g, device=DEV).to(dt) for _ in range(2))
    (q8, qs), (k8, ks), (v8, vs) = M.quant_pertoken(q), M.quant_pertoken(k), M.quant_pertensor(v)
    return [wide(q8), k8, v8, qs.to(scales), ks.to(scales), vs.to(scales)]


def check_entries(args, causal, dt, lens=None, p_round="reference"):
    kw = dict(out_dtype=dt, return_lse=True, p_round=p_round)
    at = lambda b: {} if lens is None else dict(seqlens_k=lens[b])
    out, lse = M.attention_full_int8(*args, causal, D ** -0.5, **kw, **at(slice(None)))
    for b in range(args[0].shape[0]):
        o1, l1 = M.attention_full_int8(*(a[b:b + 1] for a in args), causal, D ** -0.5, **kw, **at(slice(b, b + 1)))
        assert torch.equal(out[b:b + 1].view(torch.int16), o1.view(torch.int16)), b
        assert torch.equal(lse[b:b + 1].view(torch.int32), l1.view(torch.int32)), b
    return out, lse


# three entries of 192 query blocks: two to four rounds of 256 workgroups, the last one partial; one entry alone: one round at most.  Causal lists
# of items agree in length for a multiple of 8 K/V heads in all (lists_agree)
# query rows, keys, causal: one key block, two, three and more, full and ragged ones; rows past the end of the last query block
@pytest.mark.parametrize("Nq,Nk,causal", [(128, 64, False), (77, 65, False), (128, 300, False), (100, 500, False), (128, 128, True), (90, 91, True), (128, 700, True)])
@pytest.mark.parametrize("scales", ["of the values", torch.float32])
@pytest.mark.parametrize("p_round", ["reference", "rne"])
def test_entries_alone_give_the_same_bits(Nq, Nk, causal, scales, p_round):
    dt = torch.bfloat16 if Nk % 2 else torch.float16
    args = inputs(3, 192, 48, Nq, Nk, dt, scales if scales is torch.float32 else dt, 7 * Nq + Nk)
    _, lse = check_entries(args, causal, dt, p_round=p_round)
    assert bool(torch.isfinite(lse).all())


@pytest.mark.parametrize("scales", [torch.float16, torch.float32])
def test_several_query_blocks_per_head_causal(scales):
    """The order of the rounds (backwards every second one) with heads of several query blocks."""
    check_entries(inputs(5, 48, 48, 600, 600, torch.float16, scales, 256), True, torch.float16)


# what keeps single blocks, at as many: lengths of their own (one entry empty), causal rows above the first key, lists that do not agree in length
@pytest.mark.parametrize("H,Hkv,Nq,Nk,causal,ragged", [(192, 48, 128, 300, False, True), (192, 48, 128, 300, True, True), (192, 48, 128, 70, True, False),
                                                       (201, 67, 128, 300, True, False), (12, 12, 3000, 3000, True, False)])
def test_single_blocks_give_the_same_bits(H, Hkv, Nq, Nk, causal, ragged):
    lens = torch.tensor([Nk, 0, Nk // 2], dtype=torch.int32, device=DEV) if ragged else None
    out, lse = check_entries(inputs(3, H, Hkv, Nq, Nk, torch.float16, torch.float16, Nk), causal, torch.float16, lens)
    if ragged:
        assert not out[1].any() and bool(lse[1].isneginf().all())
    hidden = Nq - Nk if causal and not ragged else 0      # rows above the first key
    if hidden > 0:
        assert not out[:, :, :hidden].any() and bool(lse[:, :, :hidden].isneginf().all())


def test_numbers_that_are_none_stay_where_they_are():
    """Rows, keys and whole heads with scales that are not numbers or infinite: their rows' outputs, and no other block of the workgroup.  (A query row
    whose scores are all like that counts as one without keys here.)"""
    B, H = 3, 192
    args = inputs(B, H, H, 128, 200, torch.float16, torch.float16, 5)
    q8, k8, v8, qs, ks, vs = args
    clean, _ = check_entries(args, False, torch.float16)
    qs[:, 5::7, 3], qs[:, 6::7, 127], ks[:, 1::11, 150], ks[:, 2::13, 0], vs[:, 3::17] = float("nan"), float("inf"), float("nan"), float("inf"), float("nan")
    out, _ = M.attention_full_int8(*args, False, D ** -0.5, out_dtype=torch.float16, return_lse=True)
    for b in range(B):
        alone = M.attention_full_int8(*(a[b:b + 1] for a in args), False, D ** -0.5, out_dtype=torch.float16)
        assert bool(((out[b:b + 1] == alone) | (out[b:b + 1].isnan() & alone.isnan())).all())
    hit = torch.zeros((B, H, 128), dtype=torch.bool, device=DEV)
    hit[:, 5::7, 3] = hit[:, 6::7, 127] = hit[:, 1::11] = hit[:, 2::13] = hit[:, 3::17] = True
    assert torch.equal(out[~hit], clean[~hit])
    assert bool(out[:, 1::11, 4:127].isnan().all()) and bool(out[:, 3::17, 4:127].isnan().all())
