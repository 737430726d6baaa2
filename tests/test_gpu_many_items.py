"""Launches of more query blocks than workgroups are resident: a workgroup then takes several of them, and requests the next one's operands under
the last key blocks of the one before (launch_resident in csrc/intfa_launch.h).  Each batch entry alone is a launch of single blocks, which the
other tests compare with the oracle: same bits."""
import pytest
import torch

import int_flashattention_amd as M

pytestmark = pytest.mark.gpu
DEV = "cuda"

# variant, D, heads, K/V heads (three entries: two to four rounds of 256 workgroups, the last one partial; one entry alone: one round at most).  Causal lists
# of items agree in length for a multiple of 8 K/V heads in all (lists_agree)
KERNELS = [("full", 256, 192, 48)]
# query rows, keys, causal: one key block, two, three and more, full and ragged ones; rows past the end of the last query block
SHAPES = [(128, 64, False), (77, 65, False), (128, 300, False), (100, 500, False), (128, 128, True), (90, 91, True), (128, 700, True)]


@pytest.mark.parametrize("Nq,Nk,causal", SHAPES)
@pytest.mark.parametrize("variant,D,H,Hkv", KERNELS)
def test_entries_alone_give_the_same_bits(variant, D, H, Hkv, Nq, Nk, causal):
    B = 3
    g = torch.Generator(device=DEV).manual_seed(7 * Nq + Nk)
    dt = torch.bfloat16 if Nk % 2 else torch.float16
    # (query rows of a wider buffer: rows that are not back to back)
    wide = lambda x: torch.cat([x, x], dim=-1)[..., D:]
    q = torch.randn((B, H, Nq, D), generator=g, device=DEV).to(dt)
    k, v = (torch.randn((B, Hkv, Nk, D), generator=g, device=DEV).to(dt) for _ in range(2))
    if variant == "fp":
        args, fn, kw = [wide(q), k, v], M.attention, {}
    else:
        q8, qs = M.quant_pertoken(q)
        k8, ks = M.quant_pertoken(k)
        if variant == "half":
            args, fn, kw = [wide(q8), k8, v, qs, ks], M.attention_int8, {}
        else:
            v8, vs = M.quant_pertensor(v)
            args, fn, kw = [wide(q8), k8, v8, qs, ks, vs], M.attention_full_int8, dict(out_dtype=dt)
    out, lse = fn(*args, causal, D ** -0.5, return_lse=True, **kw)
    for b in range(B):
        o1, l1 = fn(*(a[b:b + 1] for a in args), causal, D ** -0.5, return_lse=True, **kw)
        assert torch.equal(out[b:b + 1].view(torch.int16), o1.view(torch.int16))
        assert torch.equal(lse[b:b + 1].view(torch.int32), l1.view(torch.int32))
    assert bool(torch.isfinite(lse).all())


def test_several_query_blocks_per_head_causal():
    """The order of the rounds (backwards every second one) with heads of several query blocks."""
    B, H, N = 5, 48, 600
    for variant, D, _, _ in KERNELS:
        g = torch.Generator(device=DEV).manual_seed(D)
        q, k, v = (torch.randn((B, H, N, D), generator=g, device=DEV).half() for _ in range(3))
        if variant == "fp":
            args, fn = [q, k, v], M.attention
        else:
            (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
            args, fn = ([q8, k8, v, qs, ks], M.attention_int8) if variant == "half" else ([q8, k8, *M.quant_pertensor(v), qs, ks], None)
            if fn is None:
                args, fn = [q8, k8, args[2], qs, ks, args[3]], M.attention_full_int8
        out = fn(*args, True, D ** -0.5)
        for b in range(B):
            assert torch.equal(out[b:b + 1].view(torch.int16), fn(*(a[b:b + 1] for a in args), True, D ** -0.5).view(torch.int16)), (variant, D, b)
