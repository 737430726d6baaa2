"""Decode-shaped calls whose K and V come to 128 MiB or more load them non-temporally: the same bits as smaller calls on the same
heads, on both sides of the line."""
import pytest
import torch

import int_flashattention_amd as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


# keys such that B H Nk D x (bytes per key and channel) lies just below, at and above 128 MiB; ragged last blocks, one split and several
@pytest.mark.parametrize("variant,D,B,H,Nk,splits", [
    ("full", 128, 8, 16, 4095, 1), ("full", 128, 8, 16, 4096, 3), ("full", 64, 16, 32, 2049, 1), ("full", 256, 4, 16, 4099, 5),
    ("half", 128, 16, 16, 1367, 2), ("half", 64, 8, 32, 2735, 1), ("half", 256, 4, 16, 2735, 2),
    ("fp", 128, 16, 16, 1024, 1), ("fp", 64, 16, 32, 1031, 3), ("fp", 256, 4, 16, 2049, 1),
])
def test_large_caches_give_the_bits_of_small_calls(variant, D, B, H, Nk, splits):
    g = torch.Generator(device=DEV).manual_seed(Nk)
    q, k, v = (torch.randn((B, H, n, D), generator=g, device=DEV).half() for n in (3, Nk, Nk))
    if variant == "fp":
        fn, args = M.attention, (q, k, v)
    else:
        (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        fn, args = M.attention_int8, (q8, k8, v, qs, ks)
        if variant == "full":
            v8, vs = M.quant_pertensor(v)
            fn, args = M.attention_full_int8, (q8, k8, v8, qs, ks, vs)
    o = fn(*args, True, D ** -0.5, num_splits=splits)
    for b in range(B):
        part = fn(*(t[b:b + 1] for t in args), True, D ** -0.5, num_splits=splits)
        assert torch.equal(o[b:b + 1], part), b
