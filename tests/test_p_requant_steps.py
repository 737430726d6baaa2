"""The requantisation of P as the kernels evaluate it (one fp16 fma, truncation by adding 1024 toward zero) against the reference's
chain (flash_atten_full_int8.py:49-51), for every fp16 probability; and the bytes the kernels produce."""
import numpy as np
import pytest
import torch

import intfa_oracle as O


def test_fma_and_magic_addition_equal_the_chain_for_every_fp16_probability():
    h = np.arange(0, 0x3C01, dtype=np.uint16).view(np.float16)            # 0 .. 1, denormals included
    chain = np.trunc(((h * np.float16(127)).astype(np.float16) + np.float16(0.5)).astype(np.float16)).astype(np.int64)
    fma = (h.astype(np.float64) * 127 + 0.5).astype(np.float16)           # exact in float64: one rounding
    magic = (1024 + np.floor(fma.astype(np.float64))).astype(np.float16)  # 1024 + fma toward zero, units of 1 from 1024 on
    assert np.array_equal(magic.view(np.uint16) & 0xFF, chain)
    assert np.array_equal(O.p_requant_reference(torch.from_numpy(h.astype(np.float32))).numpy().astype(np.int64), chain)


@pytest.mark.gpu
@pytest.mark.parametrize("D,N,heads", [(64, 32, 1), (64, 128, 300), (128, 32, 1), (128, 128, 300), (256, 32, 1), (256, 128, 200)])
def test_bytes_of_the_kernels(D, N, heads):
    """V is the identity, so an output column is one byte of P over 127 l; both divisions of labour (few heads, many heads)."""
    import int_flashattention_amd as M
    g = torch.Generator().manual_seed(5)
    Nk = 64
    q8 = torch.randint(-127, 128, (1, heads, N, D), generator=g, dtype=torch.int8)
    k8 = torch.randint(-127, 128, (1, heads, Nk, D), generator=g, dtype=torch.int8)
    v8 = torch.zeros((1, heads, Nk, D), dtype=torch.int8)
    v8[..., torch.arange(Nk), torch.arange(Nk)] = 1
    qs, ks = torch.full((1, heads, N), 0.01), torch.full((1, heads, Nk), 0.01)
    dev = [t.cuda() for t in (q8, k8, v8, qs, ks, torch.ones((1, heads)))]
    sm = 0.5
    o = M.attention_full_int8(*dev, False, sm, p_round="reference").double().cpu()[..., :Nk]
    x = torch.matmul(q8.double(), k8.double().transpose(2, 3)) * (1e-4 * sm)
    p = torch.exp(x - x.amax(-1, keepdim=True))
    got = o * 127 * p.sum(-1, keepdim=True)                               # within 127 * 2^-11 of a whole number
    assert (got - got.round()).abs().max() < 0.1
    # p of the kernel is within 2^-17 relative of this one: the byte lies between those of the two ends
    lo, hi = (O.p_requant_reference((p * (1 + s * 2.0 ** -17)).clamp(max=1.0).float()).double() for s in (-1, 1))
    assert ((got.round() >= lo) & (got.round() <= hi)).all()
