"""16-bit and 32-bit scales of the same values: the general full-int8 kernels up to head_dim 128 fold the dequantisation of the former into one instruction
per score (kScoreSeed in csrc/intfa_device.h; which calls: test_gpu_routes.py) and convert with the latter; the other kernels convert both.  Same bits,
up to the largest sums there are."""
import pytest
import torch

import int_flashattention_amd as M
from many_heads import repetitions

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D,causal,Nq,Nk", [(64, False, 300, 333), (64, True, 200, 1100), (64, True, 129, 129), (128, False, 130, 700), (128, True, 257, 257),
                                            (128, True, 90, 1000), (256, False, 130, 200), (256, True, 200, 200)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits(D, causal, Nq, Nk, dtype):
    # (head_dim 256: more than 256 query blocks of 128 rows, several per workgroup, for which causal lists take whole rounds of K/V heads)
    H = repetitions(1, 1, Nq) + 1 if D < 256 else -(-(repetitions(1, 1, Nq, rows=128) + 1) // 8) * 8
    g = torch.Generator(device=DEV).manual_seed(D + Nk)
    q8, k8, v8 = (torch.randint(-128, 128, (1, H, n, D), generator=g, device=DEV, dtype=torch.int32).to(torch.int8) for n in (Nq, Nk, Nk))
    # the largest sums of either sign: -128 * -128 and -128 * 127 throughout
    q8[:, :, ::7] = -128
    k8[:, :, ::5] = -128
    k8[:, :, 1::5] = 127
    qs, ks = (torch.rand((1, H, n), generator=g, device=DEV).mul(2e-3).to(dtype) for n in (Nq, Nk))
    ks[:, :, 3::11] *= 64
    vs = torch.rand((1, H), generator=g, device=DEV).to(dtype)
    for p_round in ("reference", "rne"):
        a, la = M.attention_full_int8(q8, k8, v8, qs, ks, vs, causal, 1.0, out_dtype=dtype, p_round=p_round, return_lse=True)
        b, lb = M.attention_full_int8(q8, k8, v8, qs.float(), ks.float(), vs.float(), causal, 1.0, out_dtype=dtype, p_round=p_round, return_lse=True)
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
        assert torch.equal(la.view(torch.int32), lb.view(torch.int32))
        assert bool(torch.isfinite(la).all()) and bool(torch.isfinite(a).all())


@pytest.mark.parametrize("causal,Nq,Nk", [(False, 130, 64), (False, 200, 333), (True, 129, 129), (True, 257, 700)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits_16bit_v(causal, Nq, Nk, dtype):
    """The pipelined half-int8 kernel."""
    H = repetitions(1, 1, Nq, rows=128) + 1
    g = torch.Generator(device=DEV).manual_seed(Nk)
    q8, k8 = (torch.randint(-128, 128, (1, H, n, 128), generator=g, device=DEV, dtype=torch.int32).to(torch.int8) for n in (Nq, Nk))
    q8[:, :, ::7] = -128
    k8[:, :, ::5] = -128
    k8[:, :, 1::5] = 127
    v = torch.randn((1, H, Nk, 128), generator=g, device=DEV).to(dtype)
    qs, ks = (torch.rand((1, H, n), generator=g, device=DEV).mul(2e-3).to(dtype) for n in (Nq, Nk))
    ks[:, :, 3::11] *= 64
    a, la = M.attention_int8(q8, k8, v, qs, ks, causal, 1.0, return_lse=True)
    b, lb = M.attention_int8(q8, k8, v, qs.float(), ks.float(), causal, 1.0, return_lse=True)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(la.view(torch.int32), lb.view(torch.int32))
    assert bool(torch.isfinite(la).all()) and bool(torch.isfinite(a).all())


@pytest.mark.parametrize("D,causal,Nq,Nk", [(64, False, 200, 300), (64, True, 130, 1100), (128, False, 200, 300), (128, True, 257, 257)])
def test_same_bits_blocked_v(D, causal, Nq, Nk):
    """One V scale per 128 keys and channel."""
    H = repetitions(1, 1, Nq, rows=128) + 1
    g = torch.Generator(device=DEV).manual_seed(Nk)
    q8, k8 = (torch.randint(-128, 128, (1, H, n, D), generator=g, device=DEV, dtype=torch.int32).to(torch.int8) for n in (Nq, Nk))
    v8, vs = M.quant_perblock_channel(torch.randn((1, H, Nk, D), generator=g, device=DEV).half(), 128)
    qs, ks = (torch.rand((1, H, n), generator=g, device=DEV).mul(2e-3).half() for n in (Nq, Nk))
    a = M.attention_full_int8(q8, k8, v8, qs, ks, vs, causal, 1.0, v_scale_block=128)
    b = M.attention_full_int8(q8, k8, v8, qs.float(), ks.float(), vs, causal, 1.0, v_scale_block=128)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and bool(torch.isfinite(a).all())
