"""The per-(batch, head) quantiser around the sizes where its launches change: a slice in the registers of one workgroup, the
two launches with a word per part, and the three with one word per slice (the smaller workspace of the C interface)."""
import ctypes

import pytest
import torch

import intfa_oracle as O
import int_flashattention_amd as M
from int_flashattention_amd import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (N * d * 2 bytes around 128 KiB; one row; more slices than workgroups are wanted; a last chunk with one row)
@pytest.mark.parametrize("B,H,N,d", [(1, 2, 1, 16), (2, 3, 511, 128), (1, 2, 512, 128), (1, 2, 513, 128), (1, 1, 1025, 64),
                                     (3, 1, 257, 256), (1, 1, 4097, 16), (1, 5, 2049, 128), (40, 64, 520, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_quant_pertensor_slice_sizes_bit_exact(B, H, N, d, dtype):
    g = torch.Generator(device=DEV).manual_seed(N + d)
    x = torch.randn((B, H, N, d), generator=g, device=DEV).to(dtype)
    x[:, :, N // 2] *= 3                                    # the maximum lies inside
    x[0, 0, -1, -1] = 30                                    # and in the very last element of one slice
    q8, s = M.quant_pertensor(x)
    cut = (slice(0, 2), slice(0, 5))
    ref8, ref_s = O.quant_pertensor(x[cut].cpu())
    assert torch.equal(s[cut].cpu(), ref_s) and torch.equal(q8[cut].cpu(), ref8)
    if B * H > 10:
        ref8, ref_s = O.quant_pertensor(x[-1:, -1:].cpu())
        assert torch.equal(s[-1:, -1:].cpu(), ref_s) and torch.equal(q8[-1:, -1:].cpu(), ref8)
    # the C interface with the smallest workspace, filled with old data
    lib = _capi.load()
    need = lib.intfa_quant_pertensor_workspace_bytes(B, H)
    ws = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    q8b, sb = torch.empty_like(q8), torch.empty_like(s)
    dt = _capi.INTFA_F16 if dtype == torch.float16 else _capi.INTFA_BF16
    rc = lib.intfa_quant_pertensor(x.data_ptr(), *x.stride()[:3], q8b.data_ptr(), sb.data_ptr(), B, H, N, d, dt, ws.data_ptr(), need,
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(q8b, q8) and torch.equal(sb, s)


# workgroups of one to four steps of rows (8 rows of head_dim 256 each; 2048 workgroups), with a last one of a single row; as one
# slice for the per-(batch, head) scale the same sizes pass 256 parts of several rounds
@pytest.mark.parametrize("steps", [1, 2, 3, 5])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_streaming_launch_sizes_bit_exact(steps, dtype):
    N = 2048 * 8 * steps + 1
    g = torch.Generator(device=DEV).manual_seed(steps)
    x = torch.randn((1, 1, N, 256), generator=g, device=DEV).to(dtype)
    x[0, 0, -1, -1] = 30
    for fn, ref in ((M.quant_pertoken, O.quant_pertoken), (M.quant_pertensor, O.quant_pertensor)):
        q8, s = fn(x)
        ref8, ref_s = ref(x.cpu())
        assert torch.equal(s.cpu(), ref_s) and torch.equal(q8.cpu(), ref8)


# 2048 pieces of 32 KiB and more, of slices that fit 256 of them: pieces wait for the maxima of their slice; one piece fewer, and a slice of
# more than 256 pieces: two passes.  Last pieces of one row, strided rows; old data in the workspace; nobody waits (the debug entry).
@pytest.mark.parametrize("H,N,d,strided", [(64, 4096, 128, False), (64, 3969, 128, True), (63, 4096, 128, False), (8, 65536, 64, False),
                                           (8, 65537, 64, False), (683, 257, 256, False), (1024, 2049, 16, True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_pieces_that_wait_for_their_slice(H, N, d, strided, dtype):
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn((1, H, N, d * (2 if strided else 1)), generator=g, device=DEV).to(dtype)[..., :d]
    x[:, :, N // 3, d // 2] = 5 + torch.arange(H, device=DEV).to(dtype) / 8      # another maximum in every slice
    x[0, -1, -1, -1] = 300
    amax = x.abs().amax((2, 3))
    want_s = (amax.float() / 127).to(dtype)
    want = (x.float() / want_s.float()[..., None, None]).to(dtype).float().round().to(torch.int32).to(torch.int8)      # (128 wraps, as in the reference)
    q8, s = M.quant_pertensor(x)
    assert torch.equal(s, want_s) and torch.equal(q8, want)
    lib = _capi.load()
    need = lib.intfa_quant_pertensor_parts_workspace_bytes(1, H, N, d)
    ws = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    for fn in (lib.intfa_quant_pertensor, lib.intfa_debug_quant_pertensor_alone):
        q8.zero_(); s.zero_()
        assert fn(x.data_ptr(), *x.stride()[:3], q8.data_ptr(), s.data_ptr(), 1, H, N, d, _capi.INTFA_F16 if dtype == torch.float16 else _capi.INTFA_BF16,
                  ws.data_ptr(), need, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
        assert torch.equal(s, want_s) and torch.equal(q8, want)


def test_pieces_that_wait_under_a_graph():
    x = torch.randn((1, 64, 4096, 128), device=DEV).half()
    M.quant_pertensor(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q8, s = M.quant_pertensor(x)
    for scale in (1.0, 0.25, 3.0):                       # (smaller maxima than those of the replay before, too)
        x.copy_(torch.randn_like(x) * scale)
        graph.replay()
        torch.cuda.synchronize()
        ref8, ref_s = M.quant_pertensor(x)
        assert torch.equal(s, ref_s) and torch.equal(q8, ref8)
