"""Split-KV: the forward that merges its partials itself (a workspace of intfa_fwd_merge_workspace_bytes) against the one
that leaves the merge to a second launch (intfa_fwd_workspace_bytes), on workspaces that hold arbitrary old data, and through
the replays of a captured graph."""
import ctypes

import pytest
import torch

import int_flashattention_amd as M
from int_flashattention_amd import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda"


def problem(variant, B, H, Nq, Nk, D, seed, lens=None):
    g = torch.Generator().manual_seed(seed)
    q, k, v = ((torch.randn((B, H, n, D), generator=g)).half().to(DEV) for n in (Nq, Nk, Nk))
    out, lse = torch.empty_like(q), torch.empty((B, H, Nq), device=DEV)
    p = _capi.FwdParams()
    keep = [q, k, v, out, lse]
    if variant != "fp":
        (q, qs), (k, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        p.q_scale, p.k_scale = qs.data_ptr(), ks.data_ptr()
        p.qs_stride_b, p.qs_stride_h, p.qs_stride_n = qs.stride()
        p.ks_stride_b, p.ks_stride_h, p.ks_stride_n = ks.stride()
        keep += [q, k, qs, ks]
    if variant == "full":
        v, vs = M.quant_pertensor(v)
        p.v_scale, (p.vs_stride_b, p.vs_stride_h) = vs.data_ptr(), vs.stride()
        keep += [v, vs]
    for name, t in (("q", q), ("k", k), ("v", v), ("o", out)):
        for axis, s in zip("bhn", t.stride()):
            setattr(p, f"{name}_stride_{axis}", s)
    p.q, p.k, p.v, p.out, p.lse = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr()
    p.batch, p.heads, p.seqlen, p.seqlen_k, p.head_dim = B, H, Nq, Nk, D
    p.scale_dtype = p.io_dtype = _capi.INTFA_F16
    p.sm_scale, p.p_round = D ** -0.5, _capi.PROUND_REFERENCE
    if lens is not None:
        t = torch.tensor(lens, dtype=torch.int32, device=DEV)
        p.seqlens_k = t.data_ptr()
        keep.append(t)
    return p, out, lse, keep


def call(variant, p, ws, nbytes):
    lib = _capi.load()
    p.workspace, p.workspace_bytes = ws.data_ptr(), nbytes
    fn = {"full": lib.intfa_fwd_full_int8, "half": lib.intfa_fwd_half_int8, "fp": lib.intfa_fwd_fp16}[variant]
    assert fn(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0


# (here for `problem`) rows behind the last one of a ragged length: every kernel writes its valid rows only, also where a head's rows are
# followed by room and not by the next head.  1 head: the decode-shaped kernels; past 512 workgroups: the general ones; 2 splits: the merges
@pytest.mark.parametrize("variant,D,H,splits", [("full", 64, 1, 1), ("full", 128, 1, 1), ("full", 256, 1, 1), ("half", 64, 1, 1), ("fp", 256, 1, 1),
                                                ("full", 64, 110, 1), ("full", 128, 110, 1), ("full", 256, 110, 1), ("half", 64, 110, 1),
                                                ("fp", 64, 300, 1), ("half", 128, 3, 1), ("fp", 128, 3, 1), ("half", 256, 110, 1), ("fp", 256, 110, 1),
                                                ("full", 128, 2, 2), ("full", 256, 2, 2), ("half", 128, 2, 2)])
def test_rows_behind_the_last_one_are_not_written(variant, D, H, splits):
    lib, N, room = _capi.load(), 130, 256
    p, out, _, keep = problem(variant, 1, H, N, N, D, D + H)
    p.num_splits = splits
    ws = torch.empty((max(16, lib.intfa_fwd_merge_workspace_bytes(ctypes.byref(p))),), dtype=torch.uint8, device=DEV)
    call(variant, p, ws, ws.numel())
    big = torch.full((1, H, room, D), 7.0, dtype=torch.float16, device=DEV)
    p.out = big.data_ptr()
    p.o_stride_b, p.o_stride_h, p.o_stride_n, _ = big.stride()
    call(variant, p, ws, ws.numel())
    torch.cuda.synchronize()
    assert torch.equal(big[:, :, :N], out) and (big[:, :, N:] == 7.0).all()


def close(a, b):
    assert torch.equal(torch.isfinite(a), torch.isfinite(b))
    f = torch.isfinite(b)
    assert (a[f].float() - b[f].float()).abs().max().item() <= 2e-3
    assert ((a[f].float() - b[f].float()).norm() / b[f].float().norm()).item() <= 1e-4


# rows of a 32-row block: one, a few (idle threads share the splits), a full block, a second block with one row; splits:
# the fewest, one more than a multiple of what a thread has in flight, the most, more than there are blocks
@pytest.mark.parametrize("variant,D,Nq,Nk,splits", [
    ("full", 128, 1, 1024, 2), ("full", 128, 33, 4096, 17), ("full", 64, 5, 8200, 64), ("full", 256, 32, 1500, 9),
    ("half", 64, 1, 5000, 33), ("half", 128, 17, 700, 5), ("half", 256, 3, 2050, 16),
    ("fp", 128, 64, 1300, 64), ("fp", 64, 9, 3001, 8), ("fp", 256, 1, 300, 3),
])
def test_merge_in_the_kernel_equals_the_merge_launch(variant, D, Nq, Nk, splits):
    lib = _capi.load()
    p, out, lse, keep = problem(variant, 2, 3, Nq, Nk, D, 7 * splits + Nq, lens=[Nk, max(1, Nk // 3)])
    p.num_splits = splits
    small, need = lib.intfa_fwd_workspace_bytes(ctypes.byref(p)), lib.intfa_fwd_merge_workspace_bytes(ctypes.byref(p))
    assert need > small
    ws = torch.empty((need,), dtype=torch.uint8, device=DEV)
    call(variant, p, ws, small)
    torch.cuda.synchronize()
    want, want_lse = out.clone(), lse.clone()
    for fill in (0, 255, None, 1):                 # None: what the call before left behind
        if fill is not None:
            ws.fill_(fill)
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        call(variant, p, ws, need)
        torch.cuda.synchronize()
        close(out, want)
        close(lse, want_lse)


# the general full-int8 kernel, a ticket per 32-row wave: more than 64 rows, a last query block with one, two and four waves of
# rows; the fewest splits, an odd number, the most, more than there are blocks; causal rows that some splits do not see
@pytest.mark.parametrize("D,Nq,Nk,splits,causal", [
    (128, 65, 1024, 2, 0), (128, 128, 8200, 64, 0), (128, 161, 700, 9, 1), (128, 512, 2048, 2, 1), (64, 129, 300, 3, 0), (64, 250, 3001, 5, 1),
])
def test_merge_in_the_general_kernel_equals_the_merge_launch(D, Nq, Nk, splits, causal):
    lib = _capi.load()
    p, out, lse, keep = problem("full", 2, 3, Nq, Nk, D, splits + Nq, lens=[Nk, max(1, Nk // 3)])
    p.num_splits, p.causal = splits, causal
    small, need = lib.intfa_fwd_workspace_bytes(ctypes.byref(p)), lib.intfa_fwd_merge_workspace_bytes(ctypes.byref(p))
    ws = torch.empty((need,), dtype=torch.uint8, device=DEV)
    call("full", p, ws, small)
    torch.cuda.synchronize()
    want, want_lse = out.clone(), lse.clone()
    for fill in (0, 255, None, 1):
        if fill is not None:
            ws.fill_(fill)
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        call("full", p, ws, need)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(lse, want_lse)          # the same sums in the same order


def test_merge_replays_from_a_graph_beside_other_calls():
    lib = _capi.load()
    p, out, lse, keep = problem("half", 1, 4, 4, 4096, 128, 3)
    p.num_splits = 8
    need = lib.intfa_fwd_merge_workspace_bytes(ctypes.byref(p))
    ws = torch.full((need,), 171, dtype=torch.uint8, device=DEV)
    call("half", p, ws, need)
    torch.cuda.synchronize()
    want, want_lse = out.clone(), lse.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call("half", p, ws, need)
    for i in range(4):
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(lse, want_lse), i
        if i == 1:
            ws.fill_(171)                          # the workspace is the caller's between replays
        call("half", p, ws, need)                  # an eager call on the same workspace
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
