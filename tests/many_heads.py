"""The general forward kernels run where the decode-shaped ones would have more workgroups of 32 query rows than are resident at once (the
lines: decode_kernel_takes in csrc/intfa_capi.hip, `pipe` in csrc/intfa_inst_f16pv.inc).  A problem small enough for the CPU oracle is
brought past a line by repeating its heads: the first ones are compared with the oracle, the others with the first ones."""
import torch

RESIDENT = 512      # workgroups: two per compute unit; head_dim 256 has one, so that this is past its line too


def repetitions(B, H, Nq, rows=32):
    """How often H heads are repeated for a grid past RESIDENT workgroups of `rows` query rows (128: past the pipelined kernel of head_dim 64)."""
    return RESIDENT // (B * H * ((Nq + rows - 1) // rows)) + 1


def repeated(reps, *tensors):
    """[B, H, ...] -> [B, reps * H, ...]; K/V heads that are repeated as often stay those of the same query heads."""
    return [t.repeat(1, reps, *([1] * (t.dim() - 2))) for t in tensors]


def first_heads(t, H):
    """The first H of the repeated heads of an output, which all others must equal bit for bit."""
    assert t.shape[1] % H == 0
    bits = t.contiguous().view(torch.int16 if t.element_size() == 2 else torch.int32)      # (NaN too)
    for r in range(H, t.shape[1], H):
        assert torch.equal(bits[:, r:r + H], bits[:, :H]), f"heads {r} .. {r + H - 1} differ from the first {H}"
    return t[:, :H]
