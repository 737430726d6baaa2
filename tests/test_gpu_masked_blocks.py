"""The masked key blocks of the general full-int8 kernel (csrc/intfa_fwd_int8.h): an instance per number of 32-key sub-tiles that a wave's rows
see, for every alignment of the causal diagonal and of a ragged end, against the oracle.  The bounds are those of test_gpu_parity.py."""
import pytest
import torch

from many_heads import first_heads, repeated, repetitions
from test_gpu_decode_forms import oracle, problem, run
from test_gpu_parity import MAX_ABS, assert_same_rounding, max_abs

pytestmark = pytest.mark.gpu
NQ = 160                                                 # a full query block and one wave of the next


@pytest.mark.parametrize("Nk,causal", [(NQ + o, True) for o in (-40, 0, 1, 31, 32, 33, 63, 64, 95, 96, 97, 127)]
                         + [(n, False) for n in (1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 193)])
@pytest.mark.parametrize("D,vb", [(64, None), (128, None), (128, 64)])
def test_alignments_of_the_mask(D, vb, Nk, causal):
    args, sm, kw = problem("full", 2, NQ, Nk, D, Nk), D ** -0.5, {}
    if vb:                                               # scale rows of 64 keys: every sub-tile is multiplied, hidden or not
        kw, args = dict(v_scale_block=vb), args[:5] + (args[5][:, :, None, None].expand(1, 2, (Nk + vb - 1) // vb, D).contiguous(),)
    out, _ = run("full", repeated(repetitions(1, 2, NQ), *args), causal, sm, torch.float16, **kw)
    out = first_heads(out, 2).float().cpu()
    hidden = NQ - Nk if causal and Nk < NQ else 0        # rows above the first key
    assert (out[:, :, :hidden] == 0).all()
    q8, k8, v8, qs, ks, vs = args
    vs = vs[:, :, 0, 0] if vb else vs
    ref = oracle((q8[:, :, hidden:], k8, v8, qs[:, :, hidden:], ks, vs), causal, sm, D)
    assert max_abs(out[:, :, hidden:], ref) <= MAX_ABS
    if Nk >= 64 and not causal:
        assert_same_rounding(out, ref)
