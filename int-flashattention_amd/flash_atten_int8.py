"""Drop-in for the reference module of the same name: ``attention_int8`` (flash_atten_int8.py:181-217)."""
from . import _capi, _host


def attention_int8(q, k, v, q_scale, k_scale, causal, sm_scale, *, num_splits=1, return_lse=False, seqlens_k=None):
    """Half-int8 attention forward: int8 q, k with per-token scales, v in fp16 (or bf16); output in v's dtype
    (fp16 in the reference, flash_atten_int8.py:188-189)."""
    native = _host._native or _host.native()
    return native.forward(_capi.VARIANT_HALF_INT8, q, k, v, q_scale, k_scale, None, causal, sm_scale, v.dtype, num_splits,
                          _capi.PROUND_REFERENCE, return_lse, None, seqlens_k)
