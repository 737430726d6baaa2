"""Drop-in for the reference module of the same name: ``attention`` (flash_atten_fp.py:155-189)."""
from . import _capi, _host


def attention(q, k, v, causal, sm_scale, *, num_splits=1, return_lse=False, seqlens_k=None):
    """fp16 (or bf16) attention forward; the output has q's dtype (flash_atten_fp.py:162)."""
    native = _host._native or _host.native()
    return native.forward(_capi.VARIANT_FP16, q, k, v, None, None, None, causal, sm_scale, q.dtype, num_splits,
                          _capi.PROUND_REFERENCE, return_lse, None, seqlens_k)
