"""Host-side plumbing shared by the entry points: the native module that checks, lays out and launches a call
(csrc/intfa_torch.cpp), loaded on first use, and the constants of the kernels' geometry."""
from __future__ import annotations

import torch  # noqa: F401  (its libraries have to be in the process before the native module's)

from . import _capi

BLOCK = 128          # query block of the kernels
MIN_HEAD_DIM = 64    # smaller head dims are zero-padded up to this (QK^T and the kept output columns are unchanged)
_VARIANT_ENUM = {"full": _capi.VARIANT_FULL_INT8, "half": _capi.VARIANT_HALF_INT8, "fp": _capi.VARIANT_FP16}

_native = None


def native():
    """The extension module behind the entry points.  Raises if it is not built: there is no other path."""
    global _native
    if _native is None:
        _capi.load()                 # (the same message as every other user of the library when nothing is built)
        try:
            from . import _native as module
        except ImportError as e:
            raise RuntimeError(f"the package's native module is not built or does not load ({e}). "
                               "Run `python -m int_flashattention_amd.build` (needs hipcc and g++).") from e
        _native = module
    return _native


def block_n(variant: str, head_dim: int) -> int:
    """Key-block length the kernel of `variant` ("full", "half", "fp") uses at `head_dim` (the reference's BLOCK_N)."""
    rc = _capi.load().intfa_fwd_block_n(_VARIANT_ENUM[variant], max(int(head_dim), MIN_HEAD_DIM))
    if rc < 0:
        _capi.check(rc, "intfa_fwd_block_n")
    return rc


def check_head_dims(q, k, v):
    """The reference's shape constraints (flash_atten_full_int8.py:189-193): AssertionError, else the head dim."""
    return native().check_head_dims(q, k, v)


def debug_qk_int32(q8: torch.Tensor, k8: torch.Tensor) -> torch.Tensor:
    """int32 accumulators S = Q8 K8^T as produced by the kernels' MFMA tile code ([Z,H,N,N])."""
    return native().debug_qk_int32(q8, k8)
