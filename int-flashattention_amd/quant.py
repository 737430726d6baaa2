"""The quantisers of the reference's harness (benchmark.py:96-107) on HIP kernels: ``quant_pertoken`` and
``quant_pertensor`` with the reference's signatures (X -> (int8 X, scale))."""
from . import _host


def quant_pertoken(x):
    """Per-row symmetric int8 (benchmark.py:96-100): scale = absmax / 127 in x's dtype, round-half-even."""
    return (_host._native or _host.native()).quant_pertoken(x)


def quant_pertensor(x):
    """One scale per (batch, head) slice (benchmark.py:102-107)."""
    return (_host._native or _host.native()).quant_pertensor(x)


def quant_perblock_channel(x, block):
    """One fp32 scale per (batch, head, block of ``block`` rows, channel) - the layout of the V scales that the
    reference's CUDA kernel reads (csrc/flash_fwd_kernel_full_qi8.h:156-160) - with the harness's formula
    (benchmark.py:102-107: absmax / 127, round-half-even) evaluated in fp32.  Returns (int8 [Z,H,N,d], fp32
    [Z,H,ceil(N/block),d]); pass both to ``attention_full_int8(..., v_scale_block=block)``."""
    return (_host._native or _host.native()).quant_perblock_channel(x, block)


def kvcache_append(k_cache, k_scale_cache, k_new, seqlens_k, v_cache=None, v_scale=None, v_new=None):
    """Quantises new keys (and values) into an int8 K/V cache in place, at each batch entry's fill position: the
    quantised-cache counterpart of the knew/vnew copy of the reference's cache kernel (csrc/flash_fwd_kernel.h:690-790).

    k_cache, v_cache: int8 [Z, H_kv, N_cache, d]; k_scale_cache: [Z, H_kv, N_cache] and v_scale: [Z, H_kv] in k_new's
    dtype; k_new, v_new: fp16/bf16 [Z, H_kv, N_new, d]; seqlens_k: int32 [Z] on the device (rows already filled) or an
    int for all entries.  K rows are quantised per token like ``quant_pertoken`` (their scales land in
    ``k_scale_cache``); V rows with the cache's existing ``v_scale`` (saturating at +-127).  Rows past the end of the
    cache are dropped.  The lengths are not advanced here: pass ``seqlens_k + N_new`` to the next forward call."""
    return (_host._native or _host.native()).kvcache_append(k_cache, k_scale_cache, k_new, seqlens_k, v_cache, v_scale, v_new)
