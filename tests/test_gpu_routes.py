"""Which forward kernel a call runs, by the names a profiler sees: the tests of the general kernels are worth something only while their
problems are past the line that sends small ones to the decode-shaped kernels."""
import torch

import pytest

import int_flashattention_amd as M
from many_heads import repetitions

pytestmark = pytest.mark.gpu
DEV = "cuda"

# variant, D, H, Nq, causal, options -> kernel and its first template arguments.  H by repetitions(): the least that is past the line, and
# the most that is not (one repetition less of one head)
N = 130
PAST = repetitions(1, 1, N)
CASES = [
    ("full", 64, PAST, N, False, {}, "fwd_full_int8_kernel<64, false"),
    ("full", 64, PAST - 1, N, False, {}, "fwd_decode_full_int8_kernel<64"),
    ("full", 128, PAST, N, True, {}, "fwd_full_int8_kernel<128, true"),
    ("full", 128, PAST - 1, N, True, {}, "fwd_decode_full_int8_kernel<128"),
    ("full", 256, PAST, N, False, {}, "fwd_full_int8_pair_kernel<false"),
    ("full", 256, 129, N, False, {}, "fwd_full_int8_pair_kernel<false, 0, 1, false, false, true>"),       # 258 query blocks: several per workgroup
    ("full", 256, 128, N, False, {}, "fwd_full_int8_pair_kernel<false, 0, 1, false, false, false>"),
    ("full", 256, 129, N, False, dict(scales=torch.float32), "fwd_full_int8_pair_kernel<false, 0, 1, false, false, true>"),
    # ... causal: two rounds of 256, whole rounds of K/V heads per XCD, lists that agree; one length for all entries, no more rows than keys
    ("full", 256, 256, N, True, {}, "fwd_full_int8_pair_kernel<true, 0, 1, false, false, true>"),
    ("full", 256, 248, N, True, {}, "fwd_full_int8_pair_kernel<true, 0, 1, false, false, false>"),
    ("full", 256, 257, N, True, {}, "fwd_full_int8_pair_kernel<true, 0, 1, false, false, false>"),
    ("full", 256, 12, 6000, True, {}, "fwd_full_int8_pair_kernel<true, 0, 1, false, false, false>"),
    ("full", 256, 129, N, False, dict(seqlens=True), "fwd_full_int8_pair_kernel<false, 0, 1, false, false, false>"),
    ("full", 256, 256, N, True, dict(keys=N - 1), "fwd_full_int8_pair_kernel<true, 0, 1, false, false, false>"),
    ("full", 256, PAST // 2, N, False, {}, "fwd_decode_full_int8_kernel<256"),
    ("full", 128, PAST, N, True, dict(v_block=128), "fwd_full_int8_kernel<128, true"),
    ("full", 128, 1, N, True, dict(v_block=64), "fwd_full_int8_kernel<128, true"),
    ("full", 128, 1, N, False, dict(num_splits=2), "fwd_full_int8_kernel<128, false"),
    ("full", 128, 1, 64, False, {}, "fwd_decode_full_int8_kernel<128"),
    # the folded dequantisation (last argument), on both sides of each line: more than two key blocks, blocks per split, 16-bit scales; head_dim 64:
    # 768 workgroups, 2048 keys, causal 640 keys and 1536 workgroups; V scales per 128 keys
    ("full", 128, PAST, 257, False, {}, "fwd_full_int8_kernel<128, false, 0, 1, false, false, 0, true>"),
    ("full", 128, PAST, 256, False, {}, "fwd_full_int8_kernel<128, false, 0, 1, false, false, 0, false>"),
    ("full", 128, PAST, 257, False, dict(scales=torch.float32), "fwd_full_int8_kernel<128, false, 0, 1, false, false, 0, false>"),
    ("full", 128, 20, 513, True, dict(num_splits=2), "fwd_full_int8_kernel<128, true, 0, 1, false, true, 0, true>"),
    ("full", 128, 20, 512, True, dict(num_splits=2), "fwd_full_int8_kernel<128, true, 0, 1, false, true, 0, false>"),
    ("full", 128, PAST, 600, False, dict(v_block=128), "fwd_full_int8_kernel<128, false, 0, 1, false, false, 1, false>"),
    ("full", 128, PAST, 600, False, dict(v_block=64), "fwd_full_int8_kernel<128, false, 0, 1, false, false, 2, false>"),
    ("full", 64, 256, 129, False, {}, "fwd_full_int8_kernel<64, false, 0, 1, false, false, 0, true>"),
    ("full", 64, 256, 128, False, {}, "fwd_full_int8_kernel<64, false, 0, 1, false, false, 0, false>"),
    ("full", 64, 256, 384, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, true>"),
    ("full", 64, 257, 384, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, false>"),
    ("full", 64, 49, 2047, False, {}, "fwd_full_int8_kernel<64, false, 0, 1, false, false, 0, false>"),
    ("full", 64, 49, 2048, False, {}, "fwd_full_int8_kernel<64, false, 0, 1, false, false, 0, true>"),
    ("full", 64, 155, 639, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, false>"),
    ("full", 64, 155, 640, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, true>"),
    ("full", 64, 255, 700, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, true>"),
    ("full", 64, 256, 700, True, {}, "fwd_full_int8_kernel<64, true, 0, 1, false, false, 0, false>"),
    ("full", 64, 300, 384, True, dict(v_block=128), "fwd_full_int8_kernel<64, true, 0, 1, false, false, 1, true>"),
    ("full", 64, 300, 128, True, dict(v_block=128), "fwd_full_int8_kernel<64, true, 0, 1, false, false, 1, false>"),
    ("full", 64, 300, 384, True, dict(v_block=128, scales=torch.float32), "fwd_full_int8_kernel<64, true, 0, 1, false, false, 1, false>"),
    ("half", 64, PAST - 1, N, False, {}, "fwd_decode_f16pv_kernel<true, 64"),
    ("half", 64, PAST, N, False, {}, "fwd_f16pv_pipe_kernel<true, 64"),
    ("half", 64, PAST, N, True, {}, "fwd_f16pv_kernel<true, 64"),                       # fewer than eight key blocks
    ("fp", 64, repetitions(1, 1, N, rows=128), N, False, {}, "fwd_f16pv_kernel<false, 64"),
    ("fp", 128, 1, 65, True, {}, "fwd_f16pv_pipe_kernel<false, 128"),
    ("half", 256, PAST // 2, N, False, {}, "fwd_decode_f16pv_kernel<true, 256"),
    ("fp", 256, PAST, N, True, {}, "fwd_f16pv_pair_kernel<false"),
]


def test_kernels_of_calls():
    from torch.profiler import ProfilerActivity, profile
    calls = []
    for variant, D, H, Nq, causal, kw, _ in CASES:
        kw = dict(kw)
        v_block, scales, Nk = kw.pop("v_block", None), kw.pop("scales", torch.float16), kw.pop("keys", Nq)
        if kw.pop("seqlens", False):
            kw["seqlens_k"] = torch.tensor([Nk], dtype=torch.int32, device=DEV)
        q, k, v = (torch.randn((1, H, n, D), device=DEV).half() for n in (Nq, Nk, Nk))
        if variant == "fp":
            calls.append(lambda a=(q, k, v, causal, 0.1), kw=kw: M.attention(*a, **kw))
            continue
        (q8, qs), (k8, ks) = M.quant_pertoken(q), M.quant_pertoken(k)
        qs, ks = qs.to(scales), ks.to(scales)
        if variant == "half":
            calls.append(lambda a=(q8, k8, v, qs, ks, causal, 0.1), kw=kw: M.attention_int8(*a, **kw))
            continue
        v8, vs = M.quant_perblock_channel(v, v_block) if v_block else M.quant_pertensor(v)
        vs = vs if v_block else vs.to(scales)
        kw["v_scale_block"] = v_block
        calls.append(lambda a=(q8, k8, v8, qs, ks, vs, causal, 0.1), kw=kw: M.attention_full_int8(*a, **kw))
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        for c in calls:
            c()
        torch.cuda.synchronize()
    ran = [e.name for e in sorted(prof.events(), key=lambda e: e.time_range.start) if "intfa::fwd_" in e.name]
    if not ran:
        pytest.skip("the profiler reports no kernels here")
    assert len(ran) == len(CASES), ran
    for case, name in zip(CASES, ran):
        assert f"intfa::{case[-1]}" in name, (case, name)
