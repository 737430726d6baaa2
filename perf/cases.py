"""The work that this package is measured on: calls of its public entry points over the sizes, types and options that a
program which runs quantised attention asks for.

Six kinds of pass ("path"):
  layer    quantise Q, K, V of a prompt and attend (what the harness of the reference does around one call)
  step     one decoding step of one layer: quantise the new query, append the new K/V row to the int8 cache, attend
  decode   attention of a few query rows against a cache that is already filled, in any of the three variants
  chunk    a chunk of a long prompt against the int8 cache that holds everything before it (causal, aligned to its end)
  prefill  attention of a whole prompt whose operands are already quantised, in any of the three variants
  quant    the input quantisers alone, on activations of a whole batch
"""
import math

import torch

import int_flashattention_amd as M

DEV = "cuda"
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
# what a drawn case may cost at most: a part of the largest listed ones
MAX_FLOPS = 4.0e11
MAX_BYTES = 6.0e8


def listed():
    return [
        # one short prompt of a small model through the whole quantised layer: four calls, little work in each
        dict(name="layer_short_prompt", path="layer", B=1, H=8, Hkv=8, Nq=250, Nk=250, D=64, dtype="float16", causal=True, v_block=0),
        # one request being generated: the smallest calls there are, grouped heads, a short cache
        dict(name="step_one_request", path="step", B=1, H=32, Hkv=8, Nq=1, Nk=1024, D=128, dtype="float16"),
        # a batch of requests at different lengths being generated, bf16 model, long caches
        dict(name="step_batch_bf16", path="step", B=16, H=32, Hkv=8, Nq=1, Nk=8192, D=128, dtype="bfloat16"),
        # one query per head against an fp16 cache, ungrouped heads: the stream of K and V at its largest
        dict(name="decode_fp16_batch", path="decode", variant="fp", B=32, H=32, Hkv=32, Nq=1, Nk=4096, D=128, dtype="float16",
             causal=False),
        # a few drafted tokens per request checked at once against a cache of ragged length, int8 K and 16-bit V
        dict(name="decode_half_drafts_ragged", path="decode", variant="half", B=4, H=16, Hkv=16, Nq=5, Nk=3001, D=64,
             dtype="float16", causal=True),
        # a chunk of a long prompt against the int8 cache
        dict(name="chunk_causal_gqa", path="chunk", variant="full", B=2, H=32, Hkv=8, Nq=512, Nk=7680, D=128, dtype="bfloat16",
             causal=True),
        # the headline configuration
        dict(name="prefill_full_b4_n4096", path="prefill", variant="full", B=4, H=32, Hkv=32, Nq=4096, Nk=4096, D=128,
             dtype="float16", causal=False),
        # half-int8, causal (a benchmark configuration)
        dict(name="prefill_half_causal", path="prefill", variant="half", B=8, H=32, Hkv=32, Nq=2048, Nk=2048, D=128,
             dtype="float16", causal=True),
        # the unquantised variant in bf16 on a causal prompt of ragged length with grouped heads
        dict(name="prefill_bf16_causal_ragged", path="prefill", variant="fp", B=2, H=32, Hkv=8, Nq=3333, Nk=3333, D=128,
             dtype="bfloat16", causal=True),
        # the grid of the reference's own benchmark script: head_dim 64
        dict(name="prefill_full_d64", path="prefill", variant="full", B=4, H=32, Hkv=32, Nq=1024, Nk=1024, D=64,
             dtype="float16", causal=False),
        # head_dim 256, bf16 (a benchmark configuration)
        dict(name="prefill_full_d256_bf16", path="prefill", variant="full", B=16, H=16, Hkv=16, Nq=1024, Nk=1024, D=256,
             dtype="bfloat16", causal=False),
        # the quantisers on the activations of the headline configuration
        dict(name="quant_qkv", path="quant", B=4, H=32, Hkv=32, Nq=4096, Nk=4096, D=128, dtype="float16", v_block=0),
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        path = rng.choice(["layer", "step", "step", "decode", "decode", "chunk", "prefill", "prefill", "prefill", "quant"])
        c = dict(path=path, dtype=rng.choice(["float16", "bfloat16"]))
        H = rng.choice([8, 12, 16, 32])
        D = rng.choice([64, 128, 128, 256]) if path in ("decode", "prefill", "quant") else rng.choice([64, 128, 128])
        group = rng.choice([1, 4])
        if path in ("decode", "prefill"):
            c["variant"] = rng.choice(["full", "half", "fp"])
        if path == "chunk":
            c["variant"] = "full"
        if path == "layer":
            N = _log(rng, 32, 1024)
            c.update(B=rng.randint(1, 2), H=H, Hkv=H, Nq=N, Nk=N, D=D, causal=rng.random() < 0.5, v_block=rng.choice([0, 128]))
        elif path == "step":
            c.update(B=_log(rng, 1, 32), H=H, Hkv=H // group, Nq=1, Nk=_log(rng, 256, 16384), D=D)
        elif path == "decode":
            c.update(B=_log(rng, 1, 32), H=H, Hkv=H // group, Nq=_log(rng, 1, 8), Nk=_log(rng, 256, 16384), D=D,
                     causal=rng.random() < 0.5)
        elif path == "chunk":
            Nq = _log(rng, 128, 2048)
            c.update(B=rng.randint(1, 4), H=H, Hkv=H // group, Nq=Nq, Nk=Nq + _log(rng, 128, 8192), D=D, causal=True)
        elif path == "prefill":
            N = _log(rng, 128, 8192)
            c.update(B=_log(rng, 1, 16), H=H, Hkv=H // group, Nq=N, Nk=N, D=D, causal=rng.random() < 0.5)
        else:
            N = _log(rng, 64, 4096)
            c.update(B=rng.randint(1, 4), H=H, Hkv=H // group, Nq=N, Nk=N, D=D, v_block=rng.choice([0, 128]))
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


def _lengths(case):
    """Rows in the cache per batch entry before a decoding step: requests of a batch are at different lengths (a quarter of
    the cache to all of it but the row of this step), one request alone is near the end."""
    B, cap = case["B"], case["Nk"]
    return [cap - 1 - (cap * 3 // 4) * i // B for i in range(B)]


def _activations(g, shape, dtype, k_outlier=False):
    """~ N(0, 1); keys also have one channel of 64 that is four times as large (projected keys have such channels)."""
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    if k_outlier:
        x[..., 5::64] *= 4.0
    return x.to(dtype)


def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    B, H, Hkv, Nq, Nk, D, path = (case[n] for n in ("B", "H", "Hkv", "Nq", "Nk", "D", "path"))
    g = torch.Generator(device=DEV).manual_seed(seed)
    s = dict(path=path, sm=D ** -0.5, causal=case.get("causal", False), v_block=case.get("v_block", 0), variant=case.get("variant"),
             dtype=dt)
    q = _activations(g, (B, H, Nq, D), dt)
    k = _activations(g, (B, Hkv, Nk, D), dt, k_outlier=True)
    v = _activations(g, (B, Hkv, Nk, D), dt)
    if path in ("layer", "quant"):
        s.update(q=q, k=k, v=v)
        return s
    if path == "step":
        # an int8 cache of Nk rows that is filled up to each request's length, and the row of this step
        lens = _lengths(case)
        kc, ksc = M.quant_pertoken(k)
        vc, vs = M.quant_pertensor(v)
        s.update(q=q, k_new=_activations(g, (B, Hkv, 1, D), dt, k_outlier=True), v_new=_activations(g, (B, Hkv, 1, D), dt),
                 kc=kc, ksc=ksc, vc=vc, vs=vs, lens=torch.tensor(lens, dtype=torch.int32, device=DEV),
                 lens_after=torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=DEV))
        return s
    if case["variant"] == "fp":
        s.update(args=(q, k, v))
        return s
    q8, qs = M.quant_pertoken(q)
    k8, ks = M.quant_pertoken(k)
    if case["variant"] == "half":
        s.update(args=(q8, k8, v, qs, ks))
    else:
        v8, vs = M.quant_pertensor(v)
        s.update(args=(q8, k8, v8, qs, ks, vs))
    return s


def _quantise_v(s):
    return M.quant_perblock_channel(s["v"], s["v_block"]) if s["v_block"] else M.quant_pertensor(s["v"])


def run(s):
    path = s["path"]
    if path == "quant":
        return [*M.quant_pertoken(s["q"]), *M.quant_pertoken(s["k"]), *_quantise_v(s)]
    if path == "layer":
        q8, qs = M.quant_pertoken(s["q"])
        k8, ks = M.quant_pertoken(s["k"])
        v8, vs = _quantise_v(s)
        return M.attention_full_int8(q8, k8, v8, qs, ks, vs, s["causal"], s["sm"], out_dtype=s["dtype"],
                                     v_scale_block=s["v_block"] or None)
    if path == "step":
        q8, qs = M.quant_pertoken(s["q"])
        M.kvcache_append(s["kc"], s["ksc"], s["k_new"], s["lens"], s["vc"], s["vs"], s["v_new"])
        o = M.attention_full_int8(q8, s["kc"], s["vc"], qs, s["ksc"], s["vs"], False, s["sm"], out_dtype=s["dtype"],
                                  num_splits="auto", seqlens_k=s["lens_after"])
        return [o, s["kc"], s["ksc"], s["vc"]]
    splits = "auto" if path in ("decode", "chunk") else 1
    if s["variant"] == "full":
        return M.attention_full_int8(*s["args"], s["causal"], s["sm"], out_dtype=s["dtype"], num_splits=splits)
    fn = M.attention if s["variant"] == "fp" else M.attention_int8
    return fn(*s["args"], s["causal"], s["sm"], num_splits=splits)


def _pairs(case):
    """Query-key pairs that the mask leaves, per head of the batch."""
    Nq, Nk = case["Nq"], case["Nk"]
    return Nq * Nk if not case.get("causal") else Nq * (Nk - Nq) + Nq * (Nq + 1) // 2


def work(case):
    B, H, Hkv, Nq, Nk, D, path = (case[n] for n in ("B", "H", "Hkv", "Nq", "Nk", "D", "path"))
    nq, nk = B * H * Nq, B * Hkv * Nk             # rows of Q and of K or V
    if path in ("layer", "quant"):
        sc = 2 * (nq + nk) + (4 * B * Hkv * -(-Nk // case["v_block"]) * D if case["v_block"] else 2 * B * Hkv)
        if path == "quant":                       # 16-bit rows in, int8 rows and scales out
            return {"bytes": 3 * D * (nq + 2 * nk) + sc, "flops": 0}
        return {"bytes": 2 * D * (nq + 2 * nk) + 2 * D * nq, "flops": 4.0 * B * H * D * _pairs(case)}
    if path == "step":
        rows = sum(n + 1 for n in _lengths(case)) * Hkv
        return {"bytes": rows * (2 * D + 2) + 4 * D * nq + B * Hkv * (6 * D + 4), "flops": 4.0 * rows * (H // Hkv) * D}
    qk, vb, sc = {"full": (1, 1, 2), "half": (1, 2, 2), "fp": (2, 2, 0)}[case["variant"]]
    return {"bytes": nq * (D * (qk + 2) + sc) + nk * (D * (qk + vb) + sc), "flops": 4.0 * B * H * D * _pairs(case)}


def tolerance(case):
    """Quantisers are defined bit for bit.  Half-int8 and fp16/bf16: P and the output are 16-bit numbers.  Full-int8: P has
    seven bits in the frame of a running maximum, so another block length or order of the keys, equally right, moves
    the output by the noise of that rounding: 5e-3 for another key block; 2e-2 to 2.5e-2 where the keys are cut into
    ranges of their own (automatic splits)."""
    path = case["path"]
    if path == "quant":
        return "exact"
    if case.get("variant", "full") != "full":
        return {"rel": 5e-3 if case["dtype"] == "float16" else 1e-2}
    if path in ("step", "chunk", "decode"):
        return {"rel": 2.5e-2, "max": 0.4}
    return {"rel": 1e-2, "max": 0.2}
