"""The work that a user of tqhip has it do, as cases that can be timed and compared.

Every case is one layer's share of something a language model with PolarQuant caches does: insert a token and
attend, attend a batch, run a chunk or a whole prompt, compress a prompt, go through the codec itself.  Sizes are
those of the benchmark configurations (28 / 4 and 32 / 8 heads, head dimension 128, three bits, up to 131 072
positions) or lie around them; lengths are mostly not multiples of anything, as a cache's length is not.

Values are seeded N(0, 1) in the model's data type; prompts that are prefilled or compressed carry one channel in a
hundred scaled by 20, as keys and values of trained models do.
"""
import math
import os
import sys

_PKG = os.path.join(os.getcwd(), "turboquant-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import torch

import tqhip

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_WORDS_OF = {1: 32, 2: 16, 3: 10, 4: 8}


def listed():
    return [
        # One token through one layer of a chat turn: key and value encoded, attention over the packed cache.  The
        # smallest call there is; latency and host time are all of it.
        {"name": "packed_step_short", "kind": "packed_step", "batch": 1, "kv_heads": 8, "n_rep": 4, "dim": 128, "bits": 3,
         "length": 1500, "dtype": "float16"},
        # The headline workload: a single-token step of a V-only cache at 32 768 positions, 28 / 4 heads.
        {"name": "vonly_step_32k", "kind": "vonly_step", "batch": 1, "kv_heads": 4, "n_rep": 7, "dim": 128, "bits": 3,
         "length": 32767, "dtype": "float16"},
        # Decode attention of a small bfloat16 batch on V-only caches with a sparse-V threshold.
        {"name": "vonly_threshold_batch", "kind": "vonly_threshold", "batch": 4, "kv_heads": 8, "n_rep": 4, "dim": 128,
         "bits": 3, "length": 9001, "dtype": "bfloat16", "threshold": 1e-5},
        # A serving loop's decode step: sixteen sequences of 4K to 32K positions, ragged, packed keys and values.
        {"name": "flash_ragged_16", "kind": "flash_ragged", "batch": 16, "kv_heads": 8, "n_rep": 4, "dim": 128, "bits": 3,
         "low": 4096, "high": 32768, "dtype": "float16"},
        # Batched generation over left-padded prompts: the attention hook with a boolean padding mask.
        {"name": "masked_batch_8", "kind": "masked_batch", "batch": 8, "kv_heads": 8, "n_rep": 4, "dim": 128, "bits": 3,
         "length": 6003, "dtype": "float16"},
        # The last 512-row chunk of a chunked prefill to 131 072 positions: encode the chunk, attend causally.
        {"name": "prefill_chunk_131k", "kind": "prefill_chunk", "kv_heads": 8, "n_rep": 4, "dim": 128, "bits": 3,
         "length": 131072, "rows": 512, "dtype": "float16"},
        # A prompt in one go into empty caches: two sequences, encode and attend causally.
        {"name": "prefill_prompt_2k", "kind": "prefill_prompt", "batch": 2, "kv_heads": 8, "n_rep": 4, "dim": 128, "bits": 3,
         "length": 2001, "dtype": "bfloat16"},
        # Compressing a prompt in the default mode: keys and values encoded, and handed back dequantised.
        {"name": "compress_prompt_10k", "kind": "compress", "batch": 1, "kv_heads": 8, "dim": 128, "bits": 3, "length": 10007,
         "dtype": "bfloat16"},
        # A token step of a V-only cache that keeps no dequantised buffer: every value is dequantised again.
        {"name": "no_buffer_step_20k", "kind": "no_buffer_step", "batch": 1, "kv_heads": 4, "dim": 128, "bits": 3,
         "length": 20003, "dtype": "float16"},
        # The reference's own chain for a decode step (pre-rotate, scores, softmax, sparse-V) at 65 536 positions.
        {"name": "composed_65k", "kind": "composed", "batch": 1, "kv_heads": 4, "n_rep": 7, "dim": 128, "bits": 3,
         "length": 65536, "dtype": "float16", "threshold": 1e-5},
        # The quantiser as an object: vectors to indices and norms, and back.
        {"name": "quantizer_100k", "kind": "quantizer", "vectors": 100003, "dim": 128, "bits": 3, "dtype": "float16"},
        # Decode attention through the hook at the other head dimensions that the caches take.
        {"name": "head_dim_64", "kind": "head_dim", "cache": "packed", "batch": 2, "kv_heads": 8, "n_rep": 4, "dim": 64,
         "bits": 4, "length": 8190, "dtype": "float16"},
    ]


def _log(rng, low, high):
    """A whole number from low to high, evenly over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["packed_step", "vonly_step", "vonly_threshold", "flash_ragged", "masked_batch", "prefill_chunk",
                       "prefill_prompt", "compress", "no_buffer_step", "composed", "quantizer", "head_dim"])
    kv, rep = rng.choice([(8, 4), (4, 7), (8, 4), (2, 6), (8, 1), (4, 8)])
    c = {"kind": kind, "kv_heads": kv, "n_rep": rep, "dim": 128, "bits": rng.choice([3, 3, 3, 2, 4]),
         "dtype": rng.choice(["float16", "bfloat16"])}
    if kind == "packed_step":
        c.update(batch=rng.choice([1, 1, 2, 4]), length=_log(rng, 64, 24000))
    elif kind == "vonly_step":
        c.update(batch=1, length=_log(rng, 500, 131000))
    elif kind == "vonly_threshold":
        c.update(batch=rng.choice([1, 2, 4, 8]), length=_log(rng, 500, 20000), threshold=rng.choice([1e-5, 1e-4]))
    elif kind == "flash_ragged":
        low = _log(rng, 200, 8000)
        c.update(batch=rng.randint(3, 24), low=low, high=low * rng.randint(2, 8))
    elif kind == "masked_batch":
        c.update(batch=rng.randint(2, 12), length=_log(rng, 300, 10000))
    elif kind == "prefill_chunk":
        rows = rng.choice([100, 256, 512, 777])
        c.update(length=_log(rng, 2048, 80000), rows=rows)
    elif kind == "prefill_prompt":
        length = _log(rng, 40, 6000)
        c.update(batch=rng.randint(1, 2 if length > 3000 else 4), length=length)
    elif kind == "compress":
        c.pop("n_rep")
        c.update(batch=1, length=_log(rng, 100, 60000), dim=rng.choice([128, 128, 64, 256]))
    elif kind == "no_buffer_step":
        c.pop("n_rep")
        c.update(batch=rng.choice([1, 2]), length=_log(rng, 300, 60000))
    elif kind == "composed":
        c.update(batch=rng.choice([1, 1, 2, 3]), length=_log(rng, 500, 65536), threshold=rng.choice([0.0, 1e-5, 1e-4]))
    elif kind == "quantizer":
        c = {"kind": kind, "vectors": _log(rng, 100, 300000), "dim": rng.choice([128, 128, 64, 256]), "bits": rng.choice([1, 2, 3, 4]),
             "dtype": rng.choice(["float16", "bfloat16", "float32"])}
    else:
        cache, dim = rng.choice([("packed", 64), ("packed", 64), ("vonly", 64), ("vonly", 256)])
        c.update(cache=cache, dim=dim, batch=rng.choice([1, 2, 4]), length=_log(rng, 300, 16000), bits=rng.choice([2, 3, 4]))
    return c


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=_DTYPES[dtype])


def _with_outliers(g, x):
    """One channel in a hundred (two of 256, at least one) scaled by 20."""
    n = max(1, x.shape[-1] // 100)
    at = torch.randperm(x.shape[-1], generator=g, device="cuda")[:n]
    x[..., at] *= 20
    return x


def _lengths(case, seed):
    """Sequence lengths of a ragged batch, evenly from low to high."""
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(case["low"], case["high"] + 1, (case["batch"],), generator=g).tolist()


def _token(g, case, heads):
    return _normal(g, (case["batch"], heads, 1, case["dim"]), case["dtype"])


def _filled(g, cache, case):
    shape = (case["batch"], case["kv_heads"], case["length"], case["dim"])
    cache.update_and_fetch(_normal(g, shape, case["dtype"]), _normal(g, shape, case["dtype"]))
    return cache


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = {"kind": kind, "case": case, "scale": 1.0 / math.sqrt(case["dim"])}
    n_q = case.get("kv_heads", 0) * case.get("n_rep", 1)
    if kind in ("packed_step", "vonly_step"):
        packed = kind == "packed_step"
        # room for the next tokens, as a program that is about to generate makes it
        if packed:
            cache = _filled(g, tqhip.TurboQuantKVCache(bits=case["bits"], fused=True), case)
            cache.reserve(case["batch"], case["kv_heads"], 256, case["dim"])
            s["written"] = [cache.k_packed.view(torch.int32), cache.k_norms, cache.v_packed.view(torch.int32), cache.v_norms]
        else:
            cache = _filled(g, tqhip.VOnlyTurboQuantCache(bits=case["bits"], fused=True), case)
            cache.reserve(case["batch"], case["kv_heads"], 256, case["dim"], dtype=_DTYPES[case["dtype"]])
            kc, tq = cache._k_cache, cache._v_tq
            s["written"] = [kc.keys, kc.values, tq.v_packed.view(torch.int32), tq.v_norms]
        s.update(cache=cache, q=_token(g, case, n_q), k=_token(g, case, case["kv_heads"]), v=_token(g, case, case["kv_heads"]))
    elif kind in ("vonly_threshold", "masked_batch", "head_dim", "composed"):
        vonly = kind == "vonly_threshold" or case.get("cache") == "vonly"
        cls = tqhip.VOnlyTurboQuantCache if vonly else tqhip.TurboQuantKVCache
        cache = _filled(g, cls(bits=case["bits"], fused=True), case)
        if kind == "vonly_threshold":
            cache.sparse_v_threshold = case["threshold"]
        mask = None
        if kind == "masked_batch":                                     # left padding: up to half of the positions
            pad = torch.randint(0, case["length"] // 2, (case["batch"], 1, 1, 1), generator=g, device="cuda")
            mask = torch.arange(case["length"], device="cuda").view(1, 1, 1, -1) >= pad
        s.update(cache=cache, q=_token(g, case, n_q), mask=mask)
    elif kind == "flash_ragged":
        lens = _lengths(case, seed)
        rows, kv, dim, bits = sum(lens), case["kv_heads"], case["dim"], case["bits"]
        cb = tqhip.quantizer.gaussian_codebook(bits)
        bd = tqhip.quantizer.gaussian_boundaries(cb)
        sides = []
        for sign_seed in (42, 43):
            signs = tqhip.random_diagonal_sign(dim, seed=sign_seed, device="cuda")
            p, n = tqhip.fused_quantize(_normal(g, (kv * rows, dim), case["dtype"]), signs, bd, dim, bits)
            sides.append((signs, p.view(kv, rows, -1), n.view(kv, rows)))
        offsets = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
        s.update(k=sides[0], v=sides[1], cb=cb, offsets=offsets, longest=max(lens),
                 q=_normal(g, (case["batch"], n_q, dim), case["dtype"]))
    elif kind == "prefill_chunk":
        rows, before = case["rows"], case["length"] - case["rows"]
        cache = tqhip.TurboQuantKVCache(bits=case["bits"], fused=True)
        shape = (1, case["kv_heads"], case["length"], case["dim"])
        k, v = (_with_outliers(g, _normal(g, shape, case["dtype"])) for _ in range(2))
        cache.update_and_fetch(k[:, :, :before].contiguous(), v[:, :, :before].contiguous())
        cache.reserve(1, case["kv_heads"], rows, case["dim"])
        s.update(cache=cache, k=k[:, :, before:].contiguous(), v=v[:, :, before:].contiguous(),
                 q=_normal(g, (1, n_q, rows, case["dim"]), case["dtype"]))
    elif kind == "prefill_prompt":
        shape = (case["batch"], case["kv_heads"], case["length"], case["dim"])
        k, v = (_with_outliers(g, _normal(g, shape, case["dtype"])) for _ in range(2))
        s.update(k=k, v=v, q=_normal(g, (case["batch"], n_q, case["length"], case["dim"]), case["dtype"]))
    elif kind == "compress":
        shape = (case["batch"], case["kv_heads"], case["length"], case["dim"])
        k, v = (_with_outliers(g, _normal(g, shape, case["dtype"])) for _ in range(2))
        s.update(k=k, v=v)
    elif kind == "no_buffer_step":
        cache = _filled(g, tqhip.VOnlyTurboQuantCache(bits=case["bits"], no_v_buffer=True), case)
        s.update(cache=cache, k=_token(g, case, case["kv_heads"]), v=_token(g, case, case["kv_heads"]))
    else:
        s.update(quantizer=tqhip.PolarQuantizer(case["dim"], bits=case["bits"]),
                 x=_with_outliers(g, _normal(g, (case["vectors"], case["dim"]), case["dtype"])))
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind, scale = s["kind"], s["scale"]
    if kind in ("packed_step", "vonly_step"):
        # insert the token and attend, then take the token back (as after a rejected draft), so that a pass can be repeated
        out = s["cache"].decode_step(s["q"], s["k"], s["v"], scale)
        s["cache"].trim(1)
        return [out] + s["written"]
    if kind in ("vonly_threshold", "masked_batch", "head_dim"):
        return tqhip.scaled_dot_product_attention(s["q"], None, None, s["cache"], scale, s["mask"])
    if kind == "flash_ragged":
        (ks, kp, kn), (vs, vp, vn) = s["k"], s["v"]
        c = s["case"]
        return tqhip.flash_decode_from_q(s["q"], ks, kp, kn, vp, vn, s["cb"], s["cb"], vs, c["dim"], c["bits"], scale,
                                         n_rep=c["n_rep"], seq_offsets=s["offsets"], max_seq_len=s["longest"],
                                         out_dtype=s["q"].dtype)
    if kind == "prefill_chunk":
        cache = s["cache"]
        k, v = cache.update_and_fetch(s["k"], s["v"])
        out = tqhip.scaled_dot_product_attention(s["q"], k, v, cache, scale, "causal")
        kp, kn, vp, vn = cache.state
        new = kp.shape[2] - s["k"].shape[2]
        cache.trim(s["k"].shape[2])
        return [out, kp[:, :, new:], kn[:, :, new:], vp[:, :, new:], vn[:, :, new:]]
    if kind == "prefill_prompt":
        cache = tqhip.TurboQuantKVCache(bits=s["case"]["bits"], fused=True)
        k, v = cache.update_and_fetch(s["k"], s["v"])
        out = tqhip.scaled_dot_product_attention(s["q"], k, v, cache, scale, "causal")
        return [out] + cache.state
    if kind == "compress":
        cache = tqhip.TurboQuantKVCache(bits=s["case"]["bits"])
        k, v = cache.update_and_fetch(s["k"], s["v"])
        return [k, v] + cache.state
    if kind == "no_buffer_step":
        k, v = s["cache"].update_and_fetch(s["k"], s["v"])
        s["cache"].trim(1)
        return [k, v]
    if kind == "composed":
        return tqhip.turboquant_attention(s["q"], s["cache"], scale, sparse_v_threshold=s["case"]["threshold"])
    indices, norms = s["quantizer"].quantize(s["x"])
    return [indices, norms, s["quantizer"].dequantize(indices, norms)]


# ------------------------------------------------------------------ what a pass cannot do without

def _row(dim, bits):
    """Bytes of one packed vector and its norm."""
    return -(-dim // _WORDS_OF[bits]) * 4 + 4


def work(case):
    kind, dim, bits = case["kind"], case["dim"], case["bits"]
    size = 4 if case["dtype"] == "float32" else 2
    packed = _row(dim, bits)
    if kind == "quantizer":
        n = case["vectors"]
        return {"bytes": n * (dim * size + 2 * (dim + 4) + 4 * dim), "flops": 0}
    kv, n_q = case["kv_heads"], case["kv_heads"] * case.get("n_rep", 1)
    if kind == "compress":
        n = 2 * case["batch"] * kv * case["length"]
        return {"bytes": n * (2 * dim * size + packed), "flops": 0}
    if kind == "no_buffer_step":
        n = case["batch"] * kv * (case["length"] + 1)
        return {"bytes": n * (packed + dim * size), "flops": 0}
    if kind == "prefill_chunk":
        rows, T = case["rows"], case["length"]
        pairs = rows * T - rows * (rows - 1) // 2
        return {"bytes": 2 * kv * T * packed + 2 * kv * rows * (dim * size + packed) + 2 * n_q * rows * dim * size, "flops": 4 * dim * n_q * pairs}
    if kind == "prefill_prompt":
        T, b = case["length"], case["batch"]
        pairs = T * (T + 1) // 2
        return {"bytes": b * (2 * kv * T * (dim * size + packed) + 2 * n_q * T * dim * size), "flops": b * 4 * dim * n_q * pairs}
    if kind == "flash_ragged":
        rows = case["batch"] * (case["low"] + case["high"]) // 2
    else:
        rows = case["batch"] * (case["length"] + (kind in ("packed_step", "vonly_step")))
    vonly = kind in ("vonly_step", "vonly_threshold") or case.get("cache") == "vonly"
    per_row = packed + (2 * dim if vonly else packed)
    extra = rows if kind == "masked_batch" else 0                      # the mask, one byte a position
    return {"bytes": rows * kv * per_row + 2 * case["batch"] * n_q * dim * size + extra, "flops": 4 * dim * n_q * rows}


def tolerance(case):
    # The codec is defined bit for bit: packed words, norms, indices and dequantised values.
    if case["kind"] in ("compress", "no_buffer_step", "quantizer"):
        return "exact"
    # Four times what the path shows against float64 arithmetic on the same packed data.  Rounding the result to the
    # data type is 2.1e-4 (float16) or 1.65e-3 (bfloat16) of that; fp16 operands of the matrix instructions bring
    # float16 results to 3e-4, and single elements of rows that span outlier channels to 9e-3 of the magnitude.
    half = case["dtype"] == "float16"
    if case["kind"] in ("composed", "head_dim"):                       # float32 fidelity up to the result
        return {"rel": 8.4e-4, "max": 2e-3} if half else {"rel": 6.6e-3, "max": 1.6e-2}
    most = 3.5e-2 if case["kind"].startswith("prefill") else 4e-3 if half else 1.6e-2
    return {"rel": 1.2e-3 if half else 6.8e-3, "max": most}
