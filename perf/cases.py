"""The workloads whose speed is tracked: what a program that keeps its KV cache compressed asks of this library.

Nine kinds of call, each through the public entry points and over the sizes that the benchmark, the tests and the
configurations of this repository use:

  attend    one fused decompress-attention step over an encoded cache                    (ops.attn_decode)
  encode    quantize + bit-pack of the keys and values of one layer                      (ops.k_quant_encode / v_quant_encode)
  codec     pack and unpack of code matrices, on the device                              (ops.encode_p / decode_p)
  host      the same through the reference's own functions, from and to host tensors     (packkv_cuda.*_encode_cpu / *_decode_cpu)
  session   a request: prompt into the growing cache, then decode steps                  (PackKVCompressedCache.update / attend)
  dense     the reference's cache contract: every update returns the dense K and V       (PackKVCache.update)
  repack    token repacking inside the encode, and a step over the repacked cache         (ops.repack_quant_encode)
  gemv      the reference's GPU ops for one decode step                                  (packkv_cuda.kq_mat_vec_mul .. fused_wv)
  record    the compression-ratio record of a layer                                      (crs.crs_evaluation_with_data)

Keys have four outlier channels per head (x10) or a per-channel scale, values are normal, as in packkv_amd/synth.py.
"""
import math

import torch

import packkv_cuda
from packkv_amd import cache as pkv_cache
from packkv_amd import crs, ops, synth

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"

# Stored bits per value of the 16-token format by code width, K with outlier channels and V normal (stream and
# block table over the number of values): what an encode has to write and an attention step to read.
K_BITS = {2: 0.5, 3: 1.6, 4: 2.8, 5: 3.8, 6: 4.8, 7: 5.8, 8: 7.0}
V_BITS = {2: 1.5, 3: 2.7, 4: 3.5, 5: 4.5, 6: 5.6, 7: 6.7, 8: 7.7}

# Most values per side of a drawn case of each kind: no drawn case costs more than the largest listed one.
MOST_VALUES = {"attend": 1 << 29, "encode": 1 << 29, "codec": 1 << 26, "host": 1 << 23, "session": 1 << 28,
               "dense": 1 << 23, "repack": 1 << 25, "gemv": 1 << 26, "record": 1 << 24}


def listed():
    return [
        # one sequence of Llama-2-7B shape, 4096 tokens: the smallest step, where launches and latency count
        {"name": "attend-1x32h-4k", "kind": "attend", "batch": 1, "q_heads": 32, "kv_heads": 32, "tokens": 4096,
         "window": 0, "rel": 0.1, "dtype": "f16"},
        # the benchmark's step: batch 16, GQA 32/8, 32768 tokens per sequence
        {"name": "attend-16x8h-32k", "kind": "attend", "batch": 16, "q_heads": 32, "kv_heads": 8, "tokens": 32768,
         "window": 0, "rel": 0.1, "dtype": "f16"},
        # an ordinary serving step: odd batch, a part-filled 16-bit window, bf16, the tighter error bound (5-bit codes)
        {"name": "attend-3x8h-11k-win", "kind": "attend", "batch": 3, "q_heads": 32, "kv_heads": 8, "tokens": 11008,
         "window": 137, "rel": 0.05, "dtype": "bf16"},
        # compressing a whole layer of the benchmark's cache
        {"name": "encode-16x8h-32k", "kind": "encode", "batch": 16, "kv_heads": 8, "tokens": 32768, "rel": 0.1,
         "dtype": "f16", "keys": "outliers"},
        # the bit-pack sweep's layer (8 heads x 16384 tokens) at its 5-bit bound, codec alone
        {"name": "codec-16k-5bit", "kind": "codec", "rows": 16384, "heads": 8, "rel": 0.05, "pack": 16},
        # the drop-in functions on host tensors, as the reference's evaluation calls them
        {"name": "host-8k", "kind": "host", "rows": 8192, "heads": 8, "rel": 0.1},
        # one user: a short odd prompt, then 24 tokens through two layers (a 64-token cut on the way)
        {"name": "session-1x509", "kind": "session", "batch": 1, "q_heads": 32, "kv_heads": 8, "layers": 2,
         "prompt": 509, "steps": 24, "rel": 0.1, "dtype": "f16"},
        # a full batch: 32 sequences, 8192-token prompt, bf16, then 24 tokens through two layers
        {"name": "session-32x8k", "kind": "session", "batch": 32, "q_heads": 32, "kv_heads": 8, "layers": 2,
         "prompt": 8192, "steps": 24, "rel": 0.1, "dtype": "bf16"},
        # the reference's generate loop: eager attention over the dense tensors that update returns
        {"name": "dense-2x3001", "kind": "dense", "batch": 2, "kv_heads": 8, "prompt": 3001, "steps": 6, "rel": 0.1,
         "dtype": "f16"},
        # tokens reordered by the median of their V codes before they are packed
        {"name": "repack-4x8k-median", "kind": "repack", "batch": 4, "kv_heads": 8, "tokens": 8192, "rel": 0.1,
         "dtype": "f16", "method": "median"},
        # the reference's throughput script: one sequence, 65536 tokens, K at 4 bits, V at 3 bits
        {"name": "gemv-64k", "kind": "gemv", "heads": 8, "rows": 65536, "k_rel": 0.1, "v_rel": 0.2, "dtype": "f16"},
        # the size record of the sweep's layer with greedy repacking
        {"name": "record-16k-greedy", "kind": "record", "batch": 1, "kv_heads": 8, "tokens": 16384, "rel": 0.1,
         "dtype": "f16", "method": "greedy"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tokens(rng, lo, hi, per_token, most, step):
    """A token count spread over the logarithm of lo..hi, a multiple of `step`, with at most `most` values in all."""
    hi = max(lo, min(hi, most // per_token))
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("attend", "attend", "encode", "codec", "host", "session", "session", "dense", "repack", "gemv", "record"))
    most = MOST_VALUES[kind]
    rel = rng.choice((0.1, 0.1, 0.05, 0.2))
    dtype = rng.choice(("f16", "bf16"))
    if kind in ("attend", "session"):
        hq, hkv = rng.choice(((32, 8), (32, 8), (32, 32), (16, 4)))
        batch = _log(rng, 1, 16 if kind == "attend" else 32)
    else:
        hq, hkv = 0, rng.choice((4, 8, 8, 32) if kind == "encode" else (4, 8, 8, 8))
        batch = _log(rng, 1, 16)
    if kind == "attend":
        return {"kind": kind, "batch": batch, "q_heads": hq, "kv_heads": hkv,
                "tokens": _tokens(rng, 256, 131072, batch * hkv * 128, most, 128), "window": rng.choice((0, rng.randint(1, 255))),
                "rel": rel, "dtype": dtype}
    if kind == "encode":
        return {"kind": kind, "batch": batch, "kv_heads": hkv, "tokens": _tokens(rng, 256, 65536, batch * hkv * 128, most, 128),
                "rel": rel, "dtype": dtype, "keys": rng.choice(("outliers", "channel_scale"))}
    if kind == "codec":
        pack = rng.choice((16, 16, 64))
        return {"kind": kind, "rows": _tokens(rng, 1024, 65536, hkv * 128, most, 8 * pack), "heads": hkv,
                "rel": rng.choice((0.2, 0.1, 0.05, 0.025)), "pack": pack}
    if kind == "host":
        return {"kind": kind, "rows": _tokens(rng, 256, 16384, hkv * 128, most, 128), "heads": hkv, "rel": rng.choice((0.1, 0.2))}
    if kind == "session":
        return {"kind": kind, "batch": batch, "q_heads": hq, "kv_heads": hkv, "layers": rng.choice((1, 2)),
                "prompt": _tokens(rng, 65, 32768, batch * hkv * 128, most, 1), "steps": rng.randint(8, 24), "rel": rel,
                "dtype": dtype}
    if kind == "dense":
        batch = min(batch, 4)
        return {"kind": kind, "batch": batch, "kv_heads": hkv, "prompt": _tokens(rng, 65, 8192, batch * hkv * 128, most, 1),
                "steps": rng.randint(2, 6), "rel": rel, "dtype": dtype}
    if kind == "repack":
        method = rng.choice(("median", "median", "greedy"))
        return {"kind": kind, "batch": batch, "kv_heads": hkv,
                "tokens": _tokens(rng, 256, 16384, batch * hkv * 128, most >> (3 if method == "greedy" else 0), 128), "rel": rel,
                "dtype": dtype, "method": method}
    if kind == "gemv":
        return {"kind": kind, "heads": 8, "rows": _tokens(rng, 1024, 65536, 1024, most, 128), "k_rel": 0.1, "v_rel": 0.2,
                "dtype": dtype}
    return {"kind": kind, "batch": min(batch, 2), "kv_heads": hkv, "tokens": _tokens(rng, 256, 16384, min(batch, 2) * hkv * 128, most, 64),
            "rel": rel, "dtype": dtype, "method": rng.choice(("none", "median", "greedy"))}


# ---- what a user's program holds before the call ----------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rotary(tokens, batch, dtype):
    """cos / sin [batch, tokens, 128] as a decoder hands them to its cache: one table, expanded over the batch."""
    inv = 1.0 / (1.0e6 ** (torch.arange(0, 128, 2, device=DEV, dtype=torch.float32) / 128))
    f = torch.outer(torch.arange(tokens, device=DEV, dtype=torch.float32), inv)
    f = torch.cat((f, f), dim=-1)
    return (f.cos().to(dtype).unsqueeze(0).expand(batch, -1, -1), f.sin().to(dtype).unsqueeze(0).expand(batch, -1, -1))


def _buffers(values, room):
    """A stream buffer of `room` bytes and its block table for one side (8192 values a block), zeroed: an encode writes
    the bytes in use only."""
    return (torch.zeros(room, dtype=torch.uint8, device=DEV), torch.zeros(values // 8192, 2, dtype=torch.uint32, device=DEV))


def _codes(x, rel):
    scale, zero = ops.quant_params(x, rel)
    return ops.quantize(x, scale, zero)[0]


def _steps(case, seed, heads):
    """The new tokens of a decode loop: [steps, batch, heads, 1, 128]."""
    return torch.randn(case["steps"], case["batch"], heads, 1, 128, generator=_gen(seed), device=DEV).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    dtype = DTYPES[case.get("dtype", "f16")]
    if kind == "attend":
        B, H, T = case["batch"], case["kv_heads"], case["tokens"]
        k, v = synth.make_kv(B, H, T + case["window"], seed=seed, dtype=dtype, device=DEV)
        s["k"] = ops.k_quant_encode(k[:, :, :T].contiguous(), case["rel"])
        s["v"] = ops.v_quant_encode(v[:, :, :T].contiguous(), case["rel"])
        if case["window"]:
            s["k_win"], s["v_win"] = k[:, :, T:].contiguous(), v[:, :, T:].contiguous()
        s["q"] = synth.make_q(B, case["q_heads"], seed=seed + 1, dtype=dtype, device=DEV)
    elif kind == "encode":
        s["k"], s["v"] = synth.make_kv(case["batch"], case["kv_heads"], case["tokens"], seed=seed, dtype=dtype, device=DEV,
                                       k_mode=case["keys"])
        bits, n = ops.bits_for_rel(case["rel"]), s["k"].numel()
        room = max(n, n // 8192 * max(ops.block_bound(True, 64, 128, bits), ops.block_bound(False, 128, 64, bits)) + 16)
        s["k_out"], s["v_out"] = _buffers(n, room), _buffers(n, room)
    elif kind in ("codec", "host"):
        k, v = synth.make_kv(1, case["heads"], case["rows"], seed=seed, device=DEV, k_mode="channel_scale")
        s["bits"] = bits = ops.bits_for_rel(case["rel"])
        host = kind == "host"
        for side, x in (("k", k), ("v", v)):
            codes = _codes(x, case["rel"])
            blk = ops.long_block_shape(side == "k", case.get("pack", 16))
            n = codes.numel() // (blk[0] * blk[1])
            room = max(codes.numel(), n * ops.block_bound_p(case.get("pack", 16), bits))
            s[side] = codes.cpu() if host else codes
            s[side + "_stream"] = torch.zeros(room, dtype=torch.uint8, device=s[side].device)
            s[side + "_info"] = torch.zeros(n, 2, dtype=torch.uint32, device=s[side].device)
            s[side + "_back"] = torch.empty_like(s[side])
    elif kind in ("session", "dense"):
        B, H, n = case["batch"], case["kv_heads"], case["prompt"]
        layers = case.get("layers", 1)
        s["prompt"] = [synth.make_kv(B, H, n, seed=seed + 100 * i, dtype=dtype, device=DEV) for i in range(layers)]
        s["cos"], s["sin"] = _rotary(n + case["steps"], B, dtype)
        s["k"], s["v"] = _steps(case, seed + 1, H), _steps(case, seed + 2, H)
        if kind == "session":
            s["q"] = _steps(case, seed + 3, case["q_heads"])
        s["config"] = pkv_cache.PackKVCacheConfig(64, 192, case["rel"], case["rel"])
    elif kind in ("repack", "record"):
        s["k"], s["v"] = synth.make_kv(case["batch"], case["kv_heads"], case["tokens"], seed=seed, dtype=dtype, device=DEV)
        s["q"] = synth.make_q(case["batch"], 4 * case["kv_heads"], seed=seed + 1, dtype=dtype, device=DEV)
    else:       # gemv
        T, H = case["rows"], case["heads"]
        k, v = synth.make_kv(1, H, T, seed=seed, dtype=dtype, device=DEV)
        s["kb"], s["vb"] = ops.bits_for_rel(case["k_rel"]), ops.bits_for_rel(case["v_rel"])
        s["k"], s["v"] = ops.k_quant_encode(k, case["k_rel"]), ops.v_quant_encode(v, case["v_rel"])
        s["q"] = torch.randn(H, 128, generator=_gen(seed + 1), device=DEV).to(dtype)
        s["w"] = torch.softmax(torch.randn(H, T, generator=_gen(seed + 2), device=DEV), dim=1).to(dtype)
        s["t"], s["kq"] = torch.empty(H, T, dtype=dtype, device=DEV), torch.empty(H, T, dtype=dtype, device=DEV)
        s["term"], s["wv"] = torch.empty(H, 128, dtype=torch.float32, device=DEV), torch.empty(H, 128, dtype=dtype, device=DEV)
    return s


# ---- one pass -----------------------------------------------------------------------------------------------

def _run_encode(s):
    out, rel = {}, s["case"]["rel"]
    for side, enc in (("k", ops.k_quant_encode), ("v", ops.v_quant_encode)):
        e = enc(s[side], rel, stream=s[side + "_out"][0], info=s[side + "_out"][1])
        out[side] = (e["size"], e["stream"], e["info"].view(torch.int32), e["scale"], e["zero"])
    return out


def _run_codec(s):
    pack, out = s["case"]["pack"], {}
    for side in ("k", "v"):
        size = ops.encode_p(side == "k", s[side], s[side + "_stream"], s[side + "_info"], pack, s["bits"])
        ops.decode_p(side == "k", s[side + "_stream"], s[side + "_info"], s[side + "_back"], pack, s["bits"])
        out[side] = (size, s[side + "_stream"], s[side + "_info"].view(torch.int32), s[side + "_back"])
    return out


def _run_host(s):
    out, (rows, hidden) = {}, s["k"].shape
    for side, enc, dec, blk in (("k", packkv_cuda.k_encode_cpu, packkv_cuda.k_decode_cpu, (64, 128)),
                                ("v", packkv_cuda.v_encode_cpu, packkv_cuda.v_decode_cpu, (128, 64))):
        stream, info, back = s[side + "_stream"], s[side + "_info"], s[side + "_back"]
        size = enc(s[side], stream, info, rows, hidden, *blk, s["bits"])
        dec(stream, info, back, rows, hidden, *blk, s["bits"])
        out[side] = (size, stream, info.view(torch.int32), back)
    return out


def _run_session(s):
    c, n = s["case"], s["case"]["prompt"]
    cache = pkv_cache.PackKVCompressedCache(c["batch"], c["kv_heads"], 128, c["layers"], s["config"],
                                            max_tokens=n + c["steps"] + 256, dtype=DTYPES[c["dtype"]], device=DEV)
    rot = {"cos": s["cos"][:, :n], "sin": s["sin"][:, :n]}
    for i, (k, v) in enumerate(s["prompt"]):
        cache.update(k, v, i, rot, return_dense=False)
    outs = []
    for t in range(c["steps"]):
        rot = {"cos": s["cos"][:, n + t:n + t + 1], "sin": s["sin"][:, n + t:n + t + 1]}
        for i in range(c["layers"]):
            cache.update(s["k"][t], s["v"][t], i, rot, return_dense=False)
            outs.append(cache.attend(s["q"][t], i))
    return {"outs": outs, "bytes": cache.cache_bytes()}


def _run_dense(s):
    c, n = s["case"], s["case"]["prompt"]
    cache = pkv_cache.PackKVCache(c["batch"], c["kv_heads"], 128, 1, config=s["config"], max_tokens=n + c["steps"] + 256)
    k, v = s["prompt"][0]
    outs = [cache.update(k, v, 0, {"cos": s["cos"][:, :n], "sin": s["sin"][:, :n]})]
    for t in range(c["steps"]):
        rot = {"cos": s["cos"][:, n + t:n + t + 1], "sin": s["sin"][:, n + t:n + t + 1]}
        outs.append(cache.update(s["k"][t], s["v"][t], 0, rot))
    return outs


def _run_repack(s):
    c = s["case"]
    k, v, perm = ops.repack_quant_encode(s["k"], s["v"], c["rel"], c["rel"], c["method"])
    out = ops.attn_decode(s["q"], k, v)
    return {"out": out, "perm": perm, "k": (k["size"], k["info"].view(torch.int32), k["scale"], k["zero"]),
            "v": (v["size"], v["info"].view(torch.int32), v["scale"], v["zero"])}


def _run_gemv(s):
    T, hidden = s["case"]["rows"], s["case"]["heads"] * 128
    k, v = s["k"], s["v"]
    packkv_cuda.kq_mat_vec_mul(k["stream"], k["info"], s["q"], s["t"], T, hidden, 64, 128, s["kb"])
    packkv_cuda.fused_kq(s["kq"], s["q"], k["zero"].reshape(-1), k["scale"].reshape(-1), s["t"])
    s["term"].zero_()
    packkv_cuda.wv_mat_vec_mul(v["stream"], v["info"], s["w"], s["term"], T, hidden, 128, 64, s["vb"])
    packkv_cuda.fused_wv(s["wv"], s["w"], v["zero"].reshape(-1), v["scale"].reshape(-1), s["term"].to(s["w"].dtype))
    return {"t": s["t"], "kq": s["kq"], "term": s["term"], "wv": s["wv"]}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attend":
        return ops.attn_decode(s["q"], s["k"], s["v"], s.get("k_win"), s.get("v_win"))
    if kind == "encode":
        return _run_encode(s)
    if kind == "codec":
        return _run_codec(s)
    if kind == "host":
        return _run_host(s)
    if kind == "session":
        return _run_session(s)
    if kind == "dense":
        return _run_dense(s)
    if kind == "repack":
        return _run_repack(s)
    if kind == "gemv":
        return _run_gemv(s)
    return crs.crs_evaluation_with_data(crs.CRConfig(64, 16, case["rel"], case["rel"], case["method"]), [s["k"]], [s["v"]])


# ---- what a pass cannot do without, and how far two correct results may lie apart ----------------------------

def _stored(bits, values):
    return (K_BITS[bits] + V_BITS[bits]) / 8 * values


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, H = case["rows"] * case["heads"] * 128, case["heads"]
        kb, vb = ops.bits_for_rel(case["k_rel"]), ops.bits_for_rel(case["v_rel"])
        return {"bytes": (K_BITS[kb] + V_BITS[vb]) / 8 * n + 8 * case["rows"] + 8 * H * case["rows"], "flops": 4 * n}
    rel_bits = ops.bits_for_rel(case["rel"])
    if kind in ("codec", "host"):
        n = case["rows"] * case["heads"] * 128
        return {"bytes": 4 * n + 2 * _stored(rel_bits, n), "flops": 0}      # codes in and out, streams out and in
    B, H = case["batch"], case["kv_heads"]
    if kind == "attend":
        n = B * H * 128 * case["tokens"]
        win = B * H * 128 * case["window"]
        return {"bytes": _stored(rel_bits, n) + 8 * B * case["tokens"] + 4 * win + 4 * B * case["q_heads"] * 128,
                "flops": 4 * B * case["q_heads"] * 128 * (case["tokens"] + case["window"])}
    if kind in ("encode", "repack"):
        n, attends = B * H * 128 * case["tokens"], int(kind == "repack")
        return {"bytes": 4 * n + (1 + attends) * (_stored(rel_bits, n) + 8 * B * case["tokens"]), "flops": attends * 16 * n}
    if kind == "record":
        return {"bytes": 4 * B * H * 128 * case["tokens"], "flops": 0}
    n, steps = B * H * 128 * case["prompt"], case["steps"]
    win = 4 * B * H * 128 * min(160, case["prompt"])
    if kind == "dense":      # the prompt in, the stream out; then every update reads the cache and writes it dense
        return {"bytes": 4 * n + _stored(rel_bits, n) + (steps + 1) * (_stored(rel_bits, n) + 4 * n), "flops": 0}
    return {"bytes": case["layers"] * (4 * n + _stored(rel_bits, n) + steps * (_stored(rel_bits, n) + win)),
            "flops": case["layers"] * steps * 4 * B * case["q_heads"] * 128 * case["prompt"]}


def tolerance(case):
    """Streams, tables, codes and sizes are exact.  Attention: fp32 sums over 16-bit softmax weights, rounded once to the
    storage type; measured against 64-bit arithmetic on the same codes, fp16 differs by up to 5.3e-4 (1.5e-3 at most in one
    value), bf16 by 2.4e-3 (6.2e-3).  The matrix-vector ops sum exact products in fp32 and round once: 2.1e-4 / 1.7e-3."""
    kind, half = case["kind"], case.get("dtype") == "f16"
    if kind in ("attend", "session", "repack"):
        return {"rel": 2e-3, "max": 6e-3} if half else {"rel": 1e-2, "max": 2.5e-2}
    if kind == "gemv":
        return {"rel": 8e-4, "max": 4e-3} if half else {"rel": 7e-3, "max": 2.5e-2}
    return "exact"
