"""The workloads this library's speed is measured on, each driven through its public entry points.

A user of the library runs quantized language models: they load GGUF blocks into QMatrix weights, multiply activations by them one
token at a time (mat-vec), a few at a time (small batches) or a prompt at a time (matrix cores), decode through a stack of layers on
an f32 or block-quantized KV cache, route tokens through experts, and dequantize tensors for the parts of a model that stay dense.
`listed` holds one or two cases of each of those, from the smallest call to the largest; `draw` gives further sizes, formats and
options of the same kinds. Weights have the statistics of trained ones (zero mean, rows of norm about one), so activations keep
their magnitude through a stack; they are made on the GPU and adopted by QMatrix.wrap_device, as a loader that streams a file into
HBM does.
"""
import math

import numpy as np
import torch

import ferric_amd as F
from ferric_amd import decode, kvquant

FORMATS = {"q8_0": F.Q8_0, "q4_k": F.Q4_K, "q6_k": F.Q6_K, "q5_k": F.Q5_K, "q4_0": F.Q4_0, "q4_1": F.Q4_1, "q5_0": F.Q5_0, "q5_1": F.Q5_1,
           "iq4_nl": F.IQ4_NL, "iq4_xs": F.IQ4_XS, "mxfp4": F.MXFP4}
BLOCK = {"q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210), "q5_k": (256, 176), "q4_0": (32, 18), "q4_1": (32, 20), "q5_0": (32, 22),
         "q5_1": (32, 24), "iq4_nl": (32, 18), "iq4_xs": (256, 136), "mxfp4": (32, 17)}
KV = {"q8_0": kvquant.Q8_0, "q4_0": kvquant.Q4_0, "q4_1": kvquant.Q4_1}
KV_BITS = {"f32": 32.0, "q8_0": 8.5, "q4_0": 4.5, "q4_1": 5.0}


# ---- the cases ------------------------------------------------------------------------------------------------------------------

def listed():
    return [
        # The smallest call of a decode step: the key or value projection of one token. Launches and the host path count.
        {"name": "proj_kv", "kind": "linear", "fmt": "q4_k", "out": 1024, "in": 5120, "rows": 1, "bits": 24, "to_host": False},
        # An ordinary projection for a few sequences decoded together, in the other common format.
        {"name": "proj_q8_b8", "kind": "linear", "fmt": "q8_0", "out": 4096, "in": 4096, "rows": 8, "bits": 24, "to_host": False},
        # A ragged width (no multiple of 1024) in a microscaling format, for two sequences.
        {"name": "proj_mxfp4_b2", "kind": "linear", "fmt": "mxfp4", "out": 9728, "in": 2560, "rows": 2, "bits": 24, "to_host": False},
        # The vocabulary head of one token, its logits read back for sampling: the largest single mat-vec.
        {"name": "head_q6k", "kind": "linear", "fmt": "q6_k", "out": 151936, "in": 5120, "rows": 1, "bits": 24, "to_host": True},
        # The Q4_K_M feed-forward block for eight sequences.
        {"name": "ffn_b8", "kind": "ffn", "fmt": "q4_k", "fmt2": "q6_k", "d": 5120, "ff": 17408, "rows": 8},
        # One projection of a 512-token prompt, bf16 activations.
        {"name": "gemm_512", "kind": "gemm", "fmt": "q4_k", "out": 5120, "in": 5120, "rows": 512, "x": "bf16"},
        # The feed-forward block of a 2048-token prompt: the largest matrix products.
        {"name": "ffn_prompt_2048", "kind": "ffn_prompt", "fmt": "q4_k", "fmt2": "q6_k", "d": 5120, "ff": 17408, "rows": 2048},
        # The routed experts of one layer for four tokens: top-k, selected gate|up + SwiGLU, selected down + weighted sum.
        {"name": "moe_t4", "kind": "moe", "fmt": "q4_k", "fmt2": "q6_k", "d": 2048, "eff": 768, "experts": 128, "k": 8, "rows": 4},
        # Four tokens generated behind a short context, each step enqueued call by call: embedding in, logits out.
        {"name": "decode_short", "kind": "decode", "layers": 8, "d": 5120, "heads": 40, "kv_heads": 8, "head_dim": 128, "ff": 17408, "vocab": 151936,
         "ctx": 128, "tokens": 4, "kv": "f32", "graph": False},
        # The same behind a long context on a block-quantized cache, each step one captured graph.
        {"name": "decode_long_q8", "kind": "decode", "layers": 4, "d": 5120, "heads": 40, "kv_heads": 8, "head_dim": 128, "ff": 17408, "vocab": 151936,
         "ctx": 32768, "tokens": 4, "kv": "q8_0", "graph": True},
        # A block of prompt rows behind an earlier one (chunked prefill, ragged counts), hidden rows in and out of host memory.
        {"name": "prefill_block", "kind": "prefill", "layers": 4, "d": 5120, "heads": 40, "kv_heads": 8, "head_dim": 128, "ff": 17408, "rows": 509,
         "past": 300, "kv": "f32"},
        # A tensor dequantized for a consumer that wants it dense: host bytes in, host floats out.
        {"name": "dequant_host", "kind": "dequant", "fmt": "q6_k", "values": 5120 * 4096},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` from lo to hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(step, round(v / step) * step), hi // step * step))


def _draw(rng):
    kind = rng.choice(["linear"] * 4 + ["ffn", "gemm", "ffn_prompt", "moe", "decode", "decode", "prefill", "dequant"])
    if kind == "linear":
        fmt = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0"] + sorted(FORMATS))
        bits = rng.choice([24, 24, 16])
        if rng.random() < 0.2:
            return {"kind": kind, "fmt": rng.choice(["q6_k", "q8_0", "q4_k"]), "out": _log(rng, 32000, 151936), "in": _log(rng, 1024, 5120, 256), "rows": 1, "bits": bits,
                    "to_host": True}
        return {"kind": kind, "fmt": fmt, "out": _log(rng, 512, 34816), "in": _log(rng, 1024, 17408, BLOCK[fmt][0]),
                "rows": rng.choice([1, 1, 1, 2, 3, 4, 5, 7, 8, 13, 16]), "bits": bits, "to_host": False}
    if kind == "ffn":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q5_k", "q6_k"]), "fmt2": rng.choice(["q4_k", "q6_k", "q8_0"]), "d": _log(rng, 1024, 5120, 256),
                "ff": _log(rng, 2048, 17408, 256), "rows": rng.choice([1, 2, 3, 4, 5, 8, 11, 16, 24, 32])}
    if kind == "gemm":
        fmt = rng.choice(["q4_k", "q5_k", "q6_k", "q8_0"])
        return {"kind": kind, "fmt": fmt, "out": _log(rng, 1024, 34816, 8), "in": _log(rng, 1024, 17408, 256), "rows": _log(rng, 16, 2048),
                "x": rng.choice(["bf16", "f32"])}
    if kind == "ffn_prompt":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q5_k", "q6_k"]), "fmt2": rng.choice(["q4_k", "q6_k", "q8_0"]), "d": _log(rng, 1024, 5120, 256),
                "ff": _log(rng, 2048, 17408, 256), "rows": _log(rng, 33, 2048)}
    if kind == "moe":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q8_0"]), "fmt2": rng.choice(["q4_k", "q6_k", "q8_0"]), "d": _log(rng, 1024, 4096, 256),
                "eff": _log(rng, 512, 2048, 256), "experts": rng.choice([16, 32, 64, 128]), "k": rng.choice([2, 4, 6, 8]), "rows": rng.choice([1, 1, 2, 3, 4, 8])}
    if kind in ("decode", "prefill"):
        head_dim = rng.choice([64, 128])
        kv_heads, group = rng.choice([4, 8]), rng.choice([1, 2, 4, 5, 8])
        c = {"kind": kind, "layers": rng.randint(1, 4), "d": _log(rng, 1024, 5120, 256), "heads": kv_heads * group, "kv_heads": kv_heads, "head_dim": head_dim,
             "ff": _log(rng, 2048, 17408, 256), "kv": rng.choice(["f32", "f32", "q8_0", "q4_0", "q4_1"])}
        if kind == "decode":
            c.update(vocab=_log(rng, 32000, 151936), ctx=_log(rng, 16, 32768), tokens=rng.randint(1, 4), graph=rng.random() < 0.5)
        else:
            c.update(rows=_log(rng, 33, 1024), past=rng.choice([0, _log(rng, 32, 1024)]))
        return c
    fmt = rng.choice(sorted(FORMATS))
    return {"kind": kind, "fmt": fmt, "values": _log(rng, 4096, 5120 * 4096, BLOCK[fmt][0])}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = {}
    for c in listed():
        most[c["kind"]] = max(most.get(c["kind"], 0), _cost(c))
    while True:
        c = _draw(rng)
        if _cost(c) <= most[c["kind"]]:
            return c


# ---- seeded inputs, made on the GPU ---------------------------------------------------------------------------------------------

class _View:
    """Device memory of the library as torch sees it (no copy); keeps its owner alive."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "strides": None, "version": 2}


def _torch_bytes(buf, nbytes):
    return torch.as_tensor(_View(buf.ptr.value, (nbytes,), "|u1", buf), device="cuda")


def _torch(t):
    """A library Tensor as a torch tensor over the same memory."""
    return torch.as_tensor(_View(t.buf.ptr.value, t.shape, "<i2" if t.dtype == np.uint16 else "<f4", t.buf), device="cuda")


def _f32(g, shape, std=1.0):
    t = F.Tensor.empty(shape)
    _torch(t).normal_(0.0, std, generator=g)
    return t


def _norm(g, n):
    t = F.Tensor.empty((n,))
    _torch(t).uniform_(0.5, 1.5, generator=g)
    return t


def _bell(g, n, width, mean, std, top):
    """n x width whole numbers 0 .. top, bell-shaped, as uint8."""
    v = torch.randn((n, width), generator=g, device="cuda", dtype=torch.float16)
    return v.mul_(std).add_(mean).round_().clamp_(0, top).to(torch.uint8)


def _halves(v):
    return v.to(torch.float16).unsqueeze(1).view(torch.uint8)


def _spread(g, n, size):
    return size * (0.75 + 0.5 * torch.rand(n, generator=g, device="cuda"))


def _blocks(fmt, n, std, g):
    """n blocks whose weights have zero mean and about the given standard deviation: [n, block bytes] uint8."""
    b = torch.empty((n, BLOCK[fmt][1]), dtype=torch.uint8, device="cuda")
    if fmt == "q8_0":
        b[:, 2:] = torch.randn((n, 32), generator=g, device="cuda", dtype=torch.float16).mul_(40).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        b[:, :2] = _halves(_spread(g, n, std / 40))
    elif fmt in ("q4_k", "q5_k"):
        # w = d * sc * q - dmin * m with m = sc and dmin = d * (middle code): zero mean
        bits = 4 if fmt == "q4_k" else 5
        mid, dev = (1 << bits) / 2 - 0.5, (1 << bits) / 6
        sc = torch.randint(16, 64, (n, 8), generator=g, device="cuda", dtype=torch.uint8)
        d = _spread(g, n, std / (40 * dev))
        b[:, 0:2], b[:, 2:4] = _halves(d), _halves(d * mid)
        b[:, 4:8] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
        q = _bell(g, n, 128, 7.5, 16 / 6, 15) | (_bell(g, n, 128, 7.5, 16 / 6, 15) << 4)
        if bits == 5:
            b[:, 16:48] = torch.randint(0, 256, (n, 32), generator=g, device="cuda", dtype=torch.uint8)
        b[:, -128:] = q
    elif fmt == "q6_k":
        # codes 0 .. 63 around 32: the low nibbles uniform, the two high bits 1 or 2 mostly
        b[:, :128] = torch.randint(0, 256, (n, 128), generator=g, device="cuda", dtype=torch.uint8)
        hi = _bell(g, n, 64, 1.5, 0.6, 3)
        for s in (2, 4, 6):
            hi |= _bell(g, n, 64, 1.5, 0.6, 3) << s
        b[:, 128:192] = hi
        b[:, 192:208] = torch.randint(48, 112, (n, 16), generator=g, device="cuda", dtype=torch.uint8)
        b[:, 208:] = _halves(_spread(g, n, std / (80 * 11)))
    elif fmt == "mxfp4":
        b[:, 1:] = torch.randint(0, 256, (n, 16), generator=g, device="cuda", dtype=torch.uint8)
        e = 128 + round(math.log2(std / 6))
        b[:, 0] = torch.randint(e - 1, e + 2, (n,), generator=g, device="cuda", dtype=torch.uint8)
    else:
        # the other four- and five-bit formats: codes uniform, an f16 scale (and offset) in front
        b[:] = torch.randint(0, 256, b.shape, generator=g, device="cuda", dtype=torch.uint8)
        d = _spread(g, n, std / {"q4_0": 4.6, "q4_1": 4.6, "q5_0": 9.2, "q5_1": 9.2, "iq4_nl": 68.0, "iq4_xs": 68.0 * 18}[fmt])
        b[:, :2] = _halves(d)
        if fmt in ("q4_1", "q5_1"):
            b[:, 2:4] = _halves(d * (-7.5 if fmt == "q4_1" else -15.5))
    return b


def _weight(g, fmt, rows, cols):
    vals, size = BLOCK[fmt]
    n = rows * cols // vals
    buf = F.DeviceBuffer(n * size)
    _torch_bytes(buf, n * size).view(n, size).copy_(_blocks(fmt, n, 1 / math.sqrt(cols), g))
    return F.QMatrix.wrap_device(buf, n * size, FORMATS[fmt], rows, cols)


def _decoder(case, g, max_len, head):
    """A stack of layers with Q4_K projections and a Q6_K down projection, random caches filled to `past` rows by the caller."""
    c = case
    d, ff, q_out, kv_out = c["d"], c["ff"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    layers = [decode.Qwen3Layer(_norm(g, d), _weight(g, "q4_k", q_out + 2 * kv_out, d), _weight(g, "q4_k", d, q_out), _norm(g, d),
                                _weight(g, "q4_k", 2 * ff, d), _weight(g, "q6_k", d, ff), _norm(g, c["head_dim"]), _norm(g, c["head_dim"]))
              for _ in range(c["layers"])]
    cfg = decode.Qwen3Cfg(d, c["heads"], c["kv_heads"], c["head_dim"], ff, eps=1e-6, rope_base=1e6)
    out_norm = _norm(g, d) if head else None
    lm_head = _weight(g, "q6_k", c["vocab"], d) if head else None
    torch.cuda.synchronize()      # the inputs above are made on torch's stream, the decoder runs on its own
    return decode.Qwen3Decoder(cfg, layers, max_len=max_len, stream=F.Stream(), output_norm=out_norm, lm_head=lm_head, kv_fmt=KV.get(c["kv"]))


def _fill(dec, case, g, past):
    """Random keys and values of `past` earlier tokens in every layer's cache."""
    width = case["kv_heads"] * case["head_dim"]
    for cache in dec.caches if past else ():
        k, v = _f32(g, (past, width), 0.5), _f32(g, (past, width), 0.5)
        if case["kv"] == "f32":
            cache.append2(k, v)
        else:
            cache[0].append(k)
            cache[1].append(v)
    torch.cuda.synchronize()
    dec.set_pos(past)


def _cache_views(dec, case):
    """The caches as torch tensors: updated state a pass leaves behind."""
    views = []
    for cache in dec.caches:
        if case["kv"] == "f32":
            views += [_torch(cache.k), _torch(cache.v)]
        else:
            views += [_torch_bytes(b, b.nbytes) for c in cache for b in (c.codes, c.scales)]
    return views


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, s = case["kind"], {"case": case}
    if kind == "linear":
        s["w"] = _weight(g, case["fmt"], case["out"], case["in"])
        s["w"].matvec_precision(case["bits"])
        s["x"] = _f32(g, (case["rows"], case["in"]))
    elif kind in ("ffn", "ffn_prompt"):
        s["gate_up"], s["down"] = _weight(g, case["fmt"], 2 * case["ff"], case["d"]), _weight(g, case["fmt2"], case["d"], case["ff"])
        s["x"] = _f32(g, (case["rows"], case["d"]))
    elif kind == "gemm":
        s["w"] = _weight(g, case["fmt"], case["out"], case["in"])
        s["x"] = _f32(g, (case["rows"], case["in"]))
        if case["x"] == "bf16":
            s["x"] = s["x"].cvt_bf16()
    elif kind == "moe":
        d, eff, ne, t = case["d"], case["eff"], case["experts"], case["rows"]
        s["gate_up"], s["down"] = _weight(g, case["fmt"], ne * 2 * eff, d), _weight(g, case["fmt2"], ne * d, eff)
        s["x"], s["logits"] = _f32(g, (t, d)), _f32(g, (t, ne), 2.0)
    elif kind == "decode":
        dec = _decoder(case, g, case["ctx"] + case["tokens"], True)
        _fill(dec, case, g, case["ctx"])
        s["dec"], s["state"] = dec, _cache_views(dec, case)
        s["x"] = torch.randn((case["tokens"], case["d"]), generator=g, device="cuda").cpu().numpy()
        if case["graph"]:
            dec.capture()
    elif kind == "prefill":
        dec = _decoder(case, g, case["past"] + case["rows"], False)
        _fill(dec, case, g, case["past"])
        s["dec"], s["state"] = dec, _cache_views(dec, case)
        s["x"] = torch.randn((case["rows"], case["d"]), generator=g, device="cuda").cpu().numpy()
    else:
        n = case["values"] // BLOCK[case["fmt"]][0]
        s["raw"] = _blocks(case["fmt"], n, 0.02, g).reshape(-1).cpu().numpy()
    torch.cuda.synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        y = s["x"].matmul_q(s["w"])
        return y.to_vec() if case["to_host"] else _torch(y)
    if kind == "ffn":
        return _torch(s["x"].ffn(s["gate_up"], s["down"]))
    if kind == "ffn_prompt":
        return _torch(s["x"].ffn_coop(s["gate_up"], s["down"]))
    if kind == "gemm":
        return _torch(s["x"].gemm_q_bf16(s["w"]) if case["x"] == "bf16" else s["x"].matmul_q_coop(s["w"]))
    if kind == "moe":
        sel = s["logits"].moe_topk(None, case["k"], False, 1.0)
        h = s["x"].matmul_q_swiglu_id(s["gate_up"], sel, case["k"], case["eff"])
        return _torch(sel), _torch(h.matmul_q_id_wsum(s["down"], sel, case["d"]))
    if kind == "decode":
        dec, logits = s["dec"], []
        dec.set_pos(case["ctx"])                     # a new continuation of the same context
        for x in s["x"]:
            dec.set_input(x)
            if case["graph"]:
                dec.step_graph()
            else:
                dec.step()
            logits.append(dec.logits.to_vec(dec.stream))
        return logits, s["state"]
    if kind == "prefill":
        s["dec"].set_pos(case["past"])
        return s["dec"].prefill(s["x"]), s["state"]
    return F.deq_raw(s["raw"], case["values"], FORMATS[case["fmt"]])


# ---- what a pass cannot do without, and what its results may differ by ----------------------------------------------------------

def _nbytes(fmt, rows, cols):
    return rows * cols // BLOCK[fmt][0] * BLOCK[fmt][1]


def work(case):
    kind = case["kind"]
    if kind in ("linear", "gemm"):
        n, k, t = case["out"], case["in"], case["rows"]
        xb = 2 if case.get("x") == "bf16" else 4
        return {"bytes": _nbytes(case["fmt"], n, k) + t * (xb * k + 4 * n), "flops": 2 * t * n * k}
    if kind in ("ffn", "ffn_prompt"):
        d, ff, t = case["d"], case["ff"], case["rows"]
        return {"bytes": _nbytes(case["fmt"], 2 * ff, d) + _nbytes(case["fmt2"], d, ff) + 8 * t * d, "flops": 6 * t * d * ff}
    if kind == "moe":
        d, eff, k, t, ne = case["d"], case["eff"], case["k"], case["rows"], case["experts"]
        used = ne * (1 - (1 - k / ne) ** t)          # distinct experts t tokens choose, in the mean
        return {"bytes": int(used * (_nbytes(case["fmt"], 2 * eff, d) + _nbytes(case["fmt2"], d, eff))) + t * (8 * d + 4 * ne + 8 * k), "flops": 6 * t * k * d * eff}
    if kind == "dequant":
        return {"bytes": _nbytes(case["fmt"], 1, case["values"]) + 4 * case["values"], "flops": 0}
    d, ff, q, kv = case["d"], case["ff"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    weights = _nbytes("q4_k", q + 2 * kv, d) + _nbytes("q4_k", d, q) + _nbytes("q4_k", 2 * ff, d) + _nbytes("q6_k", d, ff)
    macs = (q + 2 * kv) * d + d * q + 3 * d * ff
    row = 2 * kv * KV_BITS[case["kv"]] / 8           # one token's key and value in one layer's cache
    if kind == "decode":
        n, total, flops = case["tokens"], 0.0, 0.0
        for i in range(n):                            # every token reads all weights and the cache behind it
            length = case["ctx"] + i + 1
            total += case["layers"] * (weights + row * length) + _nbytes("q6_k", case["vocab"], d) + 4 * (d + case["vocab"])
            flops += case["layers"] * (2 * macs + 4 * q * length) + 2 * d * case["vocab"]
        return {"bytes": total, "flops": flops}
    t, past = case["rows"], case["past"]
    seen = t * past + t * (t + 1) // 2
    return {"bytes": case["layers"] * (weights + row * (past + t)) + 8 * t * d, "flops": case["layers"] * (2 * t * macs + 4 * q * seen)}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1e-5 if case["bits"] == 24 else 2e-4}        # f32 sums; 16-bit activations where the weight was switched to them
    if kind in ("ffn", "moe"):
        return {"rel": 1e-5}
    if kind == "gemm":
        return {"rel": 3e-3}                                         # bf16 operands, f32 sums
    if kind == "ffn_prompt":
        return {"rel": 6e-3}                                         # the same twice, and a bf16 intermediate
    if kind == "decode":
        # f32 grade through the stack; a code of the quantized cache may fall on the other side of a rounding boundary
        return {"rel": 1e-4} if case["kv"] == "f32" else {"rel": 1e-3, "differ": 5e-3}
    if kind == "prefill":
        return {"rel": 1e-2} if case["kv"] == "f32" else {"rel": 2e-2, "differ": 1e-2}
    return "exact"
