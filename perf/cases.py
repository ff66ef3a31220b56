"""The workloads this framework is timed on, each through the public Python entry points of reng_hip.

A case is a dict of plain values; its "kind" names the path:

  layer      a decoder layer's seven projections quantized in one batch (the model load)
  matrix     one weight matrix quantized, any width, pitch, element type and scale scheme
  host       one weight matrix quantized from and to host memory (the Rust binding's call)
  check      a quantized matrix looked over: its per-row error statistics and its bf16 expansion
  product    bf16 activations times fp8 weights: decode batches (m = 1 .. 64) and prefill (m > 64)
  prefill    the activation quantized per token, then the fp8 x fp8 product
  decode     one token through decoder layers: norm, q/k/v, RoPE, attention, o, gate/up, down
  attention  one query per head against a long key/value cache

Sizes are those of bench.py and the tests (Llama-3.1-8B, Qwen2.5-7B, Qwen2.5-32B layers) and, in
draw(), of the ranges around them. Weights are N(0, 0.02) with a few outlier columns, as trained
projections are; activations N(0, 1).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "reciprocating-engine_amd"))

import reng_hip as R  # noqa: E402

MAX_FINITE = {"e4m3": 240.0, "e5m2": 57344.0}
TORCH_FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def listed():
    return [
        # Model load: the seven projections of a Llama-3.1-8B layer (436 MB of bf16), bench.py's workload by the layer.
        dict(name="quantize_layer_llama8b", kind="layer", hidden=4096, inter=14336, heads=32, kv=8, hd=128,
             fmt="e4m3", scaling="pcs"),
        # The smallest quantize of bench.py: one f32 matrix, where a launch's latency counts.
        dict(name="quantize_f32_2048", kind="matrix", rows=2048, cols=2048, ld=2048, dtype="f32", fmt="e4m3",
             scaling="pcs"),
        # A width that is no multiple of a vector, under the hardware-bias scheme (one scale for the whole matrix).
        dict(name="quantize_hw_odd_width", kind="matrix", rows=4099, cols=4001, ld=4001, dtype="bf16", fmt="e4m3",
             scaling="hw"),
        # What the Rust quantize_with binding calls: host memory in, host memory out.
        dict(name="quantize_host_4096", kind="host", rows=4096, cols=4096, dtype="bf16", fmt="e4m3", scaling="pcs"),
        # After a quantize: the error report over every row and the bf16 weights an engine without fp8 would use.
        dict(name="check_down_llama8b", kind="check", rows=4096, cols=14336, fmt="e4m3"),
        # Serving one sequence: the gate projection of Llama-3.1-8B.
        dict(name="gemv_gate_llama8b", kind="product", m=1, n=14336, k=4096, fmt="e4m3"),
        # Serving small batches: Qwen2.5-7B's gate/up and down projections.
        dict(name="batch8_down_qwen7b", kind="product", m=8, n=3584, k=18944, fmt="e4m3"),
        dict(name="batch64_gate_qwen7b", kind="product", m=64, n=18944, k=3584, fmt="e4m3"),
        # A short prompt, or a large decode batch, on the bf16 matrix cores.
        dict(name="rows256_gate_llama8b", kind="product", m=256, n=14336, k=4096, fmt="e4m3"),
        # A prompt of 1024 tokens through Qwen2.5-32B's gate projection in fp8, activations quantized on the way.
        dict(name="prefill1024_gate_qwen32b", kind="prefill", m=1024, n=27648, k=5120, fmt="e4m3", afmt="e4m3"),
        # One token through four Llama-3.1-8B layers with 512 cached positions.
        dict(name="decode_4_layers_llama8b", kind="decode", layers=4, hidden=4096, inter=14336, heads=32, kv=8,
             hd=128, length=512, fmt="e4m3"),
        # One token's attention over a long context (Llama-3.1-8B heads).
        dict(name="attention_32k_llama8b", kind="attention", heads=32, kv=8, hd=128, length=32768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(v, of):
    return max(of, v // of * of)


def draw(rng):
    kind = rng.choice(["layer", "matrix", "matrix", "host", "check", "product", "product", "product", "prefill",
                       "decode", "attention"])
    fmt = "e4m3" if rng.random() < 0.75 else "e5m2"
    if kind == "layer":
        hd = rng.choice([64, 128])
        kv = rng.choice([2, 4, 8])
        heads = kv * rng.choice([2, 4, 7])
        hidden = _mult(_log(rng, 512, 4096), rng.choice([8, 64, 256]))
        inter = _mult(int(hidden * rng.uniform(2.5, 3.5)), rng.choice([8, 64, 256]))
        return dict(kind=kind, hidden=hidden, inter=inter, heads=min(heads, 32), kv=kv, hd=hd, fmt=fmt,
                    scaling=rng.choice(["pcs", "pcs", "hw", "unit"]))
    if kind in ("matrix", "host"):
        cols = _log(rng, 64, 28672)
        if rng.random() < 0.6:
            cols = _mult(cols, rng.choice([8, 64, 256]))
        rows = min(_log(rng, 64, 16384), (48 << 20) // cols)
        c = dict(kind=kind, rows=rows, cols=cols, dtype=rng.choice(["bf16", "bf16", "f32"]), fmt=fmt,
                 scaling=rng.choice(["pcs", "pcs", "hw", "unit"]))
        if kind == "matrix":   # a strided window (a tensor-parallel shard of wider rows) one time in four
            c["ld"] = cols + rng.choice([8, 64, 1024, cols]) if rng.random() < 0.25 else cols
        return c
    if kind == "check":
        cols = _log(rng, 256, 18944)
        if rng.random() < 0.7:
            cols = _mult(cols, 64)
        return dict(kind=kind, rows=min(_log(rng, 256, 18944), (58 << 20) // cols), cols=cols, fmt=fmt)
    if kind == "product":
        m = _log(rng, 1, 1024)
        k = _mult(_log(rng, 1024, 27648), rng.choice([16, 128, 256]))
        n = _log(rng, 512, 27648)
        n = _mult(n, rng.choice([1, 16, 128]))
        n = max(64, min(n, int(1.4e11 / (2.0 * m * k)), (96 << 20) // k))
        return dict(kind=kind, m=m, n=n, k=k, fmt=fmt)
    if kind == "prefill":
        m = _log(rng, 65, 2048)
        m = m if rng.random() < 0.4 else _mult(m, 64)
        k = _mult(_log(rng, 1024, 16384), rng.choice([128, 256]))
        n = _mult(_log(rng, 512, 27648), rng.choice([8, 128]))
        n = max(64, min(n, int(2.8e11 / (2.0 * m * k))))
        return dict(kind=kind, m=m, n=n, k=k, fmt=fmt, afmt=rng.choice(["e4m3", "e4m3", "e5m2"]))
    hd = rng.choice([64, 128, 128])
    kv = rng.choice([2, 4, 8])
    heads = kv * rng.choice([2, 4, 7] if kv < 8 else [2, 4])
    if kind == "decode":
        hidden = _mult(_log(rng, 1024, 5120), 128)
        return dict(kind=kind, layers=rng.choice([2, 3]), hidden=hidden, inter=_mult(int(hidden * rng.uniform(2.5, 3.5)), 128),
                    heads=heads, kv=kv, hd=hd, length=_log(rng, 16, 4096), fmt=fmt)
    return dict(kind=kind, heads=heads, kv=kv, hd=hd, length=_log(rng, 64, 32768))


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(g, rows, cols, dtype=torch.bfloat16):
    w = torch.randn(rows, cols, generator=g, device="cuda")
    w.mul_(0.02)
    w[:, :: 97] *= 4.0
    return w.to(dtype)


def _codes(w, fmt):
    """Per-row absmax codes and scales of w in plain torch: RN32(w / s) to the format, to nearest even."""
    top = MAX_FINITE[fmt]
    wf = w.float()
    s = wf.abs().amax(1) / top
    q = (wf / s[:, None]).clamp_(-top, top)
    return q.to(TORCH_FP8[fmt]).view(torch.uint8), s


def _values(codes, scales, fmt):
    """The weights that codes and scales stand for, in 64 bits."""
    return codes.view(TORCH_FP8[fmt]).float().double() * scales.double()[:, None]


def _projection(g, rows, cols, fmt):
    return _codes(_weight(g, rows, cols), fmt)


def _torch_dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _layer_shapes(c):
    q, kv = c["heads"] * c["hd"], c["kv"] * c["hd"]
    return [(q, c["hidden"]), (kv, c["hidden"]), (kv, c["hidden"]), (c["hidden"], q), (c["inter"], c["hidden"]),
            (c["inter"], c["hidden"]), (c["hidden"], c["inter"])]


def _buffers(rows, cols):
    return (torch.empty(rows * cols, dtype=torch.uint8, device="cuda"),
            torch.empty(rows, dtype=torch.float32, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda"))


def _decode_layers(c, g):
    """Per layer: [Wq; Wk; Wv] in rotation-pair order, Wo, gate/up rows alternating, Wd, norm gains, caches."""
    h, q, kv = c["hidden"], c["heads"] * c["hd"], c["kv"] * c["hd"]
    for _ in range(c["layers"]):
        kc, vc = (torch.randn(c["length"], kv, generator=g, device="cuda").bfloat16() for _ in range(2))
        yield dict(qkv=_projection(g, q + 2 * kv, h, c["fmt"]), o=_projection(g, h, q, c["fmt"]),
                   gu=_projection(g, 2 * c["inter"], h, c["fmt"]), d=_projection(g, h, c["inter"], c["fmt"]),
                   g1=1.0 + 0.1 * torch.randn(h, generator=g, device="cuda"),
                   g2=1.0 + 0.1 * torch.randn(h, generator=g, device="cuda"), kc=kc, vc=vc, k_row=kc[-1], v_row=vc[-1])


def _rope_row(c):
    """sin and cos of the last position (rotate-half, theta 500000)."""
    half = c["hd"] // 2
    d = torch.arange(c["hd"], device="cuda", dtype=torch.float64) % half
    a = (c["length"] - 1) * 500000.0 ** (-2.0 * d / c["hd"])
    return a.sin().float(), a.cos().float()


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind == "layer":
        mats = []
        for rows, cols in _layer_shapes(c):
            w = _weight(g, rows, cols)
            mats.append((w, rows, cols, *_buffers(rows, cols)))
        return dict(c, mats=mats)
    if kind == "matrix":
        return dict(c, w=_weight(g, c["rows"], c["ld"], _torch_dtype(c)), out=_buffers(c["rows"], c["cols"]))
    if kind == "host":
        w = _weight(g, c["rows"], c["cols"], _torch_dtype(c))
        w = (w.view(torch.int16) if c["dtype"] == "bf16" else w).cpu().numpy()
        return dict(c, w=w.view(np.uint16) if c["dtype"] == "bf16" else w)
    if kind == "check":
        w = _weight(g, c["rows"], c["cols"])
        codes, scales = _codes(w, c["fmt"])
        return dict(c, w=w, q=R.Quantized(c["fmt"], "pcs", c["rows"], c["cols"], codes.reshape(-1), scales,
                                          R.EXPONENT_BIAS[R.FORMAT_NAMES[c["fmt"]]]))
    if kind == "product":
        x = torch.randn(c["m"], c["k"], generator=g, device="cuda").bfloat16()
        codes, scales = _projection(g, c["n"], c["k"], c["fmt"])
        return dict(c, x=x, codes=codes, scales=scales,
                    y=torch.empty(c["m"] * c["n"], dtype=torch.bfloat16, device="cuda"))
    if kind == "prefill":
        x = torch.randn(c["m"], c["k"], generator=g, device="cuda").bfloat16()
        codes, scales = _projection(g, c["n"], c["k"], c["fmt"])
        acodes, ascales, _ = _buffers(c["m"], c["k"])
        return dict(c, x=x, codes=codes, scales=scales, acodes=acodes, ascales=ascales,
                    y=torch.empty(c["m"] * c["n"], dtype=torch.bfloat16, device="cuda"))
    if kind == "decode":
        x = torch.randn(c["hidden"], generator=g, device="cuda")
        layers = list(_decode_layers(c, g))
        sn, cs = _rope_row(c)
        bf = dict(dtype=torch.bfloat16, device="cuda")
        return dict(c, x=x, layers_=layers, sn=sn, cs=cs, scale=c["hd"] ** -0.5,
                    q=torch.empty(c["heads"] * c["hd"], **bf), a=torch.empty(c["heads"] * c["hd"], **bf),
                    act=torch.empty(c["inter"], **bf), h=torch.empty(c["hidden"], device="cuda"),
                    y=torch.empty(c["hidden"], device="cuda"),
                    ws=torch.empty(max(1, R.attention_workspace_bytes(c["heads"], c["hd"], c["length"])),
                                   dtype=torch.uint8, device="cuda"))
    if kind == "attention":
        kv = c["kv"] * c["hd"]
        q = torch.randn(c["heads"] * c["hd"], generator=g, device="cuda").bfloat16()
        return dict(c, q=q, kc=torch.randn(c["length"], kv, generator=g, device="cuda").bfloat16(),
                    vc=torch.randn(c["length"], kv, generator=g, device="cuda").bfloat16(), scale=c["hd"] ** -0.5,
                    ws=torch.empty(max(1, R.attention_workspace_bytes(c["heads"], c["hd"], c["length"])),
                                   dtype=torch.uint8, device="cuda"),
                    out=torch.empty(c["heads"] * c["hd"], dtype=torch.bfloat16, device="cuda"))
    raise ValueError(kind)


# ---------------------------------------------------------------- one pass


def run(s):
    kind = s["kind"]
    if kind == "layer":
        R.quantize_batch(s["mats"], s["fmt"], s["scaling"])
        return [(m[3], m[4], m[5]) for m in s["mats"]]
    if kind == "matrix":
        codes, scales, bias = s["out"]
        R.quantize_into(s["w"], s["rows"], s["cols"], s["fmt"], s["scaling"], 1.0, codes, scales, bias, ld=s["ld"])
        return codes, scales, bias
    if kind == "host":
        return R.quantize_host(s["w"], s["rows"], s["cols"], s["fmt"], s["scaling"])
    if kind == "check":
        mean, worst = R.row_errors(s["w"], s["q"])
        return mean, worst, s["q"].dequantize_bf16().view(torch.bfloat16)
    if kind == "product":
        return R.gemm_w8a16(s["x"], s["codes"], s["scales"], s["m"], s["n"], s["k"], s["fmt"], s["y"])
    if kind == "prefill":
        R.quantize_into(s["x"], s["m"], s["k"], s["afmt"], "pcs", 1.0, s["acodes"], s["ascales"])
        y = R.gemm_fp8_scaled(s["acodes"], s["afmt"], s["ascales"], s["codes"], s["fmt"], s["scales"], s["m"], s["n"],
                              s["k"], s["y"])
        return y, s["acodes"], s["ascales"]
    if kind == "decode":
        x, h, n, fmt = s["x"], s["hidden"], 2 * s["inter"], s["fmt"]
        for L in s["layers_"]:
            R.gemv_rmsnorm_qkv_rope(x, L["g1"], 1e-5, *L["qkv"], s["heads"], s["kv"], s["hd"], h, fmt, s["sn"],
                                    s["cs"], s["q"], L["k_row"], L["v_row"])
            R.attention_decode_split(s["q"], L["kc"], L["vc"], s["heads"], s["kv"], s["hd"], s["length"], s["scale"],
                                     s["ws"], s["a"])
            R.gemv_residual(s["a"], *L["o"], h, s["heads"] * s["hd"], fmt, x, s["h"])
            R.gemv_rmsnorm(s["h"], L["g2"], 1e-5, *L["gu"], n, h, fmt, swiglu=True, out=s["act"])
            R.gemv_residual(s["act"], *L["d"], h, s["inter"], fmt, s["h"], s["y"])
            x = s["y"]
        return s["y"], [(L["k_row"], L["v_row"]) for L in s["layers_"]]
    return R.attention_decode_split(s["q"], s["kc"], s["vc"], s["heads"], s["kv"], s["hd"], s["length"], s["scale"],
                                    s["ws"], s["out"])


# ---------------------------------------------------------------- what a pass cannot do without


def work(c):
    kind = c["kind"]
    if kind == "layer":
        return dict(bytes=sum(3 * r * k + 4 * r for r, k in _layer_shapes(c)), flops=0)
    if kind in ("matrix", "host"):
        e = 2 if c["dtype"] == "bf16" else 4
        return dict(bytes=c["rows"] * c["cols"] * (e + 1) + 4 * c["rows"], flops=0)
    if kind == "check":   # weights and codes in, bf16 weights out; scales and the two statistics per row
        return dict(bytes=5 * c["rows"] * c["cols"] + 12 * c["rows"], flops=0)
    if kind == "product":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=n * k + 4 * n + 2 * m * k + 2 * m * n, flops=2 * m * n * k)
    if kind == "prefill":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=3 * m * k + 4 * m + n * k + 4 * n + 2 * m * n, flops=2 * m * n * k)
    if kind == "decode":
        weights = sum(r * k + 4 * r for r, k in _layer_shapes(c))
        cache = 2 * 2 * c["length"] * c["kv"] * c["hd"]
        return dict(bytes=c["layers"] * (weights + cache + 8 * c["hidden"]) + 8 * c["hidden"],
                    flops=c["layers"] * (2 * sum(r * k for r, k in _layer_shapes(c))
                                         + 4 * c["length"] * c["heads"] * c["hd"]))
    return dict(bytes=4 * c["length"] * c["kv"] * c["hd"] + 4 * c["heads"] * c["hd"],
                flops=4 * c["length"] * c["heads"] * c["hd"])


def tolerance(c):
    """Codes, scales and biases are exact; the statistics are f32 over f64 sums; a bf16 product is its f32 sum
    rounded once (2^-9 of a value at most, 1.7e-3 in the 2-norm: another order of the sum moves the values that
    lie next to a rounding edge); a decode step carries such roundings through every layer after them."""
    kind = c["kind"]
    if kind in ("layer", "matrix", "host"):
        return "exact"
    if kind == "check":
        return dict(rel=1e-5, max=1e-4)
    if kind == "decode":
        return dict(rel=1e-2, max=0.1)
    return dict(rel=5e-3, max=0.02)


# ---------------------------------------------------------------- the same in 64 bits


def _scales64(w, fmt):
    """Per-row absmax scales in 64 bits."""
    return w.double().abs().amax(1) / MAX_FINITE[fmt]


def _attend64(q, kc, vc, c):
    """q [heads * hd], caches [length, kv * hd], all 64-bit: softmax(q k / sqrt(hd)) v per head."""
    heads, kv, hd = c["heads"], c["kv"], c["hd"]
    q = q.view(kv, heads // kv, hd)
    out = []
    for i in range(kv):
        k, v = kc[:, i * hd:(i + 1) * hd], vc[:, i * hd:(i + 1) * hd]
        out.append(torch.softmax(q[i] @ k.t().contiguous() * hd ** -0.5, 1) @ v.contiguous())
    return torch.cat(out).reshape(-1)


def _rope64(pairs, sn, cs, heads, hd):
    """Rows in rotation-pair order (d, d + half adjacent) to rotated heads."""
    half = hd // 2
    v = pairs.view(heads, half, 2)
    a, b = v[:, :, 0], v[:, :, 1]
    return torch.cat([a * cs[:half] - b * sn[:half], b * cs[half:] + a * sn[half:]], 1).reshape(-1)


def exact(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if c.get("scaling", "pcs") != "pcs":
        return None   # codes, and scales that are powers of two by rule
    if kind == "layer":
        out = []
        for rows, cols in _layer_shapes(c):
            out.append((None, _scales64(_weight(g, rows, cols), c["fmt"]), None))
        return out
    if kind == "matrix":
        w = _weight(g, c["rows"], c["ld"], _torch_dtype(c))
        return None, _scales64(w[:, : c["cols"]], c["fmt"]), None
    if kind == "host":
        return None, _scales64(_weight(g, c["rows"], c["cols"], _torch_dtype(c)), c["fmt"]).cpu().numpy(), None
    if kind == "check":
        w = _weight(g, c["rows"], c["cols"])
        want = _values(*_codes(w, c["fmt"]), c["fmt"])
        wd = w.double()
        rel = torch.where(wd == 0, 0.0, (want - wd).abs() / wd.abs())
        n = (wd != 0).sum(1).clamp(min=1)
        return rel.sum(1) / n, rel.amax(1), want.reshape(-1)
    if kind in ("product", "prefill"):
        x = torch.randn(c["m"], c["k"], generator=g, device="cuda").bfloat16()
        codes, scales = _projection(g, c["n"], c["k"], c["fmt"])
        a = x.double()
        if kind == "prefill":
            ac, asc = _codes(x, c["afmt"])
            a = _values(ac, asc, c["afmt"])
        y = torch.empty(c["m"], c["n"], dtype=torch.float64, device="cuda")
        for n0 in range(0, c["n"], 8192):   # a slice of the columns at a time
            v = _values(codes[n0:n0 + 8192], scales[n0:n0 + 8192], c["fmt"])
            y[:, n0:n0 + 8192] = a @ v.t()
        y = y.reshape(-1)
        return (y, None, asc.double()) if kind == "prefill" else y
    if kind == "decode":
        x = torch.randn(c["hidden"], generator=g, device="cuda").double()
        layers = list(_decode_layers(c, g))
        sn, cs = (t.double() for t in _rope_row(c))
        q, kv, hd = c["heads"] * c["hd"], c["kv"] * c["hd"], c["hd"]

        def norm(v, gain):
            return v / torch.sqrt(v.square().mean() + 1e-5) * gain.double()

        rows = []
        for L in layers:
            p = _values(*L["qkv"], c["fmt"]) @ norm(x, L["g1"])
            kc, vc = L["kc"].double(), L["vc"].double()
            kc[-1] = _rope64(p[q:q + kv], sn, cs, c["kv"], hd)
            vc[-1] = p[q + kv:]
            a = _attend64(_rope64(p[:q], sn, cs, c["heads"], hd), kc, vc, c)
            h = x + _values(*L["o"], c["fmt"]) @ a
            gu = _values(*L["gu"], c["fmt"]) @ norm(h, L["g2"])
            x = h + _values(*L["d"], c["fmt"]) @ (torch.nn.functional.silu(gu[0::2]) * gu[1::2])
            rows.append((kc[-1].clone(), vc[-1].clone()))
        return x, rows
    kv = c["kv"] * c["hd"]
    q = torch.randn(c["heads"] * c["hd"], generator=g, device="cuda").bfloat16()
    kc = torch.randn(c["length"], kv, generator=g, device="cuda").bfloat16()
    vc = torch.randn(c["length"], kv, generator=g, device="cuda").bfloat16()
    return _attend64(q.double(), kc.double(), vc.double(), c)
