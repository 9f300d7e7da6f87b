"""The work that users of the quantized-matmul library have it do, as timed cases.

A case is one pass through the public entry points at one shape.  Its kinds:

  decode      one token, one matrix: swamp_qgemv
  multi       one token, several matrices of one x: swamp_qgemv_multi
  layer       one token through a transformer layer's matrices, as an engine
              issues them: RMSNorm+QKV, O, RMSNorm+gate/up, SwiGLU+down
  logits      one token's logits: RMSNorm + the lm_head
  batch       n tokens, one matrix, fp32 activations: swamp_qgemv_batched
              (speculative verify, continuous batching, chunked prompts)
  batchlayer  n tokens through a layer's matrices with the activation
              producers between them
  prefill     m tokens, one matrix, bf16 activations: swamp_qgemm
  int8        m tokens, one matrix, activations quantized to Q8_0 by the
              device quantizer and multiplied as int8
  mlp         m tokens through a layer's feed-forward block: RMSNorm, gate,
              up, SwiGLU, down with bf16 activations
  dequant     a whole tensor dequantized to fp32 or bf16

Weights are N(0, 0.02^2) matrices quantized to GGUF blocks, activations
N(0, 1).
"""
import importlib.util
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEVICE = "cuda"
EPS = 1e-5
SIGMA = 0.02

Q4_0, Q8_0, Q4_K, Q6_K = "Q4_0", "Q8_0", "Q4_K", "Q6_K"
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}


def _package():
    if "llamanyon_rs_amd" not in sys.modules:
        path = os.path.join(ROOT, "llamanyon.rs_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("llamanyon_rs_amd", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["llamanyon_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["llamanyon_rs_amd"]


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest call of a decode step: one token's K and V projections
        # of an 8B model with grouped-query attention.
        {"name": "decode_kv_q4_0", "kind": "multi", "dtype": Q4_0, "rows": 1024, "mats": 2,
         "k": 4096},
        # One token through one 8B layer of a Q4_K_M file, whose V and down
        # projections are Q6_K in half of the layers: what decode speed is made of.
        {"name": "decode_layer_q4_k_m", "kind": "layer", "dtype": Q4_K, "dtype2": Q6_K,
         "hidden": 4096, "kv": 1024, "ffn": 14336},
        # One token's logits, the largest single matrix of a decode step.
        {"name": "decode_logits_q6_k", "kind": "logits", "dtype": Q6_K, "rows": 128256, "k": 4096},
        # Speculative verify: five tokens through the same layer.
        {"name": "verify_layer_q4_k_m", "kind": "batchlayer", "dtype": Q4_K, "dtype2": Q6_K,
         "n": 5, "hidden": 4096, "kv": 1024, "ffn": 14336},
        # Continuous batching: 16 sequences decode together, long rows.
        {"name": "batch16_down_q4_k", "kind": "batch", "dtype": Q4_K, "n": 16, "rows": 4096,
         "k": 14336},
        # A fuller batch on the widest matrix of a layer, Q8_0 weights.
        {"name": "batch48_gate_up_q8_0", "kind": "batch", "dtype": Q8_0, "n": 48, "rows": 28672,
         "k": 4096},
        # A short chat prompt handed over as fp32 activations.
        {"name": "prompt150_qkv_q4_k", "kind": "batch", "dtype": Q4_K, "n": 150, "rows": 6144,
         "k": 4096},
        # A prompt of 512 tokens, fused QKV, the benchmark's small prefill shape.
        {"name": "prefill512_qkv_q4_0", "kind": "prefill", "dtype": Q4_0, "m": 512, "rows": 6144,
         "k": 4096},
        # A ragged prompt through a Q6_K down projection of a Q4_K_M file.
        {"name": "prefill777_down_q6_k", "kind": "prefill", "dtype": Q6_K, "m": 777, "rows": 4096,
         "k": 14336},
        # The feed-forward block of an 8B layer over a prompt of 2048 tokens.
        {"name": "prefill2048_mlp_q4_k", "kind": "mlp", "dtype": Q4_K, "m": 2048, "hidden": 4096,
         "ffn": 14336},
        # The exact-integer prefill, quantizer included, the benchmark's shape.
        {"name": "int8_2048_gate_up_q4_0", "kind": "int8", "dtype": Q4_0, "m": 2048,
         "rows": 28672, "k": 4096},
        # A whole tensor back to fp32 (embedding tables, offline conversion).
        {"name": "dequant_gate_q4_k", "kind": "dequant", "dtype": Q4_K, "rows": 14336, "k": 4096,
         "out": "f32"},
    ]


def _span(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["decode", "multi", "layer", "logits", "batch", "batch", "batch",
                       "batchlayer", "prefill", "prefill", "int8", "mlp", "dequant"])
    dtype = rng.choice([Q4_0, Q8_0, Q4_K, Q6_K])
    # row lengths: whole blocks of every format, up to the 70B feed-forward's
    k = 256 * rng.choice([4, 8, 10, 11, 16, 20, 28, 32, 43, 56, 74, 112])
    if kind == "decode":
        return {"kind": kind, "dtype": dtype, "rows": _span(rng, 512, 40000), "k": k}
    if kind == "multi":
        return {"kind": kind, "dtype": dtype, "rows": _span(rng, 512, 20000),
                "mats": rng.choice([2, 3]), "k": k}
    if kind in ("layer", "batchlayer", "mlp"):
        hidden = 512 * rng.choice([4, 5, 6, 8, 10, 16])
        ffn = 512 * max(1, int(hidden * rng.uniform(2.5, 3.6)) // 512)
        if kind == "mlp":
            m = _span(rng, 100, 2048)
            while 6 * m * hidden * ffn > 7e11:
                m = m * 3 // 4
            return {"kind": kind, "dtype": dtype, "m": m, "hidden": hidden, "ffn": ffn}
        case = {"kind": kind, "dtype": dtype, "dtype2": rng.choice([dtype, Q6_K]),
                "hidden": hidden, "kv": 128 * rng.choice([2, 4, 8]), "ffn": ffn}
        if kind == "batchlayer":
            case["n"] = _span(rng, 2, 64)
        return case
    if kind == "logits":
        return {"kind": kind, "dtype": dtype, "rows": rng.choice([32000, 49155, 128256, 151937]),
                "k": 512 * rng.choice([4, 5, 6, 8, 10])}
    if kind == "batch":
        return {"kind": kind, "dtype": dtype, "n": _span(rng, 2, 256),
                "rows": _span(rng, 1000, 29000), "k": 512 * max(2, k // 512)}
    if kind in ("prefill", "int8"):
        m, rows = _span(rng, 65, 4000), _span(rng, 1000, 29000)
        while 2 * m * rows * k > 6e11:
            m = m * 3 // 4
        if kind == "int8" and dtype == Q6_K:
            dtype = Q4_0
        return {"kind": kind, "dtype": dtype, "m": m, "rows": rows, "k": k}
    return {"kind": kind, "dtype": dtype, "rows": _span(rng, 1000, 29000), "k": min(k, 8192),
            "out": rng.choice(["f32", "bf16"])}


# ------------------------------------------------- GGUF blocks (torch, device)

def _bytes(f16):
    return f16.contiguous().view(torch.uint8).reshape(f16.shape + (2,))


def _quantize(dtype, w):
    """Rows of fp32 weights to GGUF block bytes, one flat uint8 tensor."""
    rows, k = w.shape
    bs, ts = BLOCK[dtype]
    v = w.reshape(rows, k // bs, bs)
    if dtype == Q4_0:
        big = v.gather(-1, v.abs().argmax(-1, keepdim=True))
        d = (big / -8).half()
        inv = torch.where(d == 0, 0.0, 1.0 / d.float())
        q = (v * inv + 8.5).floor().clamp(0, 15).to(torch.uint8)
        out = torch.cat([_bytes(d.squeeze(-1)), q[..., 0::2] | q[..., 1::2] << 4], -1)
    elif dtype == Q8_0:
        d = v.abs().amax(-1, keepdim=True) / 127
        q = torch.where(d == 0, 0.0, v / d).round().clamp(-127, 127).to(torch.int8)
        out = torch.cat([_bytes(d.half().squeeze(-1)), q.view(torch.uint8)], -1)
    elif dtype == Q4_K:
        s = v.reshape(rows, k // bs, 8, 32)
        low = (-s.amin(-1)).clamp(min=0)
        span = (s.amax(-1) + low) / 15
        d = (span.amax(-1, keepdim=True) / 63).half()
        dm = (low.amax(-1, keepdim=True) / 63).half()
        sc = (span / d.float().clamp(min=1e-12)).round().clamp(0, 63)
        mn = (low / dm.float().clamp(min=1e-12)).round().clamp(0, 63)
        step = (d.float() * sc).clamp(min=1e-12).unsqueeze(-1)
        q = ((s + (dm.float() * mn).unsqueeze(-1)) / step).round().clamp(0, 15).to(torch.uint8)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        packed = torch.cat([sc[..., :4] | (sc[..., 4:] >> 4) << 6,
                            mn[..., :4] | (mn[..., 4:] >> 4) << 6,
                            (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4], -1)
        nib = (q[..., 0::2, :] | q[..., 1::2, :] << 4).reshape(rows, k // bs, 128)
        out = torch.cat([_bytes(d.squeeze(-1)), _bytes(dm.squeeze(-1)), packed, nib], -1)
    else:
        s = v.reshape(rows, k // bs, 16, 16)
        span = s.abs().amax(-1) / 31
        d = (span.amax(-1, keepdim=True) / 127).half()
        sc = (span / d.float().clamp(min=1e-12)).round().clamp(0, 127)
        step = (d.float() * sc).clamp(min=1e-12).unsqueeze(-1)
        q = ((s / step).round().clamp(-32, 31) + 32).to(torch.uint8)
        q = q.reshape(rows, k // bs, 2, 4, 32)
        low, high = q & 15, q >> 4
        ql = torch.cat([low[..., 0, :] | low[..., 2, :] << 4, low[..., 1, :] | low[..., 3, :] << 4], -1)
        qh = high[..., 0, :] | high[..., 1, :] << 2 | high[..., 2, :] << 4 | high[..., 3, :] << 6
        out = torch.cat([ql.reshape(rows, k // bs, 128), qh.reshape(rows, k // bs, 64),
                         sc.to(torch.uint8), _bytes(d.squeeze(-1))], -1)
    assert out.shape[-1] == ts
    return out.reshape(-1)


def _dequantize(dtype, raw, rows, k):
    """Block bytes to the fp64 weights they stand for."""
    bs, ts = BLOCK[dtype]
    b = raw.reshape(rows, k // bs, ts)

    def half_at(at):
        return b[..., at:at + 2].contiguous().view(torch.float16).double()

    if dtype == Q4_0:
        q = torch.stack([b[..., 2:] & 15, b[..., 2:] >> 4], -1).reshape(rows, k // bs, 32)
        w = (q.double() - 8) * half_at(0)
    elif dtype == Q8_0:
        w = b[..., 2:].contiguous().view(torch.int8).double() * half_at(0)
    elif dtype == Q4_K:
        p = b[..., 4:16]
        sc = torch.cat([p[..., :4] & 63, (p[..., 8:] & 15) | (p[..., :4] >> 6) << 4], -1)
        mn = torch.cat([p[..., 4:8] & 63, (p[..., 8:] >> 4) | (p[..., 4:8] >> 6) << 4], -1)
        nib = b[..., 16:].reshape(rows, k // bs, 4, 32)
        q = torch.stack([nib & 15, nib >> 4], -2).reshape(rows, k // bs, 8, 32)
        w = (half_at(0) * sc.double()).unsqueeze(-1) * q.double() \
            - (half_at(2) * mn.double()).unsqueeze(-1)
    else:
        ql = b[..., :128].reshape(rows, k // bs, 2, 2, 32)
        qh = b[..., 128:192].reshape(rows, k // bs, 2, 32)
        q = torch.stack([(ql[..., j & 1, :] >> 4 * (j >> 1) & 15) | (qh >> 2 * j & 3) << 4
                         for j in range(4)], -2).reshape(rows, k // bs, 16, 16)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        w = (half_at(208) * sc).unsqueeze(-1) * (q.double() - 32)
    return w.reshape(rows, k)


# -------------------------------------------------------------------- prepare

class _Inputs:
    """Seeded tensors on the device, in one order."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device=DEVICE)

    def weights(self, dtype, rows, k):
        step = max(1, (1 << 26) // k)
        return torch.cat([_quantize(dtype, SIGMA * self.normal(min(step, rows - r), k))
                          for r in range(0, rows, step)])

    def norm_weights(self, k):
        return 1 + 0.1 * self.normal(k)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEVICE)


def prepare(case, seed):
    gen, kind, c = _Inputs(seed), case["kind"], case
    s = {"case": case, "pkg": _package(), "stream": torch.cuda.current_stream().cuda_stream}
    if kind in ("layer", "batchlayer"):
        h, kv, f, n = c["hidden"], c["kv"], c["ffn"], c.get("n", 1)
        shapes = {"q": (c["dtype"], h, h), "k": (c["dtype"], kv, h), "v": (c["dtype2"], kv, h),
                  "o": (c["dtype"], h, h), "gate": (c["dtype"], f, h), "up": (c["dtype"], f, h),
                  "down": (c["dtype2"], h, f)}
        for name, (dtype, rows, k) in shapes.items():
            s["w_" + name] = gen.weights(dtype, rows, k)
            s["y_" + name] = _empty(n, rows)
        s["x"], s["attn"] = gen.normal(n, h), gen.normal(n, h)
        s["norm1"], s["norm2"] = gen.norm_weights(h), gen.norm_weights(h)
        s["xn"], s["xn2"], s["act"] = _empty(n, h), _empty(n, h), _empty(n, f)
        s["shapes"] = shapes
    elif kind == "mlp":
        h, f, m = c["hidden"], c["ffn"], c["m"]
        s["w_gate"], s["w_up"] = gen.weights(c["dtype"], f, h), gen.weights(c["dtype"], f, h)
        s["w_down"] = gen.weights(c["dtype"], h, f)
        s["x"], s["norm1"] = gen.normal(m, h), gen.norm_weights(h)
        s["xn"], s["act"] = _empty(m, h, dtype=torch.bfloat16), _empty(m, f, dtype=torch.bfloat16)
        s["y_gate"], s["y_up"], s["y_down"] = _empty(m, f), _empty(m, f), _empty(m, h)
    elif kind == "multi":
        s["x"] = gen.normal(1, c["k"])
        s["w"] = [gen.weights(c["dtype"], c["rows"], c["k"]) for _ in range(c["mats"])]
        s["y"] = [_empty(c["rows"]) for _ in range(c["mats"])]
    elif kind == "dequant":
        s["w"] = gen.weights(c["dtype"], c["rows"], c["k"])
        s["y"] = _empty(c["rows"], c["k"],
                        dtype=torch.float32 if c["out"] == "f32" else torch.bfloat16)
    else:
        n = c.get("n", c.get("m", 1))
        s["w"] = gen.weights(c["dtype"], c["rows"], c["k"])
        s["x"] = gen.normal(n, c["k"])
        s["y"] = _empty(n, c["rows"])
        if kind == "logits":
            s["norm1"] = gen.norm_weights(c["k"])
        elif kind == "prefill":
            s["x"] = s["x"].bfloat16()
        elif kind == "int8":
            s["xq"] = _empty(n * c["k"] // 32 * 34, dtype=torch.uint8)
    return s


# ------------------------------------------------------------------------ run

def run(s):
    c, p, st = s["case"], s["pkg"], s["stream"]
    kind = c["kind"]
    code = {Q4_0: p.Q4_0, Q8_0: p.Q8_0, Q4_K: p.Q4_K, Q6_K: p.Q6_K}
    dt = code[c["dtype"]]
    if kind == "decode":
        p.qgemv(dt, s["w"].data_ptr(), s["w"].numel(), s["x"].data_ptr(), s["y"].data_ptr(),
                c["rows"], c["k"], st)
        return s["y"]
    if kind == "multi":
        n = c["mats"]
        p.qgemv_multi([dt] * n, [w.data_ptr() for w in s["w"]], [w.numel() for w in s["w"]],
                      [c["rows"]] * n, s["x"].data_ptr(), [y.data_ptr() for y in s["y"]], c["k"],
                      st)
        return s["y"]
    if kind == "logits":
        p.qgemv_rmsnorm([dt], [s["w"].data_ptr()], [s["w"].numel()], [c["rows"]],
                        s["x"].data_ptr(), s["norm1"].data_ptr(), EPS, [s["y"].data_ptr()],
                        c["k"], st)
        return s["y"]
    if kind == "batch":
        p.qgemv_batched(dt, s["w"].data_ptr(), s["w"].numel(), s["x"].data_ptr(),
                        s["y"].data_ptr(), c["n"], c["rows"], c["k"], False, st)
        return s["y"]
    if kind == "prefill":
        p.qgemm(dt, s["w"].data_ptr(), s["w"].numel(), s["x"].data_ptr(), p.BF16,
                s["y"].data_ptr(), c["m"], c["rows"], c["k"], st)
        return s["y"]
    if kind == "int8":
        p.quantize_q8_0(s["x"].data_ptr(), p.F32, s["xq"].data_ptr(), s["x"].numel(), st)
        p.qgemm(dt, s["w"].data_ptr(), s["w"].numel(), s["xq"].data_ptr(), p.Q8_0,
                s["y"].data_ptr(), c["m"], c["rows"], c["k"], st)
        return {"x": s["xq"], "y": s["y"]}
    if kind == "dequant":
        f = p.qdequant if c["out"] == "f32" else p.qdequant_bf16
        f(dt, s["w"].data_ptr(), s["w"].numel(), s["y"].data_ptr(), s["y"].numel(), st)
        return s["y"]
    if kind == "mlp":
        h, f, m = c["hidden"], c["ffn"], c["m"]
        p.rmsnorm_rows(s["x"].data_ptr(), s["norm1"].data_ptr(), EPS, s["xn"].data_ptr(), p.BF16,
                       m, h, st)
        for name in ("gate", "up"):
            w = s["w_" + name]
            p.qgemm(dt, w.data_ptr(), w.numel(), s["xn"].data_ptr(), p.BF16,
                    s["y_" + name].data_ptr(), m, f, h, st)
        p.swiglu(s["y_gate"].data_ptr(), s["y_up"].data_ptr(), s["act"].data_ptr(), p.BF16, m * f,
                 st)
        p.qgemm(dt, s["w_down"].data_ptr(), s["w_down"].numel(), s["act"].data_ptr(), p.BF16,
                s["y_down"].data_ptr(), m, h, f, st)
        return {"gate": s["y_gate"], "up": s["y_up"], "down": s["y_down"]}

    shapes = s["shapes"]
    h, f = c["hidden"], c["ffn"]
    if kind == "layer":
        def several(names, x, norm):
            p.qgemv_rmsnorm([code[shapes[n][0]] for n in names],
                            [s["w_" + n].data_ptr() for n in names],
                            [s["w_" + n].numel() for n in names], [shapes[n][1] for n in names],
                            x.data_ptr(), norm.data_ptr(), EPS,
                            [s["y_" + n].data_ptr() for n in names], h, st)

        several(("q", "k", "v"), s["x"], s["norm1"])
        p.qgemv(dt, s["w_o"].data_ptr(), s["w_o"].numel(), s["attn"].data_ptr(),
                s["y_o"].data_ptr(), h, h, st)
        several(("gate", "up"), s["y_o"], s["norm2"])
        p.qgemv_swiglu(code[c["dtype2"]], s["w_down"].data_ptr(), s["w_down"].numel(),
                       s["y_gate"].data_ptr(), s["y_up"].data_ptr(), s["y_down"].data_ptr(), h, f,
                       False, st)
    else:
        n = c["n"]

        def batched(name, x):
            dtype, rows, k = shapes[name]
            w = s["w_" + name]
            p.qgemv_batched(code[dtype], w.data_ptr(), w.numel(), x.data_ptr(),
                            s["y_" + name].data_ptr(), n, rows, k, False, st)

        p.rmsnorm_rows(s["x"].data_ptr(), s["norm1"].data_ptr(), EPS, s["xn"].data_ptr(), p.F32,
                       n, h, st)
        for name in ("q", "k", "v"):
            batched(name, s["xn"])
        batched("o", s["attn"])
        p.rmsnorm_rows(s["y_o"].data_ptr(), s["norm2"].data_ptr(), EPS, s["xn2"].data_ptr(), p.F32,
                       n, h, st)
        batched("gate", s["xn2"])
        batched("up", s["xn2"])
        p.swiglu(s["y_gate"].data_ptr(), s["y_up"].data_ptr(), s["act"].data_ptr(), p.F32, n * f,
                 st)
        batched("down", s["act"])
    return {name: s["y_" + name] for name in shapes}


# -------------------------------------------------------- what a pass amounts to

def _wbytes(dtype, rows, k):
    bs, ts = BLOCK[dtype]
    return rows * (k // bs) * ts


def work(case):
    c, kind = case, case["kind"]
    n = c.get("n", c.get("m", 1))
    if kind in ("layer", "batchlayer"):
        h, kv, f = c["hidden"], c["kv"], c["ffn"]
        shapes = [(c["dtype"], h, h), (c["dtype"], kv, h), (c["dtype2"], kv, h),
                  (c["dtype"], h, h), (c["dtype"], 2 * f, h), (c["dtype2"], h, f)]
        values = 2 * n * h + 2 * h + n * sum(rows for _, rows, _ in shapes)
    elif kind == "mlp":
        h, f = c["hidden"], c["ffn"]
        shapes = [(c["dtype"], 2 * f, h), (c["dtype"], h, f)]
        values = n * h + h + n * (2 * f + h)
    elif kind == "multi":
        shapes = [(c["dtype"], c["rows"], c["k"])] * c["mats"]
        values = c["k"] + c["mats"] * c["rows"]
    elif kind == "dequant":
        out = 4 if c["out"] == "f32" else 2
        return {"bytes": _wbytes(c["dtype"], c["rows"], c["k"]) + out * c["rows"] * c["k"],
                "flops": 0}
    else:
        shapes = [(c["dtype"], c["rows"], c["k"])]
        values = n * c["k"] + n * c["rows"] + (c["k"] if kind == "logits" else 0)
        if kind == "prefill":
            values -= n * c["k"] // 2  # bf16 activations
    size = 4 * values + (n * c["k"] // 32 * 34 if kind == "int8" else 0)
    return {"bytes": size + sum(_wbytes(*shape) for shape in shapes),
            "flops": 2 * n * sum(rows * k for _, rows, k in shapes)}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    # about four times the error against exact() seen on each kind
    if kind in ("decode", "multi", "logits"):
        return {"rel": 1.5e-6, "max": 2e-5}  # fp32 products and sums
    if kind == "layer":
        return {"rel": 3e-6, "max": 4e-5}  # three such products in a chain
    if kind in ("batch", "batchlayer"):
        if case["n"] > 64 and case["dtype"] != Q6_K:
            return {"rel": 8e-3, "max": 6e-2}  # activations and weights in bf16
        if kind == "batch":
            return {"rel": 3e-3, "max": 2e-2}  # activations and weights in fp16
        return {"rel": 6e-3, "max": 4e-2}  # three such products in a chain
    if kind == "int8":
        return {"rel": 1.5e-6, "max": 2e-5}  # exact integer dots, fp32 sums
    if kind == "prefill":
        return {"rel": 7e-3, "max": 5e-2}  # bf16 weights, exact bf16 activations
    return {"rel": 1.6e-2, "max": 1e-1}  # mlp: bf16 activations rounded twice


def _rms64(x, w):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def exact(case, seed):
    s, c, kind = prepare(case, seed), case, case["kind"]

    def times(x, dtype, raw, rows, k):
        out = torch.empty(x.shape[0], rows, dtype=torch.float64, device=x.device)
        step = max(1, (1 << 26) // k)
        row = k // BLOCK[dtype][0] * BLOCK[dtype][1]
        for r in range(0, rows, step):
            e = min(rows, r + step)
            out[:, r:e] = x.double() @ _dequantize(dtype, raw[r * row:e * row], e - r, k).t()
        return out

    if kind == "dequant":
        w = _dequantize(c["dtype"], s["w"], c["rows"], c["k"])
        return w if c["out"] == "f32" else None
    if kind == "mlp":
        xn = _rms64(s["x"], s["norm1"])
        gate, up = (times(xn, c["dtype"], s["w_" + n], c["ffn"], c["hidden"]) for n in ("gate", "up"))
        down = times(gate / (1 + (-gate).exp()) * up, c["dtype"], s["w_down"], c["hidden"], c["ffn"])
        return {"gate": gate, "up": up, "down": down}
    if kind in ("layer", "batchlayer"):
        y = {}

        def mul(name, x):
            dtype, rows, k = s["shapes"][name]
            y[name] = times(x, dtype, s["w_" + name], rows, k)

        xn = _rms64(s["x"], s["norm1"])
        for name in ("q", "k", "v"):
            mul(name, xn)
        mul("o", s["attn"])
        xn = _rms64(y["o"], s["norm2"])
        mul("gate", xn)
        mul("up", xn)
        mul("down", y["gate"] / (1 + (-y["gate"]).exp()) * y["up"])
        return y
    x = s["x"]
    if kind == "multi":
        return [times(x, c["dtype"], w, c["rows"], c["k"])[0] for w in s["w"]]
    if kind == "logits":
        x = _rms64(x, s["norm1"])
    elif kind == "int8":
        v = x.reshape(-1, 32)
        d = v.abs().amax(-1, keepdim=True) / 127
        t = v * (1 / d)  # the quantizer's codes: round(v * (1 / d)), halves away from 0
        q = (t.abs() + 0.5).floor().clamp(max=127) * t.sign()
        x = (q.double() * d.half().double()).reshape(x.shape)
    y = times(x, c["dtype"], s["w"], c["rows"], c["k"])
    return {"x": None, "y": y} if kind == "int8" else y
