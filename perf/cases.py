"""Performance cases of the quantized-weight path, through its public entry points.

Six kinds of work, each an ordinary call of a program that uses this library:

  product   one linear layer on device buffers (Weight.matmul_dev, bit-exact)
  group     a model's linear layers as one grouped launch at batch 1..8
            (Group, or TolGroup for the tolerance-mode products)
  layer     the seven projections of one transformer layer over a prompt's
            rows (Weight.matmul_dev, bit-exact) or, with "mfma", the bf16
            matrix-core products of one or more layers (GemmGroup)
  quantize  packing an fp32 matrix into blocks (llmi_hip_quantize_dev)
  sample    one token drawn from device logits (sample_dev)
  session   a model's prompt and the decode steps after it (forward_cached),
            returning every step's logits

Shapes are those of the SmolLM2-135M and Qwen2.5-0.5B configurations in
llm-inference-cpp_amd/workloads.py and synth.py; drawn cases spread over the
same ranges with odd sizes among them.  Weights are N(0, 0.02) and activations
N(0, 1), made on the GPU from the seed alone.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-inference-cpp_amd"))

import llmi_hip as H  # noqa: E402
import synth  # noqa: E402
import workloads as W  # noqa: E402

TYPES = {"q8_0": H.Q8_0, "q4_0": H.Q4_0, "f32": H.F32}
CONFIGS = {"smollm2": synth.SMOLLM2_135M, "qwen25": synth.QWEN25_05B}
LAYERS = {"smollm2": W.SMOL_LAYER, "qwen25": W.QWEN_LAYER}
HEADS = {"smollm2": W.SMOL_HEAD, "qwen25": W.QWEN_HEAD}


def listed():
    return [
        # The smallest call: one SmolLM2 MLP matvec of a decode step; latency.
        {"name": "product_smol_up_q8_b1", "kind": "product", "type": "q8_0", "out": 1536, "in": 576, "rows": 1, "bias": False},
        # The largest single matrix of a decode step: Qwen2.5's lm_head; HBM.
        {"name": "product_qwen_head_q4_b1", "kind": "product", "type": "q4_0", "out": 151936, "in": 896, "rows": 1, "bias": False},
        # A few sequences decoded together through a matrix of ragged shape
        # (rows past the last tile, a partial last block), with a bias.
        {"name": "product_ragged_q4_b5", "kind": "product", "type": "q4_0", "out": 2749, "in": 1003, "rows": 5, "bias": True},
        # One token through every linear layer of SmolLM2 in Q4_0.
        {"name": "group_smol_q4_b1", "kind": "group", "model": "smollm2", "type": "q4_0", "layers": 30, "head": True, "rows": 1, "mode": "exact"},
        # Eight sequences' tokens through the same layers.
        {"name": "group_smol_q4_b8", "kind": "group", "model": "smollm2", "type": "q4_0", "layers": 30, "head": True, "rows": 8, "mode": "exact"},
        # A prompt of 512 tokens through one Qwen2.5 layer's projections, exact.
        {"name": "layer_qwen_q8_m512", "kind": "layer", "model": "qwen25", "type": "q8_0", "layers": 1, "rows": 512, "mode": "exact"},
        # The same prompt on the bf16 matrix-core path, all 24 layers.
        {"name": "mfma_qwen_q8_m512", "kind": "layer", "model": "qwen25", "type": "q8_0", "layers": 24, "rows": 512, "mode": "mfma"},
        # fp32 weights (--quant f32): an MLP projection over a 128-token prompt.
        {"name": "product_qwen_up_f32_m128", "kind": "product", "type": "f32", "out": 4864, "in": 896, "rows": 128, "bias": False},
        # Loading a model: packing the Qwen2.5 embedding / lm_head matrix.
        {"name": "quantize_qwen_head_q4", "kind": "quantize", "type": "q4_0", "out": 151936, "in": 896},
        # Serving: one token sampled from Qwen2.5's logits, the usual filters.
        {"name": "sample_qwen_k40_p09", "kind": "sample", "n": 151936, "temperature": 0.8, "top_k": 40, "top_p": 0.9},
        # A chat turn on SmolLM2-135M in Q8_0: 128 prompt tokens, 16 decoded, exact.
        {"name": "session_smol_q8_exact", "kind": "session", "model": "smollm2", "type": "q8_0", "layers": 30, "prompt": 128, "steps": 16, "mode": "exact"},
        # A long prompt on Qwen2.5-0.5B in Q4_0: 512 tokens, 16 tolerance-mode steps.
        {"name": "session_qwen_q4_tol", "kind": "session", "model": "qwen25", "type": "q4_0", "layers": 24, "prompt": 512, "steps": 16, "mode": "tolerance"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed cases' ranges."""
    kind = rng.choice(["product", "product", "group", "layer", "layer", "quantize", "sample", "session"])
    model = rng.choice(["smollm2", "qwen25"])
    qtype = rng.choice(["q8_0", "q4_0"])
    if kind == "product":
        qtype = rng.choice(["q8_0", "q4_0", "f32"])
        rows = rng.choice([rng.randint(1, 8), _log(rng, 9, 512)])
        out = _log(rng, 64, 151936 if rows <= 64 else 8192)
        return {"kind": kind, "type": qtype, "out": out, "in": _log(rng, 64, 4864), "rows": rows, "bias": rng.random() < 0.5}
    if kind == "group":
        mode = rng.choice(["exact", "exact", "tolerance"])
        return {"kind": kind, "model": model, "type": "q4_0" if mode == "tolerance" else qtype, "layers": rng.randint(2, 24),
                "head": rng.random() < 0.5, "rows": rng.randint(1, 8), "mode": mode}
    if kind == "layer":
        mode = rng.choice(["exact", "mfma"])
        return {"kind": kind, "model": model, "type": qtype, "layers": 1 if mode == "exact" else _log(rng, 1, 24),
                "rows": _log(rng, 17, 512), "mode": mode}
    if kind == "quantize":
        return {"kind": kind, "type": qtype, "out": _log(rng, 128, 151936), "in": _log(rng, 96, 896)}
    if kind == "sample":
        return {"kind": kind, "n": _log(rng, 32000, 151936), "temperature": round(rng.uniform(0.5, 1.2), 2),
                "top_k": rng.choice([0, 20, 40, 64]), "top_p": rng.choice([1.0, 0.9, 0.95])}
    return {"kind": kind, "model": model, "type": qtype, "layers": rng.randint(4, 24), "prompt": _log(rng, 16, 512),
            "steps": rng.randint(4, 16), "mode": rng.choice(["exact", "tolerance"])}


# ------------------------------------------------------------------ inputs


def _normal(gen, shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=gen)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _pack(w, qtype):
    torch.cuda.synchronize()
    return H.Weight.quantize_dev(w.data_ptr(), w.shape[0], w.shape[1], TYPES[qtype])


def _products(case):
    """(name, out, in, activation) of every product of a group or layer case."""
    items = []
    for i in range(case["layers"]):
        for name, out, n_in in LAYERS[case["model"]]:
            items.append((name, out, n_in, "%d.%s" % (i, W.LAYER_INPUT[name])))
    if case.get("head"):
        items.append((*HEADS[case["model"]], "head"))
    return items


def _product_inputs(case, gen):
    """Per product (fp32 weight, activation); products of one layer that read
    the same vector share it."""
    xs = {}
    for _, out, n_in, act in _products(case):
        if act not in xs:
            xs[act] = _normal(gen, (case["rows"], n_in))
        yield _normal(gen, (out, n_in), 0.02), xs[act]


def _model_tensors(case, gen):
    cfg = dict(CONFIGS[case["model"]], num_layers=case["layers"])
    tensors = [_normal(gen, shape, 0.02) if kind != "norm" else _normal(gen, shape, 0.02, 1.0)
               for _, shape, kind in synth.tensor_specs(cfg)]
    n = case["prompt"] + case["steps"]
    ids = torch.randint(0, cfg["vocab_size"], (n,), dtype=torch.int32, device="cuda", generator=gen).cpu().numpy()
    return cfg, tensors, ids


def prepare(case, seed):
    H.init(0)
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "product":
        w = _pack(_normal(gen, (case["out"], case["in"]), 0.02), case["type"])
        x = _normal(gen, (case["rows"], case["in"]))
        bias = _normal(gen, (case["out"],), 0.02) if case["bias"] else None
        y = torch.empty(case["rows"], case["out"], dtype=torch.float32, device="cuda")
        return {"kind": kind, "w": w, "x": x, "bias": bias, "y": y}
    if kind in ("group", "layer"):
        sizes = [case["rows"] * out for _, out, _, _ in _products(case)]
        y = torch.empty(sum(sizes), dtype=torch.float32, device="cuda")  # the outputs, one after another
        ws, xs = [], []
        for w, x in _product_inputs(case, gen):
            ws.append(_pack(w, case["type"]))
            xs.append(x)
        ys = torch.split(y, sizes)
        if kind == "layer" and case["mode"] == "exact":
            return {"kind": kind, "w": ws, "x": xs, "ys": ys, "y": y}
        cls = H.GemmGroup if kind == "layer" else H.TolGroup if case["mode"] == "tolerance" else H.Group
        group = cls([(w, x.data_ptr(), v.data_ptr(), case["rows"]) for w, x, v in zip(ws, xs, ys)])
        return {"kind": "launch", "group": group, "w": ws, "x": xs, "ys": ys, "y": y}
    if kind == "quantize":
        w = _normal(gen, (case["out"], case["in"]), 0.02)
        qt = TYPES[case["type"]]
        data = torch.zeros(case["out"], H.row_bytes(case["in"], qt), dtype=torch.uint8, device="cuda")
        scales = torch.zeros(case["out"], H.nblocks(case["in"]), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        return {"kind": kind, "type": qt, "w": w, "data": data, "scales": scales}
    if kind == "sample":
        logits = _normal(gen, (case["n"],), 2.0)
        buf = H.DeviceBuffer(case["n"] * 4)
        buf.upload(logits.cpu().numpy())
        target = torch.rand((), device="cuda", dtype=torch.float64, generator=gen).item()
        return {"kind": kind, "logits": buf, "n": case["n"], "target": target,
                "cfg": H.Sampling(case["temperature"], case["top_k"], case["top_p"])}
    cfg, tensors, ids = _model_tensors(case, gen)
    torch.cuda.synchronize()
    model = H.Model(cfg, [t.data_ptr() for t in tensors], TYPES[case["type"]], on_device=True)
    model.set_decode_mode(H.DECODE_TOLERANCE if case["mode"] == "tolerance" else H.DECODE_EXACT)
    return {"kind": kind, "model": model, "cache": model.new_cache(len(ids)), "ids": ids, "prompt": case["prompt"]}


def run(state):
    kind = state["kind"]
    if kind == "product":
        w, bias = state["w"], state["bias"]
        w.matmul_dev(state["x"].data_ptr(), state["x"].shape[0], None if bias is None else bias.data_ptr(), state["y"].data_ptr())
        return state["y"]
    if kind == "launch":
        state["group"].launch()
        return state["y"]
    if kind == "layer":
        for w, x, y in zip(state["w"], state["x"], state["ys"]):
            w.matmul_dev(x.data_ptr(), x.shape[0], None, y.data_ptr())
        return state["y"]
    if kind == "quantize":
        w = state["w"]
        H.check(H.load().llmi_hip_quantize_dev(w.data_ptr(), w.shape[0], w.shape[1], state["type"], state["data"].data_ptr(),
                                               state["scales"].data_ptr(), None))
        return {"data": state["data"], "scales": state["scales"]}
    if kind == "sample":
        return H.sample_dev(state["logits"], state["n"], state["cfg"], state["target"])
    model, cache, ids, n = state["model"], state["cache"], state["ids"], state["prompt"]
    cache.reset()
    logits = [model.forward_cached(cache, ids[:n])]
    for t in range(n, len(ids)):
        logits.append(model.forward_cached(cache, ids[t:t + 1]))
    return logits


# ------------------------------------------------------- what a pass needs


def _weight_bytes(out, n_in, qtype):
    if qtype == "f32":
        return 4 * out * n_in
    return out * H.row_bytes(n_in, TYPES[qtype]) + 4 * out * H.nblocks(n_in)


def work(case):
    kind = case["kind"]
    if kind == "product":
        out, n_in, rows = case["out"], case["in"], case["rows"]
        return {"bytes": _weight_bytes(out, n_in, case["type"]) + 4 * rows * (n_in + out) + (4 * out if case["bias"] else 0),
                "flops": 2 * rows * out * n_in}
    if kind in ("group", "layer"):
        rows, products = case["rows"], _products(case)
        acts = {act: n_in for _, _, n_in, act in products}
        return {"bytes": sum(_weight_bytes(o, i, case["type"]) + 4 * rows * o for _, o, i, _ in products) + 4 * rows * sum(acts.values()),
                "flops": sum(2 * rows * o * i for _, o, i, _ in products)}
    if kind == "quantize":
        return {"bytes": 4 * case["out"] * case["in"] + _weight_bytes(case["out"], case["in"], case["type"]), "flops": 0}
    if kind == "sample":
        return {"bytes": 4 * case["n"], "flops": 0}
    cfg = CONFIGS[case["model"]]
    hidden, kv = cfg["hidden_size"], cfg["num_kv_heads"] * cfg["hidden_size"] // cfg["num_heads"]
    head = HEADS[case["model"]]
    per_layer = sum(_weight_bytes(o, i, case["type"]) for _, o, i in LAYERS[case["model"]])
    elements = sum(o * i for _, o, i in LAYERS[case["model"]])
    n, steps = case["prompt"], case["steps"]
    read = (1 + steps) * (case["layers"] * per_layer + _weight_bytes(head[1], head[2], case["type"]) + 4 * head[1])
    read += sum(2 * 4 * case["layers"] * kv * (n + t) for t in range(steps + 1))
    flops = 2 * (n + steps) * case["layers"] * elements + 2 * (1 + steps) * head[1] * head[2]
    flops += 4 * case["layers"] * hidden * (n * (n + 1) // 2 + sum(n + t + 1 for t in range(steps)))
    return {"bytes": read, "flops": flops}


def tolerance(case):
    """About four times what the paths measure against `exact` (products
    1.0e-7..2.4e-7, tolerance-mode groups 2.5e-6, bf16 layers 2.3e-3, sessions
    4.4e-7 exact and 1.2e-6 in tolerance mode)."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "quantize":  # the scales are one fp32 division
        return {"rel": 2e-7}
    if kind == "session":
        return {"rel": 6e-6}
    if kind == "layer" and case["mode"] == "mfma":
        return {"rel": 1e-2, "max": 8e-2}
    if kind == "group" and case["mode"] == "tolerance":
        return {"rel": 1e-5}
    return {"rel": 1e-6}


# ------------------------------------------------------------- in 64 bits


def _blocks(w, qtype):
    """(codes, scales) of the block quantizer: 32 weights a block, the scale
    amax / 127 (Q8_0) or extreme / -8 (Q4_0) in fp32, codes rounded half away
    from zero and clamped."""
    out, n_in = w.shape
    v = torch.nn.functional.pad(w, (0, -n_in % H.BLOCK)).view(out, -1, H.BLOCK)
    peak = torch.gather(v, 2, v.abs().argmax(2, keepdim=True)).double()
    d = (peak.abs() / 127.0 if qtype == "q8_0" else peak / -8.0).float()
    d = torch.where(d == 0, torch.ones_like(d), d).double()
    lo, hi = (-127, 127) if qtype == "q8_0" else (-8, 7)
    codes = torch.empty(v.shape, dtype=torch.float64, device=w.device)
    torch.div(v.double(), d, out=codes)
    codes = (codes.sign() * (codes.abs() + 0.5).floor()).clamp(lo, hi)
    return codes, d


def _dequantized(w, qtype):
    if qtype == "f32":
        return w.double()
    codes, d = _blocks(w, qtype)
    return (codes * d).view(w.shape[0], -1)[:, :w.shape[1]]


def _matmul64(x, w, qtype):
    return x.double() @ _dequantized(w, qtype).t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    gen = _generator(seed)
    if kind == "product":
        w, x = _normal(gen, (case["out"], case["in"]), 0.02), _normal(gen, (case["rows"], case["in"]))
        # In pieces of rows: a large matrix in 64 bits is several times its size.
        y = torch.cat([_matmul64(x, p, case["type"]) for p in torch.split(w, 16384)], 1)
        if case["bias"]:
            y = _with_bias(y, x, case, seed)
        return y
    if kind in ("group", "layer"):
        return torch.cat([torch.cat([_matmul64(x, p, case["type"]) for p in torch.split(w, 16384)], 1).reshape(-1)
                          for w, x in _product_inputs(case, gen)])
    if kind == "quantize":
        w = _normal(gen, (case["out"], case["in"]), 0.02)
        scales = torch.cat([_blocks(p, case["type"])[1].flatten(1) for p in torch.split(w, 16384)])
        return {"data": None, "scales": scales}
    return _session64(case, gen)


def _with_bias(y, x, case, seed):
    gen = _generator(seed)
    _normal(gen, (case["out"], case["in"]), 0.02)
    _normal(gen, tuple(x.shape))
    return y + _normal(gen, (case["out"],), 0.02).double()


def _session64(case, gen):
    """The decoder over the whole token sequence in 64 bits, and the logits
    that the session returns: after the prompt and after each step."""
    cfg, tensors, ids = _model_tensors(case, gen)
    it = iter(tensors)
    quant = lambda w: torch.cat([_dequantized(p, case["type"]) for p in torch.split(w, 16384)])  # noqa: E731
    heads, kv_heads = cfg["num_heads"], cfg["num_kv_heads"]
    hd = cfg["hidden_size"] // heads
    n = len(ids)
    norm = lambda v, w: w.double() * v / torch.sqrt((v * v).mean(1, keepdim=True) + cfg["rms_norm_eps"])  # noqa: E731
    # The model's angles are fp32 products of the position and an fp32
    # frequency; the sines and cosines of those angles in 64 bits.
    freq = (cfg["rope_theta"] ** (-torch.arange(0, hd, 2, dtype=torch.float64) / hd)).float()
    angle = (torch.arange(n, dtype=torch.float32)[:, None] * freq).cuda().double()
    cos, sin = angle.cos(), angle.sin()

    def rope(v):  # [heads, n, hd]
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], 2)

    def split(v, h):
        return v.view(n, h, hd).transpose(0, 1).contiguous()

    embed = next(it)
    x = torch.cat([_dequantized(embed[i:i + 1], case["type"]) for i in ids.tolist()])
    mask = torch.full((n, n), -math.inf, dtype=torch.float64, device="cuda").triu(1)
    for _ in range(cfg["num_layers"]):
        ln, wq, wk, wv = (next(it) for _ in range(4))
        h = norm(x, ln)
        q, k, v = (h @ quant(w).t() for w in (wq, wk, wv))
        if cfg["qkv_bias"]:
            q, k, v = (t + next(it).double() for t in (q, k, v))
        q, k, v = rope(split(q, heads)), rope(split(k, kv_heads)), split(v, kv_heads)
        k, v = (t.repeat_interleave(heads // kv_heads, 0) for t in (k, v))
        p = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(hd) + mask, 2)
        x = x + (p @ v).transpose(0, 1).reshape(n, -1) @ quant(next(it)).t()
        ln, gate, up, down = (next(it) for _ in range(4))
        h = norm(x, ln)
        x = x + (torch.nn.functional.silu(h @ quant(gate).t()) * (h @ quant(up).t())) @ quant(down).t()
    last = norm(x, next(it))[case["prompt"] - 1:]
    logits = torch.cat([last @ _dequantized(p, case["type"]).t() for p in torch.split(embed, 16384)], 1)
    return [row for row in logits]
