"""What a program does with this framework, as cases whose time and results can be measured.

Six kinds of work, each through the entry points of the package:

  linear     one block-quantized (or fp32) Linear on a batch of rows: linear()
  layers     the Linears of a few decoder layers as one HIP graph, as a serving loop replays them:
             linear() with the fused q|k|v bias and the fused SwiGLU, captured once
  aos        a Linear on raw GGUF blocks in device memory, for programs that keep the file's format: linear_aos()
  decode     one token through a whole model, as one HIP graph of step and greedy choice: DecodeModel.greedy_graph()
  prefill    a prompt through a whole model: DecodeModel.prefill()
  attention  decode attention over a KV cache: mlq_attention_decode

Weights are random GGUF blocks with the scales that trained weights have (|N(0, 0.02)| over the code range) and codes and mins
centred on zero as a quantizer leaves them, activations are N(0, 1). The shapes are the 7B- and 8B-class ones that the benchmark uses (hidden 3584 with FFN 18944, hidden 4096 with FFN
11008 or 14336).
"""
import ctypes
import importlib
import math

import numpy as np
import torch

mlq = importlib.import_module("mini-llama_amd")
decode = importlib.import_module("mini-llama_amd.decode")

DEVICE = "cuda"
BLOCK = {"q8_0": 34, "q4_0": 18, "q4_1": 20}  # bytes of a GGUF block of 32 weights


def listed():
    return [
        # The smallest call: one decode token's k projection with its bias. Launch and host latency are all of it.
        {"name": "linear_1x512x3584_q4_0", "kind": "linear", "type": "q4_0", "m": 1, "n": 512, "k": 3584, "bias": True, "swiglu": False},
        # Every Linear of four 7B layers for one token: what single-user decoding spends most of its time on.
        {"name": "layers_1_7b_q4_0", "kind": "layers", "type": "q4_0", "m": 1, "dim": 3584, "ffn": 18944, "kv": 512, "layers": 4},
        # A few users (or a few speculated tokens) at once on an 8B model with the widest of the 4-bit formats.
        {"name": "layers_4_8b_q4_1", "kind": "layers", "type": "q4_1", "m": 4, "dim": 4096, "ffn": 14336, "kv": 1024, "layers": 4},
        # Batched decoding: 16 users on an 8B model in 8 bits.
        {"name": "layers_16_8b_q8_0", "kind": "layers", "type": "q8_0", "m": 16, "dim": 4096, "ffn": 14336, "kv": 1024, "layers": 4},
        # Batched decoding: 64 users on a 7B model in 4 bits.
        {"name": "layers_64_7b_q4_0", "kind": "layers", "type": "q4_0", "m": 64, "dim": 3584, "ffn": 18944, "kv": 512, "layers": 4},
        # An ordinary prompt through one FFN projection in 8 bits.
        {"name": "linear_512x11008x4096_q8_0", "kind": "linear", "type": "q8_0", "m": 512, "n": 11008, "k": 4096, "bias": False, "swiglu": False},
        # A long prompt, its length no round number, through the fused gate|up projection of an 8B model.
        {"name": "linear_2000x28672x4096_q4_1", "kind": "linear", "type": "q4_1", "m": 2000, "n": 28672, "k": 4096, "bias": False, "swiglu": True},
        # A prompt through a projection of a model whose weights were not quantized.
        {"name": "linear_200x4096x4096_f32", "kind": "linear", "type": "f32", "m": 200, "n": 4096, "k": 4096, "bias": False, "swiglu": False},
        # One token's FFN projection on the GGUF blocks as they lie in the file.
        {"name": "aos_1x18944x3584_q4_0", "kind": "aos", "type": "q4_0", "m": 1, "n": 18944, "k": 3584},
        # One token through a 7B-shaped model (eight of its layers, the whole vocabulary) in the middle of a conversation.
        {"name": "decode_7b_q4_0", "kind": "decode", "type": "q4_0", "dim": 3584, "ffn": 18944, "heads": 28, "kv_heads": 4, "hd": 128,
         "layers": 8, "vocab": 152064, "max_seq": 4096, "pos": 1100},
        # A long prompt through two 7B layers: large GEMMs, causal attention over 2000 positions, cache writes.
        {"name": "prefill_2000_7b_q4_0", "kind": "prefill", "type": "q4_0", "dim": 3584, "ffn": 18944, "heads": 28, "kv_heads": 4, "hd": 128,
         "layers": 2, "vocab": 32000, "max_seq": 2048, "pos": 0, "tokens": 2000},
        # One token's attention at the far end of a full 32K context.
        {"name": "attention_30000_7b", "kind": "attention", "heads": 28, "kv_heads": 4, "hd": 128, "max_seq": 32768, "pos": 29999},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layers", "layers", "aos", "decode", "prefill", "attention"])
    quant = rng.choice(["q4_0", "q8_0", "q4_1"])
    if kind == "linear":
        f32 = rng.random() < 0.2
        while True:
            m, n, k = _log(rng, 1, 256 if f32 else 2000), _log(rng, 256, 29000), _log(rng, 256, 15000)
            if rng.random() < 0.7:  # most models' widths are multiples of 32, a few are not
                n, k = n // 32 * 32, k // 32 * 32
            if m * n * k <= (4 * 10**9 if f32 else 2 * 10**11):
                break
        swiglu = n % 16 == 0 and rng.random() < 0.25
        return {"kind": kind, "type": "f32" if f32 else quant, "m": m, "n": n, "k": k, "bias": rng.random() < 0.3, "swiglu": swiglu}
    if kind == "layers":
        dim = rng.choice([896, 1536, 2048, 2560, 3072, 3584, 4096])
        return {"kind": kind, "type": quant, "m": _log(rng, 1, 64), "dim": dim, "ffn": int(dim * rng.uniform(2.6, 5.3)) // 8 * 8,
                "kv": rng.choice([128, 256, 512, 1024]), "layers": rng.randint(2, 4)}
    if kind == "aos":
        return {"kind": kind, "type": quant, "m": rng.choice([1, 1, 1, 2, 3, 4, 8, 24]), "n": _log(rng, 512, 19000), "k": _log(rng, 512, 14500) // 32 * 32}
    hd = rng.choice([64, 128, 128, 128, 256])
    kv_heads = rng.choice([2, 4, 8])
    if kind == "attention":
        max_seq = rng.choice([512, 2048, 8192, 32768])
        return {"kind": kind, "heads": kv_heads * rng.choice([1, 4, 6, 7, 8]), "kv_heads": kv_heads, "hd": hd, "max_seq": max_seq,
                "pos": min(max_seq - 1, _log(rng, 16, max_seq))}
    heads = kv_heads * rng.choice([1, 2, 4, 7])
    dim = heads * hd
    while dim > 4096 or dim < 512:
        heads = heads // 2 // kv_heads * kv_heads if dim > 4096 and heads > kv_heads else heads
        hd = 64 if dim > 4096 else 256
        heads = kv_heads * 4 if dim < 512 else heads
        dim = heads * hd
    shape = {"kind": kind, "type": quant, "dim": dim, "ffn": int(dim * rng.uniform(2.6, 5.3)) // 8 * 8, "heads": heads, "kv_heads": kv_heads,
             "hd": hd, "layers": rng.randint(1, 2), "vocab": _log(rng, 4000, 100000)}
    if kind == "decode":
        max_seq = rng.choice([1024, 4096])
        return dict(shape, layers=rng.randint(2, 6), max_seq=max_seq, pos=min(max_seq - 1, _log(rng, 1, max_seq)))
    tokens = _log(rng, 5, 1900)
    start = rng.choice([0, 0, rng.randint(1, 100)])
    return dict(shape, max_seq=2048, pos=start, tokens=tokens)


# ---- inputs -------------------------------------------------------------------------------------------------------------------


def _weight(g, kind, n, k):
    """A weight as the file or the trainer has it: fp32 [n, k], or GGUF blocks as bytes [n, blocks, block bytes]."""
    if kind == "f32":
        return torch.randn((n, k), generator=g, device=DEVICE) * 0.02
    nb = (k + 31) // 32
    raw = torch.empty((n, nb, BLOCK[kind]), dtype=torch.uint8, device=DEVICE)
    top = {"q8_0": 127.0, "q4_0": 8.0, "q4_1": 15.0}[kind]
    d = (torch.randn((n, nb, 1), generator=g, device=DEVICE) * 0.02).abs() / top
    raw[:, :, :2] = d.to(torch.float16).view(torch.uint8)
    codes = 2
    if kind == "q4_1":
        low = -7.5 * d * (1.0 + 0.1 * torch.randn((n, nb, 1), generator=g, device=DEVICE))
        raw[:, :, 2:4] = low.to(torch.float16).view(torch.uint8)
        codes = 4
    if kind == "q8_0":
        q = torch.randint(-127, 128, (n, nb, 32), generator=g, device=DEVICE, dtype=torch.int8)
        raw[:, :, codes:] = q.view(torch.uint8)
    else:  # q4_0's quantizer gives 1 .. 15 (-7 .. 7), q4_1's 0 .. 15
        q = torch.randint(1 if kind == "q4_0" else 0, 16, (2, n, nb, 16), generator=g, device=DEVICE, dtype=torch.uint8)
        raw[:, :, codes:] = q[0] | (q[1] << 4)
    return raw


def _upload(kind, raw, n, k):
    if kind == "f32":
        return mlq.TiledWeight("f32", n, k, raw.view(-1).view(torch.uint8), mlq.weight_layout("f32", n, k))
    return mlq.repack_device(kind, raw.view(-1), n, k)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _linear_inputs(case, seed):
    g = _generator(seed)
    raw = _weight(g, case["type"], case["n"], case["k"])
    x = torch.randn((case["m"], case["k"]), generator=g, device=DEVICE)
    bias = torch.randn(case["n"], generator=g, device=DEVICE) if case.get("bias") else None
    return raw, x, bias


def _layer_shapes(case):
    """(rows, columns, bias, swiglu) of a layer's four Linears: q|k|v, o, gate|up, down."""
    dim, ffn, kv = case["dim"], case["ffn"], case["kv"]
    return [(dim + 2 * kv, dim, True, False), (dim, dim, False, False), (2 * ffn, dim, False, True), (dim, ffn, False, False)]


def _layers_inputs(case, seed):
    g = _generator(seed)
    for _ in range(case["layers"]):
        for n, k, has_bias, swiglu in _layer_shapes(case):
            raw = _weight(g, case["type"], n, k)
            x = torch.randn((case["m"], k), generator=g, device=DEVICE)
            bias = torch.randn(n, generator=g, device=DEVICE) * 0.1 if has_bias else None
            yield n, k, raw, x, bias, swiglu


def _model_inputs(case, seed):
    """The model as DecodeModel takes it (everything on the device), its cache's contents before the call, and the tokens."""
    g = _generator(seed)
    dim, ffn, hd, kind = case["dim"], case["ffn"], case["hd"], case["type"]
    qd, kvd = case["heads"] * hd, case["kv_heads"] * hd

    def lin(n, k):
        return {"type": kind, "shape": (n, k), "data": _weight(g, kind, n, k)}

    def norm():
        return 1.0 + 0.1 * torch.randn(dim, generator=g, device=DEVICE)

    layers = []
    for _ in range(case["layers"]):
        layer = {"attention_norm": norm(), "ffn_norm": norm(), "wq": lin(qd, dim), "wk": lin(kvd, dim), "wv": lin(kvd, dim),
                 "wo": lin(dim, qd), "w_gate": lin(ffn, dim), "w_up": lin(ffn, dim), "w_down": lin(dim, ffn)}
        for name, n in (("bq", qd), ("bk", kvd), ("bv", kvd)):
            layer[name] = 0.1 * torch.randn(n, generator=g, device=DEVICE)
        layers.append(layer)
    config = {"vocab_size": case["vocab"], "dim": dim, "hidden_dim": ffn, "n_layers": case["layers"], "n_heads": case["heads"],
              "n_kv_heads": case["kv_heads"], "head_dim": hd, "max_seq_len": case["max_seq"], "rope_theta": 1e6, "rms_norm_eps": 1e-6,
              "rope_type": mlq.ROPE_NEOX}
    model = {"config": config, "token_embedding": torch.randn((case["vocab"], dim), generator=g, device=DEVICE), "final_norm": norm(),
             "lm_head": lin(case["vocab"], dim), "layers": layers}
    past = (case["layers"], case["pos"], case["kv_heads"], hd)
    keys = torch.randn(past, generator=g, device=DEVICE)
    values = torch.randn(past, generator=g, device=DEVICE)
    tokens = np.random.default_rng(seed).integers(0, case["vocab"], case.get("tokens", 1), dtype=np.int32)
    return model, keys, values, tokens


def _attention_inputs(case, seed):
    g = _generator(seed)
    shape = (1, case["max_seq"], case["kv_heads"], case["hd"])
    keys = torch.randn(shape, generator=g, device=DEVICE)
    values = torch.randn(shape, generator=g, device=DEVICE)
    return torch.randn((case["heads"], case["hd"]), generator=g, device=DEVICE), keys, values


# ---- what a program holds before the call -------------------------------------------------------------------------------------


def prepare(case, seed):
    return {"linear": _prepare_linear, "layers": _prepare_layers, "aos": _prepare_aos, "decode": _prepare_model, "prefill": _prepare_model,
            "attention": _prepare_attention}[case["kind"]](case, seed)


def _prepare_linear(case, seed):
    raw, x, bias = _linear_inputs(case, seed)
    return {"case": case, "w": _upload(case["type"], raw, case["n"], case["k"]), "x": x, "bias": bias,
            "act": mlq.EPI_SWIGLU if case["swiglu"] else mlq.EPI_NONE}


def _prepare_layers(case, seed):
    m, calls, need = case["m"], [], 0
    for n, k, raw, x, bias, swiglu in _layers_inputs(case, seed):
        w = _upload(case["type"], raw, n, k)
        y = torch.empty((m, n // 2 if swiglu else n), dtype=torch.float32, device=DEVICE)
        need = max(need, mlq.workspace_bytes(w, m))
        calls.append((w, x, y, bias, mlq.EPI_SWIGLU if swiglu else mlq.EPI_NONE))
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device=DEVICE)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for w, x, y, bias, act in calls:
            mlq.linear(w, x, y, stream=stream, workspace=ws, bias=bias, act=act)
    torch.cuda.current_stream().wait_stream(stream)
    return {"case": case, "graph": graph, "calls": calls, "ws": ws, "out": [c[2] for c in calls]}


def _prepare_aos(case, seed):
    raw, x, _ = _linear_inputs(case, seed)
    return {"case": case, "raw": raw.view(-1), "x": x}


def _prepare_model(case, seed):
    model, keys, values, tokens = _model_inputs(case, seed)
    dm = decode.DecodeModel(model, device=DEVICE)
    dm.keys[:, : case["pos"]] = keys
    dm.values[:, : case["pos"]] = values
    state = {"case": case, "model": dm, "tokens": tokens}
    if case["kind"] == "decode":
        state["token"] = torch.from_numpy(tokens).to(DEVICE)
        state["at"] = torch.full((1,), case["pos"], dtype=torch.int32, device=DEVICE)
        state["graph"] = dm.greedy_graph()
    return state


def _prepare_attention(case, seed):
    q, keys, values = _attention_inputs(case, seed)
    cache = mlq.MlqKvCache(keys.data_ptr(), values.data_ptr(), 1, case["max_seq"], case["kv_heads"], case["hd"])
    need = ctypes.c_size_t()
    mlq._check(mlq.lib().mlq_attention_workspace(ctypes.byref(cache), case["heads"], ctypes.byref(need)), "mlq_attention_workspace")
    return {"case": case, "q": q, "keys": keys, "values": values, "cache": cache, "out": torch.empty_like(q),
            "ws": torch.empty(max(need.value, 256), dtype=torch.uint8, device=DEVICE)}


# ---- one pass -----------------------------------------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return mlq.linear(state["w"], state["x"], bias=state["bias"], act=state["act"])
    if kind == "layers":
        state["graph"].replay()
        return state["out"]
    if kind == "aos":
        return mlq.linear_aos(case["type"], state["raw"], case["n"], case["k"], state["x"])
    if kind == "attention":
        mlq._check(mlq.lib().mlq_attention_decode(
            ctypes.byref(state["cache"]), 0, case["pos"], state["q"].data_ptr(), case["heads"], state["out"].data_ptr(),
            state["ws"].data_ptr(), state["ws"].numel(), torch.cuda.current_stream().cuda_stream), "mlq_attention_decode")
        return state["out"]
    dm = state["model"]
    if kind == "prefill":
        logits = dm.prefill(state["tokens"], case["pos"])
        return {"logits": logits, "keys": dm.keys, "values": dm.values}
    dm.token_dev.copy_(state["token"])
    dm.pos_dev.copy_(state["at"])
    state["graph"].replay()
    return {"logits": dm.logits, "keys": dm.keys, "values": dm.values, "token": dm.token_dev}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------


def _weight_bytes(kind, n, k):
    return 4 * n * k if kind == "f32" else n * ((k + 31) // 32) * BLOCK[kind]


def _linear_work(kind, m, n, k, bias=False, swiglu=False):
    return {"bytes": _weight_bytes(kind, n, k) + 4 * m * k + 4 * m * (n // 2 if swiglu else n) + (4 * n if bias else 0), "flops": 2 * m * n * k}


def work(case):
    kind = case["kind"]
    if kind in ("linear", "aos"):
        return _linear_work(case["type"], case["m"], case["n"], case["k"], case.get("bias"), case.get("swiglu"))
    if kind == "layers":
        each = [_linear_work(case["type"], case["m"], *shape) for shape in _layer_shapes(case)]
        return {key: case["layers"] * sum(e[key] for e in each) for key in ("bytes", "flops")}
    kvd = case["kv_heads"] * case["hd"]
    if kind == "attention":
        seen = case["pos"] + 1
        return {"bytes": 4 * (2 * seen * kvd + 2 * case["heads"] * case["hd"]), "flops": 4 * seen * case["heads"] * case["hd"]}
    dim, ffn, qd, rows = case["dim"], case["ffn"], case["heads"] * case["hd"], case.get("tokens", 1)
    total = {"bytes": 0, "flops": 0}
    shapes = [(qd + 2 * kvd, dim), (dim, qd), (2 * ffn, dim), (dim, ffn)]
    for n, k in shapes:
        total["bytes"] += case["layers"] * _weight_bytes(case["type"], n, k)
        total["flops"] += case["layers"] * 2 * rows * n * k
    total["bytes"] += _weight_bytes(case["type"], case["vocab"], dim) + 4 * case["vocab"] + 4 * rows * dim
    total["flops"] += 2 * case["vocab"] * dim
    pairs = rows * case["pos"] + rows * (rows + 1) // 2  # (query, key) pairs of causal attention
    total["bytes"] += case["layers"] * 4 * 2 * kvd * (case["pos"] + 2 * rows)
    total["flops"] += case["layers"] * 4 * pairs * qd
    return total


# ---- results ------------------------------------------------------------------------------------------------------------------


def tolerance(case):
    """About four times what the path shows against 64-bit arithmetic: 1.5e-7 to 7e-7 where sums are held in fp32,
    2.9e-4 (4.2e-4 behind SwiGLU) where activations and weights are rounded to fp16 once."""
    kind = case["kind"]
    if kind in ("attention", "decode") or case["type"] == "f32":
        return {"rel": 3e-6, "max": 4e-5}
    if kind == "layers":
        longest = max(case["dim"], case["ffn"])
    else:
        longest = case.get("k", 0)
    # One row, and up to 8 whose activations fit the local memory, run with fp32-class activations.
    if kind != "prefill" and case["m"] <= 8 and (case["m"] == 1 or case["m"] * longest <= 32768):
        return {"rel": 3e-6, "max": 4e-5}
    return {"rel": 1.5e-3, "max": 1.5e-2}


def _dequant(kind, raw, n, k):
    if kind == "f32":
        return raw.view(n, k).double()
    raw = raw.view(n, (k + 31) // 32, BLOCK[kind])
    d = raw[:, :, :2].contiguous().view(torch.float16).double()
    if kind == "q8_0":
        w = d * raw[:, :, 2:].contiguous().view(torch.int8).double()
    else:
        codes = raw[:, :, 2 if kind == "q4_0" else 4:]
        q = torch.cat([codes & 15, codes >> 4], dim=2).double()  # byte j holds elements j and j + 16
        w = d * (q - 8.0) if kind == "q4_0" else d * q + raw[:, :, 2:4].contiguous().view(torch.float16).double()
    return w.reshape(n, -1)[:, :k]


def _linear64(kind, raw, n, k, x, bias=None, swiglu=False):
    x = x.double()
    y = torch.empty((x.shape[0], n), dtype=torch.float64, device=x.device)
    step = max(1, 2**27 // k)
    for lo in range(0, n, step):
        hi = min(n, lo + step)
        rows = raw[lo:hi]
        y[:, lo:hi] = x @ _dequant(kind, rows, hi - lo, k).t().contiguous()
    if bias is not None:
        y += bias.double()
    if swiglu:  # rows 16t .. 16t + 7 are gates, 16t + 8 .. 16t + 15 the matching ups
        y = y.view(x.shape[0], n // 16, 2, 8)
        y = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(x.shape[0], n // 2)
    return y


def _rms(x, weight):
    return x * weight.double() / (x.square().mean(dim=-1, keepdim=True) + 1e-6).sqrt()


def _rope(x, start):
    rows, _, hd = x.shape
    freq = 1e6 ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device=x.device) / hd)
    angle = (start + torch.arange(rows, dtype=torch.float64, device=x.device))[:, None, None] * freq
    a, b = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], dim=-1)


def _attend(q, keys, values, start):
    """Causal attention of q [rows, heads, hd] at positions start.. over keys and values [positions, kv heads, hd]."""
    rows, heads, hd = q.shape
    group = heads // keys.shape[1]
    at = start + torch.arange(rows, device=q.device)[:, None]
    hidden = torch.arange(keys.shape[0], device=q.device)[None, :] > at
    out = torch.empty_like(q)
    for h in range(heads):
        s = (q[:, h] @ keys[:, h // group].t().contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1) @ values[:, h // group]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "aos"):
        raw, x, bias = _linear_inputs(case, seed)
        return _linear64(case["type"], raw, case["n"], case["k"], x, bias, case.get("swiglu", False))
    if kind == "layers":
        return [_linear64(case["type"], raw, n, k, x, bias, swiglu) for n, k, raw, x, bias, swiglu in _layers_inputs(case, seed)]
    if kind == "attention":
        q, keys, values = _attention_inputs(case, seed)
        seen = case["pos"] + 1
        return _attend(q[None].double(), keys[0, :seen].double(), values[0, :seen].double(), case["pos"])[0]
    model, keys, values, tokens = _model_inputs(case, seed)
    rows, start, heads, hd = len(tokens), case["pos"], case["heads"], case["hd"]
    shape = (case["layers"], case["max_seq"], case["kv_heads"], hd)
    cache = [torch.zeros(shape, dtype=torch.float64, device=DEVICE) for _ in range(2)]
    cache[0][:, :start] = keys
    cache[1][:, :start] = values

    def lin(w, x, bias=None):
        return _linear64(w["type"], w["data"], *w["shape"], x, bias)

    x = model["token_embedding"][torch.from_numpy(tokens).to(DEVICE).long()].double()
    for i, layer in enumerate(model["layers"]):
        h = _rms(x, layer["attention_norm"])
        q = _rope(lin(layer["wq"], h, layer["bq"]).view(rows, heads, hd), start)
        cache[0][i, start: start + rows] = _rope(lin(layer["wk"], h, layer["bk"]).view(rows, case["kv_heads"], hd), start)
        cache[1][i, start: start + rows] = lin(layer["wv"], h, layer["bv"]).view(rows, case["kv_heads"], hd)
        a = _attend(q, cache[0][i, : start + rows], cache[1][i, : start + rows], start)
        x = x + lin(layer["wo"], a.reshape(rows, heads * hd))
        h = _rms(x, layer["ffn_norm"])
        x = x + lin(layer["w_down"], torch.nn.functional.silu(lin(layer["w_gate"], h)) * lin(layer["w_up"], h))
    logits = lin(model["lm_head"], _rms(x[-1:], model["final_norm"]))[0]
    result = {"logits": logits, "keys": cache[0], "values": cache[1]}
    return dict(result, token=None) if kind == "decode" else result
