"""The workloads this framework is timed on, through its public entry points.

Each case is one call, or one step, that a program over quantized weights
makes: a decode projection, the projections of a whole decode step
(`DecodeSweep`), a prefill projection or MLP, and the mixture-of-experts MLP
of a decode token and of a prefill chunk.  Weights have the converters' byte
layouts; the sizes are those of the LLaMA-7B, LLaMA-70B and 512-expert
Qwen-MoE configurations this repository tests and benchmarks.

Decode reads every weight once per token, so the weights of a decode case are
chosen to pass the 256 MB Infinity Cache between one state and the next, as
the layers of a resident model do.
"""

import ctypes
import math

import torch
import torch.nn.functional as F

_GGUF_BYTES = {"q4_0": 18, "q8_0": 34}
_GROUP = 64  # affine-Q4 group size of the MoE converter


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest call: one GQA k/v projection of a 70B layer, one token.
        dict(name="decode_kv_1024x8192", kind="decode", fmt="q4_0", rows=1024, cols=8192, batch=1, count=1),
        # A single-sequence decode step: the projections of 8 LLaMA-7B layers and lm_head.
        dict(name="step_7b_q4_0_b1", kind="step", fmt="q4_0", hidden=4096, kv=4096, ffn=11008, layers=8,
             vocab=32000, batch=1),
        # Four sequences decoded together over 70B layers (grouped-query k/v).
        dict(name="step_70b_q4_0_b4", kind="step", fmt="q4_0", hidden=8192, kv=1024, ffn=28672, layers=2,
             vocab=32000, batch=4),
        # The 8-bit GGUF format at the largest decode batch.
        dict(name="step_7b_q8_0_b8", kind="step", fmt="q8_0", hidden=4096, kv=4096, ffn=11008, layers=4,
             vocab=32000, batch=8),
        # Per-column int8 weights (the other converter), one token through a 70B gate projection.
        dict(name="decode_int8_28672x8192", kind="decode", fmt="int8", rows=28672, cols=8192, batch=1, count=1),
        # Affine-Q4 projections of a decode token outside the experts.
        dict(name="decode_affine_32000x4096", kind="decode", fmt="affine_q4", rows=32000, cols=4096, batch=1, count=4),
        # One token through four MoE layers: router, top-10 of 512 experts, shared expert.
        dict(name="moe_decode_512x10", kind="moe_decode", layers=4, experts=512, hidden=4096, ffn=1024, top_k=10),
        # A 512-token prompt chunk over the same expert pool.
        dict(name="moe_prefill_512", kind="moe_prefill", tokens=512, experts=512, hidden=4096, ffn=1024, top_k=10),
        # A 512-token prompt chunk through a 7B MLP, the bulk of LLaMA prefill.
        dict(name="mlp_7b_q4_0_512", kind="mlp", fmt="q4_0", hidden=4096, ffn=11008, tokens=512),
        # A short prompt of no round length over 70B layers in the 8-bit format.
        dict(name="mlp_70b_q8_0_100", kind="mlp", fmt="q8_0", hidden=8192, ffn=28672, tokens=100),
        # A ragged prompt through an affine-Q4 projection.
        dict(name="prefill_affine_12288x4096_333", kind="prefill", fmt="affine_q4", rows=12288, cols=4096, tokens=333),
        # A long prompt in one chunk.
        dict(name="mlp_7b_q4_0_2048", kind="mlp", fmt="q4_0", hidden=4096, ffn=11008, tokens=2048),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer multiple of `step` in [lo, hi], log-uniform."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["decode", "step", "step", "moe_decode", "moe_prefill", "prefill", "mlp"])
    if kind == "decode":
        fmt = rng.choice(["q4_0", "q8_0", "int8", "affine_q4"])
        return dict(kind=kind, fmt=fmt, rows=_log_int(rng, 1000, 32003), cols=_log_int(rng, 2048, 14336, 256),
                    batch=rng.choice([1, 1, 2, 3, 5, 8]), count=rng.choice([1, 4]))
    if kind == "step":
        hidden = _log_int(rng, 2048, 8192, 256)
        kv = hidden if rng.random() < 0.5 else max(256, hidden // 8 // 128 * 128)
        return dict(kind=kind, fmt=rng.choice(["q4_0", "q4_0", "q8_0"]), hidden=hidden, kv=kv,
                    ffn=_log_int(rng, 2 * hidden, min(28672, 4 * hidden), 256), layers=rng.choice([2, 3]),
                    vocab=_log_int(rng, 16000, 40001), batch=rng.choice([1, 1, 2, 3, 4, 6, 8]))
    if kind == "moe_decode":
        return dict(kind=kind, layers=rng.choice([2, 4]), experts=_log_int(rng, 64, 512, 8),
                    hidden=rng.choice([2048, 4096, 4096]), ffn=rng.choice([512, 1024]), top_k=rng.randint(4, 10))
    if kind == "moe_prefill":
        return dict(kind=kind, tokens=_log_int(rng, 9, 512), experts=_log_int(rng, 64, 512),
                    hidden=rng.choice([2048, 3072, 4096]), ffn=rng.choice([512, 768, 1024]), top_k=rng.randint(4, 10))
    if kind == "prefill":
        return dict(kind=kind, fmt=rng.choice(["q4_0", "q8_0", "affine_q4"]), rows=_log_int(rng, 2000, 32003),
                    cols=_log_int(rng, 2048, 8192, 256), tokens=_log_int(rng, 9, 2048))
    hidden = _log_int(rng, 2048, 8192, 256)
    return dict(kind="mlp", fmt=rng.choice(["q4_0", "q8_0"]), hidden=hidden,
                ffn=_log_int(rng, 2 * hidden, min(28672, 3 * hidden), 256),
                tokens=_log_int(rng, 9, 2048 if hidden <= 4096 else 512))


# ------------------------------------------------- inputs, from the seed alone

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bytes(n, g):
    t = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda")
    t.random_(-(2 ** 63), None, generator=g)
    return t.view(torch.uint8)[:n]


def _uniform(shape, lo, hi, g):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g).half()


def _normal(shape, g, std=1.0):
    return (torch.randn(shape, dtype=torch.float32, device="cuda", generator=g) * std).half()


def _gguf(fmt, rows, cols, g):
    """Row-major blocks of 32 weights: an fp16 scale, then 16 bytes of 4-bit
    codes (Q4_0) or 32 int8 codes (Q8_0)."""
    n, size = rows * cols // 32, _GGUF_BYTES[fmt]
    w = _bytes(n * size, g).view(n, size)
    d = _uniform(n, 0.005, 0.02, g) if fmt == "q4_0" else _uniform(n, 0.0003, 0.001, g)
    w[:, :2] = d.view(torch.uint8).view(n, 2)
    return w.view(rows, cols // 32 * size)


def _affine(shape, g):
    """(words, scales, biases) of affine-Q4 weights: 4-bit codes around a
    group's zero point, as a quantizer of zero-mean weights leaves them."""
    *lead, cols = shape
    n = math.prod(lead)
    words = _bytes(n * cols // 2, g)
    s = _uniform((n, cols // _GROUP), 0.005, 0.02, g)
    b = (s.float() * -_uniform(s.shape, 7.0, 8.0, g).float()).half()
    return words, s, b


def _int8(rows, cols, g):
    return _bytes(rows * cols, g).view(torch.int8).view(rows, cols), _uniform((1, cols), 0.0003, 0.001, g)


def _affine_parts(case, g):
    """The stacked experts' gate/up/down, then the shared expert's."""
    E, H, Fd = case["experts"], case["hidden"], case["ffn"]
    return [_affine(s, g) for s in ([E, Fd, H], [E, Fd, H], [E, H, Fd], [Fd, H], [Fd, H], [H, Fd])]


def _sweep_shapes(case):
    H, KV, Fd = case["hidden"], case["kv"], case["ffn"]
    return {"self_attn.q_proj": (H, H), "self_attn.k_proj": (KV, H), "self_attn.v_proj": (KV, H),
            "self_attn.o_proj": (H, H), "mlp.gate_proj": (Fd, H), "mlp.up_proj": (Fd, H), "mlp.down_proj": (H, Fd)}


def _inputs(case, seed):
    """Raw inputs by name; the same for the framework's side and the 64-bit one."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("decode", "prefill"):
        rows, cols, fmt = case["rows"], case["cols"], case["fmt"]
        make = {"int8": _int8, "affine_q4": lambda m, k, r: _affine([m, k], r)}.get(fmt) or \
            (lambda m, k, r: _gguf(fmt, m, k, r))
        ws = [make(rows, cols, g) for _ in range(case.get("count", 1))]
        shape = (case["batch"], 1, cols) if kind == "decode" else (1, case["tokens"], cols)
        return {"w": ws, "x": [_normal(shape, g) for _ in ws]}
    if kind == "mlp":
        H, Fd = case["hidden"], case["ffn"]
        return {"gate": _gguf(case["fmt"], Fd, H, g), "up": _gguf(case["fmt"], Fd, H, g),
                "down": _gguf(case["fmt"], H, Fd, g), "x": _normal((1, case["tokens"], H), g, 0.3)}
    if kind == "step":
        layers = [{n: _gguf(case["fmt"], m, k, g) for n, (m, k) in _sweep_shapes(case).items()}
                  for _ in range(case["layers"])]
        H, B = case["hidden"], case["batch"]
        xs = [[_normal((B, H), g, 0.3) for _ in range(3)] for _ in layers]
        return {"layers": layers, "lm_head": _gguf(case["fmt"], case["vocab"], H, g), "xs": xs,
                "final": _normal((B, H), g)}
    if kind == "moe_decode":
        E, H = case["experts"], case["hidden"]
        return {"layers": [{"parts": _affine_parts(case, g), "router": _normal((E, H), g, 0.02),
                            "gate": _normal((1, H), g, 0.02), "x": _normal((H,), g, 0.3)}
                           for _ in range(case["layers"])]}
    T, E, H = case["tokens"], case["experts"], case["hidden"]
    parts = _affine_parts(case, g)
    val, idx = torch.randn(T, E, device="cuda", generator=g).topk(case["top_k"], dim=1)
    return {"parts": parts, "gate": _normal((1, H), g, 0.02), "x": _normal((1, T, H), g, 0.3),
            "idx": idx.to(torch.int32), "wts": torch.softmax(val, 1).half()}


# ------------------------------------------------------------ the framework's side

def _ext():
    from gdsllm_amd.runtime import ext
    return ext()


def _entry(fmt, shape, w):
    """A weight entry as ModelWeights.load_layer gives it."""
    handle = _ext().GdsBufferHandle.from_tensor
    if fmt != "affine_q4":
        return {"buffer": handle(w), "shape": list(shape), "gguf_type": fmt, "offset": 0}
    flat = [p.reshape(-1).view(torch.uint8) for p in w]
    starts = [0]
    for p in flat:
        starts.append(starts[-1] + (p.numel() + 4095) // 4096 * 4096)
    buf = torch.empty(starts[-1], dtype=torch.uint8, device="cuda")
    for p, o in zip(flat, starts):
        buf[o:o + p.numel()] = p
    return {"buffer": handle(buf), "shape": list(shape), "quant_type": "affine_q4", "weight_offset": starts[0],
            "scale_offset": starts[1], "bias_offset": starts[2], "group_size": _GROUP}


def _moe_shapes(case):
    E, H, Fd = case["experts"], case["hidden"], case["ffn"]
    return [[E, Fd, H], [E, Fd, H], [E, H, Fd], [Fd, H], [Fd, H], [H, Fd]]


def prepare(case, seed):
    raw, kind = _inputs(case, seed), case["kind"]
    if kind in ("decode", "prefill"):
        fmt, calls = case["fmt"], []
        for w, x in zip(raw["w"], raw["x"]):
            if fmt == "int8":
                weights = {"p.weight": w[0], "p.scale": w[1]}
            else:
                weights = {"p.weight": _entry(fmt, (case["rows"], case["cols"]), w)}
            calls.append((x, weights))
        return {"kind": "linear", "fmt": fmt, "calls": calls}
    if kind == "mlp":
        H, Fd = case["hidden"], case["ffn"]
        weights = {f"mlp.{n}_proj.weight": _entry(case["fmt"], s, raw[n])
                   for n, s in (("gate", (Fd, H)), ("up", (Fd, H)), ("down", (H, Fd)))}
        # the schedulers keep one scratch matrix for the dequantizing route
        scratch = torch.empty(Fd * H, dtype=torch.float16, device="cuda")
        return {"kind": kind, "x": raw["x"], "weights": weights, "scratch": scratch}
    if kind == "step":
        from gdsllm_amd.runtime.scheduler import DecodeSweep
        shapes = _sweep_shapes(case)
        layers = [{f"{n}.weight": _entry(case["fmt"], shapes[n], w) for n, w in lw.items()} for lw in raw["layers"]]
        head = _entry(case["fmt"], (case["vocab"], case["hidden"]), raw["lm_head"])
        sweep = DecodeSweep(layers, head, batch=case["batch"])
        for i, (a, o, m) in enumerate(raw["xs"]):
            sweep.attn_in[i].copy_(a)
            sweep.attn_out[i].copy_(o)
            sweep.mlp_in[i].copy_(m)
        sweep.final_in.copy_(raw["final"])
        return {"kind": kind, "sweep": sweep}
    shapes = _moe_shapes(case)
    if kind == "moe_prefill":
        names = [f"mlp.{o}.{p}_proj.weight" for o in ("switch_mlp", "shared_expert") for p in ("gate", "up", "down")]
        weights = {n: _entry("affine_q4", s, w) for n, s, w in zip(names, shapes, raw["parts"])}
        weights["mlp.shared_expert_gate.weight"] = raw["gate"]
        return {"kind": kind, "x": raw["x"], "weights": weights, "idx": raw["idx"], "wts": raw["wts"],
                "top_k": case["top_k"]}
    # moe_decode: the C interface, as a decode loop that keeps its workspace calls it
    from gdsllm_amd import AffineExperts, capi
    lib, k = capi(), case["top_k"]
    size = lib.gdsllm_moe_step_routed_workspace_size(k, case["ffn"], case["experts"])
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    layers = []
    for lw in raw["layers"]:
        structs = []
        for (w, s, b), shape in zip(lw["parts"], shapes):
            e = shape[0] if len(shape) == 3 else 1
            n, cols = shape[-2:]
            structs.append(AffineExperts(w.data_ptr(), s.data_ptr(), b.data_ptr(), n * cols // 2,
                                         n * cols // _GROUP * 2, n * cols // _GROUP * 2, e, n, cols, _GROUP))
        y = torch.empty(case["hidden"], dtype=torch.float16, device="cuda")
        idx = torch.empty(k, dtype=torch.int32, device="cuda")
        wts = torch.empty(k, dtype=torch.float16, device="cuda")
        layers.append((lw, [ctypes.byref(s) for s in structs], y, idx, wts))
    return {"kind": kind, "lib": lib, "layers": layers, "ws": ws, "size": size, "top_k": k}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        if state["fmt"] == "affine_q4":
            from gdsllm_amd.runtime.qwen_moe import affine_q4_linear as linear
        else:
            from gdsllm_amd.runtime.llama import dequant_linear as linear
        return [linear(x, weights, "p") for x, weights in state["calls"]]
    if kind == "mlp":
        from gdsllm_amd.runtime.llama import mlp
        return mlp(state["x"], state["weights"], state["scratch"])
    if kind == "step":
        s = state["sweep"]
        s.run()
        return {"q": s.q, "k": s.k, "v": s.v, "o": s.o, "h": s.h, "down": s.down, "logits": s.logits}
    if kind == "moe_prefill":
        from gdsllm_amd.runtime.qwen_moe import moe_mlp_selective
        return moe_mlp_selective(state["x"], state["weights"], None, state["idx"], state["wts"], state["top_k"])
    from gdsllm_amd import check
    stream = torch.cuda.current_stream().cuda_stream
    step, ws = state["lib"].gdsllm_moe_step_routed_affine_q4, state["ws"].data_ptr()
    outs = []
    for lw, structs, y, idx, wts in state["layers"]:
        check(step(lw["router"].data_ptr(), *structs, lw["x"].data_ptr(), state["top_k"], lw["gate"].data_ptr(),
                   y.data_ptr(), idx.data_ptr(), wts.data_ptr(), ws, state["size"], stream))
        outs.append({"y": y, "idx": idx, "wts": wts})
    return outs


# ------------------------------------------------------------ what a pass needs

def _weight_bytes(fmt, rows, cols):
    if fmt == "int8":
        return rows * cols + 2 * cols
    if fmt == "affine_q4":
        return rows * cols // 2 + 4 * rows * cols // _GROUP
    return rows * cols // 32 * _GGUF_BYTES[fmt]


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        m, k = case["rows"], case["cols"]
        n, c = case.get("batch", 1) * case.get("tokens", 1), case.get("count", 1)
        return {"bytes": c * (_weight_bytes(case["fmt"], m, k) + 2 * n * (m + k)), "flops": 2 * c * n * m * k}
    if kind == "mlp":
        H, Fd, n = case["hidden"], case["ffn"], case["tokens"]
        return {"bytes": 3 * _weight_bytes(case["fmt"], Fd, H) + 4 * n * H, "flops": 6 * n * Fd * H}
    if kind == "step":
        B, w, io, mk = case["batch"], 0, 0, 0
        for name, (m, k) in _sweep_shapes(case).items():
            w += _weight_bytes(case["fmt"], m, k)
            mk += m * k
            io += 0 if name == "mlp.up_proj" else m  # gate and up leave one h
        io += 3 * case["hidden"]
        head = _weight_bytes(case["fmt"], case["vocab"], case["hidden"])
        hio, L = case["vocab"] + case["hidden"], case["layers"]
        return {"bytes": L * (w + 2 * B * io) + head + 2 * B * hio,
                "flops": 2 * B * (L * mk + case["vocab"] * case["hidden"])}
    E, H, Fd, k = case["experts"], case["hidden"], case["ffn"], case["top_k"]
    expert = 3 * _weight_bytes("affine_q4", Fd, H)
    if kind == "moe_decode":
        L = case["layers"]
        return {"bytes": L * ((k + 1) * expert + 2 * E * H + 6 * H), "flops": 2 * L * ((k + 1) * 3 * H * Fd + E * H)}
    T = case["tokens"]
    touched = E * (1 - (1 - k / E) ** T)
    return {"bytes": (touched + 1) * expert + 4 * T * H, "flops": 6 * T * (k + 1) * H * Fd}


def tolerance(case):
    # fp16 results of fp32 sums: another order of the sums, or another rounding
    # of the weights to fp16, moves results by a last place here and there.
    # Two products in a row (an MLP, an expert) round an fp16 intermediate too.
    if case["kind"] == "moe_prefill":
        return {"rel": 2e-3, "max": 2e-2}
    if case["kind"] == "moe_decode":
        return {"rel": 2e-3, "max": 2e-2, "differ": 0.0}
    return {"rel": 1.2e-3, "max": 1e-2}


# --------------------------------------------------------- the same in 64 bits

def _w64(fmt, w, rows, cols, r0, r1):
    """Rows r0 .. r1-1 of a weight matrix, float64."""
    if fmt == "int8":
        return w[0][r0:r1].double() * w[1].double()
    if fmt == "affine_q4":
        words, s, b = w
        q = words.view(rows, cols // 2)[r0:r1]
        q = torch.stack([q & 15, q >> 4], -1).view(r1 - r0, cols // _GROUP, _GROUP).double()
        s, b = (t.view(rows, -1)[r0:r1].double().unsqueeze(-1) for t in (s, b))
        return (q * s + b).view(r1 - r0, cols)
    blk = w[r0:r1].reshape(r1 - r0, cols // 32, _GGUF_BYTES[fmt])
    d = blk[..., :2].contiguous().view(torch.float16).double()
    if fmt == "q4_0":
        q = torch.cat([blk[..., 2:] & 15, blk[..., 2:] >> 4], -1).double() - 8
    else:
        q = blk[..., 2:].contiguous().view(torch.int8).double()
    return (d * q).view(r1 - r0, cols)


def _lin64(x, fmt, w, rows, cols):
    x = x.double()
    parts = [x @ _w64(fmt, w, rows, cols, r, min(rows, r + 4096)).t() for r in range(0, rows, 4096)]
    return torch.cat(parts, -1)


def _mlp64(x, fmt, ws, H, Fd):
    g, u = _lin64(x, fmt, ws[0], Fd, H), _lin64(x, fmt, ws[1], Fd, H)
    return _lin64(F.silu(g) * u, fmt, ws[2], H, Fd)


def _expert64(parts, e, H, Fd):
    """Expert e's gate, up and down out of the stacked parts."""
    out = []
    for (w, s, b), (m, k) in zip(parts[:3], ((Fd, H), (Fd, H), (H, Fd))):
        n = m * k // 2
        out.append((w[e * n:(e + 1) * n], s.view(-1, k // _GROUP)[e * m:(e + 1) * m],
                    b.view(-1, k // _GROUP)[e * m:(e + 1) * m]))
    return out


def exact(case, seed):
    raw, kind = _inputs(case, seed), case["kind"]
    if kind in ("decode", "prefill"):
        return [_lin64(x, case["fmt"], w, case["rows"], case["cols"]) for w, x in zip(raw["w"], raw["x"])]
    if kind == "mlp":
        return _mlp64(raw["x"], case["fmt"], [raw["gate"], raw["up"], raw["down"]], case["hidden"], case["ffn"])
    if kind == "step":
        fmt, shapes = case["fmt"], _sweep_shapes(case)
        out = {n: [] for n in ("q", "k", "v", "o", "h", "down")}
        for lw, (a, o, m) in zip(raw["layers"], raw["xs"]):
            lin = lambda n, x: _lin64(x, fmt, lw[n], *shapes[n])  # noqa: E731
            for n in "qkv":
                out[n].append(lin(f"self_attn.{n}_proj", a))
            out["o"].append(lin("self_attn.o_proj", o))
            h = F.silu(lin("mlp.gate_proj", m)) * lin("mlp.up_proj", m)
            out["h"].append(h)
            out["down"].append(lin("mlp.down_proj", h))
        return dict(out, logits=_lin64(raw["final"], fmt, raw["lm_head"], case["vocab"], case["hidden"]))
    H, Fd, k = case["hidden"], case["ffn"], case["top_k"]
    if kind == "moe_decode":
        outs = []
        for lw in raw["layers"]:
            x = lw["x"].double().view(1, H)
            # the picks are those of fp16 logits, ties to the lower expert
            logits = (x @ lw["router"].double().t()).half().view(-1)
            idx = torch.sort(logits, descending=True, stable=True).indices[:k]
            wts = torch.softmax(logits[idx].double(), 0)
            y = sum(wts[j] * _mlp64(x, "affine_q4", _expert64(lw["parts"], int(idx[j]), H, Fd), H, Fd)
                    for j in range(k))
            y = y + torch.sigmoid(x @ lw["gate"].double().t()) * _mlp64(x, "affine_q4", lw["parts"][3:], H, Fd)
            outs.append({"y": y.view(-1), "idx": None, "wts": wts})
        return outs
    x = raw["x"].double().view(-1, H)
    y, wts = torch.zeros_like(x), raw["wts"].double()
    for e in raw["idx"].unique().tolist():
        tok, slot = (raw["idx"] == e).nonzero(as_tuple=True)
        y.index_add_(0, tok, wts[tok, slot].unsqueeze(1) *
                     _mlp64(x[tok], "affine_q4", _expert64(raw["parts"], e, H, Fd), H, Fd))
    y += torch.sigmoid(x @ raw["gate"].double().t()) * _mlp64(x, "affine_q4", raw["parts"][3:], H, Fd)
    return y.view(1, -1, H)
