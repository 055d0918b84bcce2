"""The work that programs have this library do, as cases that can be timed and compared.

A case is one of five kinds, each through the public Python entry points (tiny-llm_amd/__init__.py):

  decode   one decode step's projections of a stack of layers on device buffers, captured once
           into an op graph and replayed (what a device-resident decode loop does per token)
  head     one lm_head matvec on device buffers
  prefill  one layer's seven projections over a prompt of `tokens` tokens on device buffers
  host     one layer's projections on host arrays in the order in which tiny-llm's runtime calls
           the kernel registry (one token: qkv, o, gate/up pair, down; several: one matmul each)
  engine   a prompt fed token by token to the decode engine from an empty cache

Weights, activations and model files are synthetic: i4 codes uniform, scales U[0.002, 0.02], zeros
U[0, 15]; VQ2 indices uniform, codebook N(0, 0.02); activations N(0, 1).
"""
import importlib.util
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "tiny_llm_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("tiny_llm_amd", os.path.join(ROOT, "tiny-llm_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["tiny_llm_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["tiny_llm_amd"]


tq = _package()

# Layer widths (hidden, q rows, k/v rows, intermediate) of the two model sizes that the benchmark
# of this repository is built on.
SMALL = dict(hidden=896, q=896, kv=128, inter=4864)
LARGE = dict(hidden=2560, q=4096, kv=1024, inter=9728)


def listed():
    return [
        # A decode token of the 0.5B-sized model: 24 layers, each layer's seven matrices as one set
        # launch. Launch and latency bound.
        dict(name="decode_i4_set", kind="decode", fmt="i4", order="set", layers=24, group=64, **SMALL),
        # The same step of a VQ2 file.
        dict(name="decode_vq2_set", kind="decode", fmt="vq2", order="set", layers=24, group=0, **SMALL),
        # A decode token of the 4B-sized model quantized with groups of 128, in the runtime's call
        # order (qkv, o, gate/up pair, down).
        dict(name="decode_i4_g128_calls", kind="decode", fmt="i4", order="calls", layers=6, group=128, **LARGE),
        # The largest matvecs: the 4B-sized model's lm_head in both formats.
        dict(name="head_i4", kind="head", fmt="i4", rows=151936, cols=2560, group=64),
        dict(name="head_vq2", kind="head", fmt="vq2", rows=151936, cols=2560, group=0),
        # A short continuation (a few new tokens in one pass) on the 0.5B-sized model.
        dict(name="prefill_8", kind="prefill", tokens=8, group=64, **SMALL),
        # An ordinary prompt on the 4B-sized model.
        dict(name="prefill_512", kind="prefill", tokens=512, group=64, **LARGE),
        # A long ragged prompt on the 4B-sized model with groups of 128.
        dict(name="prefill_3001_g128", kind="prefill", tokens=3001, group=128, **LARGE),
        # tiny-llm's runtime on the drop-in kernels: a decode token (the smallest calls), and a
        # prompt of a VQ2 file.
        dict(name="host_i4_token", kind="host", fmt="i4", tokens=1, group=64, **SMALL),
        dict(name="host_vq2_prompt", kind="host", fmt="vq2", tokens=64, group=0, **SMALL),
        # The engine: a long prompt (attention over a growing cache), and a short one of a
        # rotated VQ2 file.
        dict(name="engine_i4_long", kind="engine", fmt="i4", layers=4, tokens=3000, heads=14, kv_heads=2, head_dim=64,
             hidden=896, inter=4864, vocab=32000),
        dict(name="engine_vq2_rotated", kind="engine", fmt="vq2", layers=8, tokens=48, heads=14, kv_heads=2,
             head_dim=64, hidden=896, inter=4864, vocab=32000),
    ]


def _spread(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _layer(rng, hi, ragged):
    """Widths of a layer between a quarter-sized model and the 4B-sized one; a third of them ragged."""
    step = rng.choice((4, 12)) if ragged else 64
    width = lambda v: max(step, int(v) // step * step)  # noqa: E731
    hidden = width(_spread(rng, 512, hi))
    q = width(hidden * rng.choice((1.0, 1.0, 1.6)))
    return dict(hidden=hidden, q=q, kv=width(q / rng.choice((1, 4, 7))), inter=width(hidden * rng.uniform(2.5, 5.5)))


def draw(rng):
    kind = rng.choice(("decode", "decode", "head", "prefill", "prefill", "host", "engine"))
    fmt = rng.choice(("i4", "i4", "vq2"))
    group = rng.choice((64, 64, 128, 32)) if fmt == "i4" else 0
    ragged = rng.random() < 0.3
    if kind == "decode":
        widths = _layer(rng, 2560, ragged)
        return dict(kind=kind, fmt=fmt, order=rng.choice(("set", "calls")),
                    layers=rng.randint(4, 24 if widths["hidden"] < 1536 else 8), group=group, **widths)
    if kind == "head":
        step = 4 if ragged else 64
        return dict(kind=kind, fmt=fmt, rows=int(_spread(rng, 16000, 151936)),
                    cols=int(_spread(rng, 512, 2560)) // step * step, group=group)
    if kind == "prefill":
        return dict(kind=kind, tokens=int(_spread(rng, 2, 3001)), group=group or 64, **_layer(rng, 2560, ragged))
    if kind == "host":
        return dict(kind=kind, fmt=fmt, tokens=rng.choice((1, int(_spread(rng, 2, 64)))), group=group,
                    **_layer(rng, 1536, ragged))
    head_dim = rng.choice((64, 64, 128))
    kv_heads = rng.choice((1, 2, 4))
    heads = kv_heads * rng.randint(2, 7 if head_dim == 64 else 3)
    return dict(kind=kind, fmt=fmt, layers=rng.randint(1, 4), tokens=int(_spread(rng, 16, 3000)), heads=heads,
                kv_heads=kv_heads, head_dim=head_dim, hidden=128 * rng.randint(4, 8), inter=256 * rng.randint(6, 19),
                vocab=rng.randint(2000, 32000))


# ---- inputs ------------------------------------------------------------------------------------

def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _i4(rows, cols, group, g):
    """i4 rows on the GPU: per group fp16 scale, fp16 zero, group / 2 code bytes."""
    groups = -(-cols // group)
    w = torch.randint(0, 256, (rows, groups, 4 + group // 2), generator=g, device="cuda", dtype=torch.uint8)
    head = torch.rand((rows, groups, 2), generator=g, device="cuda")
    head[..., 0] = 0.002 + 0.018 * head[..., 0]
    head[..., 1] *= 15.0
    w[..., :4] = head.half().view(torch.uint8)
    return w.reshape(-1)


def _vq2(rows, cols, g):
    """A VQ2 tensor on the GPU: 256 x 4 fp16 codebook, then rows x cols / 4 indices."""
    book = (0.02 * torch.randn(1024, generator=g, device="cuda")).half().view(torch.uint8)
    return torch.cat([book, torch.randint(0, 256, (rows * (cols // 4),), generator=g, device="cuda", dtype=torch.uint8)])


def _weights(case, rows, cols, g):
    return _vq2(rows, cols, g) if case.get("fmt") == "vq2" else _i4(rows, cols, case["group"], g)


def _normal(n, g):
    return torch.randn(n, generator=g, device="cuda")


# a layer's matrices in the runtime's order: name, rows, columns and which activation it reads
def _matrices(c):
    h, q, kv, i = c["hidden"], c["q"], c["kv"], c["inter"]
    return [("q", q, h, 0), ("k", kv, h, 0), ("v", kv, h, 0), ("o", h, q, 1), ("gate", i, h, 2), ("up", i, h, 2),
            ("down", h, i, 3)]


def _layer_inputs(case, seed, layer=0):
    """Weights by matrix name and the layer's four activations (tokens x width), on the GPU."""
    g = _generator(1000 * seed + layer)
    w = {name: _weights(case, rows, cols, g) for name, rows, cols, _ in _matrices(case)}
    n = case.get("tokens", 1)
    widths = (case["hidden"], case["q"], case["hidden"], case["inter"])
    return w, [_normal(n * k, g) for k in widths]


def _model(case, seed):
    make = tq.tqwen_synth.dense_i4_model
    vq2 = case["fmt"] == "vq2"
    return make(hidden=case["hidden"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                inter=case["inter"], vocab=case["vocab"], layers=case["layers"], seed=int(seed) % (1 << 30),
                max_seq_len=max(64, case["tokens"]), vq2=vq2, rotated=vq2)


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], case["tokens"]).tolist()


def _call_ops(case, w, x, y):
    """A decode layer as the runtime's calls: four launches for i4, one matvec each for VQ2."""
    p = {k: t.data_ptr() for k, t in w.items()}
    xs, ys = [t.data_ptr() for t in x], {k: t.data_ptr() for k, t in y.items()}
    h, q, kv, i, g = case["hidden"], case["q"], case["kv"], case["inter"], case["group"]
    if case["fmt"] == "vq2":
        return [tq.Op(tq.OP_VQ2_MATVEC, p[n], xs[a], ys[n], rows, cols, 1, 0) for n, rows, cols, a in _matrices(case)]
    return [tq.Op(tq.OP_I4_QKV, p["q"], xs[0], ys["q"], q, h, 1, g, p["k"], p["v"], ys["k"], ys["v"], kv),
            tq.Op(tq.OP_I4_MATVEC, p["o"], xs[1], ys["o"], h, q, 1, g),
            tq.Op(tq.OP_I4_PAIR, p["gate"], xs[2], ys["gate"], i, h, 1, g, p["up"], None, ys["up"], None, 0),
            tq.Op(tq.OP_I4_MATVEC, p["down"], xs[3], ys["down"], h, i, 1, g)]


_STREAMS = []


def _stream():
    """The one stream of a decode loop: a token's step follows the last one's."""
    if not _STREAMS:
        _STREAMS.append(tq.Stream())
    return _STREAMS[0]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "decode":
        ops, keep = [], []
        mats = _matrices(case)
        out = torch.empty((case["layers"], sum(rows for _, rows, _, _ in mats)), device="cuda")
        for layer in range(case["layers"]):
            w, x = _layer_inputs(case, seed, layer)
            y = dict(zip((m[0] for m in mats), out[layer].split([rows for _, rows, _, _ in mats])))
            keep.append((w, x))
            if case["order"] == "set":
                records = tq.i4_set([(w[n].data_ptr(), x[a].data_ptr(), y[n].data_ptr(), rows, cols)
                                     for n, rows, cols, a in mats])
                keep.append(records)
                ops.append(tq.vq2_set_op(records) if case["fmt"] == "vq2" else tq.set_op(records, case["group"]))
            else:
                ops += _call_ops(case, w, x, y)
        torch.cuda.synchronize()
        state.update(keep=keep, out=out, graph=tq.OpsGraph(ops, _stream()))
    elif kind == "head":
        g = _generator(seed)
        state.update(w=_weights(case, case["rows"], case["cols"], g), x=_normal(case["cols"], g),
                     y=torch.empty(case["rows"], device="cuda"))
    elif kind == "prefill":
        w, x = _layer_inputs(case, seed)
        n = case["tokens"]
        y = {name: torch.empty((n, rows), device="cuda") for name, rows, _, _ in _matrices(case)}
        state.update(w=w, x=x, y=y, ops=[tq.Op(tq.OP_I4_MATMUL, w[m].data_ptr(), x[a].data_ptr(), y[m].data_ptr(),
                                               rows, cols, n, case["group"]) for m, rows, cols, a in _matrices(case)])
    elif kind == "host":
        w, x = _layer_inputs(case, seed)
        state.update(w={k: t.cpu().numpy() for k, t in w.items()}, x=[t.cpu().numpy() for t in x])
    else:
        image, _, _ = _model(case, seed)
        model = tq.ModelFile.from_image(image)
        state.update(model=model, engine=tq.DecodeEngine(model), prompt=_prompt(case, seed))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        state["graph"].launch()
        return state["out"]
    if kind == "head":
        if case["fmt"] == "vq2":
            tq.matvec_vq2_dev(state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(), case["rows"], case["cols"])
        else:
            tq.matvec_i4_dev(state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(), case["rows"],
                             case["cols"], case["group"])
        return state["y"]
    if kind == "prefill":
        tq.run_ops(state["ops"], 1)
        return state["y"]
    if kind == "host":
        w, x, n, g = state["w"], state["x"], case["tokens"], case["group"]
        if n == 1 and case["fmt"] == "i4":
            q, k, v = tq.matvec_qkv_i4(w["q"], w["k"], w["v"], x[0], case["q"], case["kv"], case["hidden"], g)
            o = tq.matvec_i4(w["o"], x[1], case["hidden"], case["q"], g)
            gate, up = tq.matvec_pair_i4(w["gate"], w["up"], x[2], case["inter"], case["hidden"], g)
            down = tq.matvec_i4(w["down"], x[3], case["hidden"], case["inter"], g)
            return dict(q=q, k=k, v=v, o=o, gate=gate, up=up, down=down)
        if n == 1:
            return {m: tq.matvec_vq2(w[m], x[a], rows, cols) for m, rows, cols, a in _matrices(case)}
        if case["fmt"] == "i4":
            return {m: tq.matmul_i4(w[m], x[a], rows, cols, n, g) for m, rows, cols, a in _matrices(case)}
        return {m: tq.matmul_vq2(w[m], x[a], rows, cols, n) for m, rows, cols, a in _matrices(case)}
    engine = state["engine"]
    engine.reset()
    for token in state["prompt"]:
        engine.step(token)
    return engine.logits()


# ---- what a pass cannot do without --------------------------------------------------------------

def _weight_bytes(case, rows, cols):
    if case.get("fmt") == "vq2":
        return 2048 + rows * (cols // 4)
    return rows * -(-cols // case["group"]) * (4 + case["group"] // 2)


def work(case):
    kind = case["kind"]
    if kind == "head":
        return {"bytes": _weight_bytes(case, case["rows"], case["cols"]) + 4 * (case["rows"] + case["cols"]),
                "flops": 2 * case["rows"] * case["cols"]}
    if kind == "engine":
        c = dict(case, q=case["heads"] * case["head_dim"], kv=case["kv_heads"] * case["head_dim"], group=64)
        n, mats = c["tokens"], _matrices(c)
        token = c["layers"] * sum(_weight_bytes(c, rows, cols) for _, rows, cols, _ in mats)
        token += _weight_bytes(dict(c, fmt="i4"), c["vocab"], c["hidden"]) + 4 * c["vocab"]
        cache = c["layers"] * 2 * 4 * c["kv"] * n * (n + 1) // 2
        flops = 2 * n * (c["layers"] * sum(rows * cols for _, rows, cols, _ in mats) + c["vocab"] * c["hidden"])
        return {"bytes": n * token + cache, "flops": flops + 4 * c["layers"] * c["q"] * n * (n + 1) // 2}
    n, layers, mats = case.get("tokens", 1), case.get("layers", 1), _matrices(case)
    widths = case["hidden"] + case["q"] + case["hidden"] + case["inter"]
    per_layer = sum(_weight_bytes(case, rows, cols) + 4 * n * rows for _, rows, cols, _ in mats) + 4 * n * widths
    return {"bytes": layers * per_layer, "flops": 2 * n * layers * sum(rows * cols for _, rows, cols, _ in mats)}


# ---- comparison ----------------------------------------------------------------------------------

def tolerance(case):
    """About four times the measured distance from 64 bits. Matvecs and VQ2 products are computed in (at
    least) 32 bits: up to 5e-7. The i4 matmul rounds both operands to 16 bits: 4e-4. The engine is a chain
    of 32-bit layers: 1e-4 after 3000 tokens, whose RoPE angles are 32-bit too."""
    if case["kind"] == "prefill" or (case["kind"] == "host" and case["fmt"] == "i4" and case["tokens"] > 1):
        return {"rel": 1.6e-3, "max": 1.6e-2}
    if case["kind"] == "engine":
        return {"rel": 4e-4, "max": 4e-3}
    return {"rel": 2e-6, "max": 2e-5}


def _dense(case, w, rows, cols):
    """The matrix in 64 bits from its bytes (a uint8 tensor on the GPU)."""
    if case.get("fmt") == "vq2":
        book = w[:2048].view(torch.float16).double().reshape(256, 4)
        return book[w[2048:].long()].reshape(rows, cols)
    group = case["group"]
    w = w.reshape(rows, -1, 4 + group // 2)
    head = w[..., :4].contiguous().view(torch.float16).double()
    codes = w[..., 4:]
    q = torch.stack([codes & 15, codes >> 4], -1).reshape(rows, -1, group).double()
    return ((q - head[..., 1:]) * head[..., :1]).reshape(rows, -1)[:, :cols]


def _exact_layer(case, seed, layer):
    w, x = _layer_inputs(case, seed, layer)
    out = {}
    for m, rows, cols, a in _matrices(case):
        out[m] = x[a].double().reshape(-1, cols) @ _dense(case, w[m], rows, cols).t()
    return out


def _exact_engine(case, seed):
    """The dense decoder over the whole prompt at once in 64 bits."""
    _, cfg, tensors = _model(case, seed)
    c = dict(case, group=64)
    hd, nh, nkv, eps, n = c["head_dim"], c["heads"], c["kv_heads"], cfg["rms_norm_eps"], c["tokens"]

    def raw(name):
        return torch.frombuffer(bytearray(tensors[name][2]), dtype=torch.uint8).cuda()

    def vec(name):
        return raw(name).view(torch.float16 if tensors[name][0] == 1 else torch.float32).double()

    def mat(name, fmt=None):
        return _dense(dict(c, fmt=fmt or c["fmt"]), raw(name), *tensors[name][1])

    def project(name, x):
        if name + ".rot_sign" in tensors:
            width = x.shape[-1]
            block = next(b for b in (256, 128, 64, 32, 16, 8, 4, 2, 1) if width % b == 0)
            x = (x / vec(name + ".rot_scale") * vec(name + ".rot_sign")).reshape(n, -1, block)
            hadamard = torch.ones((1, 1), dtype=torch.float64, device="cuda")
            while hadamard.shape[0] < block:
                hadamard = torch.cat([torch.cat([hadamard, hadamard], 1), torch.cat([hadamard, -hadamard], 1)], 0)
            x = (x @ hadamard).reshape(n, width) / block ** 0.5
        return x @ mat(name + ".weight").t()

    def norm(x, w):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w

    positions = torch.arange(n, device="cuda", dtype=torch.float64)
    half = hd // 2
    angle = positions[:, None] * cfg["rope_theta"] ** (-2.0 * torch.arange(half, device="cuda").double() / hd)

    def rope(x):  # tokens x heads x head_dim
        a, b, cos, sin = x[..., :half], x[..., half:], angle.cos()[:, None], angle.sin()[:, None]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    table = mat("model.embed_tokens.weight", "i4")
    hidden = table[torch.tensor(_prompt(case, seed), device="cuda")]
    causal = positions[:, None] >= positions[None, :]
    for layer in range(c["layers"]):
        p = "model.layers.%d." % layer
        x = norm(hidden, vec(p + "input_layernorm.weight"))
        q, k, v = (project(p + "self_attn.%s_proj" % s, x) + vec(p + "self_attn.%s_proj.bias" % s) for s in "qkv")
        q, k, v = rope(q.reshape(n, nh, hd)), rope(k.reshape(n, nkv, hd)), v.reshape(n, nkv, hd)
        attended = []
        for head in range(nh):
            at = head * nkv // nh
            s = (q[:, head] @ k[:, at].t() / hd ** 0.5).masked_fill(~causal, float("-inf"))
            attended.append(torch.softmax(s, -1) @ v[:, at])
        hidden = hidden + project(p + "self_attn.o_proj", torch.cat(attended, -1))
        x = norm(hidden, vec(p + "post_attention_layernorm.weight"))
        gate, up = project(p + "mlp.gate_proj", x), project(p + "mlp.up_proj", x)
        hidden = hidden + project(p + "mlp.down_proj", gate * torch.sigmoid(gate) * up)
    return norm(hidden, vec("model.norm.weight"))[-1] @ table.t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "engine":
        return _exact_engine(case, seed)
    if kind == "head":
        g = _generator(seed)
        w, x = _weights(case, case["rows"], case["cols"], g), _normal(case["cols"], g)
        return _dense(case, w, case["rows"], case["cols"]) @ x.double()
    if kind == "decode":
        return torch.stack([torch.cat([y.reshape(-1) for y in _exact_layer(case, seed, layer).values()])
                            for layer in range(case["layers"])])
    return {m: y if kind == "prefill" else y.reshape(-1) for m, y in _exact_layer(case, seed, 0).items()}
