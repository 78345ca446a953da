"""The work that a user of the int8 taggers has them do, as cases that can be timed and compared.

Kinds of case:

* call     one whole tagger call (engine on an image batch, graph replay), reduced to two blocks: the layers of a deeper
           model repeat, and a changed rounding grows with every int8 block until it hides everything else.
* attn     the attention half of a block as the engines run it (norm + rotation + int8, QKV product with RoPE,
           attention, rotation + int8, projection added to the residual stream), in a HIP graph as the engines do.
* mlp      the MLP half (norm + rotation + int8, fc1 with SwiGLU or GELU, rotation + int8, fc2 added to the stream),
           captured in a HIP graph.
* linear   one W8A8 linear called eagerly: rotation + int8, then the int8 product with bias.
* scores   attention alone, called eagerly.
* pool     Haruka's tree-pool head over the tokens of a batch, captured in a HIP graph.
* letterbox  one host image resized and padded for Haruka on the GPU, called eagerly.

Models (dims of this package's configurations): "eva02" (EVA02-L/14: 1024 wide, 16 heads, SwiGLU hidden 2730 padded to
2816), "pixai" (1024 wide, 16 heads, GELU hidden 4736), "haruka" (EVA02-B/14: 768 wide, 12 heads, SwiGLU hidden 2048).
"""

import math

import numpy as np
import torch

from foidfinder_amd.backends.rocm.preprocess import letterbox_gpu
from foidfinder_amd.engine import Eva02Config, Eva02Int8
from foidfinder_amd.haruka import HarukaConfig, HarukaInt8
from foidfinder_amd.kernels import EPI_BIAS_F16, EPI_GELU_F16, EPI_QKV_ROPE, EPI_RESIDUAL, EPI_SWIGLU, kernels, pad_norm

DEV = "cuda"
Q_SCALE = 0.125 * math.log2(math.e)  # softmax scale x log2(e), which the QKV epilogue folds into q
MODELS = {
    "eva02": dict(dim=1024, heads=16, hidden=2730, pad=2816, act="swiglu", mlp_norm=True, eps=1e-6),
    "pixai": dict(dim=1024, heads=16, hidden=4736, pad=4736, act="gelu", mlp_norm=False, eps=1e-5),
    "haruka": dict(dim=768, heads=12, hidden=2048, pad=2048, act="swiglu", mlp_norm=True, eps=1e-6),
}


def listed():
    return [
        # one image through EVA02-L/14-448: interactive tagging, where latency and launches count
        dict(name="eva02 call, 1 image", kind="call", model="eva02", batch=1, grid=32),
        # a single W8A8 linear on one image's tokens, called from Python
        dict(name="linear 1025x1024x3072", kind="linear", rows=1025, width=1024, cols=3072),
        # EVA02-L at the benchmark's batch: large-scale tagging throughput
        dict(name="eva02 attn, 32 images", kind="attn", model="eva02", seqs=32, tokens=1025),
        dict(name="eva02 mlp, 32 images", kind="mlp", model="eva02", rows=32 * 1025),
        # small serving batches, whose products fill the GPU badly
        dict(name="eva02 attn, 3 images", kind="attn", model="eva02", seqs=3, tokens=1025),
        dict(name="eva02 mlp, 1 image", kind="mlp", model="eva02", rows=1025),
        # PixAI's windowed attention on one 1008 px image (9 windows of 24 x 24 tokens)
        dict(name="pixai attn, 1 image", kind="attn", model="pixai", seqs=9, tokens=576),
        # PixAI's MLP on one 1008 px image (GELU, the widest rotation)
        dict(name="pixai mlp, 1 image", kind="mlp", model="pixai", rows=5184),
        # PixAI's global attention: the longest sequence
        dict(name="scores 1x5184", kind="scores", seqs=1, tokens=5184, heads=16),
        # Haruka at a medium batch: 768 wide, 12 heads
        dict(name="haruka attn, 16 images", kind="attn", model="haruka", seqs=16, tokens=1025),
        # Haruka's head with its 98 782 tags
        dict(name="haruka pool, 16 images", kind="pool", batch=16, grid=32),
        # what stands before each Haruka call: one photo letterboxed to 448 px
        dict(name="letterbox 1200x900", kind="letterbox", height=900, width=1200, size=448),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "linear", "attn", "mlp", "attn", "mlp", "scores", "pool", "letterbox"])
    if kind == "call":  # EVA02 at other resolutions (112 to 448 px) and batches
        return dict(kind=kind, model="eva02", batch=_log(rng, 1, 8), grid=rng.randint(8, 32))
    if kind == "linear":
        width = rng.choice([1024, 1024, 768, 2048, 4736])
        return dict(kind=kind, rows=_log(rng, 1, 16000), width=width, cols=16 * rng.randint(48, 256))
    if kind == "scores":
        tokens = _log(rng, 64, 5184)
        most = max(1, min(32000 // tokens, 60_000_000 // tokens**2))
        return dict(kind=kind, seqs=_log(rng, 1, most), tokens=tokens, heads=rng.choice([12, 16]))
    if kind == "pool":
        return dict(kind=kind, batch=_log(rng, 1, 32), grid=rng.randint(8, 32))
    if kind == "letterbox":
        return dict(kind=kind, height=_log(rng, 200, 2000), width=_log(rng, 200, 2000), size=448)
    model = rng.choice(["eva02", "eva02", "pixai", "haruka"])
    if model == "pixai":  # windows of 24 x 24 tokens, 9 an image at 1008 px
        seqs, tokens = _log(rng, 1, 48), 576
    else:
        grid = rng.randint(8, 32)
        tokens = 1 + grid * grid
        seqs = _log(rng, 1, 32)
    if kind == "attn":
        return dict(kind=kind, model=model, seqs=seqs, tokens=tokens)
    return dict(kind=kind, model=model, rows=max(1, seqs * tokens - rng.randint(0, 63)))


# ---- inputs, from the seed alone ----


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) + 1)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * std


def _stream(g, rows, width):
    """A residual stream in fp16: unit variance, 1 % of the channels 20 times as large (activation outliers)."""
    x = _randn(g, rows, width)
    cols = torch.randperm(width, device=DEV, generator=g)[: max(1, width // 100)]
    x[:, cols] *= 20.0
    return x.half()


def _linear(g, n, k, std=0.03):
    """int8 codes as a rotated weight's (close to Gaussian, the largest near 3.3 deviations), fp32 scales and bias."""
    codes = _randn(g, n, k, std=38.0).round_().clamp_(-127, 127).to(torch.int8)
    scale = (std / 38.0) * (0.8 + 0.4 * torch.rand(n, device=DEV, generator=g))
    return codes, scale, _randn(g, n, std=0.02)


def _norm(g, n):
    return 1.0 + _randn(g, n, std=0.02), _randn(g, n, std=0.02)


def _rope(tokens):
    """cos/sin fp32 [tokens, 32] of an axial table: a class token without rotation first when tokens = 1 + grid^2."""
    side = int(round(math.sqrt(tokens)))
    cls = 0 if side * side == tokens else 1
    grid = math.isqrt(tokens - cls)
    pos = torch.arange(tokens - cls, dtype=torch.float64)
    bands = 10000.0 ** (-torch.arange(16, dtype=torch.float64) / 16)
    scale = 16.0 / max(grid, 1)
    ang = torch.cat([torch.floor(pos / grid)[:, None] * scale * bands, (pos % grid)[:, None] * scale * bands], 1)
    ang = torch.cat([torch.zeros(cls, 32, dtype=torch.float64), ang])
    return ang.cos().float().to(DEV), ang.sin().float().to(DEV)


def _fc1(g, m):
    """fc1: for SwiGLU the rows are (gate, value) pairs, zero past the hidden width."""
    if m["act"] == "gelu":
        return _linear(g, m["hidden"], m["dim"])
    w, s, b = _linear(g, 2 * m["pad"], m["dim"])
    w[2 * m["hidden"] :] = 0
    b[2 * m["hidden"] :] = 0
    return w, s, b


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        return dict(x=_stream(g, case["rows"], case["width"]), w=_linear(g, case["cols"], case["width"]))
    if kind == "scores":
        rows, c = case["seqs"] * case["tokens"], 64 * case["heads"]
        qkv = _randn(g, rows, 3 * c)
        qkv[:, :c] *= Q_SCALE
        return dict(qkv=qkv.half())
    if kind in ("attn", "mlp"):
        m = MODELS[case["model"]]
        d = m["dim"]
        rows = case["rows"] if kind == "mlp" else case["seqs"] * case["tokens"]
        s = dict(tok=_stream(g, rows, d), pos=_randn(g, d, std=0.02).half(), norm=_norm(g, d))
        if kind == "attn":
            s.update(qkv=_linear(g, 3 * d, d), proj=_linear(g, d, d), rope=_rope(case["tokens"]))
        else:
            s.update(fc1=_fc1(g, m), fc2=_linear(g, d, m["pad"]), mlp_norm=_norm(g, m["hidden"]))
        return s
    if kind == "letterbox":
        r = np.random.default_rng(seed)
        h, w = case["height"], case["width"]
        yy, xx = np.mgrid[0:h, 0:w].astype(np.float32)
        waves = [np.sin(xx / (17 + 9 * c) + r.uniform(0, 6)) * np.cos(yy / (23 + 5 * c)) for c in range(3)]
        img = 127 + 90 * np.stack(waves, -1)
        return dict(rgb=np.clip(img + r.normal(0, 12, (h, w, 1)), 0, 255).astype(np.uint8))
    if kind == "pool":
        cfg = HarukaConfig(img_size=14 * case["grid"], depth=1)
        return dict(cfg=cfg, state=_haruka_state(g, cfg), x=_stream(g, case["batch"] * cfg.tokens, cfg.dim))
    grid = case["grid"]
    img = torch.rand(case["batch"], 14 * grid, 14 * grid, 3, device=DEV, generator=g).mul_(2).sub_(1).half()
    cfg = Eva02Config(img_size=14 * grid, depth=2)
    return dict(cfg=cfg, state=_eva02_state(g, cfg), img=img)


def _put(sd, p, w):
    sd[p + ".qweight"], sd[p + ".wscale"], sd[p + ".bias"] = w


def _put_norm(sd, p, wb):
    sd[p + ".weight"], sd[p + ".bias"] = wb


def _eva02_state(g, cfg):
    d, m = cfg.dim, MODELS["eva02"]
    sd = {"patch_embed.weight": _randn(g, d, 588, std=0.06), "patch_embed.bias": _randn(g, d, std=0.02),
          "cls_token": _randn(g, d), "pos_embed": _randn(g, cfg.tokens, d, std=0.02),
          "head.weight": _randn(g, cfg.tags, d, std=0.05), "head.bias": _randn(g, cfg.tags, std=0.02)}
    _put_norm(sd, "norm", _norm(g, d))
    for i in range(cfg.depth):
        p = f"blocks.{i}."
        _put(sd, p + "attn.qkv", _linear(g, 3 * d, d))
        _put(sd, p + "attn.proj", _linear(g, d, d))
        _put(sd, p + "mlp.fc1", _fc1(g, m))
        _put(sd, p + "mlp.fc2", _linear(g, d, m["pad"]))
        for n, width in (("norm1", d), ("norm2", d), ("mlp.norm", m["hidden"])):
            _put_norm(sd, p + n, _norm(g, width))
    return sd


def _haruka_state(g, cfg):
    d, h, q, f = cfg.dim, cfg.hidden, cfg.leaves, cfg.leaf_dim
    sd = {"patch_w": _randn(g, d, 588, std=0.06 / 57.6), "patch_b": _randn(g, cfg.tokens - 1, d, std=0.02),
          "cls": _randn(g, 1, d), "pool.kv.weight": _randn(g, 2 * d, d, std=0.02),
          "pool.kv.bias": _randn(g, 2 * d, std=0.02), "pool.q_coarse": _randn(g, cfg.coarse, d),
          "pool.q_coarse_bias": -2.0 + _randn(g, cfg.coarse, std=0.1), "pool.q_child": _randn(g, q, d),
          "pool.q_child_bias": -2.0 + _randn(g, q, std=0.1), "pool.leaf.weight": _randn(g, q, d, f, std=0.02),
          "pool.leaf.bias": _randn(g, q, f, std=0.02), "head.weight": _randn(g, cfg.tags, q * f, std=0.05),
          "head.bias": _randn(g, cfg.tags, std=0.02)}
    for n in ("norm", "pool.norm", "pool.trunk_norm", "pool.child_q_norm", "pool.leaf_norm"):
        _put_norm(sd, n, _norm(g, d))
    for i in range(cfg.depth):
        p = f"blocks.{i}."
        _put(sd, p + "qkv", _linear(g, 3 * d, d))
        _put(sd, p + "proj", _linear(g, d, d))
        _put(sd, p + "fc1", _fc1(g, MODELS["haruka"]))
        _put(sd, p + "fc2", _linear(g, d, h))
        for n, width in (("norm1", d), ("norm2", d), ("mlp_norm", h)):
            _put_norm(sd, p + n, _norm(g, width))
    return sd


# ---- what a program holds before the call, and the call ----


def _captured(fn):
    """fn once on a side stream, then captured: a HIP graph and what fn returned in it."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        fn()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _empty(*shape, dtype=torch.half):
    return torch.empty(*shape, device=DEV, dtype=dtype)


@torch.no_grad()
def prepare(case, seed):
    kind, s, k = case["kind"], _inputs(case, seed), kernels()
    if kind == "linear":
        rows, width = s["x"].shape
        a8, rs = _empty(rows, width, dtype=torch.int8), _empty(rows, dtype=torch.float32)
        return dict(s, a8=a8, rs=rs, out=_empty(rows, case["cols"]))
    if kind == "scores":
        return dict(s, out=_empty(s["qkv"].shape[0], 64 * case["heads"]), tokens=case["tokens"])
    if kind == "letterbox":
        return dict(s, out=_empty(case["size"], case["size"], 3, dtype=torch.uint8))
    if kind == "call":
        eng = Eva02Int8(s["state"], s["cfg"], device=DEV)
        eng(s["img"])  # plans the batch size: buffers, tile variants, graph
        return dict(eng=eng, img=s["img"])
    if kind == "pool":
        eng, cfg = HarukaInt8(s["state"], s["cfg"], device=DEV), s["cfg"]
        x = s["x"].view(case["batch"], cfg.tokens, cfg.dim)
        graph, out = _captured(lambda: eng.pool_head(x))
        return dict(graph=graph, out=out, eng=eng, x=x)
    m = MODELS[case["model"]]
    rows, d = s["tok"].shape
    x, a8, rs = _empty(rows, d), _empty(rows, d, dtype=torch.int8), _empty(rows, dtype=torch.float32)
    o16, qkv = _empty(rows, d), _empty(rows, 3 * d)
    h16, h8 = _empty(rows, m["pad"]), _empty(rows, m["pad"], dtype=torch.int8)
    gm, bt = s["norm"]

    def rotate(src, norm):
        if d == 1024:
            k.rot_q8_1024(src, *(norm or (None, None)), a8, rs, m["eps"])
        elif norm:
            k.rot_q8_h128(src, a8, rs, *norm, d, m["eps"])
        else:
            k.rot_q8_h128(src, a8, rs)

    def linear(src, w, epi, out, rope=(None, None)):
        k.gemm_s8(src, w[0], rs, w[1], w[2], out, epi, 0, *rope, Q_SCALE)

    def attn():
        torch.add(s["tok"], s["pos"], out=x)  # the stem's sum of token and position
        rotate(x, (gm, bt))
        linear(a8, s["qkv"], EPI_QKV_ROPE, qkv, s["rope"])
        k.attention(qkv, o16, case["tokens"])
        rotate(o16, None)
        linear(a8, s["proj"], EPI_RESIDUAL, x)
        return x

    mn = pad_norm(*s["mlp_norm"], m["pad"]) if kind == "mlp" else None

    def mlp():
        torch.add(s["tok"], s["pos"], out=x)
        rotate(x, (gm, bt))
        linear(a8, s["fc1"], EPI_SWIGLU if m["act"] == "swiglu" else EPI_GELU_F16, h16)
        if m["mlp_norm"]:
            k.rot_q8_h128(h16, h8, rs, *mn, m["hidden"], m["eps"])
        else:
            k.rot_q8_h128(h16, h8, rs)
        linear(h8, s["fc2"], EPI_RESIDUAL, x)
        return x

    graph, out = _captured(attn if kind == "attn" else mlp)
    return dict(s, graph=graph, out=out, mn=mn, held=(x, a8, rs, o16, qkv, h16, h8))


@torch.no_grad()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "eng" in state:
        return state["eng"](state["img"])
    if "rgb" in state:
        letterbox_gpu(state["rgb"], state["out"].shape[0], state["out"])
        return state["out"]
    k, out = kernels(), state["out"]
    if "qkv" in state:
        k.attention(state["qkv"], out, state["tokens"])
        return out
    if state["x"].shape[1] == 1024:
        k.rot_q8_1024(state["x"], None, None, state["a8"], state["rs"])
    else:
        k.rot_q8_h128(state["x"], state["a8"], state["rs"])
    w = state["w"]
    k.gemm_s8(state["a8"], w[0], state["rs"], w[1], w[2], out, EPI_BIAS_F16, 0, None, None, 1.0)
    return out


# ---- work and tolerance ----


def _attn_work(rows, seqs_tokens, d):
    flops = 2 * rows * 4 * d * d + 4 * rows * seqs_tokens * d
    return rows * d * 4 + 4 * d * d, flops  # stream in and out in fp16, int8 weights


def _mlp_work(rows, m):
    d, h = m["dim"], m["hidden"]
    n1 = 2 * h if m["act"] == "swiglu" else h
    return rows * d * 4 + (n1 + h) * d, 2 * rows * d * (n1 + h)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, k, n = case["rows"], case["width"], case["cols"]
        return dict(bytes=2 * r * k + n * k + 8 * n + 2 * r * n, flops=2 * r * k * n)
    if kind == "scores":
        rows, c = case["seqs"] * case["tokens"], 64 * case["heads"]
        return dict(bytes=8 * rows * c, flops=4 * rows * case["tokens"] * c)
    if kind == "letterbox":
        h, w, n = case["height"], case["width"], case["size"]
        return dict(bytes=3 * (h * w + n * n), flops=0)
    if kind == "attn":
        b, f = _attn_work(case["seqs"] * case["tokens"], case["tokens"], MODELS[case["model"]]["dim"])
        return dict(bytes=b, flops=f)
    if kind == "mlp":
        b, f = _mlp_work(case["rows"], MODELS[case["model"]])
        return dict(bytes=b, flops=f)
    if kind == "pool":
        cfg = HarukaConfig(img_size=14 * case["grid"])
        rows, d, q, b = case["batch"] * cfg.tokens, cfg.dim, cfg.pool_heads * (cfg.coarse + cfg.leaves), case["batch"]
        width = cfg.leaves * cfg.leaf_dim
        return dict(bytes=2 * rows * d + 2 * cfg.tags * width + 4 * b * cfg.tags,
                    flops=4 * rows * d * q + 2 * b * cfg.tags * width)
    m, b, g = MODELS[case["model"]], case["batch"], case["grid"]
    tokens, d, tags = 1 + g * g, m["dim"], Eva02Config.tags
    rows = b * tokens
    (ab, af), (mb, mf) = _attn_work(rows, tokens, d), _mlp_work(rows, m)
    weights = ab + mb - 8 * rows * d  # the stream between the layers is not an input or output of the call
    return dict(bytes=2 * weights + 2 * b * 588 * g * g + 2 * (588 + tokens + tags) * d + 4 * b * tags,
                flops=2 * (af + mf) + 2 * rows * 588 * d + 2 * b * tags * d)


def tolerance(case):
    kind = case["kind"]
    if kind == "letterbox":
        return "exact"  # Pillow's fixed-point resize, to the byte
    if kind == "linear":
        return dict(rel=1e-3, max=2e-3)  # one rounding to fp16 of an exact integer product
    if kind == "scores":
        return dict(rel=1.2e-3, max=1e-2)  # fp16 weights and output, fp32 sums
    if kind == "pool":
        return dict(rel=4e-3, max=3e-2)  # a chain of fp16 products and norms
    if kind == "call":
        return dict(rel=3e-2, max=2e-1)  # four int8 layers: a last-bit change flips codes in all that follow
    # a last-bit change flips one code in some hundred by one step, then a product; the MLP's comes after two of them
    return dict(rel=1.2e-3, max=5e-2) if kind == "attn" else dict(rel=6e-3, max=1e-1)


# ---- the same in 64 bits, plain torch ----


def _ex_ln(x, w, b, eps):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * w.double() + b.double()


def _ex_rot(x, block):
    """Rows rotated by the block-diagonal normalized Hadamard matrix, then codes and scale per row."""
    r, c = x.shape
    v, half = x.reshape(r, c // block, block), 1
    while half < block:
        v = v.reshape(r, c // block, block // (2 * half), 2, half)
        v = torch.stack((v[..., 0, :] + v[..., 1, :], v[..., 0, :] - v[..., 1, :]), dim=-2)
        half *= 2
    v = v.reshape(r, c) / math.sqrt(block)
    scale = v.abs().amax(1).clamp_min(1e-12) / 127.0
    return torch.round(v / scale[:, None]).clamp_(-127, 127), scale


def _ex_linear(codes, scale, w):
    out = codes @ w[0].double().t()
    return out.mul_(scale[:, None]).mul_(w[1].double()).add_(w[2].double())


def _ex_attention(q, k, v, tokens, heads):
    """q (with the softmax scale), k, v [rows, C] -> [rows, C], a sequence at a time."""
    out = torch.empty_like(q)
    for a in range(0, q.shape[0], tokens):
        qs, ks, vs = (t[a : a + tokens].view(tokens, heads, 64).transpose(0, 1).contiguous() for t in (q, k, v))
        p = torch.softmax(torch.bmm(qs, ks.transpose(1, 2).contiguous()), -1)
        out[a : a + tokens] = torch.bmm(p, vs).transpose(0, 1).reshape(tokens, -1)
    return out


def _ex_attn(x, norm, eps, qkv_w, proj_w, rope, tokens, heads):
    rows, d = x.shape
    block = 1024 if d == 1024 else 128
    y = _ex_linear(*_ex_rot(_ex_ln(x, *norm, eps), block), qkv_w)
    co, si = (t.double().repeat(rows // tokens, 1)[:, None, :] for t in rope)

    def turn(t):
        a, b = t.view(rows, heads, 32, 2).unbind(-1)
        return torch.stack((a * co - b * si, a * si + b * co), -1).reshape(rows, d)

    o = _ex_attention(turn(y[:, :d]) * 0.125, turn(y[:, d : 2 * d]), y[:, 2 * d :], tokens, heads)
    return x + _ex_linear(*_ex_rot(o, block), proj_w)


def _ex_mlp(x, norm, eps, fc1, fc2, mlp_norm, m):
    y = _ex_linear(*_ex_rot(_ex_ln(x, *norm, eps), 1024 if m["dim"] == 1024 else 128), fc1)
    if m["act"] == "swiglu":
        h = y[:, 0::2] * torch.sigmoid(y[:, 0::2]) * y[:, 1::2]
    else:
        h = 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y**3)))
    if m["mlp_norm"]:
        n = m["hidden"]
        h = torch.cat([_ex_ln(h[:, :n], *mlp_norm, eps), torch.zeros_like(h[:, n:])], 1)
    return x + _ex_linear(*_ex_rot(h, 128), fc2)


def _ex_call(case, s):
    m, sd, b, g = MODELS[case["model"]], s["state"], case["batch"], case["grid"]
    d, eps, tokens = m["dim"], m["eps"], 1 + g * g
    half = lambda n: sd[n].half().double()  # noqa: E731  (what the stem and head hold in fp16)
    p = s["img"].double().view(b, g, 14, g, 14, 3).permute(0, 1, 3, 2, 4, 5).reshape(b, g * g, 588)
    x = p @ half("patch_embed.weight").t() + (sd["patch_embed.bias"] + sd["pos_embed"][1:]).double()
    x = torch.cat([(sd["cls_token"] + sd["pos_embed"][0]).double().expand(b, 1, d), x], 1).reshape(-1, d)
    for i in range(s["cfg"].depth):
        q = f"blocks.{i}."
        lw = lambda n: tuple(sd[q + n + f] for f in (".qweight", ".wscale", ".bias"))  # noqa: E731
        nw = lambda n: (sd[q + n + ".weight"], sd[q + n + ".bias"])  # noqa: E731
        x = _ex_attn(x, nw("norm1"), eps, lw("attn.qkv"), lw("attn.proj"), _rope(tokens), tokens, m["heads"])
        x = _ex_mlp(x, nw("norm2"), eps, lw("mlp.fc1"), lw("mlp.fc2"), nw("mlp.norm"), m)
    cls = _ex_ln(x.view(b, tokens, d)[:, 0], sd["norm.weight"], sd["norm.bias"], eps)
    return cls @ half("head.weight").t() + half("head.bias")


def _ex_pool(case, s):
    sd, cfg, b = s["state"], s["cfg"], case["batch"]
    d, hp, c, q, eps = cfg.dim, cfg.pool_heads, cfg.coarse, cfg.leaves, cfg.eps
    half = lambda n: sd[n].half().double()  # noqa: E731
    ln = lambda t, n: _ex_ln(t, half(n + ".weight"), half(n + ".bias"), eps)  # noqa: E731
    xn = ln(ln(s["x"].double().view(b, -1, d), "norm"), "pool.norm")
    kv = (xn @ sd["pool.kv.weight"].double().t() + sd["pool.kv.bias"].double()).view(b, -1, 2, hp, d // hp)
    key, val = kv.unbind(2)

    def attend(qs, bias):  # qs [b or 1, M, hp, e]
        lg = torch.einsum("bnhe,bmhe->bnhm", key, qs.expand(b, -1, -1, -1))
        w = torch.softmax(lg, -1) * torch.sigmoid(lg + bias.double())
        return w.sum(1).mean(1), torch.einsum("bnhm,bnhe->bmhe", w, val).reshape(b, -1, d)

    _, z = attend(sd["pool.q_coarse"].double().view(1, c, hp, -1), sd["pool.q_coarse_bias"])
    parent = ln(z, "pool.trunk_norm").repeat_interleave(q // c, 1)
    leafq = ln(parent + half("pool.q_child"), "pool.child_q_norm")
    mass, child = attend(leafq.view(b, q, hp, -1), sd["pool.q_child_bias"])
    z = ln(parent + child, "pool.leaf_norm") * (mass / (mass + 4.0))[..., None]
    leaf = torch.einsum("bqd,qdf->bqf", z, half("pool.leaf.weight")) + half("pool.leaf.bias")
    return leaf.reshape(b, -1) @ half("head.weight").t() + half("head.bias")


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "letterbox":
        return None  # bytes
    s = _inputs(case, seed)
    if kind == "linear":
        return _ex_linear(*_ex_rot(s["x"].double(), 1024 if case["width"] == 1024 else 128), s["w"])
    if kind == "scores":
        c, qkv = 64 * case["heads"], s["qkv"].double()
        q, k, v = qkv[:, :c] * math.log(2.0), qkv[:, c : 2 * c], qkv[:, 2 * c :]
        return _ex_attention(q, k, v, case["tokens"], case["heads"])
    if kind == "call":
        return _ex_call(case, s)
    if kind == "pool":
        return _ex_pool(case, s)
    m = MODELS[case["model"]]
    x = (s["tok"].double() + s["pos"].double()).half().double()
    if kind == "attn":
        return _ex_attn(x, s["norm"], m["eps"], s["qkv"], s["proj"], s["rope"], case["tokens"], m["heads"])
    return _ex_mlp(x, s["norm"], m["eps"], s["fc1"], s["fc2"], s["mlp_norm"], m)
