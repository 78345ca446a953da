"""The gfx950 kernel library behind a C ABI (include/foidfinder_rocm.h), loaded with ctypes and registered as
`torch.ops.foidfinder_rocm.*` with the reference's op schemas.

Mirrors foidfinder/backends/cuda/kernels.py:38-48 (`kernels()` -> the op namespace) and the op registration of
foidfinder/backends/cuda/csrc/kernels.cu:267-281. Every op is out-param / in-place, returns nothing, allocates
nothing and launches on the current stream, so a forward built from them can be captured in a HIP graph. Failed
preconditions raise RuntimeError, as TORCH_CHECK does in the reference.

There is no CPU fallback: without the built library every call raises.
"""

from __future__ import annotations

import ctypes
import os
from functools import cache
from pathlib import Path

import torch

LIB_PATH = Path(__file__).resolve().parent / "libfoidfinder_rocm.so"
ENV = "FOIDFINDER_ROCM_KERNELS"  # path to a prebuilt library (the reference's $FOIDFINDER_KERNELS)

# Epilogue codes (include/foidfinder_rocm.h); 0-2 as foidfinder/backends/cuda/engine.py:24.
EPI_QKV_ROPE, EPI_RESIDUAL, EPI_GELU_F16, EPI_SWIGLU, EPI_BIAS_F16, EPI_I32 = 0, 1, 2, 3, 4, 5

_vp, _i64, _f32, _int = ctypes.c_void_p, ctypes.c_int64, ctypes.c_float, ctypes.c_int
SIGNATURES = {
    "ff_abi_version": ([], _int),
    "ff_last_error": ([], ctypes.c_char_p),
    "ff_rot_q8_1024": ([_vp, _vp, _vp, _f32, _i64, _vp, _vp, _vp], _int),
    "ff_rot_q8_h128": ([_vp, _i64, _i64, _i64, _vp, _vp, _f32, _vp, _vp, _vp], _int),
    "ff_gemm_s8": ([_vp, _vp, _i64, _i64, _i64, _vp, _vp, _vp, _vp, _int, _int, _vp, _vp, _i64, _f32, _vp], _int),
    "ff_gemm_s8_variants": ([], _int),
    "ff_attention": ([_vp, _vp, _i64, _i64, _i64, _vp], _int),
    "ff_resample_u8": ([_vp, _i64, _i64, _int, _vp, _vp, _i64, _i64, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _vp],
                       _int),
    "ff_bicubic_taps": ([*[_i64] * 3, _vp, _vp, *[_i64] * 4, _vp, _vp, _i64, _vp], _int),
    "ff_layer_norm2": ([_vp, _i64, _i64, _vp, _vp, _vp, _vp, _f32, _vp, _vp], _int),
    "ff_slot_weights_blocks": ([_i64], _i64),
    "ff_slot_weights": ([_vp, _vp, _i64, _vp, _i64, _i64, _i64, _i64, _vp, _vp, _vp], _int),
    "ff_pool_weights_blocks": ([_i64], _i64),
    "ff_pool_weights": ([_vp, _vp, _i64, _vp, _i64, _vp, *[_i64] * 6, _vp, _vp, _vp], _int),
    "ff_pool_sum": ([_vp, _vp, *[_i64] * 5, _vp, _vp], _int),
    "ff_pool_values": ([_vp, _vp, _vp, _vp, *[_i64] * 5, _vp, _vp], _int),
    "ff_pool_queries": ([*[_vp] * 7, _f32, *[_i64] * 5, _vp, _vp, _vp, _vp], _int),
    "ff_pool_keys": ([_vp, _vp, _i64, _i64, _i64, _i64, _vp, _vp], _int),
    "ff_pool_tree": ([*[_vp] * 5, _i64, _f32, *[_i64] * 5, _vp, _vp], _int),
    "ff_pool_leaf": ([_vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp, _vp], _int),
    "ff_patch_embed": ([_vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp, _vp], _int),
    "ff_head": ([_vp, _i64, _vp, _vp, _f32, _vp, _vp, _i64, _i64, _i64, _vp, _vp], _int),
}
ABI_VERSION = 3


@cache
def lib() -> ctypes.CDLL:
    """The loaded C library. torch is imported first so the library binds to the HIP runtime torch already loaded."""
    path = Path(os.environ.get(ENV, LIB_PATH))
    if not path.exists():
        raise RuntimeError(f"{path} is missing: build it with `python -m foidfinder_amd.build`")
    handle = ctypes.CDLL(str(path))
    for name, (args, res) in SIGNATURES.items():
        fn = getattr(handle, name)
        fn.argtypes, fn.restype = args, res
    if handle.ff_abi_version() != ABI_VERSION:
        raise RuntimeError(f"{path}: ABI {handle.ff_abi_version()}, expected {ABI_VERSION}")
    return handle


def _check(status: int) -> None:
    if status != 0:
        raise RuntimeError(lib().ff_last_error().decode())


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def _run(name: str, dev: int, *args) -> None:
    """Calls a launching function of the library on device `dev`'s current stream, with that device current. A call is
    made of a few us of host work in all, so nothing is switched or built that is not needed: the device is entered only
    if it is not the current one already, and the stream comes as its raw handle."""
    fn = getattr(lib(), name)
    if torch.cuda.current_device() == dev:
        _check(fn(*args, torch._C._cuda_getCurrentRawStream(dev)))
        return
    with torch.cuda.device(dev):
        _check(fn(*args, torch._C._cuda_getCurrentRawStream(dev)))


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


def _on_gpu(*ts: torch.Tensor | None) -> int:
    """The device index of contiguous tensors that are all on one GPU."""
    dev = -1
    for t in ts:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("foidfinder_rocm ops take GPU tensors")
        if not t.is_contiguous():
            raise RuntimeError("foidfinder_rocm ops take contiguous tensors")
        d = t.get_device()
        if dev < 0:
            dev = d
        elif d != dev:
            raise RuntimeError("all tensors must be on one device")
    return dev


# ---- op implementations (raw; also callable directly, bypassing the dispatcher) ----


def rot_q8_1024(
    x: torch.Tensor,
    gamma: torch.Tensor | None,
    beta: torch.Tensor | None,
    out: torch.Tensor,
    row_scale: torch.Tensor,
    eps: float = 1e-5,
) -> None:
    """x fp16 [T, 1024] -> out int8 [T, 1024], row_scale fp32 [T]; LayerNorm(gamma, beta, eps) first if given."""
    dev = _on_gpu(x, gamma, beta, out, row_scale)
    _require(x.dim() == 2 and x.size(1) == 1024 and x.dtype == torch.float16, "x must be fp16 [T, 1024]")
    _require(out.dtype == torch.int8 and out.shape == x.shape, "out must be int8 [T, 1024]")
    _require(row_scale.dtype == torch.float32 and row_scale.numel() == x.size(0), "row_scale must be fp32 [T]")
    if gamma is not None:
        _require(beta is not None, "gamma and beta go together")
        _require(gamma.dtype == beta.dtype == torch.float32 and gamma.numel() == beta.numel() == 1024,
                 "gamma/beta must be fp32 [1024]")
    _run("ff_rot_q8_1024", dev, _ptr(x), _ptr(gamma), _ptr(beta), eps, x.size(0), _ptr(out), _ptr(row_scale))


def rot_q8_h128(
    x: torch.Tensor,
    out: torch.Tensor,
    row_scale: torch.Tensor,
    gamma: torch.Tensor | None = None,
    beta: torch.Tensor | None = None,
    c_real: int = 0,
    eps: float = 1e-6,
) -> None:
    """x fp16 [T, C] (C % 128 == 0) -> out int8 [T, C], row_scale fp32 [T]; LayerNorm over the first c_real columns
    (default: all) first if gamma is given. gamma/beta are fp32 [C] with zeros in columns >= c_real
    (`pad_norm` builds them)."""
    dev = _on_gpu(x, out, row_scale, gamma, beta)
    _require(x.dim() == 2 and x.dtype == torch.float16, "x must be fp16 [T, C]")
    _require(out.dtype == torch.int8 and out.shape == x.shape, "out must be int8 [T, C]")
    _require(row_scale.dtype == torch.float32 and row_scale.numel() == x.size(0), "row_scale must be fp32 [T]")
    C = x.size(1)
    cr = c_real or C
    if gamma is not None:
        _require(beta is not None, "gamma and beta go together")
        _require(gamma.dtype == beta.dtype == torch.float32 and gamma.numel() == beta.numel() == C,
                 "gamma/beta must be fp32 [C], zero past c_real")
    _run("ff_rot_q8_h128", dev, _ptr(x), x.size(0), C, cr, _ptr(gamma), _ptr(beta), eps, _ptr(out), _ptr(row_scale))


def pad_norm(weight: torch.Tensor, bias: torch.Tensor, C: int) -> tuple[torch.Tensor, torch.Tensor]:
    """LayerNorm gamma/beta over c_real columns -> fp32 [C] with zeros past c_real, as rot_q8_h128 takes them."""
    g = torch.zeros(C, dtype=torch.float32, device=weight.device)
    b = torch.zeros(C, dtype=torch.float32, device=weight.device)
    g[: weight.numel()] = weight.float().reshape(-1)
    b[: bias.numel()] = bias.float().reshape(-1)
    return g, b


def out_shape(M: int, N: int, epi: int) -> tuple[int, int]:
    return (M, N // 2) if epi == EPI_SWIGLU else (M, N)


def gemm_s8(
    A: torch.Tensor,
    W: torch.Tensor,
    row_scale: torch.Tensor,
    col_scale: torch.Tensor,
    bias: torch.Tensor,
    out: torch.Tensor,
    epi: int,
    stages: int,
    rope_cos: torch.Tensor | None,
    rope_sin: torch.Tensor | None,
    q_scale: float,
) -> None:
    """A int8 [M, K] x W int8 [N, K] -> epilogue into out. `stages` selects the tile variant (0 = default), the
    knob the engine autotunes (the reference's pipeline depth)."""
    dev = _on_gpu(A, W, row_scale, col_scale, bias, out, rope_cos, rope_sin)
    _require(A.dtype == W.dtype == torch.int8 and A.dim() == W.dim() == 2, "A and W must be int8 matrices")
    M, K = A.shape
    N = W.size(0)
    _require(W.size(1) == K, "A and W must share K")
    want = torch.int32 if epi == EPI_I32 else torch.float16
    shape = out_shape(M, N, epi)
    if out.dtype != want or tuple(out.shape) != shape:
        raise RuntimeError(f"out must be {want} {shape}")
    if epi != EPI_I32:
        _require(row_scale.dtype == col_scale.dtype == bias.dtype == torch.float32, "scales and bias must be fp32")
        _require(row_scale.numel() == M and col_scale.numel() == N and bias.numel() == N, "scale/bias sizes")
    rope_len = 0
    if epi == EPI_QKV_ROPE:
        _require(rope_cos is not None and rope_sin is not None, "QKV epilogue needs RoPE tables")
        _require(rope_cos.dtype == rope_sin.dtype == torch.float32 and rope_cos.shape == rope_sin.shape
                 and rope_cos.dim() == 2 and rope_cos.size(1) == 32, "RoPE tables must be fp32 [L, 32]")
        rope_len = rope_cos.size(0)
    _run("ff_gemm_s8", dev, _ptr(A), _ptr(W), M, N, K, _ptr(row_scale), _ptr(col_scale), _ptr(bias), _ptr(out), epi,
         stages, _ptr(rope_cos), _ptr(rope_sin), rope_len, q_scale)


def attention(qkv: torch.Tensor, out: torch.Tensor, seq_len: int) -> None:
    """qkv fp16 [T, 3C] (q rotated and pre-scaled, k rotated) -> out fp16 [T, C]; heads of 64, any seq_len."""
    dev = _on_gpu(qkv, out)
    _require(qkv.dtype == out.dtype == torch.float16, "qkv and out must be fp16")
    _require(qkv.dim() == 2 and qkv.size(1) % 192 == 0, "qkv must be [T, 3 * heads * 64]")
    C = qkv.size(1) // 3
    _require(out.shape == (qkv.size(0), C), "out must be [T, C]")
    _run("ff_attention", dev, _ptr(qkv), _ptr(out), qkv.size(0), C // 64, seq_len)


def resample_u8(src: torch.Tensor, axis: int, kk: torch.Tensor, bounds: torch.Tensor, row0: int, out: torch.Tensor,
                region: tuple[int, int, int, int]) -> None:
    """One Pillow resampling pass (include/foidfinder_rocm.h, ff_resample_u8): src uint8 [H, W, 3] -> out uint8
    [out_h, out_w, 3], `region` = (top, left, h, w) resampled along axis 0 (width) or 1 (height), the rest white."""
    dev = _on_gpu(src, kk, bounds, out)
    _require(src.dtype == out.dtype == torch.uint8 and src.dim() == out.dim() == 3 and src.size(2) == out.size(2) == 3,
             "src and out must be uint8 [rows, cols, 3]")
    _require(src.is_contiguous() and out.is_contiguous(), "src and out must be contiguous")
    _require(kk.dtype == bounds.dtype == torch.int32 and kk.dim() == 2 and bounds.dim() == 2 and bounds.size(1) == 2
             and kk.is_contiguous() and bounds.is_contiguous(), "kk int32 [n, ksize], bounds int32 [n, 2]")
    top, left, h, w = region
    n = w if axis == 0 else h
    _require(kk.size(0) >= n and bounds.size(0) >= n, "kk/bounds need a row per output index of the region")
    _run("ff_resample_u8", dev, _ptr(src), src.size(0), src.size(1), axis, _ptr(kk), _ptr(bounds), kk.size(1), row0,
         _ptr(out), out.size(0), out.size(1), top, left, h, w)


def bicubic_taps(width: tuple[int, int, int], height: tuple[int, int, int], kk_w: torch.Tensor, bounds_w: torch.Tensor,
                 kk_h: torch.Tensor, bounds_h: torch.Tensor) -> None:
    """Pillow's bicubic taps of both axes (include/foidfinder_rocm.h, ff_bicubic_taps): `width` and `height` are (input
    size, output size, shift); kk int32 [output size, ksize], bounds int32 [output size, 2]."""
    dev = _on_gpu(kk_w, bounds_w, kk_h, bounds_h)
    for (_, n, _), kk, bounds in ((width, kk_w, bounds_w), (height, kk_h, bounds_h)):
        _require(kk.dtype == bounds.dtype == torch.int32 and kk.dim() == 2 and kk.size(0) == n
                 and tuple(bounds.shape) == (n, 2), "kk int32 [n, ksize], bounds int32 [n, 2]")
    _run("ff_bicubic_taps", dev, width[0], width[1], kk_w.size(1), _ptr(kk_w), _ptr(bounds_w), width[2], height[0],
         height[1], kk_h.size(1), _ptr(kk_h), _ptr(bounds_h), height[2])


def layer_norm2(x: torch.Tensor, g1: torch.Tensor, b1: torch.Tensor, g2: torch.Tensor, b2: torch.Tensor, eps: float,
                out: torch.Tensor) -> None:
    """out = LN(fp16(LN(x; g1, b1)); g2, b2) over the last dimension of fp16 x [..., C] (fp16 params [C])."""
    dev = _on_gpu(x, g1, b1, g2, b2, out)
    C = x.size(-1)
    _require(x.dtype == out.dtype == torch.float16 and x.is_contiguous() and out.is_contiguous()
             and out.shape == x.shape, "x and out must be contiguous fp16 of one shape")
    _require(all(t.dtype == torch.float16 and t.numel() == C for t in (g1, b1, g2, b2)), "params must be fp16 [C]")
    _run("ff_layer_norm2", dev, _ptr(x), x.numel() // C, C, _ptr(g1), _ptr(b1), _ptr(g2), _ptr(b2), eps, _ptr(out))


def slot_weights_blocks(N: int) -> int:
    return lib().ff_slot_weights_blocks(N)


def slot_weights(logits: torch.Tensor, c: torch.Tensor, bias: torch.Tensor, heads: int, a_t: torch.Tensor,
                 partial: torch.Tensor) -> None:
    """Tree-pool weights (include/foidfinder_rocm.h, ff_slot_weights): logits fp16 [B, N, heads*M] + c fp32 ([heads*M]
    shared or [B, heads*M]) -> a_t fp16 [B, heads*M, N], partial fp32 [B, blocks, heads*M]."""
    dev = _on_gpu(logits, c, bias, a_t, partial)
    B, N, GM = logits.shape
    M = bias.numel()
    _require(logits.dtype == torch.float16 and logits.is_contiguous() and GM == heads * M, "logits fp16 [B, N, heads*M]")
    _require(c.dtype == bias.dtype == torch.float32 and c.is_contiguous() and bias.is_contiguous(), "c, bias fp32")
    _require(c.numel() in (GM, B * GM), "c must be [heads*M] or [B, heads*M]")
    _require(a_t.dtype == torch.float16 and a_t.is_contiguous() and a_t.shape == (B, GM, N), "a_t fp16 [B, heads*M, N]")
    _require(partial.dtype == torch.float32 and partial.is_contiguous()
             and partial.shape == (B, slot_weights_blocks(N), GM), "partial fp32 [B, blocks, heads*M]")
    _run("ff_slot_weights", dev, _ptr(logits), _ptr(c), 0 if c.numel() == GM else GM, _ptr(bias), B, N, heads, M,
         _ptr(a_t), _ptr(partial))


def pool_weights_blocks(N: int) -> int:
    return lib().ff_pool_weights_blocks(N)


def pool_fits(B: int, N: int, heads: int, leaves: int, dim: int) -> bool:
    """Whether the tree pool's kernels take B images of N tokens (others go to the library's products): 32-bit byte
    offsets within an image's tokens and weights (rows padded to 8 tokens), and at most 65535 launch rows of images and of
    16 (image, leaf) pairs each."""
    ldt = (N + 7) // 8 * 8
    return N * dim < 1 << 30 and heads * leaves * ldt < 1 << 30 and B <= 65535 and B * leaves <= 16 * 65535


def _half(shape: tuple, *ts: torch.Tensor) -> None:
    for t in ts:
        if t.dtype != torch.float16 or tuple(t.shape) != shape:
            raise RuntimeError(f"need fp16 {shape}")


def _float(numel: int, *ts: torch.Tensor) -> None:
    for t in ts:
        if t.dtype != torch.float32 or t.numel() != numel:
            raise RuntimeError(f"need fp32 of {numel} elements")


def pool_weights(xn: torch.Tensor, u: torch.Tensor, c: torch.Tensor, bias: torch.Tensor, heads: int, a_t: torch.Tensor,
                 partial: torch.Tensor) -> None:
    """Tree-pool weights from the tokens and the queries' u (include/foidfinder_rocm.h, ff_pool_weights): xn fp16
    [B, N, D], u fp16 [heads*M, D] (shared) or [B, heads*M, D], c fp32 [heads*M] or [B, heads*M], bias fp32 [M] -> a_t
    fp16 [B, heads*M, ldt], partial fp32 [B, blocks, heads*M]."""
    dev = _on_gpu(xn, u, c, bias, a_t, partial)
    B, N, D = xn.shape
    M = bias.numel()
    GM = heads * M
    _require(xn.dtype == torch.float16 and u.dtype == torch.float16 and tuple(u.shape[-2:]) == (GM, D)
             and (u.dim() == 2 or u.dim() == 3 and u.size(0) == B), "u must be fp16 [heads*M, D] or [B, heads*M, D]")
    _require(c.dtype == bias.dtype == torch.float32 and c.numel() in (GM, B * GM), "c must be fp32 [heads*M] or [B, heads*M]")
    _half((B, GM, a_t.size(-1)), a_t)
    _float(B * pool_weights_blocks(N) * GM, partial)
    _run("ff_pool_weights", dev, _ptr(xn), _ptr(u), 0 if u.dim() == 2 else GM * D, _ptr(c), 0 if c.numel() == GM else
         GM, _ptr(bias), B, N, heads, M, D, a_t.size(-1), _ptr(a_t), _ptr(partial))


def pool_sum(a_t: torch.Tensor, xn: torch.Tensor, pooled: torch.Tensor) -> None:
    """pooled fp16 [B, GM, D] = a_t xn over the N tokens of xn fp16 [B, N, D], a_t fp16 [B, GM, ldt] as pool_weights leaves
    it (ff_pool_sum)."""
    dev = _on_gpu(a_t, xn, pooled)
    B, N, D = xn.shape
    GM = a_t.size(1)
    _half((B, N, D), xn)
    _half((B, GM, a_t.size(-1)), a_t)
    _half((B, GM, D), pooled)
    _run("ff_pool_sum", dev, _ptr(a_t), _ptr(xn), B, N, GM, D, a_t.size(-1), _ptr(pooled))


def pool_values(pooled: torch.Tensor, wv: torch.Tensor, bv: torch.Tensor, partial: torch.Tensor, heads: int,
                z: torch.Tensor) -> None:
    """z fp16 [B, M, D] from pooled fp16 [B, heads*M, D], wv fp16 [D, D], bv fp32 [D] and the weights' partial sums."""
    dev = _on_gpu(pooled, wv, bv, partial, z)
    B, M, D = z.shape
    _half((B, M, D), z)
    _half((B, heads * M, D), pooled)
    _half((D, D), wv)
    _float(D, bv)
    _float(B * partial.size(1) * heads * M, partial)
    _run("ff_pool_values", dev, _ptr(pooled), _ptr(wv), _ptr(bv), _ptr(partial), partial.size(1), B, heads, M, D,
         _ptr(z))


def pool_queries(z: torch.Tensor, trunk_g: torch.Tensor, trunk_b: torch.Tensor, child: torch.Tensor,
                 child_g: torch.Tensor, child_b: torch.Tensor, bk: torch.Tensor, heads: int, eps: float,
                 parent: torch.Tensor, qleaf: torch.Tensor, cq: torch.Tensor) -> None:
    """z fp16 [B, C, D] -> parent fp16 [B, C, D], qleaf fp16 [B, Q, D], cq fp32 [B, heads*Q] (ff_pool_queries)."""
    dev = _on_gpu(z, trunk_g, trunk_b, child, child_g, child_b, bk, parent, qleaf, cq)
    B, C, D = z.shape
    Q = child.size(0)
    _half((B, C, D), z, parent)
    _half((B, Q, D), qleaf)
    _half((Q, D), child)
    _half((D,), trunk_g, trunk_b, child_g, child_b)
    _float(D, bk)
    _float(B * heads * Q, cq)
    _run("ff_pool_queries", dev, _ptr(z), _ptr(trunk_g), _ptr(trunk_b), _ptr(child), _ptr(child_g), _ptr(child_b),
         _ptr(bk), eps, B, C, Q, heads, D, _ptr(parent), _ptr(qleaf), _ptr(cq))


def pool_keys(qleaf: torch.Tensor, kT: torch.Tensor, u: torch.Tensor) -> None:
    """u fp16 [B, heads*Q, D] from qleaf fp16 [B, Q, D] and kT fp16 [heads, D, D / heads] (ff_pool_keys)."""
    dev = _on_gpu(qleaf, kT, u)
    B, Q, D = qleaf.shape
    heads = kT.size(0)
    _half((B, Q, D), qleaf)
    _half((heads, D, D // heads), kT)
    _half((B, heads * Q, D), u)
    _run("ff_pool_keys", dev, _ptr(qleaf), _ptr(kT), B, Q, heads, D, _ptr(u))


def pool_tree(parent: torch.Tensor, zc: torch.Tensor, g: torch.Tensor, b: torch.Tensor, partial: torch.Tensor,
              heads: int, eps: float, tree: torch.Tensor) -> None:
    """tree fp16 [Q, B, D] from parent fp16 [B, C, D], zc fp16 [B, Q, D] and the weights' partial sums (ff_pool_tree)."""
    dev = _on_gpu(parent, zc, g, b, partial, tree)
    B, Q, D = zc.shape
    _half((B, parent.size(1), D), parent)
    _half((B, Q, D), zc)
    _half((D,), g, b)
    _half((Q, B, D), tree)
    _float(B * partial.size(1) * heads * Q, partial)
    _run("ff_pool_tree", dev, _ptr(parent), _ptr(zc), _ptr(g), _ptr(b), _ptr(partial), partial.size(1), eps, B,
         parent.size(1), Q, heads, D, _ptr(tree))


def pool_leaf(tree: torch.Tensor, wl: torch.Tensor, bl: torch.Tensor, leaf: torch.Tensor) -> None:
    """leaf fp16 [B, Q*F] from tree fp16 [Q, B, D], wl fp16 [Q, F, D], bl fp16 [Q, F] (ff_pool_leaf)."""
    dev = _on_gpu(tree, wl, bl, leaf)
    Q, B, D = tree.shape
    F = wl.size(1)
    _half((Q, B, D), tree)
    _half((Q, F, D), wl)
    _half((Q, F), bl)
    _half((B, Q * F), leaf)
    _run("ff_pool_leaf", dev, _ptr(tree), _ptr(wl), _ptr(bl), B, Q, F, D, _ptr(leaf))


PATCH_COLS, PATCH_PAD = 588, 608  # 14 x 14 x 3, and the row length of patch_embed's weights


def pad_patch_weight(w: torch.Tensor) -> torch.Tensor:
    """Patch weights [N, 588] -> fp16 [N, 608] with zeros past column 588, as patch_embed takes them."""
    out = torch.zeros(w.size(0), PATCH_PAD, dtype=torch.half, device=w.device)
    out[:, :PATCH_COLS] = w
    return out


def patch_embed(img: torch.Tensor, w: torch.Tensor, bias_pos: torch.Tensor, cls: torch.Tensor, x: torch.Tensor) -> None:
    """x fp16 [B, 1 + grid^2, N]: the class row, then each 14 x 14 patch of img fp16 [B, S, S, 3] times w fp16 [N, 608]
    (pad_patch_weight) plus bias_pos fp16 [grid^2, N] (ff_patch_embed)."""
    dev = _on_gpu(img, w, bias_pos, cls, x)
    B, S = img.shape[:2]
    grid, N = S // 14, w.size(0)
    _half((B, grid * 14, grid * 14, 3), img)
    _half((N, PATCH_PAD), w)
    _half((grid * grid, N), bias_pos)
    _half((N,), cls)
    _half((B, 1 + grid * grid, N), x)
    _run("ff_patch_embed", dev, _ptr(img), _ptr(w), _ptr(bias_pos), _ptr(cls), B, grid, N, _ptr(x))


def head_fits(x: torch.Tensor, W: torch.Tensor) -> bool:
    """Whether `head` takes the rows x with W [N, K] (others go to the library's GEMM): up to 64 rows, and fp16, which a
    library product under autocast need not have left."""
    return x.size(0) <= 64 and x.dtype == torch.float16 and W.size(1) % 32 == 0 and W.size(1) <= 1280


def unfollowed(x: torch.Tensor) -> bool:
    """Whether x is a plain GPU tensor that nothing follows, so that an op here can take the place of a torch product: these
    ops go by addresses, past autograd (backward and forward), functorch's transforms, tracing and dispatch modes."""
    return (type(x) is torch.Tensor and x.is_cuda and not (x.requires_grad and torch.is_grad_enabled())
            and torch.autograd.forward_ad._current_level < 0 and not torch._C._functorch.is_functorch_wrapped_tensor(x)
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling()
            and torch._C._len_torch_dispatch_stack() == 0)


def head(x: torch.Tensor, W: torch.Tensor, bias: torch.Tensor, out: torch.Tensor, gamma: torch.Tensor | None = None,
         beta: torch.Tensor | None = None, eps: float = 1e-6) -> None:
    """Tag head: out fp32 [B, N] = LN(x) W^T + bias, x fp16 [B, K] with contiguous rows (any row stride from K up that is
    a multiple of 8; rows that overlap are refused), W fp16 [N, K], bias fp16 [N]; the norm (fp32 gamma, beta [K]) only if
    given (ff_head)."""
    dev = _on_gpu(W, bias, out, gamma, beta)
    B, K = x.shape
    N = W.size(0)
    _require(x.device == W.device and x.dtype == torch.float16 and x.stride(1) == 1, "x must be fp16 rows on W's device")
    _half((N, K), W)
    _half((N,), bias)
    _require(out.dtype == torch.float32 and tuple(out.shape) == (B, N), "out must be fp32 [B, N]")
    if gamma is not None:
        _require(beta is not None, "gamma and beta go together")
        _float(K, gamma, beta)
    stride = x.stride(0) if B > 1 else K  # a single row's stride says nothing
    _run("ff_head", dev, _ptr(x), stride, _ptr(gamma), _ptr(beta), eps, _ptr(W), _ptr(bias), B, N, K,
         _ptr(out))


# ---- torch.ops.foidfinder_rocm registration (schemas as kernels.cu:268-273, plus eps / the fused norm) ----

_LIB = torch.library.Library("foidfinder_rocm", "DEF")
_LIB.define(
    "gemm_s8(Tensor A, Tensor W, Tensor row_scale, Tensor col_scale, Tensor bias, Tensor(a!) out, int epi, "
    "int stages, Tensor? rope_cos, Tensor? rope_sin, float q_scale) -> ()"
)
_LIB.define("rot_q8_1024(Tensor x, Tensor? gamma, Tensor? beta, Tensor(a!) out, Tensor(b!) row_scale, "
            "float eps=1e-05) -> ()")
_LIB.define("rot_q8_h128(Tensor x, Tensor(a!) out, Tensor(b!) row_scale, Tensor? gamma=None, Tensor? beta=None, "
            "int c_real=0, float eps=1e-06) -> ()")
_LIB.define("attention(Tensor qkv, Tensor(a!) out, int seq_len) -> ()")
_LIB.impl("gemm_s8", gemm_s8, "CUDA")
_LIB.impl("rot_q8_1024", rot_q8_1024, "CUDA")
_LIB.impl("rot_q8_h128", rot_q8_h128, "CUDA")
_LIB.impl("attention", attention, "CUDA")
# Haruka's tree pool (no reference CUDA op; out-param ops in the same style)
_LIB.define("layer_norm2(Tensor x, Tensor g1, Tensor b1, Tensor g2, Tensor b2, float eps, Tensor(a!) out) -> ()")
_LIB.define("slot_weights(Tensor logits, Tensor c, Tensor bias, int heads, Tensor(a!) a_t, Tensor(b!) partial) -> ()")
_LIB.define("pool_weights(Tensor xn, Tensor u, Tensor c, Tensor bias, int heads, Tensor(a!) a_t, Tensor(b!) partial) "
            "-> ()")
_LIB.define("pool_sum(Tensor a_t, Tensor xn, Tensor(a!) pooled) -> ()")
_LIB.define("pool_values(Tensor pooled, Tensor wv, Tensor bv, Tensor partial, int heads, Tensor(a!) z) -> ()")
_LIB.define("pool_queries(Tensor z, Tensor trunk_g, Tensor trunk_b, Tensor child, Tensor child_g, Tensor child_b, "
            "Tensor bk, int heads, float eps, Tensor(a!) parent, Tensor(b!) qleaf, Tensor(c!) cq) -> ()")
_LIB.define("pool_keys(Tensor qleaf, Tensor kT, Tensor(a!) u) -> ()")
_LIB.define("pool_tree(Tensor parent, Tensor zc, Tensor g, Tensor b, Tensor partial, int heads, float eps, "
            "Tensor(a!) tree) -> ()")
_LIB.define("pool_leaf(Tensor tree, Tensor wl, Tensor bl, Tensor(a!) leaf) -> ()")
_LIB.define("patch_embed(Tensor img, Tensor w, Tensor bias_pos, Tensor cls, Tensor(a!) x) -> ()")
_LIB.define("head(Tensor x, Tensor W, Tensor bias, Tensor(a!) out, Tensor? gamma=None, Tensor? beta=None, "
            "float eps=1e-06) -> ()")
for _fn in (pool_weights, pool_sum, pool_values, pool_queries, pool_keys, pool_tree, pool_leaf, patch_embed, head):
    _LIB.impl(_fn.__name__, _fn, "CUDA")
_LIB.impl("layer_norm2", layer_norm2, "CUDA")
_LIB.impl("slot_weights", slot_weights, "CUDA")


@cache
def kernels():
    """The op namespace, loading the library (raises if it is missing). Mirrors the reference's `kernels()`."""
    lib()
    return torch.ops.foidfinder_rocm
