"""The C-ABI library without a GPU: it loads, exports every symbol include/foidfinder_rocm.h declares, and rejects
bad arguments with FF_EINVAL and a message before any HIP call (the reference raises RuntimeError via TORCH_CHECK
for the same preconditions, foidfinder/backends/cuda/csrc/kernels.cu:190-205, :222, :240, :257-258)."""

from __future__ import annotations

import re
from pathlib import Path

import pytest
import torch

from foidfinder_amd import kernels as K

HEADER = Path(__file__).resolve().parents[1] / "include" / "foidfinder_rocm.h"
FF_OK, FF_EINVAL = 0, 1


def declared() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return re.findall(r"\b(ff_\w+)\s*\(", text)


def test_library_exports_every_declared_symbol():
    names = declared()
    assert {"ff_rot_q8_1024", "ff_rot_q8_h128", "ff_gemm_s8", "ff_attention", "ff_last_error"} <= set(names)
    lib = K.lib()
    for n in names:
        assert hasattr(lib, n), n
    assert set(names) == set(K.SIGNATURES), "ctypes signatures must cover the header exactly"


def test_abi_version_and_variants():
    lib = K.lib()
    assert lib.ff_abi_version() == K.ABI_VERSION
    assert lib.ff_gemm_s8_variants() >= 1


def err(status):
    return status, K.lib().ff_last_error().decode()


def test_rot_q8_1024_rejects_bad_arguments():
    lib = K.lib()
    assert err(lib.ff_rot_q8_1024(None, None, None, 1e-5, -1, None, None, None)) == (FF_EINVAL, "rot_q8_1024: T must be >= 0")
    assert lib.ff_rot_q8_1024(None, None, None, 1e-5, 0, None, None, None) == FF_OK  # empty input: nothing to do
    assert err(lib.ff_rot_q8_1024(None, None, None, 1e-5, 4, None, None, None))[0] == FF_EINVAL
    s, m = err(lib.ff_rot_q8_1024(16, 16, None, 1e-5, 4, 16, 16, None))
    assert s == FF_EINVAL and "gamma and beta" in m
    s, m = err(lib.ff_rot_q8_1024(16, 16, 16, 0.0, 4, 16, 16, None))
    assert s == FF_EINVAL and "eps" in m
    s, m = err(lib.ff_rot_q8_1024(18, None, None, 1e-5, 4, 16, 16, None))
    assert s == FF_EINVAL and "misaligned" in m


def test_rot_q8_h128_rejects_bad_arguments():
    lib = K.lib()
    for C in (0, 100, 6272):
        s, m = err(lib.ff_rot_q8_h128(16, 4, C, 0, None, None, 0.0, 16, 16, None))
        assert s == FF_EINVAL and "C" in m
    s, m = err(lib.ff_rot_q8_h128(16, 4, 256, 300, 16, 16, 1e-6, 16, 16, None))
    assert s == FF_EINVAL and "c_real" in m


def test_gemm_s8_rejects_bad_arguments():
    lib = K.lib()

    def call(M=8, N=16, Kd=64, epi=4, variant=0, rope=(None, None, 0), ptrs=256):
        return err(lib.ff_gemm_s8(ptrs, ptrs, M, N, Kd, ptrs, ptrs, ptrs, ptrs, epi, variant, rope[0], rope[1], rope[2],
                                  1.0, None))

    assert call(Kd=100)[1] == "gemm_s8: K must be a multiple of 64"
    assert call(N=40)[1] == "gemm_s8: N must be a multiple of 16"
    assert "epilogue" in call(epi=9)[1]
    assert "variant" in call(variant=99)[1]
    assert "QKV" in call(N=48, epi=0)[1]  # N = 3C needs C % 64 == 0
    assert "RoPE" in call(N=192, epi=0)[1]
    assert "rope_len" in call(N=192, epi=0, rope=(256, 256, 1 << 24))[1]  # table bytes must fit 31 bits
    assert "rope_len" not in call(N=192, epi=0, rope=(256, 256, (1 << 24) - 1), ptrs=8)[1]  # largest accepted
    assert call(M=0) == (FF_OK, "")
    assert "misaligned" in call(ptrs=8)[1]
    assert "not supported" in call(Kd=(1 << 22) + 64)[1]  # 32-bit offsets within a tile
    assert "not supported" in call(N=(1 << 21) + 16)[1]


def test_attention_rejects_bad_arguments():
    lib = K.lib()
    assert "multiple of seq_len" in err(lib.ff_attention(16, 16, 10, 16, 3, None))[1]
    assert "heads" in err(lib.ff_attention(16, 16, 10, 0, 5, None))[1]
    assert "seq_len" in err(lib.ff_attention(16, 16, 10, 16, 0, None))[1]
    assert lib.ff_attention(None, None, 0, 16, 5, None) == FF_OK


def test_python_ops_refuse_cpu_tensors():
    x = torch.zeros(4, 1024, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="GPU tensors"):
        K.rot_q8_1024(x, None, None, torch.zeros(4, 1024, dtype=torch.int8), torch.zeros(4), 1e-5)
    with pytest.raises((RuntimeError, NotImplementedError)):  # no CPU kernel is registered for the op
        torch.ops.foidfinder_rocm.attention(torch.zeros(5, 192, dtype=torch.float16), torch.zeros(5, 64, dtype=torch.float16), 5)


def test_op_schemas_mirror_the_reference():
    ops = K.kernels()
    schema = str(ops.gemm_s8.default._schema)
    assert "Tensor(a!) out, int epi, int stages, Tensor? rope_cos, Tensor? rope_sin, float q_scale" in schema
    assert "Tensor(a!) out, Tensor(b!) row_scale" in str(ops.rot_q8_1024.default._schema)
    assert "attention(Tensor qkv, Tensor(a!) out, int seq_len)" in str(ops.attention.default._schema)


def test_resample_u8_rejects_bad_arguments():
    lib = K.lib()

    def call(src=(100, 80), axis=0, ksize=5, row0=0, out=(448, 448), region=(0, 0, 100, 40), ptrs=256):
        top, left, h, w = region
        return err(lib.ff_resample_u8(ptrs, src[0], src[1], axis, ptrs, ptrs, ksize, row0, ptrs, out[0], out[1], top,
                                      left, h, w, None))

    assert "axis" in call(axis=2)[1]
    assert "positive" in call(ksize=0)[1]
    assert "positive" in call(region=(0, 0, 0, 40))[1]
    assert "inside the output" in call(region=(400, 0, 100, 40))[1]
    assert "inside the output" in call(region=(0, -1, 10, 40))[1]
    assert "outside the source" in call(row0=1)[1]  # axis 0 reads rows row0 .. row0 + h - 1 of 100
    assert "outside the source" in call(axis=1, region=(0, 0, 10, 81))[1]  # axis 1 reads columns 0 .. w - 1 of 80
    assert "65535" in call(src=(70000, 3))[1]
    assert "null" in call(ptrs=None)[1]


def test_pool_kernels_reject_bad_arguments():
    lib = K.lib()
    assert "C <= 2048" in err(lib.ff_layer_norm2(256, 4, 100, 256, 256, 256, 256, 1e-6, 256, None))[1]
    assert "eps" in err(lib.ff_layer_norm2(256, 4, 768, 256, 256, 256, 256, 0.0, 256, None))[1]
    assert lib.ff_layer_norm2(None, 0, 768, None, None, None, None, 1e-6, None, None) == FF_OK
    assert lib.ff_slot_weights_blocks(1025) == 33 and lib.ff_slot_weights_blocks(0) == 0

    def sw(B=2, N=1025, G=16, M=18, c_stride=0, ptrs=256):
        return err(lib.ff_slot_weights(ptrs, ptrs, c_stride, ptrs, B, N, G, M, ptrs, ptrs, None))

    assert "M must be 6 or 18" in sw(M=7)[1]
    assert "bad B, N or G" in sw(N=0)[1]
    assert "c_stride" in sw(c_stride=5)[1]
    assert "LDS" in sw(G=64)[1]
    assert "null" in sw(ptrs=None)[1]
    assert sw(B=0) == (FF_OK, "")


def test_head_hands_the_row_stride_of_several_rows_to_the_library(monkeypatch):
    """Rows closer than K (an expanded or overlapping view) must reach ff_head's own check as they are: with any larger
    stride the kernel would read rows that the tensor does not hold. One row's stride is never used."""
    strides = []
    monkeypatch.setattr(K, "_on_gpu", lambda *ts: 0)
    monkeypatch.setattr(K, "_run", lambda name, dev, x, x_stride, *rest: strides.append(x_stride))
    w, b = torch.zeros(48, 64, dtype=torch.half), torch.zeros(48, dtype=torch.half)
    flat = torch.zeros(1000, dtype=torch.half)
    for x in (flat[:64].expand(16, 64), flat.as_strided((3, 64), (8, 1)), flat.as_strided((3, 64), (72, 1)),
              flat.as_strided((3, 64), (67, 1)), flat.as_strided((1, 64), (3, 1)), flat[:0].view(0, 64)):
        K.head(x, w, b, torch.zeros(x.size(0), 48))
    assert strides == [0, 8, 72, 67, 64, 64]
    for s in (0, 8, 67):
        status, msg = err(K.lib().ff_head(256, s, None, None, 1e-6, 256, 256, 3, 48, 64, 256, None))
        assert status == FF_EINVAL and "x_stride" in msg


OK_OR_NULL = "null pointer"  # with null operands, the last check of an entry whose sizes are all accepted


def tree_pool_calls(B=2, N=1025, G=16, C=6, Q=18, D=768, F=64, ptrs=None):
    """Every tree-pool entry as HarukaInt8._pool_leaves calls it, at these sizes: (name, (status, message))."""
    lib, p = K.lib(), ptrs
    ldt, nblk = (N + 7) // 8 * 8, lib.ff_pool_weights_blocks(N)
    for M in (C, Q):
        yield "weights", err(lib.ff_pool_weights(p, p, 0 if M == C else G * M * D, p, 0 if M == C else G * M, p, B, N, G, M, D,
                                                 ldt, p, p, None))
        yield "sum", err(lib.ff_pool_sum(p, p, B, N, G * M, D, ldt, p, None))
        yield "values", err(lib.ff_pool_values(p, p, p, p, nblk, B, G, M, D, p, None))
    yield "queries", err(lib.ff_pool_queries(p, p, p, p, p, p, p, 1e-6, B, C, Q, G, D, p, p, p, None))
    yield "keys", err(lib.ff_pool_keys(p, p, B, Q, G, D, p, None))
    yield "tree", err(lib.ff_pool_tree(p, p, p, p, p, nblk, 1e-6, B, C, Q, G, D, p, None))
    yield "leaf", err(lib.ff_pool_leaf(p, p, p, B, Q, F, D, p, None))


@pytest.mark.parametrize(("G", "C", "Q", "D"), [(16, 6, 18, 768), (8, 6, 18, 128), (20, 6, 18, 640), (64, 6, 6, 1024),
                                                (16, 6, 18, 2048), (2, 18, 18, 128)])
def test_pool_fits_takes_what_every_tree_pool_kernel_takes(G, C, Q, D):
    """pool_fits decides between the kernels and the library's products: at each limit of images and tokens, and on either
    side of it, it says what the entries say."""
    tokens, weights, pairs = (1 << 30) // D, (1 << 30) // (G * Q), 16 * 65535 // Q
    sizes = [(1, 1), (2, 1025), (65535, 2), (65536, 2)]
    sizes += [(1, n + d) for n in (tokens, weights) for d in (-9, -8, -7, -1, 0, 1, 7, 8, 9)]
    sizes += [(b, 2) for b in (pairs - 1, pairs, pairs + 1)]
    seen = set()
    for B, N in sizes:
        refused = [(n, m) for n, (s, m) in tree_pool_calls(B, N, G, C, Q, D) if OK_OR_NULL not in m]
        assert K.pool_fits(B, N, G, Q, D) == (not refused), (B, N, refused)
        seen.add(not refused)
    assert seen == {True, False}


def test_tree_pool_rejects_bad_arguments():
    for name, (s, m) in tree_pool_calls():
        assert s == FF_EINVAL and OK_OR_NULL in m, name
    for name, (s, m) in tree_pool_calls(B=0):
        assert (s, m) == (FF_OK, ""), name
    for name, (s, m) in tree_pool_calls(ptrs=2):  # 2-byte alignment is too little for every entry
        assert s == FF_EINVAL and "misaligned" in m, name
    for name, (s, m) in tree_pool_calls(B=-1):
        assert s == FF_EINVAL and "B" in m, name
    for name, (s, m) in [*tree_pool_calls(D=832), *tree_pool_calls(D=2176)]:  # not whole 128s, above 2048
        assert s == FF_EINVAL and "D" in m, name
    bad_heads = {name: m for name, (s, m) in tree_pool_calls(G=32)}  # heads of 24 columns
    assert all("16 columns" in bad_heads[n] for n in ("weights", "values", "queries", "keys", "tree"))
    lib = K.lib()

    def weights(u_stride=0, c_stride=0, N=1025, G=16, M=18, D=768, ldt=1032):
        return err(lib.ff_pool_weights(256, 256, u_stride, 256, c_stride, 256, 2, N, G, M, D, ldt, 256, 256, None))[1]

    assert "N * D" in weights(N=0) and "M must be" in weights(M=7) and "384" in weights(G=24, D=768)
    assert "u_stride" in weights(u_stride=5) and "u_stride" in weights(u_stride=16 * 18 * 768 + 4)
    assert "c_stride" in weights(c_stride=5)
    assert all("ldt" in weights(ldt=v) for v in (1024, 1027, 1034))

    def pool_sum(N=1025, GM=288, ldt=1032):
        return err(lib.ff_pool_sum(256, 256, 2, N, GM, 768, ldt, 256, None))[1]

    assert "GM" in pool_sum(GM=0) and "GM" in pool_sum(GM=513)
    assert "ldt" in pool_sum(ldt=1026) and "ldt" in pool_sum(ldt=1040)
    assert "M or nblk" in err(lib.ff_pool_values(256, 256, 256, 256, 0, 2, 16, 18, 768, 256, None))[1]
    assert "M or nblk" in err(lib.ff_pool_values(256, 256, 256, 256, 3, 2, 16, 65, 768, 256, None))[1]
    q = [256] * 7
    assert "C | Q" in err(lib.ff_pool_queries(*q, 1e-6, 2, 5, 18, 16, 768, 256, 256, 256, None))[1]
    assert "eps" in err(lib.ff_pool_queries(*q, 0.0, 2, 6, 18, 16, 768, 256, 256, 256, None))[1]
    assert "C | Q" in err(lib.ff_pool_tree(256, 256, 256, 256, 256, 3, 1e-6, 2, 5, 18, 16, 768, 256, None))[1]
    assert "nblk" in err(lib.ff_pool_tree(256, 256, 256, 256, 256, 0, 1e-6, 2, 6, 18, 16, 768, 256, None))[1]
    assert "eps" in err(lib.ff_pool_tree(256, 256, 256, 256, 256, 3, -1.0, 2, 6, 18, 16, 768, 256, None))[1]
    assert "F % 16" in err(lib.ff_pool_leaf(256, 256, 256, 2, 18, 20, 768, 256, None))[1]


def test_patch_embed_rejects_bad_arguments():
    def call(B=2, grid=8, N=768, img=256, w=256, bias=256, x=256):
        return err(K.lib().ff_patch_embed(img, w, bias, 256, B, grid, N, x, None))

    assert call(B=0) == (FF_OK, "")
    assert "B" in call(B=-1)[1] and "B" in call(B=65536)[1]
    assert "grid" in call(grid=0)[1] and "grid" in call(grid=2001)[1]
    assert "multiple of 128" in call(N=0)[1] and "multiple of 128" in call(N=192)[1]
    assert "null" in call(img=None)[1]
    for kw in (dict(img=258), dict(w=264), dict(bias=260), dict(x=260)):
        assert "misaligned" in call(**kw)[1]


def test_head_rejects_bad_arguments():
    def call(B=2, N=1000, Kd=1024, stride=1024, gamma=None, beta=None, eps=1e-6, x=256, w=256):
        return err(K.lib().ff_head(x, stride, gamma, beta, eps, w, 256, B, N, Kd, 256, None))

    assert call(B=0) == (FF_OK, "")
    assert "B" in call(B=65)[1] and "B" in call(B=-1)[1] and "bad N" in call(N=0)[1]
    assert "K % 32" in call(Kd=1000)[1] and "K % 32" in call(Kd=1312, stride=1312)[1]
    assert "x_stride" in call(stride=1016)[1] and "x_stride" in call(stride=1028)[1]
    assert "together" in call(gamma=256)[1] and "together" in call(beta=256)[1]
    assert "eps" in call(gamma=256, beta=256, eps=0.0)[1]
    assert "null" in call(x=None)[1]
    assert "misaligned" in call(x=264)[1] and "misaligned" in call(w=264)[1]


def test_bicubic_taps_rejects_bad_arguments():
    def call(w=(1200, 448, 13, 0), h=(900, 336, 13, 0), p=256):
        return err(K.lib().ff_bicubic_taps(*w[:3], p, 256, w[3], *h[:3], 256, 256, h[3], None))

    for bad in ((0, 448, 13, 0), (1200, 0, 13, 0), (1200, 448, 0, 0), (-5, 448, 13, 0), (1 << 20, 448, 13, 0)):
        assert "size" in call(w=bad)[1] and "size" in call(h=bad)[1]
    assert "shift" in call(w=(1200, 448, 13, -1))[1] and "shift" in call(h=(900, 336, 13, 901))[1]
    assert "null" in call(p=None)[1]
