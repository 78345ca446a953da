"""Haruka's tree-pool kernels and the tag head against float64 on the same fp16 inputs, and the pool's own chain of
kernels against the library chain, at the sizes where they can go wrong: tokens and rows that end inside a tile, one
token, one image, more rows than one tile, head widths of one and three column tiles."""

from __future__ import annotations

import pytest
import torch

from foidfinder_amd import kernels as K
from foidfinder_amd.haruka import HarukaConfig, HarukaInt8, synthetic_checkpoint

pytestmark = pytest.mark.gpu

# fp16 inputs, fp32 sums, one rounding of the result to fp16 (2^-11 relative); the sums' own error is far below.
FP16 = 2.0**-11


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


def randn(dev, *shape, std=1.0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + sum(shape))
    return torch.randn(*shape, device=dev, generator=g) * std


def close(got, want, what):
    """Within 1.5 fp16 roundings of the value, or of the result's typical size where the value is small."""
    want = want.double()
    bound = 1.5 * FP16 * torch.maximum(want.abs(), want.pow(2).mean().sqrt())
    bad = ((got.double() - want).abs() > bound).sum().item()
    assert bad == 0, f"{what}: {bad} of {want.numel()} off, worst {((got.double() - want).abs() / bound).max().item():.2f} x"


@pytest.mark.parametrize(("B", "N", "K_", "norm"), [(1, 100, 32, False), (3, 257, 1024, True), (16, 1000, 1152, False),
                                                    (17, 33, 1280, True), (33, 40, 448, False), (64, 300, 1024, True)])
def test_head(dev, B, N, K_, norm):
    stride = K_ + 64 if norm else K_  # the class tokens' rows are far apart
    x = randn(dev, B, stride, seed=1).half()[:, :K_]
    w, b = randn(dev, N, K_, std=0.05, seed=2).half(), randn(dev, N, seed=3).half()
    g, be = 1 + randn(dev, K_, std=0.1, seed=4), randn(dev, K_, std=0.1, seed=5)
    out = torch.full((B, N), float("nan"), device=dev)
    K.head(x, w, b, out, *((g, be) if norm else ()), eps=1e-6)
    xd = x.double()
    if norm:
        xd = torch.nn.functional.layer_norm(xd, (K_,), g.double(), be.double(), 1e-6).half().double()
    want = xd @ w.double().t() + b.double()
    # fp32 sums of K_ products: K_ 2^-24 of the absolute sum; with the norm an input may round the other way (one ulp)
    bound = (K_ * 2.0**-24 + (2 * FP16 if norm else 0.0)) * (xd.abs() @ w.double().abs().t() + b.double().abs())
    assert ((out.double() - want).abs() <= bound).all()


def test_head_refuses_overlapping_rows(dev):
    """Refused on the host before any launch; one row is taken whatever its stride is."""
    w, b, flat = randn(dev, 48, 64, std=0.05).half(), randn(dev, 48).half(), randn(dev, 256, seed=1).half()
    for x in (flat[:64].expand(16, 64), flat.as_strided((3, 64), (8, 1)), flat.as_strided((3, 64), (65, 1))):
        with pytest.raises(RuntimeError, match="x_stride"):
            K.head(x, w, b, torch.empty(x.size(0), 48, device=dev))
    one, two = torch.empty(1, 48, device=dev), torch.empty(1, 48, device=dev)
    K.head(flat.as_strided((1, 64), (3, 1)), w, b, one)
    K.head(flat[:64].view(1, 64), w, b, two)
    assert torch.equal(one, two)


@pytest.mark.parametrize(("B", "N", "G", "M", "D"), [(1, 1, 16, 6, 768), (2, 96, 16, 18, 768), (3, 97, 4, 18, 128),
                                                     (1, 193, 20, 18, 640), (2, 95, 64, 6, 1024)])
@pytest.mark.parametrize("shared", [True, False])
def test_pool_weights(dev, B, N, G, M, D, shared):
    xn = randn(dev, B, N, D, seed=1).half()
    u = randn(dev, *(() if shared else (B,)), G * M, D, std=0.08, seed=2).half()
    c = randn(dev, *(() if shared else (B,)), G * M, seed=3)
    bias = randn(dev, M, seed=4)
    ldt = (N + 7) // 8 * 8
    a_t = torch.full((B, G * M, ldt), float("nan"), device=dev, dtype=torch.half)
    partial = torch.full((B, K.pool_weights_blocks(N), G * M), float("nan"), device=dev)
    K.pool_weights(xn, u, c, bias, G, a_t, partial)
    lg = torch.matmul(xn.double(), u.double().transpose(-1, -2).contiguous()) + (c.double() if shared else c.double()[:, None])
    lg = lg.view(B, N, G, M)
    w = (torch.softmax(lg, -1) * torch.sigmoid(lg + bias.double())).view(B, N, G * M)
    # exp2 and rcp of ~1 ulp each, fp32 logits of size ~10 (2^-20 absolute): 1e-5 relative before the fp16 rounding
    got, want = a_t[:, :, :N].double(), w.transpose(1, 2)
    assert ((got - want).abs() <= (FP16 + 2e-5) * want + 2.0**-24).all()
    mass = w.sum(1)
    assert ((partial.double().sum(1) - mass).abs() <= 3e-5 * mass).all()
    assert (a_t[:, :, N:] == 0).all()


@pytest.mark.parametrize(("B", "N", "GM", "D"), [(1, 1, 96, 128), (2, 64, 288, 768), (3, 65, 24, 256), (2, 127, 120, 384),
                                                 (1, 1025, 512, 128), (1, 333, 97, 192 * 2)])
def test_pool_sum(dev, B, N, GM, D):
    """One token, token counts around a chunk of 64, queries that end inside a tile of 96 and past five tiles; whatever
    follows a row's N weights (zero pad, the next row) must not count."""
    xn = randn(dev, B, N, D, seed=1).half()
    a_t = torch.zeros(B, GM, (N + 7) // 8 * 8, device=dev, dtype=torch.half)
    a_t[:, :, :N] = torch.rand(B, GM, N, device=dev, generator=torch.Generator(device=dev).manual_seed(N)).half()
    pooled = torch.full((B, GM, D), float("nan"), device=dev, dtype=torch.half)
    K.pool_sum(a_t, xn, pooled)
    close(pooled, torch.matmul(a_t[:, :, :N].double().contiguous(), xn.double()), "pooled")


@pytest.mark.parametrize(("B", "C", "Q", "G", "D", "F"), [(1, 6, 18, 16, 768, 64), (3, 6, 18, 8, 128, 16),
                                                          (17, 6, 18, 20, 640, 32), (2, 3, 6, 2, 1024, 48)])
def test_pool_chain(dev, B, C, Q, G, D, F):
    """Each kernel between the products, on the previous one's actual output."""
    hd, eps, nblk = D // G, 1e-6, 3
    ln = lambda t, g, b: torch.nn.functional.layer_norm(t, (D,), g.double(), b.double(), eps)  # noqa: E731
    norm = lambda s: ((1 + randn(dev, D, std=0.1, seed=s)).half(), randn(dev, D, std=0.1, seed=s + 1).half())  # noqa: E731
    pooled, wv, bv = randn(dev, B, G * C, D, seed=1).half(), randn(dev, D, D, std=0.05, seed=2).half(), randn(dev, D, seed=3)
    partial = randn(dev, B, nblk, G * C, seed=4).abs()
    z = torch.empty(B, C, D, device=dev, dtype=torch.half)
    K.pool_values(pooled, wv, bv, partial, G, z)
    mass = partial.double().sum(1).view(B, G, C)
    want = torch.matmul(pooled.double().view(B, G, C, D), wv.double().view(G, hd, D).transpose(1, 2).contiguous())
    want = (want + mass[..., None] * bv.double().view(G, 1, hd)).transpose(1, 2).reshape(B, C, D)
    close(z, want, "values")

    trunk, childn, leafn = norm(10), norm(12), norm(14)
    child, bk = randn(dev, Q, D, seed=5).half(), randn(dev, D, seed=6)
    parent, qleaf = torch.empty_like(z), torch.empty(B, Q, D, device=dev, dtype=torch.half)
    cq = torch.empty(B, G * Q, device=dev)
    K.pool_queries(z, *trunk, child, *childn, bk, G, eps, parent, qleaf, cq)
    close(parent, ln(z.double(), *trunk), "parent")
    rep = parent.double().repeat_interleave(Q // C, 1)
    close(qleaf, ln(rep + child.double(), *childn), "leaf queries")
    want = (qleaf.double() * bk.double()).view(B, Q, G, hd).sum(-1).transpose(1, 2).reshape(B, G * Q)
    assert ((cq.double() - want).abs() <= 1e-5 * want.abs().max()).all()

    kT = randn(dev, G, D, hd, std=0.1, seed=7).half()
    u = torch.empty(B, G * Q, D, device=dev, dtype=torch.half)
    K.pool_keys(qleaf, kT, u)
    want = torch.matmul(qleaf.double().view(B, Q, G, hd).transpose(1, 2), kT.double().transpose(1, 2).contiguous())
    close(u, want.reshape(B, G * Q, D), "keys")

    zc, part2 = randn(dev, B, Q, D, seed=8).half(), randn(dev, B, nblk, G * Q, seed=9).abs()
    tree = torch.empty(Q, B, D, device=dev, dtype=torch.half)
    K.pool_tree(parent, zc, *leafn, part2, G, eps, tree)
    m = part2.double().sum(1).view(B, G, Q).mean(1)
    close(tree, (ln(rep + zc.double(), *leafn) * (m / (m + 4))[..., None]).transpose(0, 1), "tree")

    wl, bl = randn(dev, Q, F, D, std=0.05, seed=20).half(), randn(dev, Q, F, seed=21).half()
    leaf = torch.empty(B, Q * F, device=dev, dtype=torch.half)
    K.pool_leaf(tree, wl, bl, leaf)
    want = torch.matmul(tree.double(), wl.double().transpose(1, 2).contiguous()) + bl.double()[:, None]
    close(leaf, want.transpose(0, 1).reshape(B, Q * F), "leaves")


@pytest.mark.parametrize(("batch", "pool_heads", "leaf_dim"), [(1, 16, 64), (5, 8, 16), (3, 6, 64), (2, 16, 20)])
def test_pool_head_matches_library_chain(dev, monkeypatch, batch, pool_heads, leaf_dim):
    """A whole pool head on its own kernels against the library chain, which also serves the shapes that are not whole
    16-column tiles (leaves of 20 here: refused by the rule)."""
    dim = 384 if pool_heads == 6 else 768
    cfg = HarukaConfig(img_size=112, dim=dim, heads=dim // 64, depth=1, hidden=256, pool_heads=pool_heads,
                       leaf_dim=leaf_dim, tags=100)
    raw = synthetic_checkpoint(cfg, seed=3)
    eng = HarukaInt8(raw, cfg, device=dev)
    assert eng.fused_pool == (dim // pool_heads % 16 == 0 and leaf_dim % 16 == 0)
    x = randn(dev, batch, cfg.tokens, dim, seed=2).half()
    got = eng.pool_head(x)
    assert got.shape == (batch, 100) and torch.isfinite(got).all()
    if not eng.fused_pool:
        return
    monkeypatch.setattr(eng, "_pool_leaves", eng._pool_leaves_library)
    want = eng.pool_head(x)
    # the library chain rounds its logits, products and masses to fp16 at a dozen points: 4e-3 of the result's size
    rel = ((got - want).double().norm() / want.double().norm()).item()
    assert rel < 4e-3, f"fused and library pools differ by {rel:.2e}"
    monkeypatch.undo()
    monkeypatch.setattr("foidfinder_amd.haruka.pool_fits", lambda *sizes: False)  # more images or tokens than the kernels take
    assert torch.equal(eng.pool_head(x), want)


@pytest.mark.parametrize(("B", "grid", "N", "cols"),
                         [(1, 1, 128, 64), (2, 9, 128, 64), (3, 8, 768, 64), (1, 17, 384, 64), (40, 8, 1024, 64),
                          (45, 9, 768, 256), (90, 9, 384, 128), (100, 8, 1024, 512), (12, 33, 768, 256)])
def test_patch_embed(dev, B, grid, N, cols):
    """One patch, patch counts that end inside a workgroup's 64, raw pixel values, and each split of the columns: 64 a
    workgroup up to 1024 such workgroups (the fifth case has 640), past that 128, 256 or 512 in turns of 128, with a
    partial last patch block (81 and 1089 patches). The class row is copied, the others are float64's within one fp16
    rounding (fp32 sums of 588 products)."""
    workgroups = -(-grid * grid // 64) * B * (N // 64)
    assert cols == (64 if workgroups <= 1024 else next(c for c in (512, 256, 128) if N % c == 0))
    S = 14 * grid
    img = (torch.rand(B, S, S, 3, device=dev, generator=torch.Generator(device=dev).manual_seed(B)) * 255).round().half()
    w, bias = randn(dev, N, 588, std=1e-3, seed=1).half(), randn(dev, grid * grid, N, seed=2).half()
    cls = randn(dev, N, seed=3).half()
    x = torch.full((B, 1 + grid * grid, N), float("nan"), device=dev, dtype=torch.half)
    K.patch_embed(img, K.pad_patch_weight(w), bias, cls, x)
    p = img.double().view(B, grid, 14, grid, 14, 3).permute(0, 1, 3, 2, 4, 5).reshape(B, grid * grid, 588)
    want = p @ w.double().t() + bias.double()
    assert torch.equal(x[:, 0], cls.expand(B, N))
    bound = FP16 * want.abs() + 588 * 2.0**-24 * (p @ w.double().abs().t() + bias.double().abs()) + 2.0**-25
    assert ((x[:, 1:].double() - want).abs() <= bound).all()
