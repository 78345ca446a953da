"""Host-side logic on the CPU: weight conversion against the oracle, RoPE tables, configuration checks, the backend
registry and bench.py's single-GPU contract."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from foidfinder_amd import engine as E
from oracle import model as OM

ROOT = Path(__file__).resolve().parents[1]


def test_hadamard_matches_oracle():
    for n in (2, 128, 1024):
        np.testing.assert_array_equal(E.hadamard(n).numpy(), OM.hadamard(n))


def test_quantize_rows_matches_oracle(rng):
    w = (rng.standard_normal((64, 256)) * 0.02).astype(np.float32)
    q, s = E.quantize_rows_int8(torch.from_numpy(w))
    q0, s0 = OM.quantize_rows_int8(w)
    np.testing.assert_array_equal(q.numpy(), q0)
    np.testing.assert_array_equal(s.numpy(), s0)


def test_convert_checkpoint_matches_oracle_conversion():
    cfg = E.Eva02Config(img_size=56, depth=2, tags=32)
    raw = E.synthetic_checkpoint(cfg, seed=2)
    conv = E.convert_checkpoint(raw, cfg)
    ocfg = OM.Eva02Config(img_size=56, depth=2, tags=32)
    for i in range(cfg.depth):
        p = f"blocks.{i}."
        blk = {
            "qkv_w": raw[p + "attn.qkv.weight"].numpy(), "qkv_b": raw[p + "attn.qkv.bias"].numpy(),
            "proj_w": raw[p + "attn.proj.weight"].numpy(), "proj_b": raw[p + "attn.proj.bias"].numpy(),
            "fc1_w": raw[p + "mlp.fc1.weight"].numpy(), "fc1_b": raw[p + "mlp.fc1.bias"].numpy(),
            "fc2_w": raw[p + "mlp.fc2.weight"].numpy(), "fc2_b": raw[p + "mlp.fc2.bias"].numpy(),
        }
        for n in ("norm1", "norm2"):
            blk[n + "_w"], blk[n + "_b"] = raw[p + n + ".weight"].numpy(), raw[p + n + ".bias"].numpy()
        blk["mlp_norm_w"], blk["mlp_norm_b"] = raw[p + "mlp.norm.weight"].numpy(), raw[p + "mlp.norm.bias"].numpy()
        want = OM.convert_block(blk, ocfg)
        names = {"qkv": "attn.qkv", "proj": "attn.proj", "fc1": "mlp.fc1", "fc2": "mlp.fc2"}
        for short, long in names.items():
            for f in ("qweight", "wscale", "bias"):
                np.testing.assert_array_equal(conv[p + long + "." + f].numpy(), want[f"{short}.{f}"], err_msg=long + f)


def test_weight_rotation_matches_oracle_bit_for_bit(rng):
    for block, k in ((1024, 1024), (128, 2816)):
        w = (rng.standard_normal((40, k)) * 0.02).astype(np.float32)
        np.testing.assert_array_equal(E.rotate_rows64(torch.from_numpy(w), block).numpy(), OM.rotate_rows64(w, block))


def test_rope_tables_match_oracle():
    for grid in (2, 8, 32):
        c, s = E.eva02_rope_tables(grid, 16)
        c0, s0 = OM.eva02_rope_tables(grid, 16)
        np.testing.assert_array_equal(c.numpy(), c0)
        np.testing.assert_array_equal(s.numpy(), s0)


def test_config_validation():
    with pytest.raises(ValueError):
        E.Eva02Config(dim=768, heads=12).validate()
    with pytest.raises(ValueError):
        E.Eva02Config(hidden_pad=2800).validate()
    E.Eva02Config().validate()
    cfg = E.Eva02Config()
    assert cfg.tokens == 1025 and cfg.grid == 32
    ops = cfg.gemm_ops(32)
    assert sum(ops.values()) == pytest.approx(19.81e12, rel=2e-3)  # per batch-32 forward, unpadded dims
    assert cfg.attention_flops(32) == pytest.approx(3.305e12, rel=2e-3)


def test_backend_registry_without_gpu():
    from foidfinder_amd import backends

    assert backends.NAMES == ("mlx", "cuda", "rocm")
    with pytest.raises(ValueError, match="unknown backend"):
        backends.load("bogus", Path("."))
    with pytest.raises(RuntimeError):
        backends.load("cuda", Path("."))
    if not torch.cuda.is_available():
        with pytest.raises(RuntimeError, match="no AMD GPU"):
            backends.load("rocm", Path("."))
        with pytest.raises(RuntimeError, match="no supported accelerator"):
            backends.detect()


def test_model_dir_round_trip(tmp_path):
    cfg = E.Eva02Config(img_size=56, depth=1, tags=8)
    state = E.convert_checkpoint(E.synthetic_checkpoint(cfg, seed=1), cfg)
    E.save_model_dir(tmp_path, state, cfg, [f"t{i}" for i in range(8)], ["general"] * 7 + ["rating"],
                     {"general": 0.35, "rating": 0.5})
    cfg_json = (tmp_path / "config.json").read_text()
    assert '"architecture": "eva02-int8"' in cfg_json
    from safetensors.torch import load_file

    back = load_file(str(tmp_path / "model.safetensors"))
    assert set(back) == set(state)
    assert torch.equal(back["blocks.0.mlp.fc1.qweight"], state["blocks.0.mlp.fc1.qweight"])


def test_bench_refuses_more_than_one_gpu():
    r = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode == 2 and "one GPU" in r.stderr


def image_forms(B, S, device="cpu"):
    """(what, images) forms that the engines' patchify takes: dtypes, strides, storage offsets and shapes."""
    g = torch.Generator().manual_seed(B)
    base = (torch.rand(B, S, S, 3, generator=g) * 255).to(device)
    half = base.half()
    shifted = torch.zeros(half.numel() + 1, dtype=torch.half, device=device)[1:].view_as(half).copy_(half)
    wide = torch.zeros(B, S + 3, S + 5, 4, dtype=torch.half, device=device)
    wide[:, 1 : S + 1, 2 : S + 2, :3] = half
    return [("fp16", half), ("fp32", base), ("float64", base.double()), ("uint8", base.byte()),
            ("two bytes past a word", shifted), ("crop of a larger image", wide[:, 1 : S + 1, 2 : S + 2, :3]),
            ("channels first in memory", half.permute(0, 3, 1, 2).contiguous().permute(0, 2, 3, 1)),
            ("repeated image", half[:1].expand(B, S, S, 3)), ("rows of one axis", half.view(B, S, S * 3)),
            ("flat", half.view(B, -1)), ("patch grid", wide[:, 1 : S + 1, 2 : S + 2, :3].view(B, S // 14, 14, S // 14, 14, 3))]


def bare_engine(S):
    eng = object.__new__(E.Eva02Int8)
    eng.cfg = E.Eva02Config(img_size=S)
    return eng


@pytest.mark.parametrize(("B", "S"), [(1, 14), (3, 42)])
def test_stem_takes_the_images_that_patchify_takes(B, S):
    """What the stem kernel is handed is contiguous fp16 [B, S, S, 3] from a multiple of 4 bytes, and holds the pixels
    that patchify reads; shapes that patchify refuses and images that autograd follows are refused."""
    eng = bare_engine(S)
    for what, img in image_forms(B, S):
        px = eng._pixels(img)
        assert px.shape == (B, S, S, 3) and px.dtype == torch.half and px.is_contiguous(), what
        assert px.data_ptr() % 4 == 0, what
        assert torch.equal(eng.patchify(px), eng.patchify(img)), what
    for bad in (torch.zeros(B, S, S, 4), torch.zeros(B, S + 14, S, 3), torch.zeros(B, S, S)):
        for f in (eng.patchify, eng._pixels):
            with pytest.raises(RuntimeError):
                f(bad)
    followed = torch.zeros(B, S, S, 3, requires_grad=True)
    with pytest.raises(RuntimeError, match="backward"):
        eng._pixels(followed)
    with torch.no_grad():
        assert eng._pixels(followed).shape == (B, S, S, 3)


def test_stem_splits_batches_past_a_launch():
    """More images than one launch takes run in slices that cover every image once."""
    eng, B = bare_engine(14), 65535 * 2 + 3
    calls = []

    class Ops:
        @staticmethod
        def patch_embed(px, w, bias_pos, cls, x):
            calls.append((px.size(0), x.size(0), x.storage_offset()))

    eng.k, eng.patch_w = Ops, None
    eng._patch_embed(torch.zeros(1, 14, 14, 3, dtype=torch.half).expand(B, 14, 14, 3), None, None, torch.zeros(B, 2, 8))
    assert calls == [(65535, 65535, 0), (65535, 65535, 65535 * 16), (3, 3, 2 * 65535 * 16)]
