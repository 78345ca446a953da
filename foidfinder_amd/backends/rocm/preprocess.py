"""Letterbox preprocessing.

`preprocess` (PixAI, EVA02 int8): alpha composited onto white, antialiased bilinear resize on the GPU so the longer
side is `size`, pixels normalized to [-1, 1], padded with -1, NHWC fp16 (the engine's input layout); the steps of the
reference's PixAI preprocessing (foidfinder/backends/cuda/preprocess.py:16-32), at the model's own input size.

`preprocess_haruka` (Haruka): the model card's preprocessing (foidfinder/backends/mlx/haruka.py:63-72, the
reference's tests/test_haruka.py:19-34): composited onto white, Pillow bicubic resize so the longer side is `size`,
pasted centered on a white canvas, raw uint8 pixels NHWC (the normalization is folded into the patch weights). The
resize runs on the GPU (`ff_resample_u8`, two separable passes with Pillow's fixed-point taps, computed there too) and is
bit-exact with Pillow 13's `Image.resize(BICUBIC)` (the version the reference pins), as the reference's Metal resize
is (foidfinder/backends/mlx/kernels.py:75-186).
"""

from __future__ import annotations

import ctypes
import math
import threading

import numpy as np
import PIL
import torch
import torch.nn.functional as F
from PIL import Image

PILLOW_MAJOR = int(PIL.__version__.split(".")[0])


def vertical_first(w: int, h: int, nw: int, nh: int) -> bool:
    """Whether the resize resamples the height before the width (the passes do not commute: each rounds to 8 bits).
    Always the rule of Pillow 13, the version the reference pins (uv.lock) and hard-codes in its own resize: the
    vertical pass first when the height shrinks more than twice as much as the width (the reference's resize_pad,
    foidfinder/backends/mlx/kernels.py:180-182). So the served pixels do not depend on the Pillow installed here
    (Pillow 12 orders the passes by another rule and differs in the last bit on tall images such as 448 x 900)."""
    return h - nh > 0 and h - nh > (w - nw) * 2


def rgb_on_white(image: Image.Image) -> Image.Image:
    """RGB with any transparency composited onto a white background."""
    if image.mode == "RGB":
        return image
    rgba = image.convert("RGBA")
    canvas = Image.new("RGBA", rgba.size, (255, 255, 255, 255))
    canvas.alpha_composite(rgba)
    return canvas.convert("RGB")


@torch.no_grad()
def preprocess(images: list[Image.Image], size: int, device: str | torch.device = "cuda") -> torch.Tensor:
    """PIL images -> [B, size, size, 3] fp16 normalized pixels."""
    out = torch.full((len(images), size, size, 3), -1.0, device=device, dtype=torch.half)
    for b, image in enumerate(images):
        rgb = torch.from_numpy(np.array(rgb_on_white(image))).to(device, non_blocking=True)
        x = rgb.permute(2, 0, 1)[None].float().div_(255.0)
        h, w = x.shape[-2:]
        r = min(size / h, size / w)
        nh, nw = max(1, int(h * r)), max(1, int(w * r))
        if (nh, nw) != (h, w):
            x = F.interpolate(x, size=(nh, nw), mode="bilinear", align_corners=False, antialias=True)
        top, left = (size - nh) // 2, (size - nw) // 2
        out[b, top : top + nh, left : left + nw] = (x[0].permute(1, 2, 0) * 2.0 - 1.0).half()
    return out


def bicubic_taps(in_size: int, out_size: int) -> tuple[np.ndarray, np.ndarray]:
    """Pillow's bicubic filter taps along one axis (libImaging/Resample.c precompute_coeffs + normalize_coeffs_8bpc,
    a = -0.5): kk int32 [out_size, ksize] in 22-bit fixed point, bounds int32 [out_size, 2] = (first input index, tap
    count). The same float64 operations in the same order as the C code, so the taps are Pillow's to the bit."""
    scale = in_size / out_size
    filterscale = max(scale, 1.0)
    support = 2.0 * filterscale
    ksize = math.ceil(support) * 2 + 1
    center = (np.arange(out_size, dtype=np.float64) + 0.5) * scale
    first = np.maximum(np.trunc(center - support + 0.5), 0.0).astype(np.int64)
    count = np.minimum(np.trunc(center + support + 0.5).astype(np.int64), in_size) - first
    j = np.arange(ksize)
    x = np.abs(((j[None, :] + first[:, None]) - center[:, None] + 0.5) * (1.0 / filterscale))
    w = np.where(x < 1.0, (1.5 * x - 2.5) * x * x + 1.0, np.where(x < 2.0, (((x - 5.0) * x + 8.0) * x - 4.0) * -0.5, 0.0))
    w[j[None, :] >= count[:, None]] = 0.0
    total = np.zeros(out_size)
    for t in range(ksize):  # sequential sum, as the C loop
        total = total + w[:, t]
    w = np.divide(w, total[:, None], out=w.copy(), where=total[:, None] != 0.0)
    kk = np.trunc(np.where(w < 0, -0.5 + w * (1 << 22), 0.5 + w * (1 << 22))).astype(np.int32)
    return kk, np.stack([first, count], axis=1).astype(np.int32)


def taps_window(in_size: int, out_size: int, index: int) -> tuple[int, int]:
    """(first input index, one past the last) of an output index's taps: bicubic_taps' bounds, for one index."""
    scale = in_size / out_size
    support = 2.0 * max(scale, 1.0)
    center = (index + 0.5) * scale
    return max(math.trunc(center - support + 0.5), 0), min(math.trunc(center + support + 0.5), in_size)


def _as_tensor(image: np.ndarray) -> torch.Tensor:
    """The array as a tensor over the same memory, for reading only; a copy only of an array whose elements are not in
    order. PIL's arrays cannot be written, of which torch would warn, so such memory goes by its address; the tensor keeps
    the array alive."""
    image = np.require(image, requirements="C" if image.size else "CW")
    if not image.flags.writeable:
        memory = (ctypes.c_uint8 * image.nbytes).from_address(image.ctypes.data)
        memory.owner = image
        image = np.frombuffer(memory, image.dtype).reshape(image.shape)
    return torch.from_numpy(image)


class _Uploads:
    """Host images to the GPU through pinned memory: a threaded copy into a staging buffer and a DMA from it take 13 + 66
    us for 1200 x 900, the runtime's pageable copy 125, and the call returns before the DMA ends. At most BUFFERS staging
    buffers of at most LIMIT bytes are kept, for all threads and streams: a buffer is taken under the lock and handed back
    with an event recorded behind its DMA on the caller's stream, which its next user waits for. The pageable copy takes
    larger images, images up to LEAST bytes (waking the copy's threads costs more than it saves: preprocess_haruka of 448 x
    448 in 145 us staged, 127 pageable; at 600 x 448 both 190), other dtypes (which the resize refuses), and calls under
    graph capture, whose copy would read the shared buffer again on every replay."""

    BUFFERS, LEAST, LIMIT = 4, 640 << 10, 16 << 20

    def __init__(self):
        self.lock = threading.Lock()
        self.free: list[tuple[torch.Tensor, torch.cuda.Event]] = []  # oldest first

    @staticmethod
    def _buffer(n: int) -> torch.Tensor:
        """A pinned buffer of at least n bytes that serves later calls too: on the host whatever torch's default device
        is, and no inference tensor, which calls outside the inference mode could not write."""
        with torch.inference_mode(False):
            return torch.empty(1 << (n - 1).bit_length(), dtype=torch.uint8, device="cpu", pin_memory=True)

    def put(self, host: torch.Tensor, device: torch.device) -> torch.Tensor:
        if device.type == "cuda" and host.dtype == torch.uint8 and self.LEAST < host.numel() <= self.LIMIT:
            with torch.cuda.device(device):
                if not torch.cuda.is_current_stream_capturing():
                    return self._staged(host, device)
        return host.to(device)

    def _staged(self, host: torch.Tensor, device: torch.device) -> torch.Tensor:
        n, buf = host.numel(), None
        with self.lock:
            if len(self.free) >= self.BUFFERS or self.free and self.free[0][1].query():
                buf, event = self.free.pop(0)
        if buf is not None:
            event.synchronize()
        if buf is None or buf.numel() < n:
            buf = self._buffer(n)
        staged = buf[:n].view(host.shape)
        staged.copy_(host)
        out = staged.to(device, non_blocking=True)
        event = torch.cuda.Event()
        event.record()
        with self.lock:
            if len(self.free) < self.BUFFERS:
                self.free.append((buf, event))
        return out


_uploads = _Uploads()


def letterbox_gpu(rgb: np.ndarray, size: int, out: torch.Tensor) -> None:
    """uint8 [H, W, 3] -> out uint8 [size, size, 3] on the GPU: bicubic resize so the longer side is size (the other
    side int(side * ratio), at least 1), centered on white. Only the image goes to the GPU: the taps are computed there
    (ff_bicubic_taps) for two passes of ff_resample_u8."""
    from ... import kernels as K

    h, w = rgb.shape[:2]
    dev = out.device
    src = _uploads.put(_as_tensor(rgb), dev)
    if (w, h) == (size, size):
        out.copy_(src)
        return
    r = min(size / w, size / h)
    nw, nh = max(1, int(w * r)), max(1, int(h * r))
    top, left = (size - nh) // 2, (size - nw) // 2
    down_first = vertical_first(w, h, nw, nh)
    # horizontal first: only the source rows that the vertical pass reads
    row0, end = (0, h) if down_first else (taps_window(h, nh, 0)[0], taps_window(h, nh, nh - 1)[1])
    ks_w, ks_h = (2 * math.ceil(2.0 * max(n / m, 1.0)) + 1 for n, m in ((w, nw), (h, nh)))
    buf = torch.empty(nw * (ks_w + 2) + nh * (ks_h + 2), dtype=torch.int32, device=dev)
    kk_w, b_w, kk_h, b_h = buf.split([nw * ks_w, nw * 2, nh * ks_h, nh * 2])
    kk_w, b_w, kk_h, b_h = kk_w.view(nw, ks_w), b_w.view(nw, 2), kk_h.view(nh, ks_h), b_h.view(nh, 2)
    K.bicubic_taps((w, nw, 0), (h, nh, row0), kk_w, b_w, kk_h, b_h)
    if down_first:
        tmp = torch.empty(nh, w, 3, dtype=torch.uint8, device=dev)
        K.resample_u8(src, 1, kk_h, b_h, 0, tmp, (0, 0, nh, w))
        K.resample_u8(tmp, 0, kk_w, b_w, 0, out, (top, left, nh, nw))
        return
    tmp = torch.empty(end - row0, nw, 3, dtype=torch.uint8, device=dev)
    K.resample_u8(src, 0, kk_w, b_w, row0, tmp, (0, 0, end - row0, nw))
    K.resample_u8(tmp, 1, kk_h, b_h, 0, out, (top, left, nh, nw))


@torch.no_grad()
def preprocess_haruka(images: list[Image.Image], size: int, device: str | torch.device = "cuda") -> torch.Tensor:
    """PIL images -> [B, size, size, 3] uint8 letterboxed pixels on the GPU."""
    out = torch.empty(len(images), size, size, 3, dtype=torch.uint8, device=device)
    for b, image in enumerate(images):
        letterbox_gpu(np.asarray(rgb_on_white(image)), size, out[b])
    return out
