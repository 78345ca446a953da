// Pillow's separable 8-bit resampling (libImaging/Resample.c) on uint8 RGB images, for the Haruka model card's letterbox
// on the GPU (the reference's Metal version: foidfinder/backends/mlx/kernels.py:75-186): the bicubic filter's fixed-point
// taps (22 fractional bits, per output index: first input index and tap count), and one pass along one axis.
//
// A pass writes a padded canvas: bytes inside the region are sum(code * tap) + 2^21, shifted right by 22 and clipped to
// 0..255, exactly as Pillow; bytes outside are white. Every tap's source index is checked against the source image, so no
// table can make the kernel read outside it.
//
// Byte loads bound a pass (one per tap and byte: 19.9 us along the width and 7.4 along the height for 1200 x 900 -> 448),
// so a thread takes a whole pixel along the width and four bytes of a row along the height, each tap one 4-byte load: 11.0
// and 7.0 us.
#include "common.h"

namespace ff {

struct __attribute__((packed)) u32_unaligned {
  uint32_t v;
};
__device__ __forceinline__ uint32_t load_u32(const uint8_t* p) { return reinterpret_cast<const u32_unaligned*>(p)->v; }
__device__ __forceinline__ void store_u32(uint8_t* p, uint32_t v) { reinterpret_cast<u32_unaligned*>(p)->v = v; }

__device__ __forceinline__ uint32_t clip8(int ss) {
  ss >>= 22;  // arithmetic shift, as Pillow's signed accumulator
  return static_cast<uint32_t>(ss < 0 ? 0 : (ss > 255 ? 255 : ss));
}

// Along the width: one thread per canvas pixel, blockIdx.y the canvas row. Tap t of the pixel is source pixel first + t of
// row row0 + yy: its three bytes come with one 4-byte load, except for the image's last pixel, whose fourth byte would
// lie past the image.
__global__ __launch_bounds__(256) void resample_width_kernel(const uint8_t* __restrict__ src, int src_h, int src_w,
                                                             const int32_t* __restrict__ kk,
                                                             const int32_t* __restrict__ bounds, int ksize, int row0,
                                                             uint8_t* __restrict__ out, int out_w, int top, int left,
                                                             int h, int w) {
  const int x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
  if (x >= out_w) return;
  const int yy = y - top, xx = x - left;
  uint32_t c0 = 255, c1 = 255, c2 = 255;
  if (yy >= 0 && yy < h && xx >= 0 && xx < w) {
    const int first = bounds[2 * xx], taps = min(bounds[2 * xx + 1], ksize), sy = row0 + yy;
    const int32_t* k = kk + static_cast<int64_t>(xx) * ksize;
    const uint8_t* row = src + static_cast<int64_t>(sy) * src_w * 3;
    const bool row_in = sy >= 0 && sy < src_h;
    const int last = sy == src_h - 1 ? src_w - 1 : src_w;  // pixels of this row from which four bytes can be read
    int s0 = 1 << 21, s1 = 1 << 21, s2 = 1 << 21;
    for (int t = 0; t < taps; ++t) {
      const int sx = first + t;
      if (!row_in || sx < 0 || sx >= src_w) continue;
      const uint8_t* p = row + 3 * sx;
      const uint32_t v = sx < last ? load_u32(p) : p[0] | p[1] << 8 | p[2] << 16;
      const int kt = k[t];
      s0 += static_cast<int>(v & 255) * kt;
      s1 += static_cast<int>(v >> 8 & 255) * kt;
      s2 += static_cast<int>(v >> 16 & 255) * kt;
    }
    c0 = clip8(s0), c1 = clip8(s1), c2 = clip8(s2);
  }
  uint8_t* o = out + (static_cast<int64_t>(y) * out_w + x) * 3;
  o[0] = static_cast<uint8_t>(c0), o[1] = static_cast<uint8_t>(c1), o[2] = static_cast<uint8_t>(c2);
}

// Along the height: one thread per four bytes of a canvas row, blockIdx.y the row. Tap t of byte j of the region's row is
// byte j of source row row0 + first + t; four bytes inside the region are four bytes of each source row. Groups that
// cross the region's or the canvas row's edge go byte by byte.
__global__ __launch_bounds__(256) void resample_height_kernel(const uint8_t* __restrict__ src, int src_h, int src_w,
                                                              const int32_t* __restrict__ kk,
                                                              const int32_t* __restrict__ bounds, int ksize, int row0,
                                                              uint8_t* __restrict__ out, int out_w, int top, int left,
                                                              int h, int w) {
  const int j0 = 4 * (blockIdx.x * 256 + threadIdx.x), y = blockIdx.y;
  if (j0 >= 3 * out_w) return;
  const int yy = y - top, b0 = j0 - 3 * left;  // the group's first byte within the region's row
  uint8_t* o = out + static_cast<int64_t>(y) * out_w * 3 + j0;
  const bool row_in = yy >= 0 && yy < h;
  int first = 0, taps = 0;
  const int32_t* k = kk;
  if (row_in) {
    first = bounds[2 * yy], taps = min(bounds[2 * yy + 1], ksize);
    k = kk + static_cast<int64_t>(yy) * ksize;
  }
  const int64_t pitch = static_cast<int64_t>(src_w) * 3;
  if (row_in && b0 >= 0 && b0 + 4 <= 3 * w && j0 + 4 <= 3 * out_w) {  // w <= src_w: the source rows hold these bytes
    int s0 = 1 << 21, s1 = 1 << 21, s2 = 1 << 21, s3 = 1 << 21;
    for (int t = 0; t < taps; ++t) {
      const int sy = row0 + first + t;
      if (sy < 0 || sy >= src_h) continue;
      const uint32_t v = load_u32(src + sy * pitch + b0);
      const int kt = k[t];
      s0 += static_cast<int>(v & 255) * kt;
      s1 += static_cast<int>(v >> 8 & 255) * kt;
      s2 += static_cast<int>(v >> 16 & 255) * kt;
      s3 += static_cast<int>(v >> 24) * kt;
    }
    store_u32(o, clip8(s0) | clip8(s1) << 8 | clip8(s2) << 16 | clip8(s3) << 24);
    return;
  }
  for (int e = 0; e < 4 && j0 + e < 3 * out_w; ++e) {
    const int b = b0 + e;
    uint32_t v = 255;
    if (row_in && b >= 0 && b < 3 * w) {
      int ss = 1 << 21;
      for (int t = 0; t < taps; ++t) {
        const int sy = row0 + first + t;
        if (sy >= 0 && sy < src_h) ss += static_cast<int>(src[sy * pitch + b]) * k[t];
      }
      v = clip8(ss);
    }
    o[e] = static_cast<uint8_t>(v);
  }
}

// Pillow's bicubic filter (a = -0.5) at distance x.
__device__ __forceinline__ double bicubic(double x) {
  return x < 1.0 ? (1.5 * x - 2.5) * x * x + 1.0 : (x < 2.0 ? (((x - 5.0) * x + 8.0) * x - 4.0) * -0.5 : 0.0);
}

struct TapAxis {
  int in, out, ksize, shift;  // shift: subtracted from the first input indices
  int32_t *kk, *bounds;
};

// The fixed-point taps of both axes, one thread per output index (precompute_coeffs and normalize_coeffs_8bpc): every
// double operation is Pillow's, in its order (this file is built without contraction), so the taps are its bits. The
// weights are evaluated twice, for their sum and for their codes, instead of being stored in between.
__global__ __launch_bounds__(64) void bicubic_taps_kernel(TapAxis a, TapAxis b) {
  int i = blockIdx.x * 64 + threadIdx.x;
  const TapAxis t = i < a.out ? a : b;
  if (i >= a.out) i -= a.out;
  if (i >= t.out) return;
  const double scale = static_cast<double>(t.in) / static_cast<double>(t.out);
  const double filterscale = scale > 1.0 ? scale : 1.0, support = 2.0 * filterscale, step = 1.0 / filterscale;
  const double center = (static_cast<double>(i) + 0.5) * scale;
  const double lo = trunc(center - support + 0.5);
  const int first = static_cast<int>(lo > 0.0 ? lo : 0.0);
  const int end = static_cast<int>(trunc(center + support + 0.5));
  const int count = (end < t.in ? end : t.in) - first;
  auto weight = [&](int j) {
    const double x = (static_cast<double>(j + first) - center + 0.5) * step;
    return bicubic(x < 0.0 ? -x : x);
  };
  double total = 0.0;
  for (int j = 0; j < count && j < t.ksize; ++j) total = total + weight(j);
  int32_t* k = t.kk + static_cast<int64_t>(i) * t.ksize;
  for (int j = 0; j < t.ksize; ++j) {
    double w = j < count ? weight(j) : 0.0;
    if (total != 0.0) w = w / total;
    k[j] = static_cast<int32_t>(w < 0.0 ? -0.5 + w * 4194304.0 : 0.5 + w * 4194304.0);
  }
  t.bounds[2 * i] = first - t.shift;
  t.bounds[2 * i + 1] = count;
}

}  // namespace ff

using namespace ff;

extern "C" int ff_resample_u8(const uint8_t* src, int64_t src_h, int64_t src_w, int axis, const int32_t* kk,
                              const int32_t* bounds, int64_t ksize, int64_t row0, uint8_t* out, int64_t out_h,
                              int64_t out_w, int64_t top, int64_t left, int64_t h, int64_t w, void* stream) {
  clear_error();
  if (axis != 0 && axis != 1) return fail(FF_EINVAL, "resample_u8: axis must be 0 (width) or 1 (height)");
  if (src_h <= 0 || src_w <= 0 || out_h <= 0 || out_w <= 0 || h <= 0 || w <= 0 || ksize <= 0)
    return fail(FF_EINVAL, "resample_u8: sizes must be positive");
  if (src_h > 65535 || src_w > 65535 || out_h > 65535 || out_w > 65535 || ksize > 65535)
    return fail(FF_EINVAL, "resample_u8: sizes above 65535 are not supported");
  if (top < 0 || left < 0 || top + h > out_h || left + w > out_w)
    return fail(FF_EINVAL, "resample_u8: region must lie inside the output");
  if (row0 < 0 || (axis == 0 && row0 + h > src_h) || (axis == 1 && w > src_w))
    return fail(FF_EINVAL, "resample_u8: region reads outside the source");
  if (!src || !kk || !bounds || !out) return fail(FF_EINVAL, "resample_u8: null pointer");
  const hipStream_t st = as_stream(stream);
  const int sh = static_cast<int>(src_h), sw = static_cast<int>(src_w), ks = static_cast<int>(ksize),
            r0 = static_cast<int>(row0), ow = static_cast<int>(out_w), t = static_cast<int>(top),
            l = static_cast<int>(left), hi = static_cast<int>(h), wi = static_cast<int>(w);
  if (axis == 0) {
    const dim3 grid(static_cast<unsigned>((out_w + 255) / 256), static_cast<unsigned>(out_h));
    resample_width_kernel<<<grid, 256, 0, st>>>(src, sh, sw, kk, bounds, ks, r0, out, ow, t, l, hi, wi);
  } else {
    const dim3 grid(static_cast<unsigned>((3 * out_w + 1023) / 1024), static_cast<unsigned>(out_h));
    resample_height_kernel<<<grid, 256, 0, st>>>(src, sh, sw, kk, bounds, ks, r0, out, ow, t, l, hi, wi);
  }
  return check_launch("resample_u8");
}

extern "C" int ff_bicubic_taps(int64_t in_w, int64_t out_w, int64_t ksize_w, int32_t* kk_w, int32_t* bounds_w,
                               int64_t shift_w, int64_t in_h, int64_t out_h, int64_t ksize_h, int32_t* kk_h,
                               int32_t* bounds_h, int64_t shift_h, void* stream) {
  clear_error();
  for (const int64_t v : {in_w, out_w, ksize_w, in_h, out_h, ksize_h})
    if (v <= 0 || v > 65535 * 5) return fail(FF_EINVAL, "bicubic_taps: bad size");
  if (shift_w < 0 || shift_h < 0 || shift_w > in_w || shift_h > in_h) return fail(FF_EINVAL, "bicubic_taps: bad shift");
  if (!kk_w || !bounds_w || !kk_h || !bounds_h) return fail(FF_EINVAL, "bicubic_taps: null pointer");
  const TapAxis a{static_cast<int>(in_w), static_cast<int>(out_w), static_cast<int>(ksize_w), static_cast<int>(shift_w),
                  kk_w, bounds_w};
  const TapAxis b{static_cast<int>(in_h), static_cast<int>(out_h), static_cast<int>(ksize_h), static_cast<int>(shift_h),
                  kk_h, bounds_h};
  const dim3 grid(static_cast<unsigned>((out_w + out_h + 63) / 64));
  bicubic_taps_kernel<<<grid, 64, 0, as_stream(stream)>>>(a, b);
  return check_launch("bicubic_taps");
}
