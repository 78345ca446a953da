// The ViT stem: x[b, 1 + p] = patch p of image b (14 x 14 x 3 pixels) W^T + bias_pos[p], x[b, 0] = cls, straight from the
// image. As library calls it is a permuting copy of the patches (2 x the image's bytes), a product with K = 588 (rows of
// 1176 bytes, whose odd alignment costs the library its wide loads), an add and a copy of the class token.
//
// A workgroup gathers 64 patches into LDS once (84-byte runs of 14 image rows each; a row of 304 words, padded by 4 so
// that 16 rows' 16-byte chunks fall on distinct banks) and multiplies them with 64 NC columns at a time: wave w takes 16 NC
// of them against all 64 patches (v_mfma_f32_16x16x32_f16, weights as rows), its weight fragments loaded straight from
// global memory before the gather's barrier. NC = 1 while the grid is small (more workgroups, each with less to do),
// NC = 2 past that (half the LDS reads per product, which otherwise bound it). One 448 px image at 1024 columns: 8.4-9.6 us,
// mostly launch and load latency (the library calls: 21).
#include "common.h"

namespace ff {

constexpr int ST_P = 14;                      // patch side
constexpr int ST_K = ST_P * ST_P * 3;         // 588
constexpr int ST_KP = (ST_K + 31) / 32 * 32;  // 608: W's padded row length
constexpr int ST_STEPS = ST_KP / 32;          // 19
constexpr int ST_LD = ST_KP / 2 + 4;          // words per gathered row
constexpr int ST_RUN = ST_P * 3 / 2;          // 21 words of one patch row

template <int NC>
__global__ __launch_bounds__(256, 2) void patch_embed_kernel(const uint32_t* __restrict__ img, const half_t* __restrict__ w,
                                                             const half_t* __restrict__ bias_pos,
                                                             const half_t* __restrict__ cls, int grid, int N, int cols,
                                                             half_t* __restrict__ x) {
  __shared__ __attribute__((aligned(16))) uint32_t a[64 * ST_LD];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, kq = lane >> 4;
  const int np = grid * grid, p0 = 64 * blockIdx.y, b = blockIdx.z;
  const int n_begin = blockIdx.x * cols;
  half8_t f[NC][ST_STEPS];
  auto load_w = [&](int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int s = 0; s < ST_STEPS; ++s)
        f[c][s] = *reinterpret_cast<const half8_t*>(w + static_cast<int64_t>(n0 + 16 * (NC * wave + c) + i16) * ST_KP +
                                                    32 * s + 8 * kq);
  };
  load_w(n_begin);
  // gather: a thread takes one row of a patch at a time
  const uint32_t* im = img + static_cast<int64_t>(b) * grid * ST_P * grid * ST_RUN;
#pragma unroll 1
  for (int i = threadIdx.x; i < 64 * ST_P; i += 256) {
    const int r = i & 63, kh = i >> 6;
    const int p = min(p0 + r, np - 1);  // rows past the last patch repeat it and are not stored
    const uint32_t* src = im + (static_cast<int64_t>(p / grid * ST_P + kh) * grid + p % grid) * ST_RUN;
    uint32_t* dst = a + r * ST_LD + kh * ST_RUN;
    uint32_t t[ST_RUN];
#pragma unroll
    for (int j = 0; j < ST_RUN; ++j) t[j] = src[j];
#pragma unroll
    for (int j = 0; j < ST_RUN; ++j) dst[j] = t[j];
  }
  for (int i = threadIdx.x; i < 64 * (ST_KP - ST_K) / 2; i += 256)
    a[(i & 63) * ST_LD + ST_K / 2 + (i >> 6)] = 0;
  half_t* xb = x + static_cast<int64_t>(b) * (np + 1) * N;
  if (blockIdx.y == 0)
    for (int n = n_begin + threadIdx.x; n < n_begin + cols; n += 256) xb[n] = cls[n];
  __syncthreads();
#pragma unroll 1
  for (int n0 = n_begin; n0 < n_begin + cols; n0 += 64 * NC) {
    if (n0 != n_begin) load_w(n0);
    float4_t acc[NC][4] = {};
    half8_t v[2][4];
    auto read = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[s & 1][j] = *reinterpret_cast<const half8_t*>(a + (16 * j + i16) * ST_LD + 16 * s + 4 * kq);
    };
    read(0);
#pragma unroll
    for (int s = 0; s < ST_STEPS; ++s) {
      if (s + 1 < ST_STEPS) read(s + 1);
      __builtin_amdgcn_sched_barrier(0);  // one step ahead and no more (all steps' fragments would spill)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[c][s], v[s & 1][j], acc[c][j], 0, 0, 0);
    }
    // acc[c][j][i]: column n0 + 16 (NC wave + c) + 4 (lane / 16) + i of patch p0 + 16 j + lane % 16
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = p0 + 16 * j + i16, n = n0 + 16 * (NC * wave + c) + 4 * kq;
        if (p >= np) continue;
        const half4_t bp = *reinterpret_cast<const half4_t*>(bias_pos + static_cast<int64_t>(p) * N + n);
        half4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = static_cast<half_t>(acc[c][j][i] + static_cast<float>(bp[i]));
        *reinterpret_cast<half4_t*>(xb + static_cast<int64_t>(p + 1) * N + n) = o;
      }
  }
}

}  // namespace ff

using namespace ff;

extern "C" int ff_patch_embed(const void* img, const void* w, const void* bias_pos, const void* cls, int64_t B,
                              int64_t grid, int64_t N, void* x, void* stream) {
  clear_error();
  if (B < 0 || B > 65535) return fail(FF_EINVAL, "patch_embed: need 0 <= B <= 65535");
  if (grid <= 0 || grid > 2000) return fail(FF_EINVAL, "patch_embed: need 0 < grid <= 2000");
  if (N <= 0 || N % 128 != 0 || N > (1 << 20)) return fail(FF_EINVAL, "patch_embed: N must be a multiple of 128");
  if (B == 0) return FF_OK;
  if (!img || !w || !bias_pos || !cls || !x) return fail(FF_EINVAL, "patch_embed: null pointer");
  if ((reinterpret_cast<uintptr_t>(img) & 3) || (reinterpret_cast<uintptr_t>(w) & 15) ||
      (reinterpret_cast<uintptr_t>(bias_pos) & 7) || (reinterpret_cast<uintptr_t>(x) & 7))
    return fail(FF_EINVAL, "patch_embed: misaligned pointer");
  const int64_t blocks = (grid * grid + 63) / 64;
  const bool small = blocks * B * (N / 64) <= 1024;  // all workgroups of 64 columns within two rounds of the GPU's CUs
  const int64_t cols = small ? 64 : (N % 512 == 0 ? 512 : (N % 256 == 0 ? 256 : 128));
  const dim3 g(static_cast<unsigned>(N / cols), static_cast<unsigned>(blocks), static_cast<unsigned>(B));
  const hipStream_t st = as_stream(stream);
  const auto* pi = static_cast<const uint32_t*>(img);
  const auto *pw = static_cast<const half_t*>(w), *pb = static_cast<const half_t*>(bias_pos), *pc = static_cast<const half_t*>(cls);
  auto* px = static_cast<half_t*>(x);
  const int gi = static_cast<int>(grid), Ni = static_cast<int>(N), ci = static_cast<int>(cols);
  if (small)
    patch_embed_kernel<1><<<g, 256, 0, st>>>(pi, pw, pb, pc, gi, Ni, ci, px);
  else
    patch_embed_kernel<2><<<g, 256, 0, st>>>(pi, pw, pb, pc, gi, Ni, ci, px);
  return check_launch("patch_embed");
}
