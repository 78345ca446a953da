// The tag head: logits [B, N] = x [B, K] W^T + bias with a few rows of x and tens of thousands of tags, after an
// optional LayerNorm of x's rows (EVA02's final norm on the class tokens).
//
// W is read once and bounds the kernel (Haruka: 98 782 x 1152 fp16 = 228 MB, EVA02-L: 30 877 x 1024 = 63 MB), so the
// kernel is a weight stream: a persistent grid whose waves each take a 16-tag tile, load 12 of its 16 x 32 fragments
// straight from global memory into registers (12 KB in flight per wave) and multiply them with v_mfma_f32_16x16x32_f16
// by x's fragments, which every workgroup keeps in LDS in fragment order. x's rows are padded to 16, 32 or 64. Sums,
// bias and result stay fp32. Haruka's head at 16 images: 44.7-48 us (5.1-4.7 TB/s; the library product 89 us); EVA02-L's at
// one image 13.3 us with its norm (library 13.0, and five launches of 4-5 us for the norm and the casts).
#include <algorithm>

#include "common.h"

namespace ff {

constexpr int HD_KMAX = 1280;  // longest row of x: 16 rows take 40 KB of LDS
constexpr int HD_FRAGS = 12;   // W fragments a wave loads at once

// NB: 16-row tiles of x.
template <int NB>
__global__ __launch_bounds__(512, NB == 1 ? 6 : 2) void head_kernel(const half_t* __restrict__ x, int64_t x_stride,
                                                                    const float* __restrict__ gamma,
                                                                    const float* __restrict__ beta, float eps,
                                                                    const half_t* __restrict__ W,
                                                                    const half_t* __restrict__ bias, int B, int N, int K,
                                                                    float* __restrict__ out) {
  __shared__ half8_t xs[NB * 2 * HD_KMAX];  // fragment s of row tile nb, lane l: [(s NB + nb) 64 + l]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int steps = K / 32;
  // Lane l of a fragment holds row l % 16, columns 32 s + 8 (l / 16) .. + 7: chunk c = 4 s + l / 16 of 8 columns.
  if (gamma) {
    for (int r = wave; r < 16 * NB; r += 8) {  // one wave per row; lane l takes chunks l, l + 64, ...
      half8_t h[HD_KMAX / 512 + 1];
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < HD_KMAX / 512 + 1; ++k) {
        const int c = lane + 64 * k;
        h[k] = r < B && c < K / 8 ? *reinterpret_cast<const half8_t*>(x + r * x_stride + 8 * c) : half8_t{};
#pragma unroll
        for (int e = 0; e < 8; ++e) s += static_cast<float>(h[k][e]);
      }
      const float mean = wave_sum(s) / static_cast<float>(K);
      float q = 0.f;
#pragma unroll
      for (int k = 0; k < HD_KMAX / 512 + 1; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = lane + 64 * k < K / 8 ? static_cast<float>(h[k][e]) - mean : 0.f;
          q = __builtin_fmaf(d, d, q);
        }
      const float rstd = 1.f / sqrtf(wave_sum(q) / static_cast<float>(K) + eps);
#pragma unroll
      for (int k = 0; k < HD_KMAX / 512 + 1; ++k) {
        const int c = lane + 64 * k;
        if (c < K / 8) {
          half8_t y = {};
          if (r < B) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              y[e] = static_cast<half_t>((static_cast<float>(h[k][e]) - mean) * rstd * gamma[8 * c + e] + beta[8 * c + e]);
          }
          xs[((c >> 2) * NB + (r >> 4)) * 64 + (c & 3) * 16 + (r & 15)] = y;
        }
      }
    }
  } else {
    for (int i = threadIdx.x; i < 16 * NB * (K / 8); i += 512) {
      const int r = i / (K / 8), c = i % (K / 8);
      xs[((c >> 2) * NB + (r >> 4)) * 64 + (c & 3) * 16 + (r & 15)] =
          r < B ? *reinterpret_cast<const half8_t*>(x + r * x_stride + 8 * c) : half8_t{};
    }
  }
  __syncthreads();
  const int tiles = (N + 15) / 16, stride = static_cast<int>(gridDim.x) * 8;
  const int i16 = lane & 15, kq = lane >> 4;
  for (int t = static_cast<int>(blockIdx.x) * 8 + wave; t < tiles; t += stride) {
    const int n = 16 * t + i16;
    const half_t* w = W + static_cast<int64_t>(min(n, N - 1)) * K + 8 * kq;  // rows past N repeat the last, unstored
    float4_t acc[NB] = {};
    int s = 0;
    for (; s + HD_FRAGS <= steps; s += HD_FRAGS) {
      half8_t f[HD_FRAGS];
#pragma unroll
      for (int j = 0; j < HD_FRAGS; ++j) f[j] = *reinterpret_cast<const half8_t*>(w + 32 * (s + j));
#pragma unroll
      for (int j = 0; j < HD_FRAGS; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[((s + j) * NB + b) * 64 + lane], f[j], acc[b], 0, 0, 0);
    }
    for (; s + 4 <= steps; s += 4) {
      half8_t f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const half8_t*>(w + 32 * (s + j));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[((s + j) * NB + b) * 64 + lane], f[j], acc[b], 0, 0, 0);
    }
    for (; s < steps; ++s) {
      const half8_t f = *reinterpret_cast<const half8_t*>(w + 32 * s);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[(s * NB + b) * 64 + lane], f, acc[b], 0, 0, 0);
    }
    // acc[b][i]: row 16 b + 4 (lane / 16) + i of x, tag n
    if (n < N) {
      const float bn = static_cast<float>(bias[n]);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * b + 4 * kq + i;
          if (r < B) out[static_cast<int64_t>(r) * N + n] = acc[b][i] + bn;
        }
    }
  }
}

template <int NB>
static void launch_head(hipStream_t st, const half_t* x, int64_t xs, const float* g, const float* be, float eps,
                        const half_t* W, const half_t* bias, int B, int N, int K, float* out) {
  int64_t resident = resident_blocks(reinterpret_cast<const void*>(&head_kernel<NB>), 512, 0);
  if (resident <= 0) resident = 256;
  const int64_t need = ((N + 15) / 16 + 7) / 8;  // eight tiles per workgroup and turn
  head_kernel<NB><<<dim3(static_cast<unsigned>(std::min(need, resident))), 512, 0, st>>>(x, xs, g, be, eps, W, bias, B, N,
                                                                                        K, out);
}

}  // namespace ff

using namespace ff;

extern "C" int ff_head(const void* x, int64_t x_stride, const float* gamma, const float* beta, float eps, const void* W,
                       const void* bias, int64_t B, int64_t N, int64_t K, float* out, void* stream) {
  clear_error();
  if (B < 0 || B > 64) return fail(FF_EINVAL, "head: need 0 <= B <= 64");
  if (N <= 0 || N > 0x7fffff00) return fail(FF_EINVAL, "head: bad N");
  if (K <= 0 || K % 32 != 0 || K > HD_KMAX) return fail(FF_EINVAL, "head: need K % 32 == 0 and K <= 1280");
  if (x_stride < K || x_stride % 8 != 0) return fail(FF_EINVAL, "head: need x_stride >= K, a multiple of 8");
  if ((gamma == nullptr) != (beta == nullptr)) return fail(FF_EINVAL, "head: gamma and beta go together");
  if (gamma && !(eps > 0.f)) return fail(FF_EINVAL, "head: eps must be > 0");
  if (B == 0) return FF_OK;
  if (!x || !W || !bias || !out) return fail(FF_EINVAL, "head: null pointer");
  if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(W) & 15))
    return fail(FF_EINVAL, "head: misaligned pointer");
  const hipStream_t st = as_stream(stream);
  const auto *px = static_cast<const half_t*>(x), *pw = static_cast<const half_t*>(W), *pb = static_cast<const half_t*>(bias);
  const int Bi = static_cast<int>(B), Ni = static_cast<int>(N), Ki = static_cast<int>(K);
  if (B <= 16)
    launch_head<1>(st, px, x_stride, gamma, beta, eps, pw, pb, Bi, Ni, Ki, out);
  else if (B <= 32)
    launch_head<2>(st, px, x_stride, gamma, beta, eps, pw, pb, Bi, Ni, Ki, out);
  else
    launch_head<4>(st, px, x_stride, gamma, beta, eps, pw, pb, Bi, Ni, Ki, out);
  return check_launch("head");
}
