// Haruka's tree pool (foidfinder/backends/mlx/haruka.py:101-136) as a chain of a few launches. With keys and values
// never formed (logits = xn . u, u = Wk_h^T q; pooled = w^T xn, then Wv_h), the two attention levels each take:
//
//  * pool_weights: logits xn u^T on MFMA and from them the slot-sigmoid weights, transposed, in one kernel;
//  * pool_sum: the pooling product w^T xn;
//  * pool_values: the value projection of the pooled tokens plus the value bias times each query's mass;
//
// and between and after them: pool_queries (parent norm, leaf queries), pool_keys (the leaf queries' u), pool_tree (leaf
// norm times the mass gate) and pool_leaf (each leaf's own projection). At 16 images these kernels take the place of some
// 40 launches of 4-13 us, most of them a few hundred KB of element-wise work (the whole pool head 409 -> 195 us).
// The small ones (values 5.5-8.6, queries 9.0, keys 9.5, tree 9.1, leaf 5.4 us) are bounded by their launch and the round
// trips of operands that the launch before wrote.
#include <algorithm>

#include "common.h"

namespace ff {

typedef __attribute__((address_space(3))) void lds_void;
constexpr uint32_t RSRC_WORD3 = 0x00020000;  // buffer descriptor word 3: raw dword access (gfx9 family)

__device__ __forceinline__ void to_lds(const void* base, int nbytes, void* lds_dst, uint32_t voff) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, nbytes, RSRC_WORD3);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds_dst, 16, voff, 0, 0, 0);
}

constexpr int PW_TOK = 96;   // tokens per workgroup of pool_weights
constexpr int PW_SLOTS = 5;  // its LDS ring's depth

// A workgroup per (batch, block of 96 tokens). Logits of the block's tokens against all GM = G M query columns: u [GM, D] and xn
// stream through five LDS slots of 32 columns (64-byte rows, 16-byte chunks XOR-swizzled by row bits 2-3 for
// conflict-free fragment reads) filled by buffer->LDS loads, four slots ahead: both were written by the launches before,
// through other L2s, and a load takes ~0.8 us (16 x 1025 tokens, 288 columns: 24.2 us, two slots ahead 33.7; 96 columns:
// 12.3; as a library product and slot_weights 40.3 and 23.1). Rows past
// GM or the sequence read as zeros. A wave takes one 32-query tile (MFMA rows) and NT of the block's three 32-token tiles
// (MFMA columns): nine waves of three at Haruka's 288 leaf columns, nine of one at its 96 coarse columns. The fp32 logits
// go to LDS as [GM][96 + 1]; a thread then turns the M logits of a (token, head) pair into weights in place: softmax over
// the queries times sigmoid(logit + bias), from the hardware exp2 and reciprocal (each about 1 ulp). Tokens past the
// sequence get weight 0. partial[b, block, j] is column j's sum over the block's tokens, a_t[b, j, n] the weight in fp16
// (rows of ldt, their pad columns 0). GMAX bounds GM. 96 tokens, not 64: 1025 are 11 blocks then, 176 workgroups at 16
// images, one per CU, where 17 blocks would be 272, the last ones with a token each.
template <int GMAX, int NT>
constexpr int pw_waves() {
  return GMAX / 32 * (PW_TOK / 32 / NT);
}
template <int M, int GMAX, int NT>
__global__ __launch_bounds__(64 * (pw_waves<GMAX, NT>())) void pool_weights_kernel(
    const half_t* __restrict__ xn, const half_t* __restrict__ u, int64_t u_stride, const float* __restrict__ c,
    int64_t c_stride, const float* __restrict__ bias, int N, int G, int D, int ldt, half_t* __restrict__ a_t,
    float* __restrict__ partial) {
  constexpr int WV = pw_waves<GMAX, NT>(), THREADS = 64 * WV;
  constexpr int LOADS = (GMAX + PW_TOK) / 16;     // 1 KB loads per slot: 16 rows each, queries, then tokens
  constexpr int PER = (LOADS + WV - 1) / WV;      // per wave, the last only in waves below LOADS % WV (0: all)
  constexpr int SLOT = LOADS * 1024, SLOTS = PW_SLOTS;
  constexpr int LDT = PW_TOK + 1;
  constexpr int BYTES = SLOTS * SLOT > GMAX * LDT * 4 ? SLOTS * SLOT : GMAX * LDT * 4;
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[BYTES];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // 1-D grid over (batch, token block), remapped so that a batch's blocks share one XCD's L2 for its u
  const int blocks = (N + PW_TOK - 1) / PW_TOK, t = xcd_remap(blockIdx.x, gridDim.x);
  const int GM = G * M, b = t / blocks, blk = t % blocks, n0 = blk * PW_TOK;
  const int ntok = min(PW_TOK, N - n0);
  const half_t* ub = u + b * u_stride;
  const half_t* xb = xn + (static_cast<int64_t>(b) * N + n0) * D;
  const int u_bytes = GM * D * 2, x_bytes = ntok * D * 2;
  const bool full = wave + WV * (PER - 1) < LOADS;  // this wave issues PER loads per slot, else PER - 1

  auto issue = [&](int kc) __attribute__((always_inline)) {
    uint8_t* dst = lds + kc % SLOTS * SLOT;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int q = wave + WV * p;  // wave-uniform
      if (p == PER - 1 && !full) break;
      const bool tok = q >= GMAX / 16;
      const int row = 16 * q + (lane >> 2) - (tok ? GMAX : 0);
      to_lds(tok ? xb : ub, tok ? x_bytes : u_bytes, dst + q * 1024,
             static_cast<uint32_t>(row * D * 2 + kc * 64 + (((lane & 3) ^ ((row >> 2) & 3)) << 4)));
    }
  };
  auto frag = [&](const uint8_t* base, int row, int chunk) __attribute__((always_inline)) {
    return *reinterpret_cast<const half8_t*>(base + row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4));
  };
  constexpr int TS = PW_TOK / 32 / NT;  // waves per query tile
  const int qt = wave / TS, t0 = wave % TS * NT, fr = lane & 31, fh = lane >> 5;
  float16_t acc[NT] = {};
  const int chunks = D / 32;  // at least four (D % 128 == 0)
#pragma unroll
  for (int i = 0; i < SLOTS - 1; ++i)
    if (i < chunks) issue(i);
  for (int kc = 0; kc < chunks; ++kc) {
    // slot kc has landed once only the SLOTS - 2 slots after it have loads outstanding
    if (kc + SLOTS - 2 >= chunks)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else if (full)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SLOTS - 2) * PER) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SLOTS - 2) * (PER - 1)) : "memory");
    __builtin_amdgcn_s_barrier();  // and every wave has read slot kc - 1, which slot kc + SLOTS - 1 takes over
    asm volatile("" ::: "memory");
    const uint8_t* su = lds + kc % SLOTS * SLOT;
    const uint8_t* sx = su + GMAX * 64;
    half8_t uf[2], xf[2][NT];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      uf[ks] = frag(su, 32 * qt + fr, 2 * ks + fh);
#pragma unroll
      for (int i = 0; i < NT; ++i) xf[ks][i] = frag(sx, 32 * (t0 + i) + fr, 2 * ks + fh);
    }
    if (kc + SLOTS - 1 < chunks) issue(kc + SLOTS - 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(uf[ks], xf[ks][i], acc[i], 0, 0, 0);
  }
  __syncthreads();  // the slots are read: the logits take their place
  float* tile = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = 32 * qt + 8 * (r >> 2) + 4 * fh + (r & 3);
      if (j < GM) tile[j * LDT + 32 * (t0 + i) + fr] = acc[i][r];
    }
  const float* cb = c + b * c_stride;
  __syncthreads();
  for (int p = threadIdx.x; p < PW_TOK * G; p += THREADS) {
    const int t = p % PW_TOK, h = p / PW_TOK;
    float l[M], w[M], mx = -INFINITY, s = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      l[m] = tile[(h * M + m) * LDT + t] + cb[h * M + m];
      mx = fmaxf(mx, l[m]);
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      w[m] = __builtin_amdgcn_exp2f((l[m] - mx) * LOG2E);
      s += w[m];
    }
    const float inv = __builtin_amdgcn_rcpf(s);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float gate = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(__builtin_fmaf(-l[m], LOG2E, -bias[m] * LOG2E)));
      tile[(h * M + m) * LDT + t] = t < ntok ? w[m] * inv * gate : 0.f;
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < GM; j += THREADS) {
    float s = 0.f;
#pragma unroll 8
    for (int t = 0; t < PW_TOK; ++t) s += tile[j * LDT + t];
    partial[(static_cast<int64_t>(b) * blocks + blk) * GM + j] = s;
  }
  // a query row per wave and pass, two tokens (4 bytes) per lane, up to the row's (even) pitch: past the sequence the
  // tile holds zeros
  const int t2 = 2 * lane;
  if (t2 < PW_TOK && t2 < ldt - n0)
    for (int j = wave; j < GM; j += WV)
      *reinterpret_cast<half2_t*>(a_t + (static_cast<int64_t>(b) * GM + j) * ldt + n0 + t2) =
          half2_t{static_cast<half_t>(tile[j * LDT + t2]), static_cast<half_t>(tile[j * LDT + t2 + 1])};
}

// pooled[b, j, d] = sum_n a_t[b, j, n] xn[b, n, d]: a workgroup per (batch, 96 queries j, 64 SUB columns d), wave w the 32
// columns 32 w against the three 32-query tiles (columns as MFMA rows, queries as columns), the tokens in chunks of 64
// through four LDS slots, three ahead (a load takes ~0.8 us: its rows come from other L2s). xn's rows are the product's k:
// its fragments come through the transposing ds_read_b64_tr_b16, which hands a lane 4 consecutive tokens of one column
// (slot u of lane half f: token 8 f + u of 16, so that a_t's fragments are 16-byte reads; 8-byte ones, which conflict
// two ways, made LDS the bound at 21 and 23 us a launch). Tokens past the sequence
// read as zero rows of xn against finite weights (a_t's zero pad, or the next row); queries past GM read as zeros and are
// not stored. SUB = 3 where 192 divides D (Haruka's 768: 64 and 192 workgroups at 16 images for the 96 coarse and 288 leaf
// queries, one per CU), else 2.
// 16 images, 96 and 288 queries, per launch: 17.1 and 19.0 us; as a library product 15.9 and 28.2; two slots of 128
// columns 16.0 and 21.3.
constexpr int PS_J = 96, PS_N = 64, PS_SLOTS = 4;

// The eight transposing reads of a chunk's 64 tokens, four columns' 16 tokens in x[tt][0] (tokens 0-3 of each lane half's 8)
// and x[tt][1] (4-7), and the wait for them. One block: the results are the compiler's only once they have arrived, and
// (as inline asm) its wait-insertion pass does not drain the buffer->LDS loads in flight before them.
__device__ __forceinline__ void tr_read_chunk(half4_t (&x)[4][2], uint32_t lds_addr) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:512\n\t"
      "ds_read_b64_tr_b16 %2, %8 offset:2048\n\t"
      "ds_read_b64_tr_b16 %3, %8 offset:2560\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:4096\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:4608\n\t"
      "ds_read_b64_tr_b16 %6, %8 offset:6144\n\t"
      "ds_read_b64_tr_b16 %7, %8 offset:6656\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[2][0]), "=&v"(x[2][1]), "=&v"(x[3][0]),
        "=&v"(x[3][1])
      : "v"(lds_addr)
      : "memory");
}

template <int SUB>
__global__ __launch_bounds__(128 * SUB) void pool_sum_kernel(const half_t* __restrict__ a_t, const half_t* __restrict__ xn,
                                                             int N, int GM, int D, int ldt,
                                                             half_t* __restrict__ pooled) {
  constexpr int WV = 2 * SUB, XB = PS_N * 128;             // waves; bytes of 64 columns of a chunk (rows of 128)
  constexpr int LOADS = SUB * 8 + PS_J * PS_N * 2 / 1024;  // 1 KB loads per slot, 8 rows each: xn by 64 columns, then a_t
  constexpr int PER = LOADS / WV, SLOT = LOADS * 1024;
  static_assert(LOADS % WV == 0, "every wave issues as many loads");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[PS_SLOTS * SLOT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 31, fh = lane >> 5;
  // 1-D grid over (batch, query tile, column tile), a batch's workgroups on one XCD
  const int td = D / (64 * SUB), tj = (GM + PS_J - 1) / PS_J, t = xcd_remap(blockIdx.x, gridDim.x);
  const int b = t / (td * tj), j0 = t / td % tj * PS_J, d0 = t % td * 64 * SUB;
  const half_t* xb = xn + static_cast<int64_t>(b) * N * D + d0;
  const half_t* ab = a_t + (static_cast<int64_t>(b) * GM + j0) * ldt;
  const int a_bytes = (GM - j0) * ldt * 2;

  // 16-byte chunk c of row r sits at slot c ^ 2 (r & 2) of xn's rows (the four rows of a transposing read on distinct
  // banks) and at c ^ ((r >> 1) & 7) of a_t's
  auto issue = [&](int chunk) __attribute__((always_inline)) {
    uint8_t* dst = lds + chunk % PS_SLOTS * SLOT;
    const int n0 = chunk * PS_N;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int q = wave + WV * p;  // wave-uniform
      if (q < 8 * SUB) {
        const int r = 8 * (q & 7) + (lane >> 3), c = (lane & 7) ^ ((r & 2) << 1);
        to_lds(xb + static_cast<int64_t>(n0) * D, (N - n0) * D * 2 - d0 * 2, dst + q * 1024,
               static_cast<uint32_t>(r * D * 2 + (q >> 3) * 128 + c * 16));
      } else {
        const int r = 8 * (q - 8 * SUB) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        to_lds(ab, a_bytes, dst + q * 1024, static_cast<uint32_t>(r * ldt * 2 + n0 * 2 + c * 16));
      }
    }
  };
  const int row = 8 * fh + ((lane & 15) >> 2), col = 32 * (wave & 1) + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const uint32_t xoff =
      static_cast<uint32_t>((wave >> 1) * XB + row * 128 + (((col >> 3) ^ ((row & 2) << 1)) << 4) + (col & 7) * 2);
  float16_t acc[3] = {};
  const int chunks = (N + PS_N - 1) / PS_N;
#pragma unroll
  for (int i = 0; i < PS_SLOTS - 1; ++i)
    if (i < chunks) issue(i);
  for (int k = 0; k < chunks; ++k) {
    // chunk k has landed once only the PS_SLOTS - 2 chunks after it have loads outstanding
    if (k + PS_SLOTS - 2 >= chunks)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((PS_SLOTS - 2) * PER) : "memory");
    __builtin_amdgcn_s_barrier();  // and every wave has read chunk k - 1
    asm volatile("" ::: "memory");
    if (k + PS_SLOTS - 1 < chunks) issue(k + PS_SLOTS - 1);
    const uint8_t* sl = lds + k % PS_SLOTS * SLOT;
    const uint32_t xa = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)sl)) + xoff;
    half8_t w[4][3];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int r = 32 * i + fr;
        w[tt][i] = *reinterpret_cast<const half8_t*>(sl + SUB * XB + r * 128 + (((2 * tt + fh) ^ ((r >> 1) & 7)) << 4));
      }
    half4_t x[4][2];
    tr_read_chunk(x, xa);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      const half4_t lo = x[tt][0], hi = x[tt][1];
      const half8_t xf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf, w[tt][i], acc[i], 0, 0, 0);
    }
  }
  // acc[i][4 q + e]: column d0 + 32 wave + 8 q + 4 (lane / 32) + e of query j0 + 32 i + lane % 32
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int j = j0 + 32 * i + fr;
    if (j >= GM) continue;
    half_t* o = pooled + (static_cast<int64_t>(b) * GM + j) * D + d0 + 32 * wave + 4 * fh;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      half4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = static_cast<half_t>(acc[i][4 * q + e]);
      *reinterpret_cast<half4_t*>(o + 8 * q) = v;
    }
  }
}

// One 16 x 16 product tile over K (K % 32 == 0, columns contiguous) by 4 waves: wave w takes the 32-column steps w,
// w + 4, ...; lane l's pointers are at its row (l % 16) and column 8 (l / 16). The waves' sums meet in LDS; every lane of
// wave 0 returns D[a row 4 (l / 16) + i][b row l % 16].
__device__ __forceinline__ float4_t tile16(const half_t* a, const half_t* b, int K, float4_t (&part)[4][64]) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float4_t acc = {};
  const int steps = K / 32;
#pragma unroll 6
  for (int s = wave; s < steps; s += 4)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const half8_t*>(a + 32 * s),
                                                 *reinterpret_cast<const half8_t*>(b + 32 * s), acc, 0, 0, 0);
  part[wave][lane] = acc;
  __syncthreads();
  return part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
}

// z[b, m, h hd + e] = sum_d pooled[b, h M + m, d] wv[h hd + e, d] + mass[b, h, m] bv[h hd + e], the mass summed from the
// weights' partial sums. Grid (hd / 16, ceil(B M / 16), G).
__global__ __launch_bounds__(256) void pool_values_kernel(const half_t* __restrict__ pooled, const half_t* __restrict__ wv,
                                                          const float* __restrict__ bv, const float* __restrict__ partial,
                                                          int nblk, int B, int G, int M, int hd, half_t* __restrict__ z) {
  __shared__ float4_t part[4][64];
  __shared__ float mass[16];
  const int lane = threadIdx.x & 63, D = G * hd, R = B * M;
  const int e0 = 16 * blockIdx.x, r0 = 16 * blockIdx.y, h = blockIdx.z;
  {
    const int r = min(r0 + static_cast<int>(threadIdx.x >> 4), R - 1);
    const float* p = partial + (static_cast<int64_t>(r / M) * nblk * G + h) * M + r % M;
    float s = 0.f;
    for (int k = threadIdx.x & 15; k < nblk; k += 16) s += p[static_cast<int64_t>(k) * G * M];
    s = s + dpp<DPP_XOR15>(s);
    s = s + dpp<DPP_XOR7>(s);
    s = s + dpp<DPP_XOR3>(s);
    s = s + dpp<DPP_XOR1>(s);
    if ((threadIdx.x & 15) == 0) mass[threadIdx.x >> 4] = s;
  }
  const int r = min(r0 + (lane & 15), R - 1);
  const half_t* pa = wv + static_cast<int64_t>(h * hd + e0 + (lane & 15)) * D + 8 * (lane >> 4);
  const half_t* pb = pooled + (static_cast<int64_t>(r / M) * G * M + h * M + r % M) * D + 8 * (lane >> 4);
  const float4_t v = tile16(pa, pb, D, part);
  if (threadIdx.x >= 64 || r0 + (lane & 15) >= R) return;
  const int e = h * hd + e0 + 4 * (lane >> 4);
  half4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = static_cast<half_t>(__builtin_fmaf(mass[lane & 15], bv[e + i], v[i]));
  *reinterpret_cast<half4_t*>(z + static_cast<int64_t>(r0 + (lane & 15)) * D + e) = o;
}

struct Norm {
  const half_t *g, *b;
};

// Rows held two columns per lane and step, c = 2 (lane + 64 k), D <= 128 PER. The kernels load everything a row needs
// (operands, affine vectors) before their first reduction, so one round trip covers all of it.
template <int PER>
__device__ __forceinline__ void load_pairs(half2_t (&x)[PER], const half_t* row, int D) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = 2 * (lane + 64 * k);
    x[k] = c < D ? *reinterpret_cast<const half2_t*>(row + c) : half2_t{};
  }
}
// LayerNorm: v = (v - mean) rstd g + b. Columns past D hold zeros.
template <int PER>
__device__ __forceinline__ void norm_row(float (&v)[PER][2], int D, const half2_t (&g)[PER], const half2_t (&b)[PER],
                                         float eps) {
  const int lane = threadIdx.x & 63;
  float s = 0.f, q = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) s += v[k][0] + v[k][1];
  const float mean = wave_sum(s) / static_cast<float>(D);
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float d = 2 * (lane + 64 * k) < D ? v[k][e] - mean : 0.f;
      q = __builtin_fmaf(d, d, q);
    }
  const float rstd = 1.f / sqrtf(wave_sum(q) / static_cast<float>(D) + eps);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (2 * (lane + 64 * k) < D) {
#pragma unroll
      for (int e = 0; e < 2; ++e)
        v[k][e] = (v[k][e] - mean) * rstd * static_cast<float>(g[k][e]) + static_cast<float>(b[k][e]);
    }
  }
}
template <int PER>
__device__ __forceinline__ void store_row2(const float (&v)[PER][2], half_t* row, int D) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = 2 * (lane + 64 * k);
    if (c < D) *reinterpret_cast<half2_t*>(row + c) = half2_t{static_cast<half_t>(v[k][0]), static_cast<half_t>(v[k][1])};
  }
}

// One wave per (batch, leaf q): its parent is coarse query m = q C / Q. parent[b, m] = LN(z[b, m]; trunk), qleaf[b, q] =
// LN(parent + child[q]; childn), cq[b, h Q + q] = sum over head h's columns of qleaf bk (the keys' bias term).
template <int PER>
__global__ __launch_bounds__(64) void pool_queries_kernel(const half_t* __restrict__ z, Norm trunk,
                                                          const half_t* __restrict__ child, Norm childn,
                                                          const float* __restrict__ bk, float eps, int C, int Q, int G,
                                                          int D, half_t* __restrict__ parent, half_t* __restrict__ qleaf,
                                                          float* __restrict__ cq) {
  __shared__ float prod[128 * PER];
  const int q = blockIdx.x, b = blockIdx.y, lane = threadIdx.x, m = q / (Q / C), hd = D / G;
  half2_t x[PER], ch[PER], tg[PER], tb[PER], cg[PER], cb[PER];
  load_pairs(x, z + (static_cast<int64_t>(b) * C + m) * D, D);
  load_pairs(tg, trunk.g, D);
  load_pairs(tb, trunk.b, D);
  load_pairs(ch, child + static_cast<int64_t>(q) * D, D);
  load_pairs(cg, childn.g, D);
  load_pairs(cb, childn.b, D);
  float v[PER][2], kb[PER][2];
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      v[k][e] = static_cast<float>(x[k][e]);
      kb[k][e] = 2 * (lane + 64 * k) < D ? bk[2 * (lane + 64 * k) + e] : 0.f;
    }
  norm_row(v, D, tg, tb, eps);
  if (q % (Q / C) == 0) store_row2(v, parent + (static_cast<int64_t>(b) * C + m) * D, D);
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e)  // the parent as stored
      v[k][e] = static_cast<float>(static_cast<half_t>(v[k][e])) + static_cast<float>(ch[k][e]);
  norm_row(v, D, cg, cb, eps);
  store_row2(v, qleaf + (static_cast<int64_t>(b) * Q + q) * D, D);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = 2 * (lane + 64 * k);
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (c < D) prod[c + e] = static_cast<float>(static_cast<half_t>(v[k][e])) * kb[k][e];
  }
  __syncthreads();
  for (int h0 = 0; h0 < G; h0 += 16) {  // four lanes per head
    const int h = h0 + (lane >> 2);
    float s = 0.f;
    if (h < G)
      for (int e = lane & 3; e < hd; e += 4) s += prod[h * hd + e];
    s = s + dpp<DPP_XOR3>(s);
    s = s + dpp<DPP_XOR1>(s);
    if (h < G && (lane & 3) == 0) cq[(static_cast<int64_t>(b) * G + h) * Q + q] = s;
  }
}

// u[b, h Q + q, d] = sum_e qleaf[b, q, h hd + e] kT[h, d, e]: one wave per 16 (batch, query) rows x 64 columns d of a head,
// K = hd in steps of 16 (v_mfma_f32_16x16x16_f16: lane l holds 4 columns 4 (l / 16) .. of row l % 16). Grid
// (ceil(D / 256), ceil(B Q / 16), G), wave w the w-th 64 columns.
__global__ __launch_bounds__(256) void pool_keys_kernel(const half_t* __restrict__ qleaf, const half_t* __restrict__ kT,
                                                        int B, int Q, int G, int hd, half_t* __restrict__ u) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, D = G * hd, R = B * Q;
  const int d0 = 256 * blockIdx.x + 64 * wave, r0 = 16 * blockIdx.y, h = blockIdx.z, i16 = lane & 15, kq = lane >> 4;
  if (d0 >= D) return;
  const int r = min(r0 + i16, R - 1);
  const half_t* pq = qleaf + static_cast<int64_t>(r) * D + h * hd + 4 * kq;
  float4_t acc[4] = {};
#pragma unroll 3
  for (int k = 0; k < hd; k += 16) {
    const half4_t x = *reinterpret_cast<const half4_t*>(pq + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = min(d0 + 16 * i + i16, D - 1);
      const half4_t w = *reinterpret_cast<const half4_t*>(kT + (static_cast<int64_t>(h) * D + d) * hd + 4 * kq + k);
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x16f16(w, x, acc[i], 0, 0, 0);
    }
  }
  if (r0 + i16 >= R) return;
  half_t* o = u + (static_cast<int64_t>(r / Q) * G * Q + h * Q + r % Q) * D + d0 + 4 * kq;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (d0 + 16 * i >= D) break;
    half4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = static_cast<half_t>(acc[i][e]);
    *reinterpret_cast<half4_t*>(o + 16 * i) = v;
  }
}

// One wave per (batch, leaf): tree[q, b] = LN(parent[b, q C / Q] + zc[b, q]; leafn) * mass / (mass + 4), mass the leaf's
// weight sum averaged over the heads.
template <int PER>
__global__ __launch_bounds__(64) void pool_tree_kernel(const half_t* __restrict__ parent, const half_t* __restrict__ zc,
                                                       Norm leafn, const float* __restrict__ partial, int nblk, float eps,
                                                       int C, int Q, int G, int D, half_t* __restrict__ tree) {
  const int q = blockIdx.x, b = blockIdx.y, B = gridDim.y, lane = threadIdx.x;
  half2_t x[PER], y[PER], g[PER], be[PER];
  load_pairs(x, parent + (static_cast<int64_t>(b) * C + q / (Q / C)) * D, D);
  load_pairs(y, zc + (static_cast<int64_t>(b) * Q + q) * D, D);
  load_pairs(g, leafn.g, D);
  load_pairs(be, leafn.b, D);
  float s = 0.f;
#pragma unroll 5
  for (int i = lane; i < nblk * G; i += 64) s += partial[(static_cast<int64_t>(b) * nblk * G + i) * Q + q];
  const float mass = wave_sum(s) / static_cast<float>(G);
  float v[PER][2];
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e) v[k][e] = static_cast<float>(x[k][e]) + static_cast<float>(y[k][e]);
  norm_row(v, D, g, be, eps);
  const float gate = mass / (mass + 4.f);
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int e = 0; e < 2; ++e) v[k][e] = v[k][e] * gate;
  store_row2(v, tree + (static_cast<int64_t>(q) * B + b) * D, D);
}

// leaf[b, q F + f] = sum_d tree[q, b, d] wl[q, f, d] + bl[q, f]. Grid (F / 16, ceil(B / 16), Q).
__global__ __launch_bounds__(256) void pool_leaf_kernel(const half_t* __restrict__ tree, const half_t* __restrict__ wl,
                                                        const half_t* __restrict__ bl, int B, int Q, int F, int D,
                                                        half_t* __restrict__ leaf) {
  __shared__ float4_t part[4][64];
  const int lane = threadIdx.x & 63, f0 = 16 * blockIdx.x, b0 = 16 * blockIdx.y, q = blockIdx.z;
  const int b = min(b0 + (lane & 15), B - 1);
  const float4_t v = tile16(wl + (static_cast<int64_t>(q) * F + f0 + (lane & 15)) * D + 8 * (lane >> 4),
                            tree + (static_cast<int64_t>(q) * B + b) * D + 8 * (lane >> 4), D, part);
  if (threadIdx.x >= 64 || b0 + (lane & 15) >= B) return;
  const int f = q * F + f0 + 4 * (lane >> 4);
  half4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = static_cast<half_t>(v[i] + static_cast<float>(bl[f + i]));
  *reinterpret_cast<half4_t*>(leaf + static_cast<int64_t>(b) * Q * F + f) = o;
}

}  // namespace ff

using namespace ff;

static bool al(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// The shapes all of the pool's kernels share: D = G hd columns in whole 32-column steps and 16-column head tiles.
static const char* pool_shape(int64_t B, int64_t G, int64_t D) {
  if (B < 0 || B > 65535) return "need 0 <= B <= 65535";
  if (G <= 0 || G > 64 || D <= 0 || D > 2048 || D % 128 != 0 || D % G != 0 || (D / G) % 16 != 0)
    return "need 0 < G <= 64 heads of a multiple of 16 columns, D % 128 == 0, D <= 2048";
  return nullptr;
}
#define FF_POOL_CHECK(name, ...)                                                        \
  if (const char* m = pool_shape(__VA_ARGS__)) return fail(FF_EINVAL, std::string(name ": ") + m)

extern "C" int64_t ff_pool_weights_blocks(int64_t N) { return N > 0 ? (N + PW_TOK - 1) / PW_TOK : 0; }

extern "C" int ff_pool_weights(const void* xn, const void* u, int64_t u_stride, const float* c, int64_t c_stride,
                               const float* bias, int64_t B, int64_t N, int64_t G, int64_t M, int64_t D, int64_t ldt,
                               void* a_t, float* partial, void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_weights", B, G, D);
  if (N <= 0 || N > (int64_t(1) << 30) / D) return fail(FF_EINVAL, "pool_weights: need 0 < N * D <= 2^30");
  if (M != 6 && M != 18) return fail(FF_EINVAL, "pool_weights: M must be 6 or 18 (the tree pool's query counts)");
  if (G * M > 384) return fail(FF_EINVAL, "pool_weights: G*M above 384");
  if ((u_stride != 0 && u_stride < G * M * D) || u_stride % 8 != 0 || (c_stride != 0 && c_stride < G * M))
    return fail(FF_EINVAL, "pool_weights: u_stride must be 0 or >= G*M*D, c_stride 0 or >= G*M");
  if (ldt < N || ldt % 2 != 0 || ldt > (N + 7) / 8 * 8)
    return fail(FF_EINVAL, "pool_weights: need ldt even and N <= ldt <= the next multiple of 8");
  if (B == 0) return FF_OK;
  if (!xn || !u || !c || !bias || !a_t || !partial) return fail(FF_EINVAL, "pool_weights: null pointer");
  if (!al(xn, 16) || !al(u, 16) || !al(a_t, 4)) return fail(FF_EINVAL, "pool_weights: misaligned pointer");
  const int64_t blocks = ff_pool_weights_blocks(N) * B;
  if (blocks > 0x7fffffff) return fail(FF_EINVAL, "pool_weights: too many token blocks");
  const dim3 grid(static_cast<unsigned>(blocks));
  const hipStream_t st = as_stream(stream);
  const auto *px = static_cast<const half_t*>(xn), *pu = static_cast<const half_t*>(u);
  auto* pa = static_cast<half_t*>(a_t);
  const int Ni = static_cast<int>(N), Gi = static_cast<int>(G), Di = static_cast<int>(D), li = static_cast<int>(ldt);
#define FF_PW(MM, GMAX, NT)                                                                                           \
  pool_weights_kernel<MM, GMAX, NT><<<grid, 64 * (pw_waves<GMAX, NT>()), 0, st>>>(px, pu, u_stride, c, c_stride, bias, \
                                                                                  Ni, Gi, Di, li, pa, partial)
  if (M == 6 && G * M <= 96)
    FF_PW(6, 96, 1);
  else if (M == 6)
    FF_PW(6, 384, 3);
  else if (G * M <= 288)
    FF_PW(18, 288, 3);
  else
    FF_PW(18, 384, 3);
#undef FF_PW
  return check_launch("pool_weights");
}

extern "C" int ff_pool_sum(const void* a_t, const void* xn, int64_t B, int64_t N, int64_t GM, int64_t D, int64_t ldt,
                           void* pooled, void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_sum", B, 1, D);
  // a batch's tokens and weights span less than 2^31 bytes: their lengths are signed 32-bit numbers in the kernel
  if (N <= 0 || N >= ((int64_t(1) << 30) + D - 1) / D) return fail(FF_EINVAL, "pool_sum: need 0 < N * D < 2^30");
  if (GM <= 0 || GM > 512) return fail(FF_EINVAL, "pool_sum: need 0 < GM <= 512");
  if (ldt != (N + 7) / 8 * 8) return fail(FF_EINVAL, "pool_sum: ldt must be N rounded up to a multiple of 8");
  if (GM * ldt >= (int64_t(1) << 30)) return fail(FF_EINVAL, "pool_sum: need GM * ldt < 2^30");
  if (B == 0) return FF_OK;
  if (!a_t || !xn || !pooled) return fail(FF_EINVAL, "pool_sum: null pointer");
  if (!al(a_t, 16) || !al(xn, 16) || !al(pooled, 8)) return fail(FF_EINVAL, "pool_sum: misaligned pointer");
  const int sub = D % 192 == 0 ? 3 : 2;
  const int64_t blocks = B * ((GM + PS_J - 1) / PS_J) * (D / (64 * sub));
  if (blocks > 0x7fffffff) return fail(FF_EINVAL, "pool_sum: too many tiles");
  const dim3 grid(static_cast<unsigned>(blocks));
  const auto *pa = static_cast<const half_t*>(a_t), *px = static_cast<const half_t*>(xn);
  auto* po = static_cast<half_t*>(pooled);
  const int Ni = static_cast<int>(N), Gi = static_cast<int>(GM), Di = static_cast<int>(D), li = static_cast<int>(ldt);
  if (sub == 3)
    pool_sum_kernel<3><<<grid, 384, 0, as_stream(stream)>>>(pa, px, Ni, Gi, Di, li, po);
  else
    pool_sum_kernel<2><<<grid, 256, 0, as_stream(stream)>>>(pa, px, Ni, Gi, Di, li, po);
  return check_launch("pool_sum");
}

extern "C" int ff_pool_values(const void* pooled, const void* wv, const float* bv, const float* partial, int64_t nblk,
                              int64_t B, int64_t G, int64_t M, int64_t D, void* z, void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_values", B, G, D);
  if (M <= 0 || M > 64 || nblk <= 0 || nblk > (1 << 24)) return fail(FF_EINVAL, "pool_values: bad M or nblk");
  const int64_t rows = (B * M + 15) / 16;
  if (rows > 65535) return fail(FF_EINVAL, "pool_values: B*M too large");
  if (B == 0) return FF_OK;
  if (!pooled || !wv || !bv || !partial || !z) return fail(FF_EINVAL, "pool_values: null pointer");
  if (!al(pooled, 16) || !al(wv, 16) || !al(z, 8)) return fail(FF_EINVAL, "pool_values: misaligned pointer");
  const int hd = static_cast<int>(D / G);
  const dim3 grid(static_cast<unsigned>(hd / 16), static_cast<unsigned>(rows), static_cast<unsigned>(G));
  pool_values_kernel<<<grid, 256, 0, as_stream(stream)>>>(
      static_cast<const half_t*>(pooled), static_cast<const half_t*>(wv), bv, partial, static_cast<int>(nblk),
      static_cast<int>(B), static_cast<int>(G), static_cast<int>(M), hd, static_cast<half_t*>(z));
  return check_launch("pool_values");
}

extern "C" int ff_pool_queries(const void* z, const void* trunk_g, const void* trunk_b, const void* child,
                               const void* child_g, const void* child_b, const float* bk, float eps, int64_t B, int64_t C,
                               int64_t Q, int64_t G, int64_t D, void* parent, void* qleaf, float* cq, void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_queries", B, G, D);
  if (C <= 0 || Q <= 0 || Q > 65535 || Q % C != 0) return fail(FF_EINVAL, "pool_queries: need C | Q");
  if (!(eps > 0.f)) return fail(FF_EINVAL, "pool_queries: eps must be > 0");
  if (B == 0) return FF_OK;
  if (!z || !trunk_g || !trunk_b || !child || !child_g || !child_b || !bk || !parent || !qleaf || !cq)
    return fail(FF_EINVAL, "pool_queries: null pointer");
  for (const void* p : {z, trunk_g, trunk_b, child, child_g, child_b, const_cast<const void*>(parent),
                        const_cast<const void*>(qleaf)})
    if (!al(p, 4)) return fail(FF_EINVAL, "pool_queries: misaligned pointer");
  const dim3 grid(static_cast<unsigned>(Q), static_cast<unsigned>(B));
  const Norm t{static_cast<const half_t*>(trunk_g), static_cast<const half_t*>(trunk_b)};
  const Norm n{static_cast<const half_t*>(child_g), static_cast<const half_t*>(child_b)};
  const auto *pz = static_cast<const half_t*>(z), *pc = static_cast<const half_t*>(child);
  auto *pp = static_cast<half_t*>(parent), *pq = static_cast<half_t*>(qleaf);
  const int Ci = static_cast<int>(C), Qi = static_cast<int>(Q), Gi = static_cast<int>(G), Di = static_cast<int>(D);
  if (D <= 768)
    pool_queries_kernel<6><<<grid, 64, 0, as_stream(stream)>>>(pz, t, pc, n, bk, eps, Ci, Qi, Gi, Di, pp, pq, cq);
  else
    pool_queries_kernel<16><<<grid, 64, 0, as_stream(stream)>>>(pz, t, pc, n, bk, eps, Ci, Qi, Gi, Di, pp, pq, cq);
  return check_launch("pool_queries");
}

extern "C" int ff_pool_keys(const void* qleaf, const void* kT, int64_t B, int64_t Q, int64_t G, int64_t D, void* u,
                            void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_keys", B, G, D);
  if (Q <= 0 || Q > 65535) return fail(FF_EINVAL, "pool_keys: bad Q");
  const int64_t rows = (B * Q + 15) / 16;
  if (rows > 65535) return fail(FF_EINVAL, "pool_keys: B*Q too large");
  if (B == 0) return FF_OK;
  if (!qleaf || !kT || !u) return fail(FF_EINVAL, "pool_keys: null pointer");
  if (!al(qleaf, 8) || !al(kT, 8) || !al(u, 8)) return fail(FF_EINVAL, "pool_keys: misaligned pointer");
  const dim3 grid(static_cast<unsigned>((D + 255) / 256), static_cast<unsigned>(rows), static_cast<unsigned>(G));
  pool_keys_kernel<<<grid, 256, 0, as_stream(stream)>>>(static_cast<const half_t*>(qleaf), static_cast<const half_t*>(kT),
                                                        static_cast<int>(B), static_cast<int>(Q), static_cast<int>(G),
                                                        static_cast<int>(D / G), static_cast<half_t*>(u));
  return check_launch("pool_keys");
}

extern "C" int ff_pool_tree(const void* parent, const void* zc, const void* g, const void* b, const float* partial,
                            int64_t nblk, float eps, int64_t B, int64_t C, int64_t Q, int64_t G, int64_t D, void* tree,
                            void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_tree", B, G, D);
  if (C <= 0 || Q <= 0 || Q > 65535 || Q % C != 0) return fail(FF_EINVAL, "pool_tree: need C | Q");
  if (nblk <= 0 || nblk > (1 << 24)) return fail(FF_EINVAL, "pool_tree: bad nblk");
  if (!(eps > 0.f)) return fail(FF_EINVAL, "pool_tree: eps must be > 0");
  if (B == 0) return FF_OK;
  if (!parent || !zc || !g || !b || !partial || !tree) return fail(FF_EINVAL, "pool_tree: null pointer");
  for (const void* p : {parent, zc, g, b, const_cast<const void*>(tree)})
    if (!al(p, 4)) return fail(FF_EINVAL, "pool_tree: misaligned pointer");
  const dim3 grid(static_cast<unsigned>(Q), static_cast<unsigned>(B));
  const Norm n{static_cast<const half_t*>(g), static_cast<const half_t*>(b)};
  const auto *pp = static_cast<const half_t*>(parent), *pz = static_cast<const half_t*>(zc);
  auto* pt = static_cast<half_t*>(tree);
  const int nb = static_cast<int>(nblk), Ci = static_cast<int>(C), Qi = static_cast<int>(Q), Gi = static_cast<int>(G),
            Di = static_cast<int>(D);
  if (D <= 768)
    pool_tree_kernel<6><<<grid, 64, 0, as_stream(stream)>>>(pp, pz, n, partial, nb, eps, Ci, Qi, Gi, Di, pt);
  else
    pool_tree_kernel<16><<<grid, 64, 0, as_stream(stream)>>>(pp, pz, n, partial, nb, eps, Ci, Qi, Gi, Di, pt);
  return check_launch("pool_tree");
}

extern "C" int ff_pool_leaf(const void* tree, const void* wl, const void* bl, int64_t B, int64_t Q, int64_t F, int64_t D,
                            void* leaf, void* stream) {
  clear_error();
  FF_POOL_CHECK("pool_leaf", B, 1, D);
  if (Q <= 0 || Q > 65535 || F <= 0 || F % 16 != 0 || F > 65536) return fail(FF_EINVAL, "pool_leaf: need F % 16 == 0");
  if (B == 0) return FF_OK;
  if (!tree || !wl || !bl || !leaf) return fail(FF_EINVAL, "pool_leaf: null pointer");
  if (!al(tree, 16) || !al(wl, 16) || !al(leaf, 8)) return fail(FF_EINVAL, "pool_leaf: misaligned pointer");
  const dim3 grid(static_cast<unsigned>(F / 16), static_cast<unsigned>((B + 15) / 16), static_cast<unsigned>(Q));
  pool_leaf_kernel<<<grid, 256, 0, as_stream(stream)>>>(static_cast<const half_t*>(tree), static_cast<const half_t*>(wl),
                                                        static_cast<const half_t*>(bl), static_cast<int>(B),
                                                        static_cast<int>(Q), static_cast<int>(F), static_cast<int>(D),
                                                        static_cast<half_t*>(leaf));
  return check_launch("pool_leaf");
}
