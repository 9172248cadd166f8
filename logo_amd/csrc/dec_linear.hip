// Linear layers of a decode step (a few token rows) for gfx950:
//   y = x W^T, W [N, K] bf16 as nn.Linear holds it, x [M, K] with M <= 16,
// with what surrounds each of them in the decoder fused in: the RMSNorm of
// the input row (logo/modules/layernorm.py:17-22), the residual add behind
// the output (logo/modeling_logo.py:58-66), and the SwiGLU of a stacked
// gate / up projection (logo/modules/mlp.py:24-27).
//
// Bound: reading W once.  A step of the 24-layer 1.5B model reads 2.6 GB of
// weights, 103 MB a layer in four products, so each product lasts 4-15 us and
// its start-up matters as much as its rate.  Hence:
//   * a workgroup takes 16 rows of W and its eight waves split K, so a product
//     of 2048 columns still has 1024 waves; their sums meet in LDS, in wave
//     order;
//   * every wave issues its whole W tile (up to 16 rows x 256 k) at once as
//     streaming buffer_load ... lds copies, each covering rows by 512
//     contiguous bytes, before anything happens to x: no registers, and the
//     matrix is in flight while the norm's row statistics are formed.  (W
//     straight to registers in the MFMA's layout, 64 bytes a row and load,
//     measured 19 against 15 us on the gate / up product.);
//   * the MFMA (16x16x32) takes W as its A operand and x as B, x straight from
//     L2 in the operand layout (lane i + 16 G: row i, k 8 G .. 8 G + 7 of the
//     step), rows past M zero.
// The norm is recomputed by each workgroup from the rows it reads anyway,
// which saves its launch (about 5 us each, two a layer).
// Four rows, graph-replayed launches over weights larger than the caches,
// against the library's GEMM with its separate norm / SwiGLU / add launches:
// [6152, 2048] with norm 15.7 -> 10.4 us, [2048, 2048] with the add 10.4 -> 5.8,
// 2 x [5632, 2048] norm and SwiGLU 21.4 -> 15.1, [2048, 5632] with the add
// 13.7 -> 10.0, [32000, 2048] 33.6 -> 25.9 (5.1 TB/s); the whole decode step
// 2089 -> 1480 us.
#include <math.h>

#include <algorithm>

#include "capi.hpp"
#include "common.hpp"

// every product and sum outside the MFMA rounds as its own eager bf16 op
#pragma clang fp contract(off)

namespace logo {

struct DecLinArgs {
  const bf16* x;       // [M, K], row stride ldx
  int64_t ldx;
  const bf16* w;       // [N, K] (SwiGLU: [2 N, K], gate rows then up rows)
  const bf16* norm_w;  // [K] or null
  float eps;
  const bf16* resid;   // [M, N] dense or null
  bf16* y;             // [M, N] dense
  int m, n, k;
  int stages;          // W tiles a wave has: 1 where its k range is one batch, else 2
};

constexpr int kDlRows = 16;   // rows of W per workgroup (GLU: 8 gate rows, then their 8 up rows)
constexpr int kDlWaves = 8;   // waves, which split K

// Waits for LDS accesses only and meets the other waves (the W copies in
// flight into the waves' own tiles go on).
__device__ __forceinline__ void dl_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A wave's W tile: 16 rows x U k steps of 32 in LDS, row r's 16-byte chunk c at
// chunk c ^ (r & (4 U - 1)), so that the 16 rows of an operand read fall in
// distinct banks.  One buffer_load ... lds fills 1 KB: 16 / U rows of 64 U
// contiguous bytes each (512 at U = 8).
template <int U>
struct DlTile {
  static constexpr int CH = 4 * U, RPI = 64 / CH, BYTES = kDlRows * CH * 16;
  __device__ __forceinline__ static void issue(char* t, __amdgpu_buffer_rsrc_t r, const uint32_t (&rowoff)[16 / RPI],
                                               int k0, int ns) {
    const int j = threadIdx.x & 63;
#pragma unroll
    for (int b = 0; b < 16 / RPI; ++b) {
      const int row = RPI * b + j / CH;
      const int ch = (j % CH) ^ (row & (CH - 1));
      // chunks past the wave's range read its last one (never used)
      buf_load_lds16_nt(r, reinterpret_cast<bf16*>(t + 1024 * b), rowoff[b] + 2 * k0 + 16 * min(ch, 4 * ns - 1));
    }
  }
  __device__ __forceinline__ static bf16x8 row(const char* t, int u, int i, int G) {
    return lds_load(reinterpret_cast<const bf16x8*>(t + 16 * (CH * i + ((4 * u + G) ^ (i & (CH - 1))))));
  }
};

// U: k steps per batch; NORM: RMSNorm of x first (then
// each wave's k range is one batch).
template <int U, bool NORM, bool GLU>
__global__ __launch_bounds__(64 * kDlWaves) void dec_linear_kernel(const DecLinArgs a) {
  constexpr int NW = kDlWaves, NO = GLU ? kDlRows / 2 : kDlRows;  // NO: output columns
  using TL = DlTile<U>;
  constexpr int RPI = TL::RPI;
  extern __shared__ __attribute__((aligned(16))) char dl_smem[];  // NW x a.stages of TL::BYTES
  __shared__ float part[NW][16][kDlRows];
  __shared__ float sq[NW][16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, G = l >> 4;
  const int n0 = blockIdx.x * NO;
  const int steps_all = a.k >> 5;
  const int per = (steps_all + NW - 1) / NW;
  const int s_lo = min(wave * per, steps_all), s_hi = min(s_lo + per, steps_all);
  const int nb = (s_hi - s_lo + U - 1) / U;  // batches of this wave
  // W rows as the copies see them, from the workgroup's first one; rows past N
  // read the last one, their columns are not stored
  const bf16* w0 = a.w + (int64_t)n0 * a.k;
  uint32_t rowoff[16 / RPI];
#pragma unroll
  for (int b = 0; b < 16 / RPI; ++b) {
    const int r = RPI * b + l / TL::CH;
    const int row = min(GLU ? r & 7 : r, a.n - 1 - n0) + (GLU && r >= 8 ? a.n : 0);
    rowoff[b] = (uint32_t)row * (uint32_t)a.k * 2;
  }
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w0), (short)0, -1, kBufRsrcWord3);
  const bool xin = i < a.m;
  const bf16* xp = a.x + (int64_t)(xin ? i : 0) * a.ldx + 8 * G;
  bf16x8 xv[U];
  auto load_x = [&](int s0, int ns) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      xv[u] = bf16x8{};
      if (u < ns && xin) xv[u] = *reinterpret_cast<const bf16x8*>(xp + 32 * (s0 + u));
    }
  };
  f32x4 acc = f32x4{};
  char* const tile = dl_smem + wave * a.stages * TL::BYTES;
  bf16x8 g8[NORM ? U : 1];
  if (nb > 0) {
    load_x(s_lo, min(U, s_hi - s_lo));
    if constexpr (NORM) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (u < s_hi - s_lo) g8[u] = *reinterpret_cast<const bf16x8*>(a.norm_w + 32 * (s_lo + u) + 8 * G);
    }
    TL::issue(tile, rsrc, rowoff, 32 * s_lo, min(U, s_hi - s_lo));
    if (!NORM && nb > 1) TL::issue(tile + TL::BYTES, rsrc, rowoff, 32 * (s_lo + U), min(U, s_hi - s_lo - U));
  } else {
    load_x(0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORM) {
    // sum of squares of each row: over the lane's elements, the four lanes of a row, the waves
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf((float)xv[u][e], (float)xv[u][e], ss);
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (G == 0) sq[wave][i] = ss;
    dl_barrier();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) ss += lds_load(&sq[w][i]);
    const float r = rsqrtf(ss / (float)a.k + a.eps);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < s_hi - s_lo) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[u][e] = (bf16)((float)g8[u][e] * bfr((float)xv[u][e] * r));
      }
  }
  for (int bt = 0; bt < nb; ++bt) {
    const int s0 = s_lo + U * bt, ns = min(U, s_hi - s0);
    if (bt > 0) load_x(s0, ns);
    // all copies have landed, this batch's and the next one's: past the first
    // batch, x of this one was loaded behind them, and loads return in order.  So
    // a range of three batches (K = 5632) copies two, computes, copies the third
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* t = tile + (bt & 1) * TL::BYTES;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < ns) {
        const bf16x8 wv = TL::row(t, u, i, G);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv[u], acc, 0, 0, 0);
      }
    if (!NORM && bt + 2 < nb) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tile's reads are done
      TL::issue(tile + (bt & 1) * TL::BYTES, rsrc, rowoff, 32 * (s0 + 2 * U), min(U, s_hi - s0 - 2 * U));
    }
  }
  // lane (i, G) holds W rows 4 G .. + 3 of x row i
  *reinterpret_cast<f32x4*>(&part[wave][i][4 * G]) = acc;
  __syncthreads();
  static_assert(16 * NO <= 64 * NW, "one output element a thread");
  const int m = tid / NO, no = tid % NO, n = n0 + no;
  if (m >= a.m || n >= a.n) return;
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) s += part[w][m][no];
  s = bfr(s);
  float out = s;
  if constexpr (GLU) {
    float u = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) u += part[w][m][NO + no];
    out = bfr(s / (1.f + expf(-s))) * bfr(u);
  } else if (a.resid != nullptr) {
    out = (float)a.resid[(int64_t)m * a.n + n] + s;
  }
  a.y[(int64_t)m * a.n + n] = (bf16)out;
}

template <int U, bool NORM, bool GLU>
static hipError_t dl_launch(DecLinArgs a, hipStream_t st) {
  constexpr int NO = GLU ? kDlRows / 2 : kDlRows;
  a.stages = a.k <= U * kDlWaves * 32 ? 1 : 2;
  const size_t smem = (size_t)kDlWaves * a.stages * DlTile<U>::BYTES;
  auto kern = dec_linear_kernel<U, NORM, GLU>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)((a.n + NO - 1) / NO)), dim3(64 * kDlWaves), smem, st, a);
  return hipSuccess;
}

template <int U>
static hipError_t dl_dispatch(const DecLinArgs& a, bool glu, hipStream_t st) {
  if (a.norm_w) return glu ? dl_launch<U, true, true>(a, st) : dl_launch<U, true, false>(a, st);
  return glu ? dl_launch<U, false, true>(a, st) : dl_launch<U, false, false>(a, st);
}

}  // namespace logo

using namespace logo;

extern "C" int logo_dec_linear(const void* x, int64_t ldx, const void* w, const void* norm_w, float eps,
                               const void* resid, void* y, int m, int n, int k, int glu, int dtype, void* stream) {
  LOGO_REQUIRE(dtype == LOGO_DTYPE_BF16, "only bf16 tensors are supported");
  LOGO_REQUIRE(m >= 0 && m <= 16, "m (%d) must be in [0, 16]", m);
  LOGO_REQUIRE(n >= 1 && k >= 32 && k % 32 == 0, "n must be positive and k (%d) a positive multiple of 32", k);
  LOGO_REQUIRE(n < (1 << 28) && k < (1 << 28), "n and k must be below 2^28");
  // the copies address W from the workgroup's first row by 32-bit offsets
  LOGO_REQUIRE(((int64_t)(glu ? n : 0) + 16) * k * 2 < ((int64_t)1 << 32), "W is too large");
  LOGO_REQUIRE(!glu || n % 8 == 0, "the SwiGLU form needs n (%d) a multiple of 8", n);
  LOGO_REQUIRE(ldx >= k && ldx % 8 == 0, "ldx must hold a row and be a multiple of 8");
  LOGO_REQUIRE(norm_w == nullptr || k <= 8 * kDlWaves * 32, "k (%d) must be at most 2048 with a norm", k);
  LOGO_REQUIRE(!(glu && resid), "the SwiGLU form takes no residual");
  LOGO_REQUIRE(m == 0 || (x && w && y), "null pointer argument");
  LOGO_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w) % 16 == 0, "x, w and norm_w must be 16-byte aligned");
  if (m == 0) return LOGO_OK;
  DecLinArgs a{};
  a.x = static_cast<const bf16*>(x);
  a.ldx = ldx;
  a.w = static_cast<const bf16*>(w);
  a.norm_w = static_cast<const bf16*>(norm_w);
  a.eps = eps;
  a.resid = static_cast<const bf16*>(resid);
  a.y = static_cast<bf16*>(y);
  a.m = m;
  a.n = n;
  a.k = k;
  hipStream_t st = as_stream(stream);
  const bool wide = k > 4 * kDlWaves * 32;  // eight steps a wave
  LOGO_HIP_CHECK(wide ? dl_dispatch<8>(a, glu != 0, st) : dl_dispatch<4>(a, glu != 0, st));
  LOGO_LAUNCH_CHECK("dec_linear_kernel");
  return LOGO_OK;
}
