// LoGo's global re-parameterisation and the rotary embedding of its inputs and
// outputs, in one pass over the activations (logo/layers/logo.py:86-94,
// :112-158; logo/modules/rotary.py:81-106):
//
//   global_maps_kernel      xr = rope(x), y = rope(x W_h)     (q, k)
//                           y = x W_h                         (v)
//   global_maps_bwd_kernel  dg = rope^T(dy), dx = dg W_h^T + rope^T(dxr),
//                           dW_h = x^T dg                     (q, k; v without the rotations)
//
// for up to three [N, H_i, D] tensors in one launch.  The steps as separate
// kernels (head_linear, head_linear_grad_acc, head_linear_dw, RoPE) are bound
// by memory and read or write every tensor of q and k two to three times more:
// 14 and 23 passes over a [N, H, D] tensor in the two directions against 8 and
// 12 here.  Every rounding of theirs is kept (the product to bf16 before its
// rotation, both rotations as their eager bf16 ops, the sum of two bf16
// gradients), as is the order of the sums: the results are the same bits.
//
// A workgroup of 8 waves owns one head and a run of tokens, kGmRows at a time;
// W_h stays in registers as MFMA operands for all of them (wave w: 32 tokens,
// w & 3, times half of the output columns, w >> 2).  A row is moved in 16-byte
// chunks, eight lanes a half row: lane (row, c) holds chunk c of both halves, the pair
// that a rotation mixes, so that both rotations are register arithmetic on
// coalesced loads and stores, with one load of cos / sin for both; between the
// lanes and the MFMA operands the rows go through LDS.  The product is taken
// transposed (W as the left operand), which leaves each lane four adjacent
// columns of one token: 8-byte LDS stores.  The next rows load while the
// current ones are computed; one workgroup a CU has 100 KB in flight.
//
// 32768 tokens, 3 x 16 heads of 128: forward 385 -> 237 us (1.07 GB, 4.5 TB/s),
// backward 703 -> 412 + 42 us for the sum of the partials (1.7 GB); 6002 tokens:
// forward 101 -> 59 us.
#include "capi.hpp"
#include "common.hpp"

namespace logo {

int device_cus();  // sq_attn.hip

constexpr int kGmRows = 128;      // tokens per pass
constexpr int kGmThreads = 512;
constexpr int kGmChunk = 1024;    // tokens of one partial weight gradient (as head_linear_dw)

struct GmTensor {
  const bf16* x;   // [N, H, D]
  const bf16* w;   // [H, D, D]
  bf16* xr;        // forward: rope(x), or null (no rotation)
  bf16* y;         // forward: the mapped rows
  const bf16* da;  // backward: gradient of xr (of x itself without rotation)
  const bf16* dg;  // backward: gradient of y
  bf16* dx;        // backward: dx[n * lddx + h * D + c]
  bf16* dw;        // backward: [H, D, D], or null
  int heads;
  int rope;
};

struct GmArgs {
  GmTensor t[3];
  const bf16* cos;  // [N, D]
  const bf16* sin;
  int64_t n;
  int64_t lddx;
  float* part;   // backward: [sum H_i, nchunk, D, D]
  int nchunk;
  int runs;      // token runs (workgroups) per head
  int64_t run;   // tokens per run (a multiple of kGmRows; of kGmChunk in the backward)
};

// The head of the workgroup: its tensor and the head's index in it.
__device__ __forceinline__ const GmTensor& gm_tensor(const GmArgs& a, int& h) {
  int ti = 0;
  while (ti < 2 && h >= a.t[ti].heads) h -= a.t[ti++].heads;
  return a.t[ti];
}

// Workgroup barrier for LDS only (a __syncthreads() would also wait for the
// next pass's copies into LDS).
__device__ __forceinline__ void gm_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Rows [t0, min(t0 + rows, n)) of a [n, ld] tensor from column col0 as a
// buffer: loads past them return zeros, stores past them are dropped, without
// a branch (so that every pass has the same number of operations in flight).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gm_rows(const bf16* p, int64_t ld, int64_t col0, int64_t t0, int rows,
                                                          int64_t n) {
  const int64_t left = n - t0;
  const int r = left < rows ? (left > 0 ? (int)left : 0) : rows;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p + t0 * ld + col0), (short)0,
                                           (int)((int64_t)r * ld * sizeof(bf16)), kBufRsrcWord3);
}
// Waits until at most N memory operations of this wave, its last ones, are on
// their way.  The first pass has no stores behind its loads and waits for all.
template <int N>
__device__ __forceinline__ void gm_wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
constexpr int kNt = 2;  // streaming accesses
template <int AUX>
__device__ __forceinline__ bf16x8 gm_ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX));
}
template <int AUX>
__device__ __forceinline__ void gm_st(__amdgpu_buffer_rsrc_t r, uint32_t off, bf16x8 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, AUX);
}

// y^T = W^T x^T per 32 tokens: bound by memory (8 passes over [N, H, D]).
template <int D>
__global__ __launch_bounds__(kGmThreads, 2) void global_maps_kernel(const GmArgs a) {
  constexpr int RS = D + 8;    // padded LDS row: conflict-free 16-byte reads and 8-byte stores
  constexpr int HC = D / 16;   // 16-byte chunks of half a row
  constexpr int NIT = kGmRows * HC / kGmThreads;  // chunk pairs per lane
  constexpr int DS = D / 16, CT = D / 64;
  static_assert(NIT >= 1 && kGmRows * HC % kGmThreads == 0, "");
  __shared__ __attribute__((aligned(16))) bf16 xt[kGmRows * RS];
  __shared__ __attribute__((aligned(16))) bf16 ot[kGmRows * RS];
  int h = blockIdx.x / a.runs;
  const int64_t t_lo = (int64_t)(blockIdx.x % a.runs) * a.run;
  const int64_t t_hi = t_lo + a.run < a.n ? t_lo + a.run : a.n;
  if (t_lo >= t_hi) return;
  const GmTensor& t = gm_tensor(a, h);
  const int64_t ld = (int64_t)t.heads * D;
  const int64_t hoff = (int64_t)h * D;
  const bool rope = t.xr != nullptr;
  // The loads are issued on every path, of no rows where there are none to load:
  // behind a branch, the waits would count for the path without them.
  const int64_t cs_hi = rope ? t_hi : 0;
  const int tid = threadIdx.x, pr = tid / HC, pc = 8 * (tid % HC);  // lane's row and chunk (first pair)
  constexpr int PSTEP = kGmThreads / HC;
  uint32_t xo[NIT], co[NIT];  // byte offsets of the lane's chunks in a pass's rows
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    xo[it] = (uint32_t)((pr + PSTEP * it) * (int)ld + pc) * 2;
    co[it] = (uint32_t)((pr + PSTEP * it) * D + pc) * 2;
  }
  auto load_x = [&](int64_t t0, bf16x8 (&v)[NIT][2]) {
    const auto r = gm_rows(t.x, ld, hoff, t0, kGmRows, t_hi);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      v[it][0] = gm_ld<kNt>(r, xo[it]);
      v[it][1] = gm_ld<kNt>(r, xo[it] + D);
    }
  };
  bf16x8 nx[NIT][2];
  load_x(t_lo, nx);
  // W_h as the left operand: output column 32 ct + i, k = 16 s + 8 g + ...
  const bf16* wh = t.w + (int64_t)h * D * D;
  constexpr int NW = D * D / 8 / kGmThreads;
  bf16x8 wv[NW];
#pragma unroll
  for (int k = 0; k < NW; ++k) wv[k] = *reinterpret_cast<const bf16x8*>(wh + 8 * (tid + kGmThreads * k));
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    const int idx = tid + kGmThreads * k, r = idx / (D / 8), c8 = (idx % (D / 8)) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) ot[(c8 + j) * RS + r] = wv[k][j];
  }
  __syncthreads();
  const int wave = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int tg = 32 * (wave & 3), c0 = 32 * CT * (wave >> 2);
  bf16x8 wf[CT][DS];
#pragma unroll
  for (int u = 0; u < CT; ++u)
#pragma unroll
    for (int s = 0; s < DS; ++s)
      wf[u][s] = lds_load(reinterpret_cast<const bf16x8*>(ot + (c0 + 32 * u + i) * RS + 16 * s + 8 * g));
  __syncthreads();
  for (int64_t t0 = t_lo; t0 < t_hi; t0 += kGmRows) {
    bf16x8 x[NIT][2], cs[NIT][4];
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        x[it][e] = nx[it][e];
        *reinterpret_cast<bf16x8*>(xt + (pr + PSTEP * it) * RS + pc + e * D / 2) = x[it][e];
      }
    gm_barrier();  // the rows are in xt; every lane has read its chunks of ot
    {
      const auto rc = gm_rows(a.cos, D, 0, t0, kGmRows, cs_hi), rs = gm_rows(a.sin, D, 0, t0, kGmRows, cs_hi);
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          cs[it][e] = gm_ld<0>(rc, co[it] + e * D);
          cs[it][2 + e] = gm_ld<0>(rs, co[it] + e * D);
        }
    }
    load_x(t0 + kGmRows, nx);
    f32x16 acc[CT];
#pragma unroll
    for (int u = 0; u < CT; ++u) acc[u] = f32x16{};
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const bf16x8 xv = lds_load(reinterpret_cast<const bf16x8*>(xt + (tg + i) * RS + 16 * s + 8 * g));
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[u] = mfma32(wf[u][s], xv, acc[u]);
    }
    // acc[u] item 4m + e of lane (i, g): column c0 + 32u + 8m + 4g + e, token tg + i
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)acc[u][4 * m + e];
        *reinterpret_cast<bf16x4*>(ot + (tg + i) * RS + c0 + 32 * u + 8 * m + 4 * g) = v;
      }
    gm_barrier();  // the product is in ot; xt is free
    const auto ry = gm_rows(t.y, ld, hoff, t0, kGmRows, a.n);
    const auto rx = gm_rows(rope ? t.xr : t.y, ld, hoff, t0, kGmRows, a.n);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      bf16x8 y1 = lds_load(reinterpret_cast<const bf16x8*>(ot + (pr + PSTEP * it) * RS + pc));
      bf16x8 y2 = lds_load(reinterpret_cast<const bf16x8*>(ot + (pr + PSTEP * it) * RS + pc + D / 2));
      if (rope) {
        rope_chunk<false>(x[it][0], x[it][1], cs[it][0], cs[it][1], cs[it][2], cs[it][3]);
        rope_chunk<false>(y1, y2, cs[it][0], cs[it][1], cs[it][2], cs[it][3]);
        gm_st<kNt>(rx, xo[it], x[it][0]);
        gm_st<kNt>(rx, xo[it] + D, x[it][1]);
      }
      gm_st<kNt>(ry, xo[it], y1);
      gm_st<kNt>(ry, xo[it] + D, y2);
    }
  }
}

// Bound by memory (12 passes over [N, H, D] and the partial weight gradients).
// x comes by global -> LDS copies (it is an operand of dW only); dW_h is kept
// over kGmChunk tokens in registers, wave w the 32 x 64 block (w & 3, w >> 2),
// both operands read transposed.
constexpr size_t kGmBwdSmem = (size_t)(3 * kGmRows * 128 + kGmRows * (128 + 8)) * sizeof(bf16);

template <int D>
__global__ __launch_bounds__(kGmThreads, 2) void global_maps_bwd_kernel(const GmArgs a) {
  static_assert(D == 128 && kGmRows == 128 && kGmThreads == 512, "");
  constexpr int RS = D + 8, HC = D / 16, NIT = kGmRows * HC / kGmThreads, DS = D / 16, CT = D / 64;
  constexpr int PSTEP = kGmThreads / HC, TILE = 64 * D;
  using Geo = TileGeom<D, kSwz>;
  extern __shared__ __attribute__((aligned(16))) char gm_smem[];
  bf16* const smem = reinterpret_cast<bf16*>(gm_smem);
  bf16* const dgt = smem;              // two 64-row tiles of dg
  bf16* const xt = smem + 2 * TILE;    // two buffers of two tiles of x
  bf16* const ot = smem + 6 * TILE;    // dg W^T, padded rows
  int h = blockIdx.x / a.runs;
  const int hg = h;
  const int64_t t_lo = (int64_t)(blockIdx.x % a.runs) * a.run;
  const int64_t t_hi = t_lo + a.run < a.n ? t_lo + a.run : a.n;
  if (t_lo >= t_hi) return;
  const GmTensor& t = gm_tensor(a, h);
  const int64_t ld = (int64_t)t.heads * D;
  const int64_t hoff = (int64_t)h * D;
  const bool rope = t.rope != 0, with_dw = t.dw != nullptr;
  const int64_t cs_hi = rope ? t_hi : 0, x_hi = with_dw ? t_hi : 0;  // loads on every path, as in the forward
  const int tid = threadIdx.x, pr = tid / HC, pc = 8 * (tid % HC);
  const int wave = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int tg = 32 * (wave & 3), c0 = 32 * CT * (wave >> 2);
  uint32_t xo[NIT], co[NIT], so[NIT];  // byte offsets of the lane's chunks in a pass's rows
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    xo[it] = (uint32_t)((pr + PSTEP * it) * (int)ld + pc) * 2;
    so[it] = (uint32_t)((pr + PSTEP * it) * (int)a.lddx + pc) * 2;
    co[it] = (uint32_t)((pr + PSTEP * it) * D + pc) * 2;
  }
  bf16x8 nda[NIT][2], ndg[NIT][2], cs[NIT][4];
  auto load_d = [&](int64_t t0) {
    const auto rg = gm_rows(t.dg, ld, hoff, t0, kGmRows, t_hi), ra = gm_rows(t.da, ld, hoff, t0, kGmRows, t_hi);
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        ndg[it][e] = gm_ld<kNt>(rg, xo[it] + e * D);
        nda[it][e] = gm_ld<kNt>(ra, xo[it] + e * D);
      }
  };
  auto load_cs = [&](int64_t t0) {
    const auto rc = gm_rows(a.cos, D, 0, t0, kGmRows, cs_hi), rs = gm_rows(a.sin, D, 0, t0, kGmRows, cs_hi);
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        cs[it][e] = gm_ld<0>(rc, co[it] + e * D);
        cs[it][2 + e] = gm_ld<0>(rs, co[it] + e * D);
      }
  };
  TileBufDma<D, kGmThreads / 64> dma;
  dma.init((int)ld);
  auto load_x = [&](int64_t t0, int b) {
#pragma unroll
    for (int th = 0; th < 2; ++th)
      dma.issue(xt + (2 * b + th) * TILE, gm_rows(t.x, ld, hoff, t0 + 64 * th, 64, x_hi));
  };
  load_d(t_lo);
  load_cs(t_lo);
  load_x(t_lo, 0);
  // W_h as the left operand of dx^T = W dg^T: row c0 + 32 u + i, k = 16 s + 8 g + ...
  const bf16* wh = t.w + (int64_t)h * D * D;
  bf16x8 wf[CT][DS];
#pragma unroll
  for (int u = 0; u < CT; ++u)
#pragma unroll
    for (int s = 0; s < DS; ++s)
      wf[u][s] = *reinterpret_cast<const bf16x8*>(wh + (c0 + 32 * u + i) * D + 16 * s + 8 * g);
  wait_vmem();
#pragma unroll
  for (int u = 0; u < CT; ++u)
#pragma unroll
    for (int s = 0; s < DS; ++s) asm("" : "+v"(wf[u][s]));  // landed here, or every pass would wait for them
  // transposed reads (as TileReader::tr, for this wave's column blocks): block
  // w & 3 of x, blocks 2 (w >> 2) + u of dg; row reads of dg
  int xq[2], go[CT][2], ro[DS];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int r = 4 * g + ((l & 15) >> 2) + 8 * e, c = 16 * ((l >> 4) & 1) + 4 * (l & 3);
    xq[e] = Geo::off(r, (tg + c) >> 3) + (c & 7);
#pragma unroll
    for (int u = 0; u < CT; ++u) go[u][e] = Geo::off(r, (c0 + 32 * u + c) >> 3) + (c & 7);
  }
#pragma unroll
  for (int s = 0; s < DS; ++s) ro[s] = tg * D + Geo::off(i, 2 * s + g);
  // opaque: each offset stays one register, the constant part of an address in
  // the instruction (folded into them, the sums don't fit in registers)
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    asm("" : "+v"(xq[e]));
#pragma unroll
    for (int u = 0; u < CT; ++u) asm("" : "+v"(go[u][e]));
  }
#pragma unroll
  for (int s = 0; s < DS; ++s) asm("" : "+v"(ro[s]));
  auto tr = [](const bf16* p, const int (&o)[2]) {
    const bf16x4 lo = ds_read_tr((const lds_bf16x4*)(p + o[0])), hi = ds_read_tr((const lds_bf16x4*)(p + o[1]));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  f32x16 dw[CT];
#pragma unroll
  for (int u = 0; u < CT; ++u) dw[u] = f32x16{};
  int b = 0;
  for (int64_t t0 = t_lo; t0 < t_hi; t0 += kGmRows, b ^= 1) {
    gm_wait_loads<2 * NIT>();  // all but the last pass's stores: x is in LDS, the other rows in registers
    bf16x8 da[NIT][2];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int r = pr + PSTEP * it;
      if (rope) {
        rope_chunk<true>(ndg[it][0], ndg[it][1], cs[it][0], cs[it][1], cs[it][2], cs[it][3]);
        rope_chunk<true>(nda[it][0], nda[it][1], cs[it][0], cs[it][1], cs[it][2], cs[it][3]);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        da[it][e] = nda[it][e];
        *reinterpret_cast<bf16x8*>(dgt + (r >> 6) * TILE + Geo::off(r & 63, pc / 8 + e * HC)) = ndg[it][e];
      }
    }
    gm_barrier();  // dg and x are there; every lane has read its chunks of ot
    const bool more = t0 + kGmRows < t_hi;
    load_d(t0 + kGmRows);
    load_x(t0 + kGmRows, b ^ 1);
    f32x16 acc[CT];
#pragma unroll
    for (int u = 0; u < CT; ++u) acc[u] = f32x16{};
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const bf16x8 v = lds_load(reinterpret_cast<const bf16x8*>(dgt + ro[s]));
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[u] = mfma32(wf[u][s], v, acc[u]);
    }
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)acc[u][4 * m + e];
        *reinterpret_cast<bf16x4*>(ot + (tg + i) * RS + c0 + 32 * u + 8 * m + 4 * g) = v;
      }
    load_cs(t0 + kGmRows);  // behind the product, whose registers are free now
    if (with_dw) {
#pragma unroll
      for (int th = 0; th < 2; ++th)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const bf16x8 xv = tr(xt + (2 * b + th) * TILE + 16 * ks * D, xq);
#pragma unroll
          for (int u = 0; u < CT; ++u) dw[u] = mfma32(xv, tr(dgt + th * TILE + 16 * ks * D, go[u]), dw[u]);
        }
      if (!more || (t0 + kGmRows) % kGmChunk == 0) {
        // dw[u] item 4m + e of lane (i, g): row 32 (wave & 3) + 8m + 4g + e, column c0 + 32u + i
        float* p = a.part + ((int64_t)hg * a.nchunk + t0 / kGmChunk) * D * D;
        int o = (tg + 4 * g) * D + c0 + i;
        asm("" : "+v"(o));  // the addresses of this rare branch aren't kept over the passes
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int jj = 0; jj < 16; ++jj) {
            p[o + (8 * (jj / 4) + jj % 4) * D + 32 * u] = dw[u][jj];
            dw[u][jj] = 0.f;
          }
      }
    }
    gm_barrier();  // the product is in ot; dgt and x's buffer are free
    const auto rx = gm_rows(t.dx, a.lddx, hoff, t0, kGmRows, a.n);
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf16x8 y = lds_load(reinterpret_cast<const bf16x8*>(ot + (pr + PSTEP * it) * RS + pc + e * D / 2));
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = (bf16)((float)y[j] + (float)da[it][e][j]);
        gm_st<0>(rx, so[it] + e * D, y);
      }
  }
}

// dw[h, d, e] = sum over chunks, in chunk order, of the heads of all tensors;
// four elements a thread, eight chunks' loads in flight.
template <int D>
__global__ __launch_bounds__(64) void global_maps_dw_reduce_kernel(const GmArgs a) {
  const int64_t idx = ((int64_t)blockIdx.x * 64 + threadIdx.x) * 4;
  const int hg = (int)(idx / (D * D)), de = (int)(idx % (D * D));
  int h = hg;
  const GmTensor& t = gm_tensor(a, h);
  if (h >= t.heads || t.dw == nullptr) return;
  const float* p = a.part + (int64_t)hg * a.nchunk * D * D + de;
  f32x4 s{};
  int k = 0;
  for (; k + 8 <= a.nchunk; k += 8, p += 8 * D * D) {
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = ld_nt(reinterpret_cast<const f32x4*>(p + j * D * D));
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[j];
  }
  for (; k < a.nchunk; ++k, p += D * D) s += ld_nt(reinterpret_cast<const f32x4*>(p));
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (bf16)s[e];
  *reinterpret_cast<bf16x4*>(t.dw + (int64_t)h * D * D + de) = o;
}

// Token runs per head: the count that ends first when the workgroups of all
// heads take turns on the CUs, a run taking its passes and about one more for
// W_h and the ends of its pipeline.
static int gm_runs(int heads, int64_t units, int unit_passes) {
  const int cus = std::max(device_cus(), 1);
  int64_t best = 1, best_cost = INT64_MAX;
  for (int64_t r = 1; r <= units && r <= 256; ++r) {
    const int64_t turns = (heads * r + cus - 1) / cus;
    const int64_t cost = turns * ((units + r - 1) / r * unit_passes + 1);
    if (cost < best_cost) best = r, best_cost = cost;
  }
  return (int)best;
}

}  // namespace logo

using namespace logo;

static int gm_check(const void* cos, const void* sin, bool rope, int64_t n_tokens, int dtype) {
  LOGO_REQUIRE(dtype == LOGO_DTYPE_BF16, "only bf16 tensors are supported");
  // (no tokens: the weight gradients asked for would not be written)
  LOGO_REQUIRE(n_tokens >= 1 && n_tokens < ((int64_t)1 << 31), "n_tokens must be in [1, 2^31)");
  LOGO_REQUIRE(!rope || (cos && sin), "null cos / sin");
  LOGO_REQUIRE(((uintptr_t)cos | (uintptr_t)sin) % 16 == 0, "cos and sin must be 16-byte aligned");
  return LOGO_OK;
}

static void gm_split(GmArgs& a, int heads, int64_t unit) {
  const int64_t units = (a.n + unit - 1) / unit;
  a.runs = gm_runs(heads, units, (int)(unit / kGmRows));
  a.run = (units + a.runs - 1) / a.runs * unit;
}

extern "C" int logo_global_maps(const void* x0, const void* w0, void* xr0, void* y0, int h0, const void* x1,
                                const void* w1, void* xr1, void* y1, int h1, const void* x2, const void* w2,
                                void* xr2, void* y2, int h2, const void* cos, const void* sin, int64_t n_tokens,
                                int d, int dtype, void* stream) {
  const void* xs[3] = {x0, x1, x2};
  const void* ws[3] = {w0, w1, w2};
  void* xrs[3] = {xr0, xr1, xr2};
  void* ys[3] = {y0, y1, y2};
  const int hs[3] = {h0, h1, h2};
  LOGO_REQUIRE(d == 64 || d == 128, "head dim %d unsupported (64 or 128)", d);
  const int rc = gm_check(cos, sin, xr0 || xr1 || xr2, n_tokens, dtype);
  if (rc != LOGO_OK) return rc;
  GmArgs a{};
  int nt = 0, heads = 0;
  for (int i = 0; i < 3; ++i) {
    if (xs[i] == nullptr) continue;
    LOGO_REQUIRE(ws[i] && ys[i] && hs[i] >= 1 && hs[i] <= 4096, "tensor %d: null weight / output or bad head count", i);
    LOGO_REQUIRE(((uintptr_t)xs[i] | (uintptr_t)ws[i] | (uintptr_t)xrs[i] | (uintptr_t)ys[i]) % 16 == 0,
                 "tensor %d: pointers must be 16-byte aligned", i);
    GmTensor& t = a.t[nt++];
    t.x = static_cast<const bf16*>(xs[i]);
    t.w = static_cast<const bf16*>(ws[i]);
    t.xr = static_cast<bf16*>(xrs[i]);
    t.y = static_cast<bf16*>(ys[i]);
    t.heads = hs[i];
    heads += hs[i];
  }
  if (heads == 0) return LOGO_OK;
  a.cos = static_cast<const bf16*>(cos);
  a.sin = static_cast<const bf16*>(sin);
  a.n = n_tokens;
  gm_split(a, heads, kGmRows);
  const dim3 grid((unsigned)(heads * a.runs));
  if (d == 128) hipLaunchKernelGGL(global_maps_kernel<128>, grid, dim3(kGmThreads), 0, as_stream(stream), a);
  else hipLaunchKernelGGL(global_maps_kernel<64>, grid, dim3(kGmThreads), 0, as_stream(stream), a);
  LOGO_LAUNCH_CHECK("global_maps_kernel");
  return LOGO_OK;
}

extern "C" int logo_global_maps_bwd(const void* x0, const void* w0, const void* da0, const void* dg0, void* dx0,
                                    void* dw0, int h0, int rope0, const void* x1, const void* w1, const void* da1,
                                    const void* dg1, void* dx1, void* dw1, int h1, int rope1, const void* x2,
                                    const void* w2, const void* da2, const void* dg2, void* dx2, void* dw2, int h2,
                                    int rope2, const void* cos, const void* sin, int64_t lddx, void* workspace,
                                    int64_t n_tokens, int d, int dtype, void* stream) {
  const void* xs[3] = {x0, x1, x2};
  const void* ws[3] = {w0, w1, w2};
  const void* das[3] = {da0, da1, da2};
  const void* dgs[3] = {dg0, dg1, dg2};
  void* dxs[3] = {dx0, dx1, dx2};
  void* dws[3] = {dw0, dw1, dw2};
  const int hs[3] = {h0, h1, h2}, ropes[3] = {rope0, rope1, rope2};
  LOGO_REQUIRE(d == 128, "head dim %d unsupported (128)", d);
  const int rc = gm_check(cos, sin, rope0 || rope1 || rope2, n_tokens, dtype);
  if (rc != LOGO_OK) return rc;
  GmArgs a{};
  int nt = 0, heads = 0;
  bool any_dw = false;
  for (int i = 0; i < 3; ++i) {
    if (xs[i] == nullptr) continue;
    LOGO_REQUIRE(ws[i] && das[i] && dgs[i] && dxs[i] && hs[i] >= 1 && hs[i] <= 4096,
                 "tensor %d: null argument or bad head count", i);
    LOGO_REQUIRE(((uintptr_t)xs[i] | (uintptr_t)ws[i] | (uintptr_t)das[i] | (uintptr_t)dgs[i] | (uintptr_t)dxs[i]) %
                         16 == 0,
                 "tensor %d: pointers must be 16-byte aligned", i);
    LOGO_REQUIRE(lddx >= (int64_t)hs[i] * d && lddx % 8 == 0 && lddx < ((int64_t)1 << 23),
                 "dx's row stride must cover heads * d and be a multiple of 8 below 2^23");
    GmTensor& t = a.t[nt++];
    t.x = static_cast<const bf16*>(xs[i]);
    t.w = static_cast<const bf16*>(ws[i]);
    t.da = static_cast<const bf16*>(das[i]);
    t.dg = static_cast<const bf16*>(dgs[i]);
    t.dx = static_cast<bf16*>(dxs[i]);
    t.dw = static_cast<bf16*>(dws[i]);
    t.heads = hs[i];
    t.rope = ropes[i];
    heads += hs[i];
    any_dw |= dws[i] != nullptr;
  }
  LOGO_REQUIRE(!any_dw || (workspace && (uintptr_t)workspace % 16 == 0), "workspace must be 16-byte aligned memory");
  if (heads == 0) return LOGO_OK;
  a.cos = static_cast<const bf16*>(cos);
  a.sin = static_cast<const bf16*>(sin);
  a.lddx = lddx;
  a.part = static_cast<float*>(workspace);
  a.n = n_tokens;
  a.nchunk = (int)((n_tokens + kGmChunk - 1) / kGmChunk);
  gm_split(a, heads, kGmChunk);
  auto kern = global_maps_bwd_kernel<128>;
  LOGO_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGmBwdSmem));
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(kern, dim3((unsigned)(heads * a.runs)), dim3(kGmThreads), kGmBwdSmem, st, a);
  LOGO_LAUNCH_CHECK("global_maps_bwd_kernel");
  if (any_dw) {
    hipLaunchKernelGGL(global_maps_dw_reduce_kernel<128>, dim3((unsigned)(heads * (128 * 128 / 256))), dim3(64), 0,
                       st, a);
    LOGO_LAUNCH_CHECK("global_maps_dw_reduce_kernel");
  }
  return LOGO_OK;
}
