// Query-sparse causal attention in fp32, forward, dq and dk/dv, for gfx950
// (logo/ops/selected_full_attn.py:33-337 with fp32 dots, P kept in fp32 for PV,
// :93-99).  Every product on v_mfma_f32_16x16x4_f32, nothing rounded below fp32.
//
// Bound: the fp32 MFMA rate (154 TFLOP/s in a large product on this part), once
// there are waves enough: a 16-row tile costs a wave 64 MFMAs (2048 cycles) per
// 16 keys at D = 128, so calls of a few thousand tokens are bound by their
// longest wave and by the latencies that too few waves leave open.  Hence a
// workgroup of eight waves shares one tile's work:
//   fwd, dq : RW row waves of 16 compacted rows x KG key groups, each group
//             walking every KG-th 16-key tile through its own two LDS stages;
//             the groups' partial results are combined through LDS at the end.
//   dk/dv   : NP pairs of waves, 16 keys each, x RG row groups, each taking
//             every RG-th step of 16 rows; in a pair wave A computes S, P and
//             dV, wave B dP, dS and dK, P passing through LDS.  (One wave per 16
//             keys with both accumulators needs 230 registers at D = 128, two
//             waves a SIMD.)
// RW / KG and NP / RG follow from the size of the call (dispatch_rows,
// dispatch_dkv).
// All partial sums are added in a fixed order.
// Measured against 16 rows or keys a wave, 64 a workgroup, no key or row groups:
// T = 4096, 16 heads, D = 128, a quarter of the rows, forward + backward 1238 to
// 1306 -> 715 to 821 us on the boxes measured; 512 tokens, 4 heads, D = 64: the
// three kernels 34 + 42 + 36 -> 13 + 13 + 12 us.  At T = 8192 the matrix units are
// 54 / 75 / 79% busy (forward, dq, dk/dv); the forward's waves meet at a barrier
// every 16 keys and do their softmax together.  Running S of the next tile beside
// the softmax of the current one measured no faster.
#include "sq_attn.hpp"

#include <algorithm>

namespace logo {
namespace f32 {

constexpr int KT = 16;  // keys per tile (fwd, dq), rows per step (dk/dv), keys per pair (dk/dv)
constexpr int kWaves = 8;

// c[n] += a[n] b over a 16-deep k step (lane group G holds k = 4 G + e in element
// e), element by element over all accumulators: an MFMA that continues the accumulator of the one before it waits
// for it, one of another accumulator does not.
template <int N>
__device__ __forceinline__ void mma_cols(const f32x4 (&a)[N], const f32x4 b, f32x4* c) {
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int n = 0; n < N; ++n) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n][s], b[s], c[n], 0, 0, 0);
}

// max / sum over the four lanes of a column (i, i + 16, i + 32, i + 48)
__device__ __forceinline__ float swap16_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float swap16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float col_max(float x) { return pair_max(swap16_max(x)); }
__device__ __forceinline__ float col_sum(float x) { return pair_sum(swap16_sum(x)); }

// exp2 of four scores.  The hardware's exp2 flushes results below 2^-126, where a
// probability still gives a gradient if dO v is large, so a wave with a score
// there takes exp2f (whose other results are the hardware's).  At T = 4096, 16
// heads, D = 128, a quarter of the rows, forward + backward 792 us with the
// hardware's exp2, 802 so, 814 with exp2f in every wave.
__device__ __forceinline__ f32x4 exp2_4(f32x4 x) {
  if (__ballot(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])) < -126.f)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = exp2f(x[j]);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = fast_exp2(x[j]);
  }
  return x;
}

__device__ __forceinline__ void barrier_all() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// 16 rows of D floats in LDS, in 1 KB blocks of RPB whole rows 1 KB + 16 RPB
// bytes apart; the 16-byte chunk ch of row r sits at chunk ch ^ (r % RPB) of its
// row.  The 16 lanes of an operand read then cover all banks once, and every
// read is a lane offset plus an immediate.
template <int D>
struct Tile {
  static constexpr int RB = 4 * D, RPB = 1024 / RB, BLK = 1024 + 16 * RPB, NBLK = KT / RPB, BYTES = NBLK * BLK;
  static constexpr int KS = D / 16, DT = D / 16;
  int row_off, tr_off[RPB];
  __device__ __forceinline__ void init() {
    const int l = threadIdx.x & 63, i = l & 15, G = l >> 4;
    row_off = (i / RPB) * BLK + (i % RPB) * RB + 16 * (G ^ (i % RPB));
#pragma unroll
    for (int e = 0; e < RPB; ++e) tr_off[e] = (4 * G / RPB) * BLK + e * RB + 16 * ((i >> 2) ^ e) + 4 * (i & 3);
  }
  // lane (i, G): elements 16 ks + 4 G .. + 3 of row i
  __device__ __forceinline__ f32x4 row(const char* t, int ks) const {
    return lds_load(reinterpret_cast<const f32x4*>(t + row_off + 64 * ks));
  }
  // lane (i, G): column 16 dt + i of rows 4 G .. 4 G + 3
  __device__ __forceinline__ f32x4 tr(const char* t, int dt) const {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = lds_load(reinterpret_cast<const float*>(t + tr_off[e % RPB] + (e / RPB) * BLK + 64 * dt));
    return v;
  }
  // Block b of the tile by one wave: rowoff(r) is the byte offset of row r from the buffer's base
  template <typename F>
  __device__ __forceinline__ static void copy_block(char* t, int b, __amdgpu_buffer_rsrc_t rsrc, F rowoff) {
    constexpr int CH = RB / 16;
    const int j = threadIdx.x & 63, r = RPB * b + j / CH, pc = j % CH;
    buf_load_lds16(rsrc, reinterpret_cast<bf16*>(t + BLK * b), rowoff(r) + 16 * (uint32_t)(pc ^ (r % RPB)));
  }
};

// sum over k of rows of t times b, as two interleaved chains of MFMAs
template <int D>
__device__ __forceinline__ f32x4 row_product(const Tile<D>& tl, const char* t, const f32x4 (&b)[Tile<D>::KS]) {
  f32x4 x[2] = {f32x4{}, f32x4{}};
#pragma unroll
  for (int ks = 0; ks < Tile<D>::KS; ks += 2) {
    const f32x4 r0 = tl.row(t, ks), r1 = tl.row(t, ks + 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(r0[e], b[ks][e], x[0], 0, 0, 0);
      x[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(r1[e], b[ks + 1][e], x[1], 0, 0, 0);
    }
  }
  return x[0] + x[1];
}

// acc[dt] += (columns 16 dt .. of t)^T x for every column block
template <int D>
__device__ __forceinline__ void tr_product(const Tile<D>& tl, const char* t, const f32x4 x, f32x4 (&acc)[Tile<D>::DT]) {
#pragma unroll
  for (int dt = 0; dt < Tile<D>::DT; dt += 2) {
    const f32x4 v[2] = {tl.tr(t, dt), tl.tr(t, dt + 1)};
    mma_cols<2>(v, x, &acc[dt]);
  }
}

// The rows of a fwd / dq workgroup: 16 RW of a kBQ-row tile of the
// compaction's tile list, heaviest first.
template <int RW>
struct Rows {
  QTile<true> qt;
  int r0, r_end, sub;
  __device__ __forceinline__ bool init(const AttnArgs& a) {
    constexpr int SUB = kBQ / (16 * RW);
    int rank, hq;
    xcd_remap(blockIdx.x, a.hq, rank, hq);
    qt.rank = rank;
    qt.hq = hq;
    qt.lane_sel = a.lanes > 1 ? hq : 0;
    const int32_t* meta = a.meta + (int64_t)qt.lane_sel * a.meta_stride;
    const int nt = meta[1];
    const int32_t* cu_q = meta + kMetaHdr;
    const int32_t* cu_tq = cu_q + (a.nseq + 1);
    qt.q_end = cu_q[a.nseq];
    qt.ntile = nt;
    qt.trank = rank / SUB;
    sub = SUB - 1 - rank % SUB;  // the tile's latest rows first
    if (qt.trank >= nt) return false;
    const int tile = nt - 1 - qt.trank;
    qt.s = seg_of(cu_tq, a.nseq, tile);
    qt.r0 = cu_q[qt.s] + (tile - cu_tq[qt.s]) * kBQ;
    qt.r_end = min(qt.r0 + kBQ, cu_q[qt.s + 1]);
    qt.bos = a.cu[qt.s];
    qt.seqlen = a.cu[qt.s + 1] - qt.bos;
    qt.h = hq / a.g;
    qt.rv = row_view<true>(a, qt.lane_sel, qt.bos);
    r0 = qt.r0 + 16 * RW * sub;
    r_end = min(r0 + 16 * RW, qt.r_end);
    return true;
  }
};

// Zero rows of unselected tokens, by the first part of each tile (rows counted
// in bf16-sized units: D floats are 2 D of them).
template <int D, int RW>
__device__ __forceinline__ void zero_rows(const AttnArgs& a, void* out, float* lse, const Rows<RW>& rw, bool have) {
  if (!have) zero_empty_lane<2 * D>(a, static_cast<bf16*>(out), lse, rw.qt, 64 * kWaves);
  else if (rw.sub == 0) zero_unselected<2 * D>(a, static_cast<bf16*>(out), lse, rw.qt, 64 * kWaves);
}

// Forward (DQ = false): o and lse.  dq (DQ = true): dS^T = P^T (dP^T - delta),
// dQ^T += K^T dS^T.  S^T = K Q^T, so a lane's query is its column i.
template <int D, int RW, bool DQ>
__global__ __launch_bounds__(64 * kWaves) void f32_rows_kernel(const AttnArgs a) {
  using TL = Tile<D>;
  constexpr int KG = kWaves / RW, KS = TL::KS, DT = TL::DT;
  constexpr int NB = (TL::NBLK + RW - 1) / RW;  // tile blocks a wave copies
  const float* q = reinterpret_cast<const float*>(a.q);
  const float* dout = reinterpret_cast<const float*>(a.dout);
  float* out = reinterpret_cast<float*>(DQ ? a.dq : a.o);
  float* const lse_out = DQ ? nullptr : a.lse;
  Rows<RW> rows;
  if (!rows.init(a)) {
    zero_rows<D, RW>(a, out, lse_out, rows, false);
    return;
  }
  zero_rows<D, RW>(a, out, lse_out, rows, true);
  if (rows.r0 >= rows.r_end) return;  // a part past the end of a short tile
  const QTile<true>& qt = rows.qt;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, G = l >> 4;
  const int rw = wave % RW, kg = wave / RW;
  const int hq = qt.hq;
  const int rw0 = rows.r0 + 16 * rw;
  const bool wave_active = rw0 < rows.r_end;
  const int r = rw0 + i;
  const bool valid = r < rows.r_end;
  const int64_t t = valid ? qt.rv.token(r) : 0;
  const int p = valid ? qt.rv.posn(r) : -1;
  const int p_lo = wave_active ? qt.rv.posn(rw0) : 0;
  const int p_hi = wave_active ? qt.rv.posn(min(rw0 + 15, rows.r_end - 1)) : -1;
  const int ntl = (qt.rv.posn(rows.r_end - 1) + KT) / KT;  // key tiles the workgroup's rows see
  const int nit = (ntl + KG - 1) / KG;
  const float c = a.scale_log2;
  const int stride = a.h * D;
  const int64_t kv0 = ((int64_t)qt.bos * a.h + qt.h) * D;
  const float* k0 = reinterpret_cast<const float*>(a.k) + kv0;
  const float* v0 = reinterpret_cast<const float*>(a.v) + kv0;
  char* const stage0 = logo_smem + kg * 4 * TL::BYTES;
  TL tl;
  tl.init();
  // the group's waves copy its K and V tile `it` (keys past the segment read
  // its last key: masked)
  auto copy = [&](int it) {
    const int kt = KT * (KG * it + kg);
    if (kt >= KT * ntl) return;
    const int last = min(KT - 1, qt.seqlen - 1 - kt);
    char* const st = stage0 + 2 * (it & 1) * TL::BYTES;
    const auto rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(k0 + (int64_t)kt * stride), (short)0,
                                                      last * stride * 4 + TL::RB, kBufRsrcWord3);
    const auto rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(v0 + (int64_t)kt * stride), (short)0,
                                                      last * stride * 4 + TL::RB, kBufRsrcWord3);
    auto off = [&](int row) { return (uint32_t)(min(row, last) * stride * 4); };
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (TL::NBLK % RW == 0 || rw + RW * b < TL::NBLK) {
        TL::copy_block(st, rw + RW * b, rk, off);
        TL::copy_block(st + TL::BYTES, rw + RW * b, rv, off);
      }
  };
  copy(0);

  f32x4 qreg[KS], dreg[DQ ? KS : 1];
  const int64_t qoff = (t * a.hq + hq) * D + 4 * G;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qreg[ks] = valid ? *reinterpret_cast<const f32x4*>(q + qoff + 16 * ks) : f32x4{};
    if constexpr (DQ) dreg[ks] = valid ? *reinterpret_cast<const f32x4*>(dout + qoff + 16 * ks) : f32x4{};
  }
  const float lse = DQ && valid ? a.lse[(int64_t)hq * a.n + r] : 0.f;
  const float dlt = DQ && valid ? a.delta[(int64_t)hq * a.n + r] : 0.f;
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{};
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's keys only

  for (int it = 0; it < nit; ++it) {
    const int kt = KT * (KG * it + kg);
    barrier_all();  // tile `it` has landed; every wave is done with the other stage
    if (it + 1 < nit) copy(it + 1);
    if (kt > p_hi) continue;  // (wave-uniform) no row sees these keys
    const char* kb = stage0 + 2 * (it & 1) * TL::BYTES;
    const char* vb = kb + TL::BYTES;
    // item j is key kt + 4 G + j
    const bool mask = kt + KT - 1 > p_lo;
    f32x4 s = f32x4{};
    if constexpr (DQ) {
      f32x4 dp = f32x4{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const f32x4 kr = tl.row(kb, ks), vr = tl.row(vb, ks);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[e], qreg[ks][e], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e], dreg[ks][e], dp, 0, 0, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] = fmaf(s[j], c, -lse);
      s = exp2_4(s);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (mask && kt + 4 * G + j > p) s[j] = 0.f;
        s[j] *= dp[j] - dlt;
      }
      tr_product<D>(tl, kb, s, acc);
    } else {
      s = row_product<D>(tl, kb, qreg) * c;
      if (mask)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (kt + 4 * G + j > p) s[j] = -INFINITY;
      const float m_new = fmaxf(m_run, col_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
      // a query that has seen no key keeps m = -inf, P and l zero through base 0
      const float base = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = exp2f(m_run - base);
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] -= base;
      s = exp2_4(s);
      l_run = l_run * alpha + ((s[0] + s[1]) + (s[2] + s[3]));
      m_run = m_new;
      if (__ballot(alpha != 1.f)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
      }
      tr_product<D>(tl, vb, s, acc);
    }
  }

  // Combine the key groups: every wave leaves its partial as [wave][dt][lane],
  // then the waves of a row group share its column blocks.
  constexpr int PW = DT * 64;  // f32x4 per wave
  f32x4* const part = reinterpret_cast<f32x4*>(logo_smem);
  float* const stat = reinterpret_cast<float*>(logo_smem + (size_t)kWaves * PW * sizeof(f32x4));  // m, l [wave][16]
  barrier_all();
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) part[wave * PW + dt * 64 + l] = acc[dt];
  if constexpr (!DQ) {
    const float ls = col_sum(l_run);
    if (G == 0) {
      stat[wave * 32 + i] = m_run;
      stat[wave * 32 + 16 + i] = ls;
    }
  }
  __syncthreads();
  if (!valid) return;
  float w[KG], inv = 1.f;
  if constexpr (DQ) {
#pragma unroll
    for (int k = 0; k < KG; ++k) w[k] = a.scale;
  } else {
    float m = -INFINITY, ls = 0.f;
#pragma unroll
    for (int k = 0; k < KG; ++k) m = fmaxf(m, stat[(k * RW + rw) * 32 + i]);
#pragma unroll
    for (int k = 0; k < KG; ++k) {
      w[k] = exp2f(stat[(k * RW + rw) * 32 + i] - m);
      ls = fmaf(w[k], stat[(k * RW + rw) * 32 + 16 + i], ls);
    }
    inv = 1.f / ls;
    if (G == 0 && kg == 0) a.lse[(int64_t)hq * a.n + r] = m + log2f(ls);
  }
  float* const orow = out + (t * a.hq + hq) * D + 4 * G;
#pragma unroll
  for (int d0 = 0; d0 < DT; d0 += KG) {
    const int dt = d0 + kg;
    if (DT % KG != 0 && dt >= DT) break;
    f32x4 sum = f32x4{};
#pragma unroll
    for (int k = 0; k < KG; ++k) sum += part[(k * RW + rw) * PW + dt * 64 + l] * w[k];
    *reinterpret_cast<f32x4*>(orow + 16 * dt) = sum * inv;
  }
}

// ---------------------------------------------------------------------------
// dk / dv: S = Q K^T, P, dP = dO V^T, dS; dV^T += dO^T P, dK^T += Q^T dS,
// summed over the query heads of the GQA group.
// ---------------------------------------------------------------------------
// Step t of a row group is its rows 16 (RG t + rg) ..; q and dO tiles pass
// through a ring of three.  One barrier a step, in its middle: before it wave A
// has left P(t) in LDS and tile t + 1 has landed; after it wave B takes P(t),
// and tile t + 2 may replace tile t - 1, which no wave reads any more.
template <int D>
constexpr size_t dkv_group_bytes() { return 3 * 2 * (size_t)Tile<D>::BYTES + 3 * 3 * KT * sizeof(float); }

template <int D, int NP>
__global__ __launch_bounds__(64 * kWaves) void f32_dkv_kernel(const AttnArgs a) {
  using TL = Tile<D>;
  constexpr int RG = kWaves / (2 * NP), KS = TL::KS, DT = TL::DT;
  constexpr int GW = 2 * NP;  // waves of a row group, which copy its tiles
  constexpr int NB = (2 * TL::NBLK + GW - 1) / GW;
  constexpr int SUB = kBKV / (KT * NP);  // workgroups per kBKV-key tile
  int rank, h;
  xcd_remap(blockIdx.x, a.h, rank, h);
  const int tile = rank / SUB;
  if (tile >= a.meta[2]) return;
  const int32_t* cu_tk = a.meta + kMetaHdr + 2 * (a.nseq + 1);
  const int s = seg_of(cu_tk, a.nseq, tile);
  const int bos = a.cu[s];
  const int seqlen = a.cu[s + 1] - bos;
  const int k0 = (tile - cu_tk[s]) * kBKV + KT * NP * (rank % SUB);
  if (k0 >= seqlen) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 15, G = l >> 4;
  const bool role_b = wave & 1;
  const int pair = (wave >> 1) % NP, rg = wave / GW, gw = wave % GW;
  const int kw0 = k0 + KT * pair;
  const int key = kw0 + i;
  const bool valid_k = key < seqlen;
  const bool pair_keys = kw0 < seqlen;
  const float c = a.scale_log2;
  char* const ring = logo_smem + rg * dkv_group_bytes<D>();
  float* const sstat = reinterpret_cast<float*>(ring + 3 * 2 * TL::BYTES);  // [slot][lse | delta | pos][16]
  f32x4* const pbuf = reinterpret_cast<f32x4*>(logo_smem + RG * dkv_group_bytes<D>()) + (wave >> 1) * 2 * 64;
  TL tl;
  tl.init();

  f32x4 kv[KS];  // A: K, B: V
  {
    const float* src = reinterpret_cast<const float*>(role_b ? a.v : a.k) +
                       ((int64_t)(bos + min(key, seqlen - 1)) * a.h + h) * D + 4 * G;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kv[ks] = valid_k ? *reinterpret_cast<const f32x4*>(src + 16 * ks) : f32x4{};
  }
  f32x4 acc[DT];  // A: dV, B: dK
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{};

  for (int gg = 0; gg < a.g; ++gg) {
    const int hq = h * a.g + gg;
    const int lane_sel = a.lanes > 1 ? hq : 0;
    const int32_t* cu_q = a.meta + (int64_t)lane_sel * a.meta_stride + kMetaHdr;
    const RowView<true> rv = row_view<true>(a, lane_sel, bos);
    const int rq_end = __builtin_amdgcn_readfirstlane(cu_q[s + 1]);
    const int rq0 = __builtin_amdgcn_readfirstlane(wave_lower_bound(rv.ps, cu_q[s], rq_end, k0));
    if (rq0 >= rq_end) continue;  // no row of this head sees these keys
    const int nt = (rq_end - rq0 + KT * RG - 1) / (KT * RG);  // steps, the same for every group
    // rows before lb0 see none of the pair's keys
    const int lb0 = __builtin_amdgcn_readfirstlane(wave_lower_bound(rv.ps, rq0, rq_end, kw0));
    const float* lse_h = a.lse + (int64_t)hq * a.n;
    const float* delta_h = a.delta + (int64_t)hq * a.n;
    // 32-bit byte offsets from the head's first row (the launcher checks that
    // the tensors are below 4 GB)
    const uint32_t row_bytes = (uint32_t)a.hq * D * 4;
    const auto rq = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(reinterpret_cast<const float*>(a.q) + (int64_t)hq * D), (short)0, -1, kBufRsrcWord3);
    const auto ro = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(reinterpret_cast<const float*>(a.dout) + (int64_t)hq * D), (short)0, -1, kBufRsrcWord3);
    auto row_of = [&](int t) { return rq0 + KT * (RG * t + rg); };  // first row of step t
    // lanes i: token and statistic of row i of step t, loaded a step before use.
    // Rows past the end repeat the last one at position -1: they see no key.
    // Wave gw = 0 of a group loads lse and the positions, gw = 1 delta.
    auto load_tok = [&](int t) { return (int)rv.token(min(row_of(t) + i, rq_end - 1)); };
    auto copy = [&](int t, int slot, int tok) {
      char* const dst = ring + slot * 2 * TL::BYTES;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int b = gw + GW * n;  // q blocks, then dO blocks
        if (2 * TL::NBLK % GW == 0 || b < 2 * TL::NBLK) {
          const bool isq = b < TL::NBLK;
          TL::copy_block(dst + (isq ? 0 : TL::BYTES), isq ? b : b - TL::NBLK, isq ? rq : ro,
                         [&](int row) { return (uint32_t)__shfl(tok, row) * row_bytes; });
        }
      }
    };
    struct Stat {
      float x;
      int pos;
    };
    auto load_stat = [&](int t) {
      const int rr = row_of(t) + i, rc = min(rr, rq_end - 1);
      Stat st{0.f, -1};
      if (gw == 0) {
        st.x = lse_h[rc];
        st.pos = rr < rq_end ? rv.posn(rr) : -1;
      } else if (gw == 1) {
        st.x = delta_h[rc];
      }
      return st;
    };
    auto store_stat = [&](int slot, const Stat& st) {
      if (gw > 1 || G != 0) return;
      sstat[(3 * slot + gw) * KT + i] = st.x;
      if (gw == 0) reinterpret_cast<int*>(sstat)[(3 * slot + 2) * KT + i] = st.pos;
    };

    {
      const Stat s0 = load_stat(0), s1 = load_stat(1);
      copy(0, 0, load_tok(0));
      store_stat(0, s0);
      if (nt > 1) {
        copy(1, 1, load_tok(1));
        store_stat(1, s1);
      }
    }
    int tok = load_tok(2);
    barrier_all();
    int slot = 0;
    for (int t = 0; t < nt; ++t) {
      const int nslot = slot == 2 ? 0 : slot + 1, pslot = slot == 0 ? 2 : slot - 1;
      const char* qb = ring + slot * 2 * TL::BYTES;
      const char* ob = qb + TL::BYTES;
      const float* st = sstat + 3 * slot * KT;
      const bool more = t + 2 < nt;
      Stat sn{};
      if (more) sn = load_stat(t + 2);
      const bool live = pair_keys && row_of(t) < rq_end && row_of(t) + KT > lb0;
      f32x4 x = f32x4{};  // A: S then P, B: dP then dS; item j is row 4 G + j of the step, column `key`
      if (live) {
        x = row_product<D>(tl, role_b ? ob : qb, kv);
        if (!role_b) {
          const f32x4 l4 = lds_load(reinterpret_cast<const f32x4*>(st + 4 * G));
          const int4 p4 = lds_load(reinterpret_cast<const int4*>(st + 2 * KT + 4 * G));
          const int pq[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = fmaf(x[j], c, -l4[j]);
          x = exp2_4(x);
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = valid_k && key <= pq[j] ? x[j] : 0.f;
          pbuf[(t & 1) * 64 + l] = x;
        }
      }
      barrier_all();
      if (more) {
        store_stat(pslot, sn);
        copy(t + 2, pslot, tok);
        tok = load_tok(t + 3);
      }
      if (live) {
        if (role_b) {
          const f32x4 pr = pbuf[(t & 1) * 64 + l];
          const f32x4 d4 = lds_load(reinterpret_cast<const f32x4*>(st + KT + 4 * G));
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = pr[j] * (x[j] - d4[j]);
        }
        const char* tb = role_b ? qb : ob;
        tr_product<D>(tl, tb, x, acc);
      }
      slot = nslot;
    }
    barrier_all();  // the rings are free for the next head
  }

  // lane (i, G) holds columns 16 dt + 4 G .. + 3 of key `key`; the row groups
  // of a pair are added through LDS
  const float mul = role_b ? a.scale : 1.f;
  float* const dst = reinterpret_cast<float*>(role_b ? a.dk : a.dv) + ((int64_t)(bos + key) * a.h + h) * D + 4 * G;
  if constexpr (RG == 1) {
    if (!valid_k) return;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(dst + 16 * dt) = acc[dt] * mul;
  } else {
    constexpr int PW = DT * 64;
    f32x4* const part = reinterpret_cast<f32x4*>(logo_smem);
    __syncthreads();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) part[wave * PW + dt * 64 + l] = acc[dt];
    __syncthreads();
    if (!valid_k) return;
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += RG) {
      const int dt = d0 + rg;
      f32x4 sum = f32x4{};
#pragma unroll
      for (int k = 0; k < RG; ++k) sum += part[(k * GW + gw) * PW + dt * 64 + l];
      *reinterpret_cast<f32x4*>(dst + 16 * dt) = sum * mul;
    }
  }
}

// delta = rowsum(o * dO) per compacted row: D / 4 lanes of 16 bytes a row
template <int D>
__global__ __launch_bounds__(256) void f32_delta_kernel(const AttnArgs a) {
  constexpr int LPR = D / 4, RPB = 256 / LPR;
  const int hq = blockIdx.y, lane_sel = a.lanes > 1 ? hq : 0;
  const int sq = a.meta[(int64_t)lane_sel * a.meta_stride];
  const int r = blockIdx.x * RPB + threadIdx.x / LPR, c = threadIdx.x % LPR;
  if ((int)blockIdx.x * RPB >= sq) return;
  const bool ok = r < sq;
  const int64_t off = ((ok ? a.q_idx[(int64_t)lane_sel * a.n + r] : 0) * a.hq + hq) * D + 4 * c;
  const f32x4 o = ok ? *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.o) + off) : f32x4{};
  const f32x4 d = ok ? *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.dout) + off) : f32x4{};
  float acc = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = fmaf(o[e], d[e], acc);
  acc = group_sum<LPR>(acc);
  if (ok && c == 0) a.delta[(int64_t)hq * a.n + r] = acc;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <int D, int RW>
constexpr size_t rows_smem() {
  return std::max((size_t)(kWaves / RW) * 4 * Tile<D>::BYTES,
                  (size_t)kWaves * Tile<D>::DT * 64 * sizeof(f32x4) + kWaves * 32 * sizeof(float));
}
template <int D, int NP>
constexpr size_t dkv_smem() {
  constexpr int RG = kWaves / (2 * NP);
  return std::max(RG * dkv_group_bytes<D>() + (size_t)(kWaves / 2) * 2 * 64 * sizeof(f32x4),
                  RG == 1 ? (size_t)0 : (size_t)kWaves * Tile<D>::DT * 64 * sizeof(f32x4));
}

template <int D, int RW, bool DQ>
int launch_rows(const AttnArgs& a, hipStream_t st) {
  const int64_t nblk = (kBQ / (16 * RW)) * ((a.n + kBQ - 1) / kBQ + a.nseq) * a.hq;
  LOGO_REQUIRE(nblk < ((int64_t)1 << 31), "grid too large");
  auto kern = f32_rows_kernel<D, RW, DQ>;
  LOGO_HIP_CHECK(allow_smem(kern, rows_smem<D, RW>()));
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(64 * kWaves), (rows_smem<D, RW>()), st, a);
  LOGO_LAUNCH_CHECK("f32_rows_kernel");
  return LOGO_OK;
}

template <int D, int NP>
int launch_dkv(const AttnArgs& a, hipStream_t st) {
  const int64_t nblk = (kBKV / (KT * NP)) * ((a.n + kBKV - 1) / kBKV + a.nseq) * a.h;
  LOGO_REQUIRE(nblk < ((int64_t)1 << 31), "grid too large");
  auto kern = f32_dkv_kernel<D, NP>;
  LOGO_HIP_CHECK(allow_smem(kern, dkv_smem<D, NP>()));
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(64 * kWaves), (dkv_smem<D, NP>()), st, a);
  LOGO_LAUNCH_CHECK("f32_dkv_kernel");
  return LOGO_OK;
}

// Row waves per workgroup: as many as leave two workgroups a CU, taking a third
// of the (token, head) rows as selected (the count is on the device), within
// the LDS of the key groups.
template <int D, bool DQ>
int dispatch_rows(const AttnArgs& a, hipStream_t st) {
  constexpr int RW_MIN = D / 64;  // 128 KB of tiles
  const int64_t per_cu = a.n * a.hq / 3 / 32 / std::max(device_cus(), 1);
  if constexpr (RW_MIN <= 1)
    if (per_cu < 2) return launch_rows<D, 1, DQ>(a, st);
  if constexpr (RW_MIN <= 2)
    if (per_cu < 4) return launch_rows<D, 2, DQ>(a, st);
  return launch_rows<D, 4, DQ>(a, st);
}

// Pairs per workgroup: as many as leave four workgroups a CU.
template <int D>
int dispatch_dkv(const AttnArgs& a, hipStream_t st) {
  const int64_t per_cu = a.n * a.h / KT / std::max(device_cus(), 1);
  if constexpr (D <= 64)
    if (per_cu < 8) return launch_dkv<D, 1>(a, st);
  if constexpr (D <= 128)
    if (per_cu < 16) return launch_dkv<D, 2>(a, st);
  return launch_dkv<D, 4>(a, st);
}

template <int D>
int launch(const AttnArgs& a, hipStream_t st, int phase) {
  if (phase == kPhaseFwd) return dispatch_rows<D, false>(a, st);
  if (phase == kPhaseDq) return dispatch_rows<D, true>(a, st);
  if (phase == kPhaseDkv) return dispatch_dkv<D>(a, st);
  constexpr int RPB = 256 / (D / 4);
  hipLaunchKernelGGL((f32_delta_kernel<D>), dim3((unsigned)((a.n + RPB - 1) / RPB), a.hq), dim3(256), 0, st, a);
  LOGO_LAUNCH_CHECK("f32_delta_kernel");
  return LOGO_OK;
}

}  // namespace f32

bool f32_applies(const AttnArgs& a, int d, int dtype, bool sparse) {
  return dtype == LOGO_DTYPE_F32 && sparse && a.window < 0 && a.n * a.hq * d * (int64_t)sizeof(float) < ((int64_t)1 << 32);
}

int f32_launch(const AttnArgs& a, hipStream_t st, int phase, int d) {
  return d == 64 ? f32::launch<64>(a, st, phase) : d == 128 ? f32::launch<128>(a, st, phase)
                                                             : f32::launch<256>(a, st, phase);
}

}  // namespace logo
