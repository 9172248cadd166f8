// Query-sparse / dense causal attention at head dim 256 in 16-bit types,
// forward and backward, for gfx950 (logo/ops/selected_full_attn.py:33-337; the
// reference takes any K <= 256 in one block, :344).  The tuned kernels'
// scheme with 32x32x16 MFMAs, cut for 256 columns:
//   fwd, dq : 4 waves x 32 compacted rows per workgroup, one wave per SIMD;
//             64-key K / V tiles (two LDS slots each, 128 KB), walked in
//             32-key halves: the S (dP) MFMAs of the next half run with the
//             softmax arithmetic of the current one, then its PV (K^T dS)
//             MFMAs.  Q (and dO) sit in registers, dQ in AGPRs.
//   dk/dv   : two pairs of waves x 32 keys; in a pair one wave computes S, P
//             and dV, the other dP, dS and dK, P passing through LDS; 32
//             gathered rows of q and dO a step.
// An operand read from LDS feeds one MFMA here (the wave's registers hold no
// second row block), 1 KB per 32 cycles and SIMD: all of the LDS bandwidth at the
// MFMA peak, so about half of that peak is the most this form can reach.
// Bound: waits.  One wave a SIMD is resident; at T = 8192, 16 heads, a quarter of
// the rows it waits 40 / 33 / 34% of its time (forward, dq, dk/dv: for barriers,
// the copies behind them, LDS operands) with the matrix units 26 / 37 / 32%, the
// VALU 20 / 16 / 25% and the LDS 13 / 19 / 22% busy.  Forward + backward there:
// 784 to 897 us on the boxes measured, 1825 to 1866 on the generic kernels (16
// rows or keys a wave on 16x16 MFMAs, one LDS operand read per half as many FLOPs,
// no pipelining); 4001 tokens, 4 heads, forward only with split key ranges: 70
// against 227 us; a few hundred tokens are bound by the launches either way.
// Numerics are the generic kernels' but for three things: S from the unscaled
// inputs, scaled in fp32; P and dS rounded to the input type.  The dP accumulators
// start from -delta; the forward's running maximum may lag by up to 2^8 (o is
// 0.05% further from float64 so, relative to its error of 1.9e-3; dq, dk and dv as
// near); the hardware's exp2 flushes P below 2^-126, as in the kernels of dim 64
// and 128.  q and dO rows are gathered in place (no compacted copies).
#include "sq_attn.hpp"

#include <algorithm>

namespace logo {
namespace wide {

constexpr int D = 256, DS = D / 16, DT = D / 32;
using GT = TileGeom<D, kSwz>;
constexpr int kHalf = 32;  // keys per half tile (fwd, dq); query rows per step (dk/dv)

// Operand reads from swizzled tiles (TileReader's, with the column blocks that
// differ by 128 columns sharing a lane offset: the swizzle leaves bit 4 of the
// chunk alone).
struct Reader {
  int row_off[DS / 2], tr_off[DT];
  __device__ __forceinline__ void init() {
    const int l = threadIdx.x & 63, i = l & 31, g = l >> 5, G = l >> 4, j = l & 15;
#pragma unroll
    for (int ks = 0; ks < DS / 2; ++ks) row_off[ks] = GT::off(i, 2 * ks + g);
#pragma unroll
    for (int dt = 0; dt < DT / 2; ++dt)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 4 * g + (j >> 2) + 8 * h, col = 32 * dt + 16 * (G & 1) + 4 * (j & 3);
        tr_off[2 * dt + h] = GT::off(row, col >> 3) + (col & 7);
      }
  }
  template <typename E>
  __device__ __forceinline__ typename Elem<E>::x8 row(const bf16* tile, int rbase, int ks) const {
    return lds_load(reinterpret_cast<const typename Elem<E>::x8*>(tile + rbase * D + 128 * (ks >> 3) + row_off[ks & 7]));
  }
  template <typename E>
  __device__ __forceinline__ typename Elem<E>::x8 tr(const bf16* tile, int r0, int dt) const {
    using L4 = std::conditional_t<Elem<E>::kHalf, lds_hf16x4, lds_bf16x4>;
    const bf16* t = tile + r0 * D + 128 * (dt >> 2);
    const auto lo = ds_read_tr((const L4*)(t + tr_off[2 * (dt & 3)]));
    const auto hi = ds_read_tr((const L4*)(t + tr_off[2 * (dt & 3) + 1]));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// The copies of one step may still be in flight at its end (one 64-row tile is
// eight loads a wave); everything older has landed.
__device__ __forceinline__ void step_end(bool newest_in_flight) {
  if (newest_in_flight) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Output rows of a workgroup (128 x 256 in LDS, kSwz 64-row tiles) to the
// scattered token rows, 32 lanes a row.
template <bool SPARSE, bool NT>
__device__ __forceinline__ void store_rows(const bf16* blk, const AttnArgs& a, const QTile<SPARSE>& qt, bf16* out) {
  const int ch = threadIdx.x & 31, nrow = qt.r_end - qt.r0;
  for (int r = threadIdx.x >> 5; r < nrow; r += 8) {
    const int64_t tok = qt.rv.token(qt.r0 + r);
    const u32x4 v = *reinterpret_cast<const u32x4*>(blk + (r >> 6) * GT::ELEMS + GT::off(r & 63, ch));
    u32x4* const p = reinterpret_cast<u32x4*>(out + (tok * a.hq + qt.hq) * D + 8 * ch);
    if constexpr (NT) st_nt(p, v);
    else *p = v;
  }
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
// Step (t, H) of key tile t: X: S of the next half ((t, 1) or (t + 1, 0)) with
// P of half (t, H); Y: O += V^T P of half (t, H) with the mask and row max of
// the next half; then the next half's statistics (lazy rescale, as the tuned
// forward).  V(t + 1) is copied during (t, 0), K(t + 2) during (t, 1): each
// two steps ahead of its first read, into the slot whose last read was the
// step before.
template <typename EL, bool SPARSE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void w256_fwd_kernel(const AttnArgs a) {
  using E8 = typename Elem<EL>::x8;
  using E4 = typename Elem<EL>::x4;
  constexpr int NX = DS, NY = 2 * DT, PF = 4;
  bf16* const smem = dyn_smem();
  auto tileK = [&](int b) { return smem + b * GT::ELEMS; };
  auto tileV = [&](int b) { return smem + (2 + b) * GT::ELEMS; };
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  QTile<SPARSE> qt;
  if (!qt.init(a, wave, i, false, 32, false, true)) {
    if constexpr (SPARSE) zero_empty_lane<D>(a, a.o, a.lse, qt, 256);
    return;
  }
  const int hq = qt.hq, p = qt.p;
  E8 qreg[DS];
  {
    const bf16* qrow = a.q + (qt.t * a.hq + hq) * D + 8 * g;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) qreg[ds] = qt.valid ? *reinterpret_cast<const E8*>(qrow + 16 * ds) : E8{};
  }
  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x16{};
  f32x16 sb[2];  // S of half H (index H) and of the next half
  E8 pb[2];      // P of the current half, one per 16-key step
  float m_run = -INFINITY, l_run = 0.f, base = 0.f;
  const float c = a.scale_log2;

  Reader rd;
  rd.init();
  const int64_t rstride = (int64_t)a.h * D;
  const bf16* kbase = a.k + ((int64_t)qt.bos * a.h + qt.h) * D;
  const bf16* vbase = a.v + ((int64_t)qt.bos * a.h + qt.h) * D;
  const int seqlen = qt.seqlen;
  TileBufDma<D, 4> dma;
  dma.init((int)rstride);
  auto load_one = [&](bf16* tile, const bf16* src, int j0) {
    if (j0 + 64 <= seqlen) dma.issue(tile, src + j0 * rstride);
    else dma.issue_clamped(tile, src + j0 * rstride, seqlen - 1 - j0);
  };
  const int kv_lo = qt.kv_lo;
  const int nt = (qt.kv_hi - kv_lo + 63) >> 6;
  const bool desc = qt.desc;
  auto ph = [&](int t) { return desc ? nt - 1 - t : t; };
  const int hw_hi = qt.wave_active ? min(2 * nt, ((qt.pmax - kv_lo) >> 5) + 1) : 0;  // halves this wave's rows see

  auto step = [&](auto par_tag, auto h_tag, int t) {
    constexpr int PAR = decltype(par_tag)::value, H = decltype(h_tag)::value;  // PAR: t & 1
    bool newest = false;
    if (H == 0) {
      if ((newest = t + 1 < nt)) load_one(tileV(PAR ^ 1), vbase, kv_lo + 64 * ph(t + 1));
    } else {
      if ((newest = t + 2 < nt)) load_one(tileK(PAR), kbase, kv_lo + 64 * ph(t + 2));
    }
    const bf16* kx = tileK(H == 0 ? PAR : PAR ^ 1) + (H == 0 ? 32 * D : 0);
    const bf16* vy = tileV(PAR) + 32 * D * H;
    const int hx = t >= 0 ? 2 * ph(t) + H : -1;
    const int hn = H == 0 ? 2 * ph(t) + 1 : (t + 1 < nt ? 2 * ph(t + 1) : -1);
    const int j0n = kv_lo + 32 * hn;
    auto body = [&](auto dox_tag, auto dov_tag, auto mask_tag) {
      constexpr bool DOX = decltype(dox_tag)::value, DOV = decltype(dov_tag)::value, MASK = decltype(mask_tag)::value;
      E8 op[NX + NY];
      auto load_op = [&](auto s_c) {
        constexpr int S = decltype(s_c)::value;
        if constexpr (S < NX) {
          if constexpr (DOX) op[S] = rd.template row<EL>(kx, 0, S);
        } else {
          if constexpr (DOV) op[S] = rd.template tr<EL>(vy, 16 * ((S - NX) / DT), (S - NX) % DT);
        }
      };
      static_for<PF>([&](auto s_c) { load_op(s_c); });
      const int hi = p - j0n - 4 * g;
      float mx = -INFINITY, psum = 0.f;
      static_for<NX + NY>([&](auto s_c) {
        constexpr int S = decltype(s_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        float spv = 0.f;
        if constexpr (DOV && S < 16) {
          spv = sb[H][S];
          pin(spv);
        }
        if constexpr (S < NX) {
          if constexpr (DOX) sb[H ^ 1] = mfma32(op[S], qreg[S], S == 0 ? f32x16{} : sb[H ^ 1]);
        } else {
          constexpr int Y = S - NX;
          if constexpr (DOV) oacc[Y % DT] = mfma32(op[S], pb[Y / DT], oacc[Y % DT]);
          // mask and max of the next half, two slots behind its last MFMA
          constexpr int I0 = Y < 2 ? 0 : ((Y - 2) * 16 + 13) / 14, I1 = Y < 1 ? 0 : ((Y - 1) * 16 + 13) / 14;
          if constexpr (DOX)
            static_for<I1 - I0>([&](auto e_c) {
              constexpr int JJ = I0 + decltype(e_c)::value;
              float sv = sb[H ^ 1][JJ];
              if constexpr (MASK) {
                pin(sv);
                constexpr int off = 8 * (JJ / 4) + (JJ % 4);
                if (!(off <= hi)) sv = -INFINITY;
                sb[H ^ 1][JJ] = sv;
              }
              mx = max3_f32(mx, sv, sv);
            });
        }
        if constexpr (DOV) {
          if constexpr (S < 16) {
            float pv = fast_exp2(fmaf(spv, c, -base));
            pin(pv);
            sb[H][S] = pv;
          }
          if constexpr (S >= 1 && S <= 16) {
            psum += sb[H][S - 1];
            if constexpr (S % 8 == 0) {
              pb[S / 8 - 1] = acc_to<EL>(sb[H], S / 8 - 1);
              pin(pb[S / 8 - 1]);
            }
            pin(psum);
          }
        }
        if constexpr (S + PF < NX + NY) load_op(std::integral_constant<int, S + PF>{});
      });
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DOV) l_run += psum;
      if constexpr (DOX) {
        const float mxs = pair_max(mx) * c;
        const bool any_grow = __ballot(mxs - m_run > 8.f);
        const float m_new = any_grow ? fmaxf(m_run, mxs) : m_run;
        const float nbase = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - nbase);
        l_run *= alpha;
        m_run = m_new;
        base = nbase;
        if (__ballot(alpha != 1.f)) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
        }
      }
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    const bool dox = hn >= 0 && hn < hw_hi, dov = hx >= 0 && hx < hw_hi;
    const bool maskn = j0n + 31 > qt.pmin;
    if (dox && dov) {
      if (maskn) body(T_{}, T_{}, T_{});
      else body(T_{}, T_{}, F_{});
    } else if (dox) {
      body(T_{}, F_{}, T_{});
    } else if (dov) {
      body(F_{}, T_{}, F_{});
    }
    step_end(newest);
  };

  load_one(tileK(0), kbase, kv_lo + 64 * ph(0));
  load_one(tileV(0), vbase, kv_lo + 64 * ph(0));
  step_end(false);
  step(BufTag<1>{}, BufTag<1>{}, -1);  // S of half (0, 0); copies K(1)
  for (int t = 0; t < nt; t += 2) {
    step(BufTag<0>{}, BufTag<0>{}, t);
    step(BufTag<0>{}, BufTag<1>{}, t);
    if (t + 1 < nt) {
      step(BufTag<1>{}, BufTag<0>{}, t + 1);
      step(BufTag<1>{}, BufTag<1>{}, t + 1);
    }
  }

  float l_tot = pair_sum(l_run);
  if constexpr (SPARSE)
    if (qt.piece == 0) zero_unselected<D>(a, a.o, a.lse, qt, 256);
  if (qt.nsplit > 1) {  // as the tuned forward: partials by piece, combined by the last to arrive
    constexpr int OF = DT * 16 * 64;
    float* const part0 = a.part + (int64_t)(hq * 2 * a.split_cap + qt.trank * qt.nper) * 4 * (OF + 64);
    {
      float* po = part0 + (int64_t)qt.piece * 4 * (OF + 64) + wave * (OF + 64);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) st_agent(po + (dt * 16 + e) * 64 + l, oacc[dt][e]);
      st_agent(po + OF + l, g == 0 ? m_run : l_tot);
    }
    if (!split_arrive(a.cnt + hq * 2 * a.split_cap + qt.trank, qt.nsplit, reinterpret_cast<int*>(smem))) return;
    float w[kMaxSplit], mx = -INFINITY, lsum = 0.f;
    for (int pc = 0; pc < qt.nsplit; ++pc) {
      const float* po = part0 + (int64_t)pc * 4 * (OF + 64) + wave * (OF + 64);
      const float mc = ld_agent(po + OF + i), lc = ld_agent(po + OF + 32 + i);
      if (lc > 0.f) mx = fmaxf(mx, mc);
    }
    for (int pc = 0; pc < qt.nsplit; ++pc) {
      const float* po = part0 + (int64_t)pc * 4 * (OF + 64) + wave * (OF + 64);
      const float mc = ld_agent(po + OF + i), lc = ld_agent(po + OF + 32 + i);
      w[pc] = lc > 0.f ? fast_exp2(mc - mx) : 0.f;
      lsum = fmaf(w[pc], lc, lsum);
    }
    // in piece order, whichever arrived last; one 16-float block at a time
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      f32x16 sum = f32x16{};
      for (int pc = 0; pc < qt.nsplit; ++pc) {
        const float* po = part0 + (int64_t)pc * 4 * (OF + 64) + wave * (OF + 64) + dt * 16 * 64;
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[e] = fmaf(w[pc], ld_agent(po + e * 64 + l), sum[e]);
      }
      oacc[dt] = sum;
    }
    l_tot = lsum;
    m_run = mx;
  }
  const float inv = qt.valid ? 1.f / l_tot : 0.f;
  if (qt.valid && g == 0) a.lse[(int64_t)hq * a.n + qt.r] = m_run + log2f(l_tot);
  __syncthreads();  // every wave is done with the K / V tiles
  const int row = 32 * wave + i;
  bf16* const orow = smem + (row >> 6) * GT::ELEMS;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      E4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (EL)(oacc[dt][4 * q4 + e] * inv);
      *reinterpret_cast<E4*>(orow + GT::off(row & 63, 4 * dt + q4) + 4 * g) = v;
    }
  __syncthreads();
  store_rows<SPARSE, false>(smem, a, qt, a.o);
}

// ---------------------------------------------------------------------------
// delta = rowsum(o * dO) per compacted row: 32 lanes of 16 bytes a row
// ---------------------------------------------------------------------------
template <typename EL, bool SPARSE>
__global__ __launch_bounds__(256) void w256_delta_kernel(const AttnArgs a) {
  using E8 = typename Elem<EL>::x8;
  constexpr int R = 2;  // rows per thread, RPB apart
  constexpr int RPB = 8;
  const int hq = blockIdx.y, lane_sel = a.lanes > 1 ? hq : 0;
  const int sq = a.meta[(int64_t)lane_sel * a.meta_stride];
  const int r0 = blockIdx.x * RPB * R + (threadIdx.x >> 5), c = threadIdx.x & 31;
  if ((int)(blockIdx.x * RPB * R) >= sq) return;
  E8 ov[R], dv[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int r = r0 + k * RPB;
    const bool ok = r < sq;
    const int64_t t = ok ? (SPARSE ? a.q_idx[(int64_t)lane_sel * a.n + r] : (int64_t)r) : 0;
    const int64_t off = (t * a.hq + hq) * D + 8 * c;
    ov[k] = ok ? *reinterpret_cast<const E8*>(a.o + off) : E8{};
    dv[k] = ok ? *reinterpret_cast<const E8*>(a.dout + off) : E8{};
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = fmaf((float)ov[k][e], (float)dv[k][e], acc);
    acc = group_sum<32>(acc);
    const int r = r0 + k * RPB;
    if (r < sq && c == 0) a.delta[(int64_t)hq * a.n + r] = acc;
  }
}

// ---------------------------------------------------------------------------
// dq
// ---------------------------------------------------------------------------
// Step (t, H): X: S / dP of the next half (K rows in even slots, V rows in odd
// ones) with P = exp2(S c - lse) and dS = P dP of half (t, H); Y: dQ += K^T dS
// of half (t, H).  K(t + 1) is copied during (t, 0), after K(t - 1)'s last
// read; V(t + 2) during (t, 1).
template <typename EL, bool SPARSE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void w256_dq_kernel(const AttnArgs a) {
  using E8 = typename Elem<EL>::x8;
  using E4 = typename Elem<EL>::x4;
  constexpr int NX = 2 * DS, NY = 2 * DT, PF = 4;
  bf16* const smem = dyn_smem();
  auto tileK = [&](int b) { return smem + b * GT::ELEMS; };
  auto tileV = [&](int b) { return smem + (2 + b) * GT::ELEMS; };
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  QTile<SPARSE> qt;
  if (!qt.init(a, wave, i, false, 32, false, true)) {
    if constexpr (SPARSE) zero_empty_lane<D>(a, a.dq, nullptr, qt, 256);
    return;
  }
  const int hq = qt.hq, p = qt.p;
  E8 qreg[DS], doreg[DS];
  {
    const int64_t off = (qt.t * a.hq + hq) * D + 8 * g;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      qreg[ds] = qt.valid ? *reinterpret_cast<const E8*>(a.q + off + 16 * ds) : E8{};
      doreg[ds] = qt.valid ? *reinterpret_cast<const E8*>(a.dout + off + 16 * ds) : E8{};
    }
  }
  const float lse = qt.valid ? a.lse[(int64_t)hq * a.n + qt.r] : 0.f;
  const float dlt = qt.valid ? a.delta[(int64_t)hq * a.n + qt.r] : 0.f;
  const float c = a.scale_log2;
  f32x16 c_del;
#pragma unroll
  for (int j = 0; j < 16; ++j) c_del[j] = -dlt;
  f32x16 dqacc[DT];  // AGPRs
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dqacc[dt] = f32x16{};
  f32x16 sp[2][2];  // [half parity][S, dP]
  E8 dsb[2];

  Reader rd;
  rd.init();
  const int64_t rstride = (int64_t)a.h * D;
  const bf16* kbase = a.k + ((int64_t)qt.bos * a.h + qt.h) * D;
  const bf16* vbase = a.v + ((int64_t)qt.bos * a.h + qt.h) * D;
  const int seqlen = qt.seqlen;
  TileBufDma<D, 4> dma;
  dma.init((int)rstride);
  auto load_one = [&](bf16* tile, const bf16* src, int j0) {
    if (j0 + 64 <= seqlen) dma.issue(tile, src + j0 * rstride);
    else dma.issue_clamped(tile, src + j0 * rstride, seqlen - 1 - j0);
  };
  const int kv_lo = qt.kv_lo;
  const int nt = (qt.kv_hi - kv_lo + 63) >> 6;
  const bool desc = qt.desc;
  auto ph = [&](int t) { return desc ? nt - 1 - t : t; };
  const int hw_hi = qt.wave_active ? min(2 * nt, ((qt.pmax - kv_lo) >> 5) + 1) : 0;

  auto step = [&](auto par_tag, auto h_tag, int t) {
    constexpr int PAR = decltype(par_tag)::value, H = decltype(h_tag)::value;
    bool newest = false;
    if (H == 0) {
      if (t + 1 < nt) load_one(tileK(PAR ^ 1), kbase, kv_lo + 64 * ph(t + 1));
    } else {
      if ((newest = t + 2 < nt)) load_one(tileV(PAR), vbase, kv_lo + 64 * ph(t + 2));
    }
    const bf16* kx = tileK(H == 0 ? PAR : PAR ^ 1) + (H == 0 ? 32 * D : 0);
    const bf16* vx = tileV(H == 0 ? PAR : PAR ^ 1) + (H == 0 ? 32 * D : 0);
    const bf16* ky = tileK(PAR) + 32 * D * H;
    const int hx = t >= 0 ? 2 * ph(t) + H : -1;
    const int hn = H == 0 ? 2 * ph(t) + 1 : (t + 1 < nt ? 2 * ph(t + 1) : -1);
    const int j0h = kv_lo + 32 * hx;
    auto body = [&](auto dox_tag, auto dov_tag, auto mask_tag) {
      constexpr bool DOX = decltype(dox_tag)::value, DOV = decltype(dov_tag)::value, MASK = decltype(mask_tag)::value;
      E8 op[NX + NY];
      auto load_op = [&](auto s_c) {
        constexpr int S = decltype(s_c)::value;
        if constexpr (S < NX) {
          if constexpr (DOX) op[S] = rd.template row<EL>(S % 2 ? vx : kx, 0, S / 2);
        } else {
          if constexpr (DOV) op[S] = rd.template tr<EL>(ky, 16 * ((S - NX) / DT), (S - NX) % DT);
        }
      };
      static_for<PF>([&](auto s_c) { load_op(s_c); });
      const int hi = p - j0h - 4 * g;
      static_for<NX + NY>([&](auto s_c) {
        constexpr int S = decltype(s_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        // item JJ: P in slot 2 JJ, dS in slot 2 JJ + 1, groups of eight packed a slot later
        constexpr int JJ = S / 2;
        float sv = 0.f;
        if constexpr (DOV && S < NX && S % 2 == 0) {
          sv = sp[H][0][JJ];
          pin(sv);
        }
        if constexpr (S < NX) {
          if constexpr (DOX) {
            if constexpr (S % 2 == 0) sp[H ^ 1][0] = mfma32(op[S], qreg[JJ], JJ == 0 ? f32x16{} : sp[H ^ 1][0]);
            else sp[H ^ 1][1] = mfma32(op[S], doreg[JJ], JJ == 0 ? c_del : sp[H ^ 1][1]);
          }
          if constexpr (DOV) {
            if constexpr (S % 2 == 0) {
              float pv = fast_exp2(fmaf(sv, c, -lse));
              if constexpr (MASK) {
                constexpr int off = 8 * (JJ / 4) + (JJ % 4);
                if (!(off <= hi)) pv = 0.f;
              }
              sp[H][0][JJ] = pv;
            } else {
              float dsv = sp[H][0][JJ] * sp[H][1][JJ];
              pin(dsv);
              sp[H][1][JJ] = dsv;
            }
          }
        } else {
          constexpr int Y = S - NX;
          if constexpr (DOV) mfma32_agpr_ready(dqacc[Y % DT], op[S], dsb[Y / DT]);
        }
        if constexpr (DOV && (S == 16 || S == 32)) {
          dsb[S / 16 - 1] = acc_to<EL>(sp[H][1], S / 16 - 1);
          pin(dsb[S / 16 - 1]);
        }
        if constexpr (S + PF < NX + NY) load_op(std::integral_constant<int, S + PF>{});
      });
      __builtin_amdgcn_sched_barrier(0);
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    const bool dox = hn >= 0 && hn < hw_hi, dov = hx >= 0 && hx < hw_hi;
    const bool mask = j0h + 31 > qt.pmin;
    if (dox && dov) {
      if (mask) body(T_{}, T_{}, T_{});
      else body(T_{}, T_{}, F_{});
    } else if (dox) {
      body(T_{}, F_{}, F_{});
    } else if (dov) {
      body(F_{}, T_{}, T_{});
    }
    step_end(newest);
  };

  load_one(tileK(0), kbase, kv_lo + 64 * ph(0));
  load_one(tileV(0), vbase, kv_lo + 64 * ph(0));
  step_end(false);
  step(BufTag<1>{}, BufTag<1>{}, -1);  // S / dP of half (0, 0); copies V(1)
  for (int t = 0; t < nt; t += 2) {
    step(BufTag<0>{}, BufTag<0>{}, t);
    step(BufTag<0>{}, BufTag<1>{}, t);
    if (t + 1 < nt) {
      step(BufTag<1>{}, BufTag<0>{}, t + 1);
      step(BufTag<1>{}, BufTag<1>{}, t + 1);
    }
    agpr_acc_drain();  // the epilogue reads dQ: on every path, ahead of any copy placed for it
  }
  if constexpr (SPARSE)
    if (qt.piece == 0) zero_unselected<D>(a, a.dq, nullptr, qt, 256);
  if (qt.nsplit > 1) {
    constexpr int PQF = 4 * DT * 16 * 64;  // floats per piece
    float* const part0 = a.part + (int64_t)(hq * 2 * a.split_cap + qt.trank * qt.nper) * PQF;
    {
      float* pq = part0 + (int64_t)qt.piece * PQF + wave * (DT * 16 * 64);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) st_agent(pq + (dt * 16 + e) * 64 + l, dqacc[dt][e]);
    }
    if (!split_arrive(a.cnt + hq * 2 * a.split_cap + qt.trank, qt.nsplit, reinterpret_cast<int*>(smem))) return;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      f32x16 sum = f32x16{};
      for (int pc = 0; pc < qt.nsplit; ++pc) {
        const float* pq = part0 + (int64_t)pc * PQF + wave * (DT * 16 * 64) + dt * 16 * 64;
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[e] += ld_agent(pq + e * 64 + l);
      }
      dqacc[dt] = sum;
    }
  }
  __syncthreads();  // every wave is done with the K / V tiles
  const int row = 32 * wave + i;
  bf16* const orow = smem + (row >> 6) * GT::ELEMS;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      E4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (EL)(dqacc[dt][4 * q4 + e] * a.scale);
      *reinterpret_cast<E4*>(orow + GT::off(row & 63, 4 * dt + q4) + 4 * g) = v;
    }
  __syncthreads();
  store_rows<SPARSE, true>(smem, a, qt, a.dq);
}

// ---------------------------------------------------------------------------
// dk / dv
// ---------------------------------------------------------------------------
// 64 keys per workgroup (half a kBKV tile): two pairs of waves, 32 keys each.
// dK and dV of 32 keys would take one wave's 256 AGPRs and leave it no room
// for K, V and the scores (that form spilled them), so a pair shares them:
//   wave A: S(t), P(t) -> LDS (fp32), dV += dO(t - 1)^T P(t - 1);  K in registers
//   wave B: dP(t), dS(t - 1) = P(t - 1) (dP(t - 1) - delta), dK += Q(t - 1)^T dS(t - 1);  V in registers
// with t the step of 32 query rows: 32 MFMAs each, every lane of B reading the
// P values that the same lane of A wrote.  q and dO rows pass through rings of
// four 32-row tiles: t - 1 and t in use, t + 1 landing, t + 2 issued in step t.
constexpr int kRing = 4, kTileElems = kHalf * D, kKeysWG = 64;
constexpr size_t kPBytes = (size_t)2 * 2 * 64 * 16 * sizeof(float);  // [parity][pair][item group][lane] x 4
constexpr size_t kDkvSmem = 2 * kRing * kTileElems * sizeof(bf16) + kPBytes + kRing * 3 * kHalf * sizeof(float);

template <typename EL, bool SPARSE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void w256_dkv_kernel(const AttnArgs a) {
  using E8 = typename Elem<EL>::x8;
  using E4 = typename Elem<EL>::x4;
  constexpr int RS = kHalf;
  bf16* const smem = dyn_smem();  // the q ring, then the dO ring
  char* const sP = logo_smem + 2 * kRing * kTileElems * sizeof(bf16);
  float* const sStat = reinterpret_cast<float*>(sP + kPBytes);  // ring of [lse][delta][pos]
  auto sQ = [&](int t) { return smem + (t & (kRing - 1)) * kTileElems; };
  auto sO = [&](int t) { return smem + (kRing + (t & (kRing - 1))) * kTileElems; };
  auto stat = [&](int t) { return sStat + (t & (kRing - 1)) * 3 * RS; };

  int rank, h;
  xcd_remap(blockIdx.x, a.h, rank, h);
  const int32_t* meta0 = a.meta;
  const int tile = rank >> 1;  // early key blocks (most queries) first
  if (tile >= meta0[2]) return;
  const int32_t* cu_tk = meta0 + kMetaHdr + 2 * (a.nseq + 1);
  const int s = seg_of(cu_tk, a.nseq, tile);
  const int k0 = (tile - cu_tk[s]) * kBKV + kKeysWG * (rank & 1);
  const int bos = a.cu[s];
  const int seqlen = a.cu[s + 1] - bos;
  if (k0 >= seqlen) return;
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, i = l & 31, g = l >> 5;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int pair = wave >> 1;
  const int kw0 = k0 + 32 * pair;
  const bool wave_active = kw0 < seqlen;
  const int kw_last = min(kw0 + 31, seqlen - 1);
  const int key = kw0 + i;
  const bool valid_k = key < seqlen;
  const float c = a.scale_log2;

  Reader rd;
  rd.init();
  auto first = [](int k) constexpr { return k < 2 ? 0 : k > 15 ? 16 : ((k - 2) * 16 + 13) / 14; };  // first item of slot k
  auto pbuf = [&](int par, int m) { return reinterpret_cast<f32x4*>(sP) + ((par * 2 + pair) * 4 + m) * 64 + l; };

  // One role's whole walk, up to its accumulators in LDS.  The roles are
  // separate code (with their own registers) that meets at the same barriers.
  auto walk = [&](auto role_tag) {
    constexpr bool ROLE_B = decltype(role_tag)::value;
    E8 kv[DS];  // A: K, B: V
    {
      const bf16* src = (ROLE_B ? a.v : a.k) + ((int64_t)(bos + min(key, seqlen - 1)) * a.h + h) * D + 8 * g;
  #pragma unroll
      for (int ds = 0; ds < DS; ++ds) kv[ds] = valid_k ? *reinterpret_cast<const E8*>(src + 16 * ds) : E8{};
    }
    f32x16 acc[DT];  // A: dV, B: dK (AGPRs)
  #pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
    f32x16 sd[2];  // A: S of step t in sd[0]; B: dP of steps t, t - 1 by parity
    E8 pb[2];      // A: P(t - 1) packed

    for (int gg = 0; gg < a.g; ++gg) {
      const int hq = h * a.g + gg;
      const int lane_sel = a.lanes > 1 ? hq : 0;
      const int32_t* cu_q = a.meta + (int64_t)lane_sel * a.meta_stride + kMetaHdr;
      const RowView<SPARSE> rv = row_view<SPARSE>(a, lane_sel, bos);
      const int q_lo = cu_q[s], rq_end = cu_q[s + 1];
      auto lb_pos = [&](int lo, int hi, int x) {
        return SPARSE ? wave_lower_bound(rv.ps, lo, hi, x) : min(max(q_lo + x, lo), hi);
      };
      const int rq0 = lb_pos(q_lo, rq_end, k0);
      if (rq0 >= rq_end) continue;  // (uniform) no row of this head sees these keys
      const int nt = (rq_end - rq0 + RS - 1) / RS;
      // steps before t_lo see none of this pair's keys, rows from lb1 on all of them
      int t_lo = nt, lb1 = rq_end;
      if (wave_active) {
        const int lb0 = lb_pos(rq0, rq_end, kw0);
        lb1 = lb_pos(lb0, rq_end, kw_last);
        t_lo = (lb0 - rq0) / RS;
      }
      const float* lse_h = a.lse + (int64_t)hq * a.n;
      const float* delta_h = a.delta + (int64_t)hq * a.n;
      // q and dO rows of head hq: 32-bit byte offsets from the head's first row
      // (the launcher checks that the tensors are below 4 GB)
      const int row_bytes = a.hq * D * 2;
      const auto rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a.q + (int64_t)hq * D), (short)0, -1,
                                                        kBufRsrcWord3);
      const auto ro = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a.dout + (int64_t)hq * D), (short)0, -1,
                                                        kBufRsrcWord3);
      // token of row i of step t, loaded a step ahead of the copy that uses it
      // (the low half of the index: as a 64-bit load, whose dead half's register
      // is used again, it had every step wait for its own copies: 42% of the
      // wave time was waiting, forward + backward took 876 us in place of 822 us
      // at T = 8192, 16 heads, a quarter of the rows)
      auto load_tok = [&](int t) {
        const int r = min(rq0 + RS * t + i, rq_end - 1);
        return SPARSE ? reinterpret_cast<const int*>(rv.qi)[2 * r] : r;
      };
      // a statistic of row i of step t: lse in wave 0, delta in wave 1, the
      // position in wave 2 (rows past the end repeat the last one, at position
      // -1: they see no key); one load on every path, for the count at the end
      // of the step
      const int* const stat_src = wave == 1                  ? reinterpret_cast<const int*>(delta_h)
                                  : (SPARSE && wave >= 2) ? reinterpret_cast<const int*>(rv.ps)
                                                          : reinterpret_cast<const int*>(lse_h);
      auto load_stat = [&](int t) { return stat_src[min(rq0 + RS * t + i, rq_end - 1)]; };
      auto store_stat = [&](int t, int v) {
        const int rr = rq0 + RS * t + i;
        if (wave == 2) v = rr >= rq_end ? -1 : SPARSE ? v : rv.posn(rr);
        if (wave < 3 && l < RS) reinterpret_cast<int*>(stat(t))[RS * wave + l] = v;
      };
      auto load_tile = [&](int t, int tok) {  // wave w copies rows 8 w .. 8 w + 7, two a load
  #pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int r = 8 * wave_s + 2 * k;
          const int t0 = __builtin_amdgcn_readlane(tok, r), t1 = __builtin_amdgcn_readlane(tok, r + 1);
          const uint32_t off = (uint32_t)(g ? t1 : t0) * (uint32_t)row_bytes + 16 * (uint32_t)(i ^ GT::swz(r + g));
          buf_load_lds16(rq, sQ(t) + r * D, off);
          buf_load_lds16(ro, sO(t) + r * D, off);
        }
      };

      // wave A's step: X: S(t); Y: dV(t - 1) with P(t)
      auto step_a = [&](auto par_tag, auto doy_tag, auto mask_tag, int t) {
        constexpr int PAR = decltype(par_tag)::value;
        constexpr bool DOY = decltype(doy_tag)::value, MASK = decltype(mask_tag)::value;
        constexpr int PF = 4;
        const bf16* qb = sQ(t);
        const bf16* ob = sO(t - 1);
        const float* st = stat(t);
        E8 op[2 * DS];
        E8 pn[2];
        f32x4 l4[4];
        int4 p4[4];
        auto load_op = [&](auto s_c) {
          constexpr int S = decltype(s_c)::value, K = S % DS;
          if constexpr (S < DS) {
            op[S] = rd.template row<EL>(qb, 0, K);
          } else {
            if constexpr (DOY) op[S] = rd.template tr<EL>(ob, 16 * (K / DT), K % DT);
          }
        };
        static_for<PF>([&](auto s_c) { load_op(s_c); });
        static_for<2 * DS>([&](auto s_c) {
          constexpr int S = decltype(s_c)::value, K = S % DS;
          constexpr int I0 = first(K), NI = first(K + 1) - I0;
          __builtin_amdgcn_sched_barrier(0);
          float sv[2];
          if constexpr (S >= DS)
            static_for<NI>([&](auto e_c) {
              constexpr int E = decltype(e_c)::value;
              sv[E] = sd[0][I0 + E];
              pin(sv[E]);
            });
          if constexpr (S < DS) {
            sd[0] = mfma32(op[S], kv[K], K == 0 ? f32x16{} : sd[0]);
          } else {
            if constexpr (DOY) mfma32_agpr_ready(acc[K % DT], op[S], pb[K / DT]);
          }
          if constexpr (S + PF < 2 * DS) load_op(std::integral_constant<int, S + PF>{});
          if constexpr (S >= 8 && S < 12) {  // item j of an accumulator is query row rowmap(g, j)
            l4[S - 8] = lds_load(reinterpret_cast<const f32x4*>(st + 8 * (S - 8) + 4 * g));
            if constexpr (MASK) p4[S - 8] = lds_load(reinterpret_cast<const int4*>(st + 2 * RS + 8 * (S - 8) + 4 * g));
          }
          if constexpr (S >= DS) {
            static_for<NI>([&](auto e_c) {
              constexpr int E = decltype(e_c)::value, JJ = I0 + E;
              float pv = fast_exp2(fmaf(sv[E], c, -l4[JJ / 4][JJ % 4]));
              if constexpr (MASK) {
                const int4 q4 = p4[JJ / 4];
                const int pq = JJ % 4 == 0 ? q4.x : JJ % 4 == 1 ? q4.y : JJ % 4 == 2 ? q4.z : q4.w;
                if (!(key <= pq)) pv = 0.f;
              }
              pin(pv);
              sd[0][JJ] = pv;
              // a group of four leaves for wave B, a group of eight is packed
              if constexpr (JJ % 4 == 3)
                *pbuf(PAR, JJ / 4) = f32x4{sd[0][JJ - 3], sd[0][JJ - 2], sd[0][JJ - 1], sd[0][JJ]};
              if constexpr (JJ % 8 == 7) pn[JJ / 8] = acc_to<EL>(sd[0], JJ / 8);
            });
          }
        });
        __builtin_amdgcn_sched_barrier(0);
        pb[0] = pn[0];
        pb[1] = pn[1];
      };
      // wave B's step: X: dP(t) with dS(t - 1); Y: dK(t - 1)
      auto step_b = [&](auto par_tag, auto doy_tag, int t) {
        constexpr int PAR = decltype(par_tag)::value;
        constexpr bool DOY = decltype(doy_tag)::value;
        constexpr int PF = 4;
        const bf16* ob = sO(t);
        const bf16* qb = sQ(t - 1);
        const float* st = stat(t - 1) + RS;
        E8 op[2 * DS];
        E8 db[2];
        f32x4 d4[4], p4[4];
        auto load_op = [&](auto s_c) {
          constexpr int S = decltype(s_c)::value, K = S % DS;
          if constexpr (S < DS) {
            op[S] = rd.template row<EL>(ob, 0, K);
          } else {
            if constexpr (DOY) op[S] = rd.template tr<EL>(qb, 16 * (K / DT), K % DT);
          }
        };
        static_for<PF>([&](auto s_c) { load_op(s_c); });
        if constexpr (DOY) {
  #pragma unroll
          for (int m = 0; m < 4; ++m) {
            p4[m] = lds_load(pbuf(PAR ^ 1, m));
            d4[m] = lds_load(reinterpret_cast<const f32x4*>(st + 8 * m + 4 * g));
          }
        }
        static_for<2 * DS>([&](auto s_c) {
          constexpr int S = decltype(s_c)::value, K = S % DS;
          constexpr int I0 = first(K), NI = first(K + 1) - I0;
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (S < DS) {
            sd[PAR] = mfma32(op[S], kv[K], K == 0 ? f32x16{} : sd[PAR]);
          } else {
            if constexpr (DOY) mfma32_agpr_ready(acc[K % DT], op[S], db[K / DT]);
          }
          if constexpr (S + PF < 2 * DS) load_op(std::integral_constant<int, S + PF>{});
          if constexpr (DOY && S < DS)
            static_for<NI>([&](auto e_c) {
              constexpr int JJ = I0 + decltype(e_c)::value;
              float dsv = p4[JJ / 4][JJ % 4] * (sd[PAR ^ 1][JJ] - d4[JJ / 4][JJ % 4]);
              pin(dsv);
              sd[PAR ^ 1][JJ] = dsv;
              if constexpr (JJ % 8 == 7) {
                db[JJ / 8] = acc_to<EL>(sd[PAR ^ 1], JJ / 8);
                pin(db[JJ / 8]);
              }
            });
        });
        __builtin_amdgcn_sched_barrier(0);
      };
      {
        const int tok0 = load_tok(0), tok1 = load_tok(1), st0 = load_stat(0), st1 = load_stat(1);
        load_tile(0, tok0);
        load_tile(1, tok1);
        store_stat(0, st0);
        store_stat(1, st1);
      }
      int tok[2] = {load_tok(2), load_tok(3)}, stn[2] = {0, load_stat(2)};
      step_end(false);
      // landed here: pending at the loop's entry, each turn would wait for all
      asm volatile("" : "+v"(tok[0]), "+v"(tok[1]), "+v"(stn[1]));
      using T_ = std::true_type;
      using F_ = std::false_type;
      // step t; the last (t = nt) finishes step nt - 1 (what it forms of step nt
      // comes from old tiles and is never used)
      // Step t copies the rows of step t + 2 and loads the statistics of t + 3 and
      // the tokens of t + 4 (past the end: of the last row, into free slots), so
      // that a step waits for nothing that it issued itself: at its end the copies
      // of step t - 1 have landed, behind which 12 operations were issued (10
      // without token indices to load).
      auto step = [&](auto par_tag, int t) {
        constexpr int PAR = decltype(par_tag)::value;
        asm volatile("" ::: "memory");
        load_tile(t + 2, tok[PAR]);
        asm volatile("" ::: "memory");
        stn[PAR] = load_stat(t + 3);
        tok[PAR] = load_tok(t + 4);
        asm volatile("" ::: "memory");
        const bool dox = t >= t_lo && t < nt, doy = t - 1 >= t_lo && t >= 1 && t <= nt;
        if constexpr (!ROLE_B) {
          const bool mask = rq0 + RS * t < lb1 || rq0 + RS * (t + 1) > rq_end;
          if (doy) {
            if (mask) step_a(par_tag, T_{}, T_{}, t);
            else step_a(par_tag, T_{}, F_{}, t);
          } else if (dox) {
            step_a(par_tag, F_{}, T_{}, t);
          }
        } else {
          if (doy) step_b(par_tag, T_{}, t);
          else if (dox) step_b(par_tag, F_{}, t);
        }
        store_stat(t + 2, stn[PAR ^ 1]);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(SPARSE ? 12 : 10) : "memory");
      };
      for (int t = 0; t <= nt; t += 2) {
        step(BufTag<0>{}, t);
        step(BufTag<1>{}, t + 1);  // (may be past the last: on every path, for the waits' counts)
        agpr_acc_drain();  // the accumulators may be read next
      }
    }
    step_end(false);
    {
      bf16* const blk = smem + (ROLE_B ? GT::ELEMS : 0);
      const int row = 32 * pair + i;
      const float mul = ROLE_B ? a.scale : 1.f;
  #pragma unroll
      for (int dt = 0; dt < DT; ++dt)
  #pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          E4 v;
  #pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (EL)(acc[dt][4 * q4 + e] * mul);
          *reinterpret_cast<E4*>(blk + GT::off(row, 4 * dt + q4) + 4 * g) = v;
        }
    }
  };
  if (wave_s & 1) walk(std::true_type{});
  else walk(std::false_type{});
  __syncthreads();
  // dV (waves A) and dK (waves B) leave as whole rows through LDS
  {
    const int ch = tid & 31, nkey = min(kKeysWG, seqlen - k0);
    for (int r = tid >> 5; r < nkey; r += 8) {
      const int64_t off = ((int64_t)(bos + k0 + r) * a.h + h) * D + 8 * ch;
      st_nt(reinterpret_cast<u32x4*>(a.dv + off), *reinterpret_cast<const u32x4*>(smem + GT::off(r, ch)));
      st_nt(reinterpret_cast<u32x4*>(a.dk + off), *reinterpret_cast<const u32x4*>(smem + GT::ELEMS + GT::off(r, ch)));
    }
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
constexpr size_t kRowSmem = (size_t)4 * GT::ELEMS * sizeof(bf16);

template <typename EL, bool SPARSE>
int launch_rows(const AttnArgs& a_in, hipStream_t st, bool bwd) {
  AttnArgs a = a_in;
  split_setup(a, 1, bwd ? dq_part_floats(D) : fwd_part_floats(D, 4));
  // A piece starts with the loads of its rows and leaves 133 KB of partials: about
  // the time of 400 keys.  Time over the generic kernels', forward and backward of
  // 500 to 8192 tokens in one and six segments, 4 to 32 heads, 5 to 60 % of the rows:
  // 0.622x with at least 320 keys (256: 0.623x; 448, and 1024 where the pieces take
  // turns on the CUs: 0.633x); 0.655x without a least size, up to 1.34x.
  a.split_keys = LOGO_WIDE_SPLIT_KEYS;
  a.round_rows /= 2;  // one 128-row workgroup per CU in a round
  const int64_t nblk = std::max<int64_t>((a.n + kBQ - 1) / kBQ + a.nseq, 2 * a.split_cap) * a.hq;
  LOGO_REQUIRE(nblk < ((int64_t)1 << 31), "grid too large");
  auto kern = bwd ? w256_dq_kernel<EL, SPARSE> : w256_fwd_kernel<EL, SPARSE>;
  LOGO_HIP_CHECK(allow_smem(kern, kRowSmem));
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), kRowSmem, st, a);
  LOGO_LAUNCH_CHECK("w256 forward / dq kernel");
  return LOGO_OK;
}

template <typename EL, bool SPARSE>
int launch(const AttnArgs& a, hipStream_t st, int phase) {
  if (phase == kPhaseFwd || phase == kPhaseDq) return launch_rows<EL, SPARSE>(a, st, phase == kPhaseDq);
  if (phase == kPhaseDelta) {
    hipLaunchKernelGGL((w256_delta_kernel<EL, SPARSE>), dim3((unsigned)((a.n + 15) / 16), a.hq), dim3(256), 0, st, a);
    LOGO_LAUNCH_CHECK("w256_delta_kernel");
    return LOGO_OK;
  }
  const int64_t nblk = 2 * ((a.n + kBKV - 1) / kBKV + a.nseq) * a.h;  // two workgroups per 128-key tile
  LOGO_REQUIRE(nblk < ((int64_t)1 << 31), "grid too large");
  auto kern = w256_dkv_kernel<EL, SPARSE>;
  LOGO_HIP_CHECK(allow_smem(kern, kDkvSmem));
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), kDkvSmem, st, a);
  LOGO_LAUNCH_CHECK("w256_dkv_kernel");
  return LOGO_OK;
}

}  // namespace wide

bool wide_applies(const AttnArgs& a, int d, int dtype) {
  return d == wide::D && dtype != LOGO_DTYPE_F32 && a.window < 0 &&
         a.n * a.hq * wide::D * (int64_t)sizeof(bf16) < ((int64_t)1 << 32);
}

size_t wide_workspace_bytes(int hq) {
  const int cap = split_cap_for(hq, 1);
  if (cap < 2) return 0;
  return 2 * split_cnt_bytes() +
         (size_t)hq * 2 * cap * std::max(fwd_part_floats(wide::D, 4), dq_part_floats(wide::D)) * sizeof(float);
}

int wide_launch(const AttnArgs& a, hipStream_t st, int phase, bool sparse, bool half) {
  if (half) return wide::launch<f16, true>(a, st, phase);
  return sparse ? wide::launch<bf16, true>(a, st, phase) : wide::launch<bf16, false>(a, st, phase);
}

}  // namespace logo
