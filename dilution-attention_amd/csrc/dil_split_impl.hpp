// The forward's passes with split walks (dil_walk.hpp): statistics, demand and
// output of one 32-row or 32-key tile per workgroup.
#pragma once

#include "dil_walk.hpp"

namespace dil {

namespace {

// ---------------------------------------------------------------------------
// row statistics (+ pk)

template <typename CT, int D, bool PK>
__global__ __launch_bounds__(kThreads, 1) void fwd_stats_split(FwdParams P) {
  __shared__ float m_s[kSplitWaves][kTileQ], mx_s[kSplitWaves][kTileQ], l_s[kSplitWaves][kTileQ];
  __shared__ __attribute__((aligned(16))) floatx4 pk_s[PK ? kSplitWaves : 1][PK ? 4 * kDTiles<D> : 1][64];
  // late (long) row tiles first
  const WorkItem item = xcd_work_item(P.groups, P.n, true, true, true);
  if (!item.valid) return;
  const int64_t slice = item.slice;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const int r0 = item.idx * kTileQ, C = static_cast<int>(P.C), Tk = static_cast<int>(P.Tk);
  const int qa0 = static_cast<int>(P.q0) + r0;
  const int kend = min(qa0 + kTileQ - 1, static_cast<int>(P.q0) + C - 1) / kTileK + 1;
  const int kfull = (qa0 + 1) / kTileK;            // tiles below need no mask
  const CT* qs = static_cast<const CT*>(P.q) + P.qv.slice(slice);
  const CT* ks = static_cast<const CT*>(P.k) + P.kv.slice(slice);
  const CT* kts = PK ? static_cast<const CT*>(P.kt) + slice * P.t_sn : nullptr;
  RowFrag<CT, D> qf;
  const bool row_ok = r0 + l32 < C;
  global_row_frag<CT, D>(qf, qs, r0 + l32, C - 1, P.qv.sr, h);
  const int my_q = qa0 + l32;
  float m = -INFINITY, mx = -INFINITY, l0 = 0.f, l1 = 0.f;
  floatx16 pka[PK ? kDTiles<D> : 1];
#pragma unroll
  for (int t = 0; t < (PK ? kDTiles<D> : 1); ++t) pka[t] = floatx16{};
  const float thresh = kLazyMax / P.c;

  using F = WalkFrags<CT, D, PK>;
  auto load = [&](F& f, int kt) {
    global_row_frag<CT, D>(f.row, ks, kt * kTileK + rho(l32), Tk - 1, P.kv.sr, h);
    if constexpr (PK) {
#pragma unroll
      for (int t = 0; t < kDTiles<D>; ++t)
        global_t_frags<CT, D, false>(f.t[t], kts + static_cast<int64_t>(kt) * kTileK * D, 32 * t + l32, h);
    }
  };
  auto step = [&](const F& f, int kt) {
    const floatx16 acc = mma_rows<CT, D>(f.row, qf, floatx16{});
    float a[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = acc[i];
    if (kt >= kfull) {
      const int dq = kt * kTileK + 8 * h - my_q;       // key - query for register i: perm_row(i, 0) + dq
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (16 * (i >> 3) + (i & 7) + dq > 0) a[i] = -INFINITY;
    }
    float tmax = fmaxf(fmaxf(a[0], a[1]), a[2]);
#pragma unroll
    for (int i = 3; i < 15; i += 2) tmax = fmaxf(fmaxf(tmax, a[i]), a[i + 1]);
    tmax = fmaxf(tmax, a[15]);
    const HalfPair tp = halves(tmax);                  // one running max per query (both halves)
    tmax = fmaxf(tp.lo, tp.hi);
    mx = fmaxf(mx, tmax);
    // a masked tile can hold no key of a query (then tmax is -inf and m stays)
    const bool take = tmax > m + thresh || (m == -INFINITY && tmax > -INFINITY);
    if (__any(take)) {
      const float mnew = take ? tmax : m;
      const float alpha = take ? (m == -INFINITY ? 0.f : fast_exp2((m - mnew) * P.c)) : 1.f;
      l0 *= alpha;
      l1 *= alpha;
      if constexpr (PK) {
#pragma unroll
        for (int t = 0; t < kDTiles<D>; ++t) pka[t] *= alpha;
      }
      m = mnew;
    }
    const float mc = m == -INFINITY ? 0.f : m * P.c;
    float e[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) e[i] = fast_exp2(fmaf(a[i], P.c, -mc));
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      l0 += e[i];
      l1 += e[i + 1];
    }
    if constexpr (PK) {
#pragma unroll
      for (int s = 0; s < kSlots<CT>; ++s) {
        const auto bfr = acc_frag<CT>(e, s);
#pragma unroll
        for (int t = 0; t < kDTiles<D>; ++t) pka[t] = Mma<CT>::mma(f.t[t][s], bfr, pka[t]);
      }
    }
  };
  walk_tiles<kWalkAhead<CT, D>, F>(wave, kend, load, step);

  const HalfPair lp = halves(l0 + l1);                 // the halves share m
  if (h == 0) {
    m_s[wave][l32] = m;
    mx_s[wave][l32] = mx;
    l_s[wave][l32] = lp.lo + lp.hi;
  }
  if constexpr (PK) {
#pragma unroll
    for (int t = 0; t < kDTiles<D>; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        pk_s[wave][4 * t + j][lane] = floatx4{pka[t][4 * j], pka[t][4 * j + 1], pka[t][4 * j + 2], pka[t][4 * j + 3]};
  }
  __syncthreads();
  // the waves' sums against the largest offset (a wave without keys has none)
  float M = m_s[0][l32], mxt = mx_s[0][l32], f[kSplitWaves], l = 0.f;
#pragma unroll
  for (int w = 1; w < kSplitWaves; ++w) {
    M = fmaxf(M, m_s[w][l32]);
    mxt = fmaxf(mxt, mx_s[w][l32]);
  }
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) {
    const float mw = m_s[w][l32];
    f[w] = mw == -INFINITY ? 0.f : fast_exp2((mw - M) * P.c);
    l = fmaf(l_s[w][l32], f[w], l);
  }
  if (wave == 0 && h == 0 && row_ok) {
    // re-referenced to the exact row maximum: p = 2^(a c - rmax) / rden
    P.rmax[slice * P.C + r0 + l32] = mxt * P.c;
    P.rden[slice * P.C + r0 + l32] = l * fast_exp2((M - mxt) * P.c);
  }
  if constexpr (PK) {
    if (row_ok) {
      const float pf = P.scale / l;
      float* dst = P.pk + (slice * P.C + r0 + l32) * D;
#pragma unroll
      for (int c = 0; c < kDTiles<D>; ++c) {
        const int q = wave + kSplitWaves * c;          // chunk: head dims 32 (q / 4) + 8 (q % 4) + 4 h + [0, 4)
        floatx4 v = pk_s[0][q][lane] * f[0];
#pragma unroll
        for (int w = 1; w < kSplitWaves; ++w) v += pk_s[w][q][lane] * f[w];
        const int d = 32 * (q >> 2) + 8 * (q & 3) + 4 * h;
        if (d < D) *reinterpret_cast<floatx4*>(dst + d) = v * pf;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// demand checkpoints and totals: one workgroup per 32 keys, a quarter of the
// row blocks per wave

constexpr int kSplitDemandBlocks = 256;                // row blocks a workgroup keeps the sums of (32 KB)

// Whether a chunk that starts past row 0 splits its demand walks.  The pass has a
// workgroup per 32 keys, of which a chunk has more than row tiles (split_walks
// counts those), each with a shorter walk: up to 3 blocks are one step per wave
// and nothing is won.  fwd_demand, us, split / whole (key tiles x row blocks):
//   bf16 64:  260x10 8.2 / 10.3, 656x10 11.3 / 11.6, 832x4 8.1 / 7.1, 2160x10 20 / 14, 16256x4 58 / 27
//   bf16 32:  1040x10 8.6 / 11.3, 2624x10 15.4 / 16.1, 4160x10 20 / 16, 4304x19 27.2 / 27.4, 4032x32 30 / 35
//   bf16 128: 269x19 15 / 17, 540x10 15 / 12, 1008x32 36 / 26
//   fp32 64:  516x4 11.0 / 11.6, 656x10 22 / 22, 1016x4 16 / 12;  fp32 128: 269x19 36 / 52, 540x10 34 / 31
//   split 64: 269x19 15 / 19, 540x10 15 / 13, 1008x32 36 / 28;  split 128: 260x10 16 / 16, 540x10 24 / 17
template <typename CT, int D>
inline bool split_demand_tiles(int64_t n, int64_t blocks, int64_t Tk) {
  constexpr bool kNarrow = std::is_same_v<CT, __bf16> && D <= 32;      // the longer walks pay for more key tiles
  constexpr int64_t kTiles = std::is_same_v<CT, float>     ? (D <= 64 ? 640 : 512)
                             : std::is_same_v<CT, split32> ? (D <= 32 ? 512 : 320)
                                                           : (D <= 32 ? 2048 : D <= 64 ? 640 : 384);
  const int64_t limit = kNarrow && blocks >= 16 ? 2 * kTiles : kTiles;
  return blocks > 3 && n * ((Tk + kTileK - 1) / kTileK) <= limit;
}

template <typename CT, int D>
__global__ __launch_bounds__(kThreads, 1) void fwd_demand_split(FwdParams P) {
  extern __shared__ float csum_s[];                    // [row block][32 keys]: column sums of p
  __shared__ double tot_s[kSplitWaves][kTileK];
  __shared__ __attribute__((aligned(16))) float st_s[kSplitWaves][2][kTileQ];
  const WorkItem item = xcd_work_item(P.kgroups, P.n, false, true, true);   // early keys (long walks) first
  if (!item.valid) return;
  const int64_t slice = item.slice;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const int C = static_cast<int>(P.C), q0 = static_cast<int>(P.q0), Tk = static_cast<int>(P.Tk), nb = static_cast<int>(P.nb);
  const int key0 = item.idx * kTileK, key = key0 + l32;
  const bool key_ok = key < Tk;
  // first block whose last row reaches the first key; the blocks in quarters
  const int t = key0 - q0 - (kTileQ - 1);
  const int b0 = t > 0 ? (t + kTileQ - 1) / kTileQ : 0;
  const int per = (max(nb - b0, 0) + kSplitWaves - 1) / kSplitWaves;
  const int b_lo = min(b0 + wave * per, nb), b_hi = min(b_lo + per, nb);
  const CT* qs = static_cast<const CT*>(P.q) + P.qv.slice(slice);
  const float* rmax = P.rmax + slice * P.C;
  const float* rden = P.rden + slice * P.C;
  RowFrag<CT, D> kf;
  global_row_frag<CT, D>(kf, static_cast<const CT*>(P.k) + P.kv.slice(slice), key, Tk - 1, P.kv.sr, h);
  // the carried demand, read by all 4 waves before the barrier: total may be the
  // same memory (a prefill chunk advances its demand in place), and the last wave
  // stores it after the barrier, whatever the other waves have reached
  const float demand0 = (P.demand_in != nullptr && key < q0 && key_ok) ? P.demand_in[slice * P.din_sn + key] : 0.f;
  struct F {
    RowFrag<CT, D> row;
    float lse;
  };
  auto load = [&](F& f, int b) {
    const int r = b * kTileQ + l32;
    global_row_frag<CT, D>(f.row, qs, r, C - 1, P.qv.sr, h);
    f.lse = r < C ? rmax[r] + __log2f(rden[r]) : INFINITY;
  };
  double run = 0.0;
  int buf = 0;
  auto step = [&](const F& f, int b) {
    st_s[wave][buf][l32] = f.lse;                      // within the wave: no barrier
    const floatx16 acc = mma_rows<CT, D>(f.row, kf, floatx16{});   // register i <-> row acc_row(i, h)
    float p[16];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const floatx4 r = *reinterpret_cast<const floatx4*>(&st_s[wave][buf][8 * u + 4 * h]);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * u + e] = fast_exp2(fmaf(acc[4 * u + e], P.c, -r[e]));
    }
    buf ^= 1;
    if (key0 + kTileK - 1 > q0 + b * kTileQ) {
      const int dq = key - q0 - b * kTileQ - 4 * h;    // key - row for register i: dq - (8 (i >> 2) + (i & 3))
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (dq > 8 * (i >> 2) + (i & 3)) p[i] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] += p[i + 8];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] += p[i + 4];
    const HalfPair cp = halves((p[0] + p[1]) + (p[2] + p[3]));
    const float s = cp.lo + cp.hi;
    if (h == 0) csum_s[(b - b0) * kTileK + l32] = s;
    run += static_cast<double>(s);
  };
  {
    // the wave's blocks one after the other, the next one's operands a step ahead
    F f[2];
    if (b_lo < b_hi) load(f[0], b_lo);
    for (int b = b_lo; b < b_hi; b += 2) {
      if (b + 1 < b_hi) load(f[1], b + 1);
      step(f[0], b);
      if (b + 1 < b_hi) {
        if (b + 2 < b_hi) load(f[0], b + 2);
        step(f[1], b + 1);
      }
    }
  }
  if (h == 0) tot_s[wave][l32] = run;
  __syncthreads();
  // demand entering the wave's first block: the carried demand and the earlier quarters
  double at = static_cast<double>(demand0);
  for (int w = 0; w < wave; ++w) at += tot_s[w][l32];
  if (key_ok && h == 0) {
    float* ccol = P.carry + slice * P.nb * P.Tk + key;
    for (int b = b_lo; b < b_hi; ++b) {
      ccol[static_cast<int64_t>(b) * P.Tk] = static_cast<float>(at);
      at += static_cast<double>(csum_s[(b - b0) * kTileK + l32]);
    }
    if (wave == kSplitWaves - 1) P.total[slice * P.tot_sn + key] = static_cast<float>(at);
  }
}

// ---------------------------------------------------------------------------
// output pass

template <typename CT, int D>
__global__ __launch_bounds__(kThreads, 1) void fwd_out_split(FwdParams P) {
  __shared__ __attribute__((aligned(16))) float lse_s[kTileQ];
  __shared__ float ssum_s[kSplitWaves][kTileQ];
  __shared__ __attribute__((aligned(16))) floatx4 o_s[kSplitWaves][4 * kDTiles<D>][64];
  const WorkItem item = xcd_work_item(P.groups, P.n, true, true, true);
  if (!item.valid) return;
  const int64_t slice = item.slice;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const float hf = static_cast<float>(h);
  const int r0 = item.idx * kTileQ, C = static_cast<int>(P.C), Tk = static_cast<int>(P.Tk);
  const int qa0 = static_cast<int>(P.q0) + r0;
  const int kend = min(qa0 + kTileQ - 1, static_cast<int>(P.q0) + C - 1) / kTileK + 1;
  const int kfull = (qa0 + 1) / kTileK;
  const CT* qs = static_cast<const CT*>(P.q) + P.qv.slice(slice);
  const CT* ks = static_cast<const CT*>(P.k) + P.kv.slice(slice);
  const CT* vts = static_cast<const CT*>(P.vt) + slice * P.t_sn;
  const float* c_row = P.carry + (slice * P.nb + item.idx) * P.Tk;
  RowFrag<CT, D> qf;                                   // QS order: register i of half h <-> row 16 h + i
  global_row_frag<CT, D>(qf, qs, r0 + qsig(l32), C - 1, P.qv.sr, h);
  if (threadIdx.x < kTileQ) {
    const int r = r0 + threadIdx.x;
    lse_s[threadIdx.x] = r < C ? P.rmax[slice * P.C + r] + __log2f(P.rden[slice * P.C + r]) : INFINITY;
  }
  typename Mma<CT>::frag ident[kSlots<CT>];
#pragma unroll
  for (int s = 0; s < kSlots<CT>; ++s) ident[s] = ident_qs<CT>(l32, h, s);
  floatx16 o[kDTiles<D>];
#pragma unroll
  for (int t = 0; t < kDTiles<D>; ++t) o[t] = floatx16{};
  float rsum = 0.f;
  __syncthreads();

  struct F {
    WalkFrags<CT, D, true> w;
    float cin;
  };
  auto load = [&](F& f, int kt) {
    const int key = kt * kTileK + rho(l32);
    global_row_frag<CT, D>(f.w.row, ks, key, Tk - 1, P.kv.sr, h);
    f.cin = key < Tk ? c_row[key] : 0.f;
#pragma unroll
    for (int t = 0; t < kDTiles<D>; ++t)
      global_t_frags<CT, D, false>(f.w.t[t], vts + static_cast<int64_t>(kt) * kTileK * D, 32 * t + l32, h);
  };
  auto step = [&](const F& f, int kt) {
    const floatx16 acc = mma_rows<CT, D>(qf, f.w.row, floatx16{});
    float lse[16], p[16], x[16];
    lds_read16(lse_s + 16 * h, lse);
#pragma unroll
    for (int i = 0; i < 16; ++i) p[i] = fast_exp2(fmaf(acc[i], P.c, -lse[i]));
    if (kt >= kfull) {
      const int dk = kt * kTileK + rho(l32) - qa0 - 16 * h;   // key - query(i) = dk - i
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (dk > i) p[i] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = p[i];
    scan_incl_qs(x, f.cin + kEps, hf);                        // demand + p + eps
#pragma unroll
    for (int i = 0; i < 16; ++i) p[i] *= fast_rcp(x[i]);      // share
    // transposed: queries in lanes, keys (natural order) in registers
    floatx16 xt = floatx16{};
#pragma unroll
    for (int s = 0; s < kSlots<CT>; ++s) xt = Mma<CT>::mma_bexact(acc_frag<CT>(p, s), ident[s], xt);
    float xv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) xv[i] = xt[i];
#pragma unroll
    for (int s = 0; s < kSlots<CT>; ++s) {
      const auto af = acc_frag<CT>(xv, s);
#pragma unroll
      for (int t = 0; t < kDTiles<D>; ++t) o[t] = Mma<CT>::mma(af, f.w.t[t][s], o[t]);
    }
    rsum += sum16(xv);
  };
  walk_tiles<kWalkAhead<CT, D>, F>(wave, kend, load, step);

  const HalfPair rp = halves(rsum);
  if (h == 0) ssum_s[wave][l32] = rp.lo + rp.hi;
#pragma unroll
  for (int t = 0; t < kDTiles<D>; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o_s[wave][4 * t + j][lane] = floatx4{o[t][4 * j], o[t][4 * j + 1], o[t][4 * j + 2], o[t][4 * j + 3]};
  __syncthreads();
  auto sum_of = [&](int row) { return (ssum_s[0][row] + ssum_s[1][row]) + (ssum_s[2][row] + ssum_s[3][row]); };
  if (threadIdx.x < kTileQ && r0 + threadIdx.x < C) P.ssum[slice * P.C + r0 + threadIdx.x] = sum_of(threadIdx.x);
  const int64_t out0 = P.ov.slice(slice) + r0 * P.ov.sr + l32;
#pragma unroll
  for (int c = 0; c < kDTiles<D>; ++c) {
    const int q = wave + kSplitWaves * c;              // chunk: head dim 32 (q / 4) + l32, rows 8 (q % 4) + 4 h + [0, 4)
    const floatx4 v = (o_s[0][q][lane] + o_s[1][q][lane]) + (o_s[2][q][lane] + o_s[3][q][lane]);
    if (32 * (q >> 2) + l32 < D) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 8 * (q & 3) + 4 * h + e;
        if (r0 + row < C)
          store_as(P.out, out0 + row * P.ov.sr + 32 * (q >> 2), P.odt, v[e] * (1.f / (sum_of(row) + kEps)));
      }
    }
  }
}

}  // namespace
}  // namespace dil
