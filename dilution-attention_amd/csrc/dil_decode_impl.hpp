// Cached decode step: one new query row per (batch, head) slice against
// `length` cached keys, with the per-key fp32 demand vector advanced in place.
//
// Reference behaviour: /root/reference/src/dilution/kernels.py:937-991
// (_dilution_decode) and :994-1038 (dilution_decode_step).  The reference runs
// one program per slice; here the keys are split into chunks so the grid fills
// 256 CUs, in three launches:
//
//   dec_stats  (chunks x n): a_j = q.k_j * scale*log2e -> fp32 scratch AFF,
//                            chunk-local (max, sum 2^(a-max))
//   dec_apply  (chunks x n): combine the chunk statistics -> lse; for every key
//                            p = 2^(a-lse), share = p / (committed + p + eps),
//                            chunk partials sum(share), sum(share * v);
//                            committed += p stored in place
//   dec_finish (n):          out = sum(share * v) / (sum(share) + eps) in the
//                            query dtype
//
// and slices of short contexts in one (dec_one).
//
// q1 is read in its own dtype and the output stored in it, whatever the
// caches' dtype (the reference loads q1 as fp32 and stores into q1.dtype,
// kernels.py:953, 1029).
//
// HBM bytes per key: K and V rows (2*D*elt) + demand read+write (8) + AFF
// write+read (8).  K and V are streamed once with 16-byte non-temporal loads.
#pragma once

#include "dil_common.hpp"
#include "dil_internal.hpp"
#include "dil_variant.hpp"

namespace dil {

namespace {

// Measured on MI355X at 128K context, B16 H16 d64 bf16 (sweep over 128-1024
// threads, 1-4 rows in flight, 512-8192-key chunks): 1024-thread workgroups
// over 2048-key chunks stream fastest.  With the affinities and shares of a chunk
// in LDS (one key per thread: one exponential a key instead of one a lane, and
// full-line stores of the affinities and the demand) the step takes 1450 us
// where it took 1510, 6.1 TB/s; 64 bytes of rows in flight per lane.
constexpr int kDecThreads = 1024;
constexpr int kDecWaves = kDecThreads / 64;
template <int DT> constexpr int kDecUnroll = DT == DT_F32 ? 2 : 4;   // cached rows in flight per lane (64 bytes)

// Keys per workgroup.  At most 2048 (the sweep above), and as many chunks as
// fill whole rounds of the workgroups the GPU holds at once (two 1024-thread
// workgroups per CU, 256 CUs): a partial last round streams at a fraction of
// HBM speed, and a small batch x context would leave CUs idle.  At least 256
// keys.  The rule is computed alike on the host and, for a length held in
// device memory, by the kernels, so both give the same chunks (and the same
// bits) at the same live length.  kDecResident is MI355X's figure (256 CUs x
// 2 workgroups); on a part with another CU count the rule still gives correct
// results, only the last round may then be partly filled.
constexpr int64_t kDecResident = 512;
constexpr int64_t kDecMaxChunk = 2048;
constexpr int64_t kDecMinChunk = 256;

// The chunk count that fills whole rounds: never below the 2048-key count,
// and non-decreasing in `length`.
__host__ __device__ inline int64_t decode_target_chunks(int64_t n, int64_t length) {
  const int64_t base = (length + kDecMaxChunk - 1) / kDecMaxChunk;     // chunks at the largest size
  const int64_t rounds = (n * base + kDecResident - 1) / kDecResident;
  const int64_t target = rounds * kDecResident / n;
  return target < base ? base : target;
}

__host__ __device__ inline int64_t decode_chunk(int64_t n, int64_t length) {
  if (length < 1 || n < 1) return kDecMinChunk;
  const int64_t target = decode_target_chunks(n, length);
  const int64_t chunk = (length + target - 1) / target;
  return chunk < kDecMinChunk ? kDecMinChunk : chunk;
}

// Chunks per slice in the grid and the scratch: exact for a host length; for
// a device-resident live length up to `length`, the largest count of any live
// length.  A live length L <= length has at most target(L) <= target(length)
// chunks (the target does not decrease with the length), and at most one per
// 256 keys.
inline int64_t decode_chunks(int64_t n, int64_t length, bool device_length) {
  if (length < 1) return 1;
  if (!device_length) {
    const int64_t chunk = decode_chunk(n, length);
    return (length + chunk - 1) / chunk;
  }
  const int64_t per_min = (length + kDecMinChunk - 1) / kDecMinChunk;
  const int64_t target = decode_target_chunks(n < 1 ? 1 : n, length);
  return per_min < target ? per_min : target;
}

template <int D>
struct DecLayout {
  static constexpr int kLanesPerRow = D / 8;          // each lane owns 8 consecutive d
  static constexpr int kRowsPerWave = 64 / kLanesPerRow;
  static constexpr int kRowsPerBlock = kRowsPerWave * kDecWaves;
};

// Sum over the kLanesPerRow lanes that share one cached row, with DPP lane
// moves within a 16-lane row (no LDS traffic) and, for 32 lanes, one lane
// shuffle across two rows.  The full sum is guaranteed only in the first lane
// of each row group (lane % LPR == 0), the only lane that consumes it.
template <int LPR>
__device__ __forceinline__ float row_reduce(float x) {
  constexpr int kQuadXor1 = 0xB1;      // quad_perm [1, 0, 3, 2]
  constexpr int kQuadXor2 = 0x4E;      // quad_perm [2, 3, 0, 1]
  constexpr int kRowShl4 = 0x104;      // row_shl:4
  constexpr int kRowShl8 = 0x108;      // row_shl:8
  if constexpr (LPR >= 2)
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), kQuadXor1, 0xF, 0xF, true));
  if constexpr (LPR >= 4)
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), kQuadXor2, 0xF, 0xF, true));
  if constexpr (LPR >= 8)
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), kRowShl4, 0xF, 0xF, true));
  if constexpr (LPR >= 16)
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), kRowShl8, 0xF, 0xF, true));
  if constexpr (LPR >= 32) x += __shfl_down(x, 16, 64);   // across the two 16-lane DPP rows (head_dim 256)
  return x;
}

// 8 cached elements as loaded: converted where they are used, so that a deep
// unroll holds 4 registers a row for 16-bit caches
template <int DT> using DecRaw = std::conditional_t<DT == DT_F32, floatx8, u16x8>;
template <int DT>
__device__ __forceinline__ DecRaw<DT> load_raw_stream(const void* base, int64_t idx) {
  if constexpr (DT == DT_F32) {
    const floatx4* p = reinterpret_cast<const floatx4*>(static_cast<const float*>(base) + idx);
    const floatx4 a = __builtin_nontemporal_load(p), b = __builtin_nontemporal_load(p + 1);
    return floatx8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  } else {
    return __builtin_nontemporal_load(reinterpret_cast<const u16x8*>(static_cast<const uint16_t*>(base) + idx));
  }
}
template <int DT>
__device__ __forceinline__ float raw_at(const DecRaw<DT>& r, int e) {
  if constexpr (DT == DT_F32) return r[e];
  else return DT == DT_BF16 ? bf16_bits_to_f32(r[e]) : f16_bits_to_f32(r[e]);
}

// The workgroup's walk over `count` rows from element `base` on (this lane's 8
// elements of row 0): load() takes the first rows, ahead of what they wait for,
// and walk() hands every row to f(row, elements); rows past the end are read as
// the last one (a test around each load made the loads wait for one another:
// 9.6 us to 13 for 16 slices of 1000 keys).  Two rows a lane are enough for a
// 256-key chunk at head_dim 64.
template <int D, int DT>
struct RowStream {
  static constexpr int U = kDecUnroll<DT>, kRows = DecLayout<D>::kRowsPerBlock;
  const void* src;
  int64_t base;
  int first, count;
  DecRaw<DT> r[U];
  __device__ __forceinline__ RowStream(const void* s, int64_t b, int wave, int lane, int n)
      : src(s), base(b), first(wave * DecLayout<D>::kRowsPerWave + lane / DecLayout<D>::kLanesPerRow), count(n) {}
  __device__ __forceinline__ void at(int jb) {
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = row(jb + u * kRows);
  }
  __device__ __forceinline__ DecRaw<DT> row(int j) {
    return load_raw_stream<DT>(src, base + static_cast<int64_t>(min(j, count - 1)) * D);
  }
  __device__ __forceinline__ void load() {
    if (count <= 0) return;
    if (U == 2 || count > 2 * kRows) {
      at(first);
    } else {
      r[0] = row(first);
      r[1] = row(first + kRows);
    }
  }
  template <typename F>
  __device__ __forceinline__ void walk(F&& f) {
    if (U > 2 && count <= 2 * kRows) {
      if (count <= 0) return;
      f(first, r[0]);
      f(first + kRows, r[1]);
      return;
    }
    for (int jb = first; jb < count; jb += U * kRows) {
      if (jb != first) at(jb);
#pragma unroll
      for (int u = 0; u < U; ++u) f(jb + u * kRows, r[u]);
    }
  }
};

// The live length: `length`, or the device-resident value clamped to
// [0, length] (the scratch and the grid are sized for `length`).
__device__ __forceinline__ int64_t live_length(const int64_t* dlen, int64_t length) {
  return dlen == nullptr ? length : max(int64_t{0}, min(*dlen, length));
}
__device__ __forceinline__ int live_chunks(int64_t live, int64_t chunk) {
  return static_cast<int>((live + chunk - 1) / chunk);
}

// ---------------------------------------------------------------------------
// short contexts: a slice's whole step in one workgroup
//
// The three launches of the chunked step cost more than the work while a slice
// is short.  Here one workgroup reads a slice's K rows, keeps the affinities in
// LDS (no scratch in memory), reduces max and sum, turns them into shares (one
// key per thread, the demand advanced there) and reads the V rows, the first of
// them before the reductions.  The production operator only.

// The most keys a slice may hold for this form; above, and for the other
// operators, the chunked step.  Computed alike on the host and, for a
// device-resident length, in the kernels.  One workgroup streams ~54 GB/s, so
// with few slices the chunked step's many workgroups catch up at a few hundred
// KB of K and V; from 160 slices on HBM bounds both and this form saves the
// launches and the affinities' way through memory.  The workgroups run in rounds
// of 256; where the last round leaves more than 3/16 of the rounds' places empty
// the lead is gone above 768 KB (two rounds), 1 MB (three) or 2 MB a slice.  us
// per step from memory, chunked -> here:
//   bf16 64:  16 slices 512 keys 10.3 -> 6.4, 1000 11.2 -> 9.2, 2000 11.8 -> 13.9;
//             64 slices 1000 12.6 -> 9.8, 2000 16.8 -> 15.1, 4000 21 -> 26;
//             128 slices 2000 20 -> 18, 4000 31 -> 32; 192 slices 8000 76 -> 68;
//             256 slices 1000 20 -> 14, 4000 54 -> 44, 16000 198 -> 170;
//             288 slices 2000 41 -> 33, 4000 61 -> 62, 8000 113 -> 122; 512 slices 8000 186 -> 171;
//             520 slices 2000 63 -> 54, 4000 107 -> 106, 8000 192 -> 211, 16000 371 -> 424;
//             640 slices 8000 231 -> 224, 16000 452 -> 456; 832 slices 8000 299 -> 297, 16000 586 -> 605;
//             1024 slices 4000 186 -> 174, 16000 722 -> 701; 2048 slices 16000 1433 -> 1408
//   bf16 128: 16 slices 512 12 -> 9, 1000 13 -> 14; 64 slices 1000 15 -> 15; 520 slices 2000 112 -> 103,
//             4000 198 -> 204, 16000 715 -> 843; 640 slices 16000 876 -> 898; 1024 slices 16000 1393 -> 1370
//   fp32 64:  16 slices 512 13 -> 12, 1000 13 -> 18; 128 slices 512 16 -> 14, 1000 23 -> 25;
//             256 slices 4000 107 -> 96; 520 slices 2000 131 -> 122, 4000 232 -> 248, 16000 864 -> 996;
//             1024 slices 16000 1687 -> 1529
constexpr int64_t kOneMaxKeys = 16384;                  // affinities a workgroup holds (64 KB of LDS)
template <int D, int DT>
__host__ __device__ inline int64_t one_max_keys(int64_t n) {
  constexpr int64_t kKeyBytes = 2 * D * (DT == DT_F32 ? 4 : 2);
  if (n > 256) {
    const int64_t places = (n + 255) / 256 * 256;
    if (n >= 512 && 16 * n >= 13 * places) return kOneMaxKeys;
    const int64_t keys = (n < 512 ? int64_t{768} : n < 768 ? int64_t{1024} : int64_t{2048}) * 1024 / kKeyBytes;
    return keys < kOneMaxKeys ? keys : kOneMaxKeys;
  }
  if (n >= 160) return kOneMaxKeys;
  const int64_t keys = (DT == DT_F32 ? (256 + n) << 10 : (272 + 3 * n) << 10) / kKeyBytes;
  return keys < 4096 ? keys : 4096;
}

struct OneSlice {
  const void* q1;
  int qdt;
  int64_t q_sn;
  const void* kc;
  const void* vc;
  int64_t kv_sn;
  float* committed;
  int64_t c_sn;
  void* out;
  int64_t o_sn;
  float qscale;
};

template <int D, int DT>
__device__ __forceinline__ void one_slice(const OneSlice& A, int64_t slice, int live, float* a_s) {
  using L = DecLayout<D>;
  __shared__ float sm[kDecWaves], ss[kDecWaves];
  __shared__ float red[kDecWaves][D + 1];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int sub = lane % L::kLanesPerRow, rw = lane / L::kLanesPerRow;
  float* crow = A.committed + slice * A.c_sn;
  const int64_t base = slice * A.kv_sn + sub * 8;

  float q[8];
  load8_f32(A.q1, slice * A.q_sn + sub * 8, A.qdt, q);
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] *= A.qscale;

  float m = -INFINITY;
  {
    RowStream<D, DT> k(A.kc, base, wave, lane, live);
    k.load();
    k.walk([&](int j, const DecRaw<DT>& r) {
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(q[e], raw_at<DT>(r, e), dot);
      const float a = row_reduce<L::kLanesPerRow>(dot);
      if (sub == 0 && j < live) {
        a_s[j] = a;
        m = fmaxf(m, a);
      }
    });
  }
  RowStream<D, DT> v(A.vc, base, wave, lane, live);
  v.load();                                             // in flight over the reductions
  float c0 = t < live ? crow[t] : 0.f;
  const float wm = wave_max(m);
  if (lane == 0) sm[wave] = wm;
  __syncthreads();
  float M = sm[0];
#pragma unroll
  for (int w = 1; w < kDecWaves; ++w) M = fmaxf(M, sm[w]);
  float l = 0.f;
  for (int j = t; j < live; j += kDecThreads) l += fast_exp2(a_s[j] - M);
  l = wave_sum(l);
  if (lane == 0) ss[wave] = l;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kDecWaves; ++w) tot += ss[w];
  const float lse = M + __log2f(tot);
  float ssum = 0.f;
  for (int j = t; j < live; j += kDecThreads) {
    const float p = fast_exp2(a_s[j] - lse);
    const float cm = j == t ? c0 : crow[j];
    const float sh = p * fast_rcp(cm + p + kEps);
    crow[j] = cm + p;
    a_s[j] = sh;
    ssum += sh;
  }
  ssum = wave_sum(ssum);
  if (lane == 0) red[wave][D] = ssum;
  __syncthreads();
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  v.walk([&](int j, const DecRaw<DT>& r) {
    if (j < live) {
      const float sh = a_s[j];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(sh, raw_at<DT>(r, e), acc[e]);
    }
  });
#pragma unroll
  for (int o = L::kLanesPerRow; o < 64; o <<= 1) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], o, 64);
  }
  if (rw == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[wave][sub * 8 + e] = acc[e];
  }
  __syncthreads();
  if (t < D) {
    float x = 0.f, s = 0.f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
      x += red[w][t];
      s += red[w][D];
    }
    store_as(A.out, slice * A.o_sn + t, A.qdt, x / (s + kEps));
  }
}

template <int D, int DT>
__global__ __launch_bounds__(kDecThreads) void dec_one(OneSlice A, int64_t length, int64_t slice0,
                                                       const int64_t* __restrict__ dlen) {
  extern __shared__ float one_s[];
  one_slice<D, DT>(A, slice0 + blockIdx.x, static_cast<int>(live_length(dlen, length)), one_s);
}

// Chunk statistics: softmax bids (max, sum 2^(a - max)) in log2 units; ratio
// bids (0 or the minimum of a for minshift, sum of the numerators) in natural
// units; none for the elementwise bids.
// ONE: a device-resident length that may be short: then one workgroup per slice
// does the whole step and the output launch has nothing to do.  The launch's first
// workgroups take the slices, one each, as they are dealt to the XCDs in turn: the
// first workgroup of every slice would put them on one XCD for 8 chunks a slice (160
// slices of 8000 keys, head_dim 128, of at most 20000, took 296 us so, and take 122).
template <int D, int DT, int BID = BID_SOFTMAX, bool ONE = false>
__global__ __launch_bounds__(kDecThreads) void dec_stats(
    const void* __restrict__ q1, int qdt, int64_t q_sn, const void* __restrict__ kc, int64_t kv_sn,
    float* __restrict__ aff, float2* __restrict__ part, int64_t length, int64_t chunk, int nchunk,
    float qscale, int64_t slice0, int64_t nslices, const int64_t* __restrict__ dlen,
    OneSlice one) {
  using L = DecLayout<D>;
  const int64_t slice = slice0 + blockIdx.y;
  const int c = blockIdx.x;
  if constexpr (ONE) {
    extern __shared__ float one_s[];
    const int64_t live = live_length(dlen, length);
    if (live <= one_max_keys<D, DT>(nslices)) {
      const unsigned block = blockIdx.y * gridDim.x + blockIdx.x;
      if (block < gridDim.y) one_slice<D, DT>(one, slice0 + block, static_cast<int>(live), one_s);
      return;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane % L::kLanesPerRow, rw = lane / L::kLanesPerRow;
  const int64_t live = live_length(dlen, length);
  if (dlen != nullptr) chunk = decode_chunk(nslices, live);
  if (c >= live_chunks(live, chunk)) return;             // past the live length: no statistics
  const int64_t j0 = c * chunk;
  const int64_t j1 = min(j0 + chunk, live);
  const int count = static_cast<int>(j1 - j0);
  RowStream<D, DT> rows(kc, slice * kv_sn + j0 * D + sub * 8, wave, lane, count);
  rows.load();

  float q[8];
  load8_f32(q1, slice * q_sn + sub * 8, qdt, q);        // q1 in its own dtype, as fp32
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] *= qscale;

  // the affinities of the chunk, then one key per thread: full-line stores and
  // one exponential per key
  __shared__ float a_s[kDecMaxChunk];
  rows.walk([&](int j, const DecRaw<DT>& r) {
    float dot = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) dot = fmaf(q[e], raw_at<DT>(r, e), dot);
    const float a = row_reduce<L::kLanesPerRow>(dot);
    if (sub == 0 && j < count) a_s[j] = a;
  });
  __syncthreads();
  float* arow = aff + slice * length + j0;
  float m = BID == BID_MINSHIFT ? INFINITY : -INFINITY, s = 0.f;
  for (int j = threadIdx.x; j < count; j += kDecThreads) {
    const float a = a_s[j];
    arow[j] = a;
    if constexpr (bid_ratio<BID>()) {
      if constexpr (BID == BID_MINSHIFT) m = fminf(m, a);
      s += bid_f<BID>(a);
    } else if constexpr (BID == BID_SOFTMAX) {
      const float mn = fmaxf(m, a);
      if (mn > -INFINITY) {
        s = s * fast_exp2(m - mn) + fast_exp2(a - mn);
        m = mn;
      }
    }
  }
  if constexpr (BID != BID_SOFTMAX) {
    const float wmn = -wave_max(-m);
    const float wsum = wave_sum(s);
    __shared__ float vm[kDecWaves], vs[kDecWaves];
    if (lane == 0) { vm[wave] = wmn; vs[wave] = wsum; }
    __syncthreads();
    if (threadIdx.x == 0) {
      float bm = INFINITY, bs = 0.f;
      for (int w = 0; w < kDecWaves; ++w) {
        bm = fminf(bm, vm[w]);
        bs += vs[w];
      }
      part[slice * nchunk + c] = make_float2(bm, bs);
    }
    return;
  }
  const float wm = wave_max(m);
  float ws = wave_sum(m == -INFINITY ? 0.f : s * fast_exp2(m - wm));
  __shared__ float sm[kDecWaves], ss[kDecWaves];
  if (lane == 0) { sm[wave] = wm; ss[wave] = ws; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float bm = -INFINITY;
    for (int w = 0; w < kDecWaves; ++w) bm = fmaxf(bm, sm[w]);
    float bs = 0.f;
    for (int w = 0; w < kDecWaves; ++w)
      if (sm[w] > -INFINITY) bs += ss[w] * fast_exp2(sm[w] - bm);
    part[slice * nchunk + c] = make_float2(bm, bs);
  }
}

template <int D, int DT, int BID = BID_SOFTMAX, int SHARE = SHARE_INCL>
__global__ __launch_bounds__(kDecThreads) void dec_apply(
    const void* __restrict__ vc, int64_t kv_sn, float* __restrict__ committed, int64_t c_sn,
    const float* __restrict__ aff, const float2* __restrict__ part, float* __restrict__ part_out,
    int64_t length, int64_t chunk, int nchunk, float shift, int64_t slice0, int64_t nslices,
    const int64_t* __restrict__ dlen, int64_t one_max) {
  using L = DecLayout<D>;
  const int64_t slice = slice0 + blockIdx.y;
  const int c = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane % L::kLanesPerRow, rw = lane / L::kLanesPerRow;
  // the scratch strides keep `length` and `nchunk` (the maxima); the walk
  // covers the live length only
  const int64_t live = live_length(dlen, length);
  if (dlen != nullptr) chunk = decode_chunk(nslices, live);
  if (live <= one_max) return;                            // dec_stats did the whole step
  const int nlive = live_chunks(live, chunk);
  if (c >= nlive) return;
  const int64_t j0 = c * chunk;
  const int count = static_cast<int>(min(j0 + chunk, live) - j0);
  const float* arow = aff + slice * length + j0;
  float* crow = committed + slice * c_sn + j0;
  // this thread's keys (one or two), which do not wait for the statistics
  constexpr int kOwn = static_cast<int>(kDecMaxChunk / kDecThreads);
  float av[kOwn], cv[kOwn];
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    const int j = min(static_cast<int>(threadIdx.x) + u * kDecThreads, count - 1);
    av[u] = arow[j];
    cv[u] = crow[j];
  }
  // and the first V rows, when every workgroup of the grid starts at once (in a
  // later round the CU's other workgroup covers the wait, and the earlier loads
  // cost 1.4%: 128 slices of 8192 keys 55 -> 53 us, 256 of 131072 1450 -> 1470)
  RowStream<D, DT> rows(vc, slice * kv_sn + j0 * D + sub * 8, wave, lane, count);
  const bool ahead = nslices * nlive <= kDecResident;
  if (ahead) rows.load();

  // Combine the chunk statistics of this slice (every wave redundantly).
  float m = -INFINITY, s = 0.f;
  for (int i = lane; i < nlive; i += 64) {
    const float2 ps = part[slice * nchunk + i];
    const float mn = fmaxf(m, ps.x);
    if (mn > -INFINITY) {
      s = s * fast_exp2(m - mn) + ps.y * fast_exp2(ps.x - mn);
      m = mn;
    }
  }
  const float gm = wave_max(m);
  const float gs = wave_sum(m == -INFINITY ? 0.f : s * fast_exp2(m - gm));
  float lse = gm + __log2f(gs);
  // row parameters of the other bids (natural-unit affinities in AFF)
  float r0 = 0.f, r1 = 0.f;
  const float lshift = __log2f(shift);
  if constexpr (BID != BID_SOFTMAX) {
    float mn = INFINITY, sm = 0.f;
    for (int i = lane; i < nlive; i += 64) {
      const float2 ps = part[slice * nchunk + i];
      mn = fminf(mn, ps.x);
      sm += ps.y;
    }
    mn = -wave_max(-mn);
    sm = wave_sum(sm);
    const float rden = BID == BID_MINSHIFT ? fmaxf(sm - static_cast<float>(live) * mn, 0.f)
                                           : (BID == BID_EXPSHIFT ? shift : sm);
    bid_row_params<BID>(BID == BID_MINSHIFT ? mn : 0.f, rden, static_cast<float>(live), true, r0, r1);
  }

  __shared__ float sh_s[kDecMaxChunk];
  __shared__ float red[kDecWaves][D + 1];
  // one key per thread: its share, and the demand advanced
  float ssum = 0.f;
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    const int j = threadIdx.x + u * kDecThreads;
    if (j >= count) break;
    const float a = av[u], cm = cv[u];
    float p;
    if constexpr (BID == BID_SOFTMAX) p = fast_exp2(a - lse);
    else p = bid_p<BID>(a, kLog2e, 1.f, r0, r1, lshift);
    float sh;
    if constexpr (SHARE == SHARE_INCL) sh = p * fast_rcp(cm + p + kEps);
    else if constexpr (SHARE == SHARE_EXCL) sh = p * fast_rcp(cm + kEps);
    else sh = p;
    crow[j] = cm + p;
    sh_s[j] = sh;
    ssum += sh;
  }
  ssum = wave_sum(ssum);
  if (lane == 0) red[wave][D] = ssum;
  __syncthreads();
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (!ahead) rows.load();
  rows.walk([&](int j, const DecRaw<DT>& r) {
    if (j < count) {
      const float sh = sh_s[j];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(sh, raw_at<DT>(r, e), acc[e]);
    }
  });
  // Reduce over lanes holding the same d-slice, then over waves.
#pragma unroll
  for (int o = L::kLanesPerRow; o < 64; o <<= 1) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], o, 64);
  }
  if (rw == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[wave][sub * 8 + e] = acc[e];
  }
  __syncthreads();
  for (int i = threadIdx.x; i <= D; i += kDecThreads) {
    float t = 0.f;
    for (int w = 0; w < kDecWaves; ++w) t += red[w][i];
    part_out[(slice * nchunk + c) * (D + 1) + i] = t;
  }
}

constexpr int kFinishThreads = 512;
// One workgroup per slice: the chunk partials' columns (D of share V, one of the
// shares) summed by kGroups threads each, every kGroups-th chunk per thread and
// two in flight, then over the groups; always in the same order.  One thread
// per column walked up to 512 chunks alone: one slice of 131072 keys took
// 52 us a step, 27 with the groups.
template <int D>
__global__ __launch_bounds__(kFinishThreads) void dec_finish(const float* __restrict__ part_out, int nchunk,
                                                  void* __restrict__ out, int64_t o_sn, int dt,
                                                  int64_t length, int64_t chunk,
                                                  const int64_t* __restrict__ dlen, int64_t one_max) {
  constexpr int kCols = D + 1, kGroups = kFinishThreads / kCols < 16 ? kFinishThreads / kCols : 16;
  __shared__ float red[kGroups][kCols];
  const int64_t slice = blockIdx.x;
  const int64_t live = live_length(dlen, length);
  if (live <= one_max) return;                            // dec_stats did the whole step
  if (dlen != nullptr) chunk = decode_chunk(gridDim.x, live);   // one workgroup per slice
  const int nlive = live_chunks(live, chunk);
  const int g = threadIdx.x / kCols, col = threadIdx.x % kCols;
  if (g < kGroups) {
    const float* p = part_out + slice * nchunk * kCols + col;   // slice stride: the maximum
    float t0 = 0.f, t1 = 0.f;
    int i = g;
    for (; i + kGroups < nlive; i += 2 * kGroups) {
      t0 += p[static_cast<int64_t>(i) * kCols];
      t1 += p[static_cast<int64_t>(i + kGroups) * kCols];
    }
    if (i < nlive) t0 += p[static_cast<int64_t>(i) * kCols];
    red[g][col] = t0 + t1;
  }
  __syncthreads();
  if (threadIdx.x < D) {
    float x = 0.f, tot = 0.f;
#pragma unroll
    for (int w = 0; w < kGroups; ++w) {
      x += red[w][threadIdx.x];
      tot += red[w][D];
    }
    store_as(out, slice * o_sn + threadIdx.x, dt, x / (tot + kEps));
  }
}

template <int D, int DT, int BID = BID_SOFTMAX, int SHARE = SHARE_INCL>
int launch_decode(const DecodeArgs& a) {
  // with a device-resident length the kernels choose the chunk from the live
  // length; the grid and scratch cover every live length up to a.length
  const int64_t chunk = decode_chunk(a.n, a.length);
  const int nchunk = static_cast<int>(decode_chunks(a.n, a.length, a.dlen != nullptr));
  char* ws = static_cast<char*>(a.workspace);
  float* aff = reinterpret_cast<float*>(ws);
  size_t off = align_up(sizeof(float) * a.n * a.length);
  float2* part = reinterpret_cast<float2*>(ws + off);
  off += align_up(sizeof(float2) * a.n * nchunk);
  float* part_out = reinterpret_cast<float*>(ws + off);
  // softmax bids keep log2-unit affinities, the others natural units
  const float qscale = (BID == BID_SOFTMAX ? kLog2e : 1.f) / sqrtf(static_cast<float>(D));
  hipStream_t st = static_cast<hipStream_t>(a.stream);
  const OneSlice one{a.q1, a.q_dtype, a.q_sn, a.k_cache, a.v_cache, a.kv_sn, a.committed, a.c_sn, a.out, a.o_sn, qscale};
  int64_t one_max = -1;                                   // a device-resident length the first launch may finish
  if constexpr (BID == BID_SOFTMAX && SHARE == SHARE_INCL) {
    const int64_t keys = one_max_keys<D, DT>(a.n);
    if (a.length <= keys) {
      const size_t lds = sizeof(float) * static_cast<size_t>((a.length + 63) / 64 * 64);
      slice_batches(a.n, [&](int64_t s0, unsigned ns) {
        DIL_TIMED("dec_one", st, (dec_one<D, DT><<<dim3(ns), kDecThreads, lds, st>>>(one, a.length, s0, a.dlen)));
      });
      return static_cast<int>(hipGetLastError());
    }
    if (a.dlen != nullptr) one_max = keys;
  }
  slice_batches(a.n, [&](int64_t s0, unsigned ns) {
    auto stats = [&](auto with_one, size_t lds) {
      DIL_TIMED("dec_stats", st,
                (dec_stats<D, DT, BID, decltype(with_one)::value><<<dim3(nchunk, ns), kDecThreads, lds, st>>>(
                    a.q1, a.q_dtype, a.q_sn, a.k_cache, a.kv_sn, aff, part, a.length, chunk, nchunk,
                    qscale, s0, a.n, a.dlen, one)));
    };
    if constexpr (BID == BID_SOFTMAX && SHARE == SHARE_INCL) {
      if (one_max >= 0) {
        stats(std::true_type{}, sizeof(float) * static_cast<size_t>((one_max + 63) / 64 * 64));
        return;
      }
    }
    stats(std::false_type{}, 0);
  });
  slice_batches(a.n, [&](int64_t s0, unsigned ns) {
    DIL_TIMED("dec_apply", st,
              (dec_apply<D, DT, BID, SHARE><<<dim3(nchunk, ns), kDecThreads, 0, st>>>(
                  a.v_cache, a.kv_sn, a.committed, a.c_sn, aff, part, part_out, a.length, chunk, nchunk,
                  a.var.shift, s0, a.n, a.dlen, one_max)));
  });
  DIL_TIMED("dec_finish", st,
            (dec_finish<D><<<dim3(static_cast<unsigned>(a.n)), kFinishThreads, 0, st>>>(part_out, nchunk, a.out, a.o_sn,
                                                                                    a.q_dtype, a.length, chunk, a.dlen,
                                                                                    one_max)));
  return static_cast<int>(hipGetLastError());
}

}  // namespace
}  // namespace dil
