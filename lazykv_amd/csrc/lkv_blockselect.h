// Top-K of one KV head's float32 bounds inside one workgroup, for launches that select and then
// use the selection in the same workgroup (the fused select + decode launch).
//
// The rule is lkv_bound_topk's: the k candidates with the highest bound, ties at the threshold
// taken towards the lower candidate index, reported in ascending index order. Each thread holds a
// contiguous run of up to KPT candidates as order-preserving integer keys. The k-th best candidate
// (key, index) is found by range-adaptive radix select: a pass histograms the live key range into at
// most 2048 bins scaled to that range and keeps the bin holding the k-th key. When that bin's keys are
// all taken the selection is complete; when it holds at most 64 keys every wave ranks them for itself,
// one lane each, with the keys handed round by v_readlane. Three passes narrow any 32-bit range to one
// value, so the loop is capped at four.
//
// What bounds it is the chain of phases, not bytes: each is one LDS round trip and one barrier, 0.2 to
// 1.4 us in a decode launch of 512 threads. So
//   - the first range starts at the least of the threads' own largest keys (second largest) when there
//     are at least k (k / 2) of them: that many keys lie above it. With k of 512 threads that leaves
//     about a third of the keys to the histogram, whose LDS atomics to random bins are its cost;
//   - the ranking of the boundary bin gives the k-th candidate itself, (key, index), and a thread then
//     takes every key above one threshold: no bitmap, no second barrier, two instructions a key.
#pragma once

#include "lkv_common.h"

namespace lkv {

constexpr int kSelBins = 2048;
constexpr int kSelPasses = 4;
constexpr int kSelRank = 64;  // a boundary bin of up to this many keys is ranked, a lane each

__device__ __forceinline__ uint32_t orderable_bits(uint32_t u) { return (u & 0x80000000u) ? ~u : (u | 0x80000000u); }
__device__ __forceinline__ uint32_t orderable_key(float f) { return orderable_bits(__float_as_uint(f)); }

template <int NT, int KPT>
struct SelectLds {
  static constexpr int kWaves = NT / 64;
  static constexpr int kBpt = kSelBins / NT;     // bins a thread owns
  static_assert(kBpt == 2 || kBpt == 4 || kBpt == 8, "256, 512 or 1024 threads");
  alignas(16) uint32_t hist[kSelBins];
  uint32_t list_key[kSelRank];  // the boundary bin's keys and candidate indices, in any order
  uint32_t list_id[kSelRank];
  uint32_t mm[2 * kWaves];
  uint32_t scan[3][kWaves];
  uint32_t info[4];  // boundary bin, keys above it, keys in it, boundary-list length
};

// What one thread contributes: bit u of `take` marks candidate i0 + u as selected; the selected
// candidates of the thread occupy consecutive output positions from `pos`.
struct SelectPick {
  uint32_t take;
  int pos;
  int i0;
};

// Exclusive prefix sum over the workgroup's threads in thread order; `slots` holds one word per
// wave and is read after the barrier inside. The caller separates reuses of `slots` by a barrier.
// SCALAR_WAVE reads the wave index into a scalar register, so that `w < wave` is a scalar compare
// instead of a lane mask per w that the compiler may keep live across the passes (a launch with
// little else to hold gains; inside the decode launch it measured slower).
template <int NT, bool SCALAR_WAVE = false>
__device__ __forceinline__ uint32_t workgroup_exclusive_sum(uint32_t v, uint32_t* slots, uint32_t* total) {
  const int lane = threadIdx.x & 63;
  const int wave = SCALAR_WAVE ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : (int)(threadIdx.x >> 6);
  const uint32_t x = wave_inclusive_sum(v);
  if (lane == 63) slots[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const uint32_t s = slots[w];
    if (w < wave) before += s;
    all += s;
  }
  *total = all;
  return before + x - v;
}

// A thread's kBpt bins, as vector LDS accesses.
template <int B>
__device__ __forceinline__ void read_bins(const uint32_t* p, uint32_t (&c)[B]) {
#pragma unroll
  for (int i = 0; i < B; i += 4) {
    if constexpr (B == 2) {
      const uint2 x = *(const uint2*)p;
      c[0] = x.x;
      c[1] = x.y;
    } else {
      const uint4 x = *(const uint4*)(p + i);
      c[i] = x.x;
      c[i + 1] = x.y;
      c[i + 2] = x.z;
      c[i + 3] = x.w;
    }
  }
}
template <int B>
__device__ __forceinline__ void clear_bins(uint32_t* p) {
  if constexpr (B == 2) {
    *(uint2*)p = make_uint2(0u, 0u);
  } else {
#pragma unroll
    for (int i = 0; i < B; i += 4) *(uint4*)(p + i) = make_uint4(0u, 0u, 0u, 0u);
  }
}

// The need-th best of the m <= kSelRank listed candidates by (key desc, index asc), found by every wave
// for itself: lane e ranks entry e, the entries handed round by v_readlane.
__device__ __forceinline__ void rank_boundary(const uint32_t* list_key, const uint32_t* list_id, int m_, int need, int lane, uint32_t* tk,
                                              int* tid) {
  const int m = __builtin_amdgcn_readfirstlane(m_);
  const uint32_t ek = lane < m ? list_key[lane] : 0u, ei = lane < m ? list_id[lane] : 0xffffffffu;
  int rank = 0;
  for (int e = 0; e < m; ++e) {
    const uint32_t sk = (uint32_t)__builtin_amdgcn_readlane((int)ek, e), si = (uint32_t)__builtin_amdgcn_readlane((int)ei, e);
    rank += (sk > ek) | ((sk == ek) & (si < ei));
  }
  const uint64_t at = __ballot(lane < m && rank == need - 1);
  const int src = at != 0 ? __ffsll((unsigned long long)at) - 1 : 0;
  *tk = (uint32_t)__builtin_amdgcn_readlane((int)ek, src);
  *tid = __builtin_amdgcn_readlane((int)ei, src);
}

// Select k of the n bounds at `bound_h` (n <= NT * KPT; the row is readable in whole 16-byte
// vectors up to a multiple of 4 when `aligned`). Every thread of the workgroup must call it.
template <int NT, int KPT, bool SCALAR_WAVE = false>
__device__ __forceinline__ SelectPick block_top_k(const float* __restrict__ bound_h, bool aligned, int n, int k, SelectLds<NT, KPT>& L) {
  static_assert(KPT % 4 == 0 && KPT <= 32, "a thread's slots are tracked in 32-bit masks, loaded 4 at a time");
  constexpr int kWaves = NT / 64;
  constexpr int kBpt = SelectLds<NT, KPT>::kBpt;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // Keys per thread: a multiple of 4, so a thread's run is whole 16-byte vectors.
  const int npt = ((n + NT - 1) / NT + 3) & ~3;
  const int i0 = threadIdx.x * npt;
  const int nlive = max(0, min(npt, n - i0));
  uint32_t key[KPT];
  if (aligned) {
#pragma unroll
    for (int u = 0; u < KPT; u += 4) {
      float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
      if (u < nlive) f = *(const float4*)(bound_h + i0 + u);  // within the row's padding to 4
      key[u] = orderable_key(f.x);
      key[u + 1] = orderable_key(f.y);
      key[u + 2] = orderable_key(f.z);
      key[u + 3] = orderable_key(f.w);
    }
  } else {
#pragma unroll
    for (int u = 0; u < KPT; ++u) key[u] = u < nlive ? orderable_key(bound_h[i0 + u]) : 0u;
  }
  const uint32_t live = nlive >= 32 ? 0xffffffffu : (1u << nlive) - 1u;  // bit u: slot u holds a candidate
  // While the loads are in flight: this thread's bins for the first pass.
  clear_bins<kBpt>(L.hist + threadIdx.x * kBpt);
  // This thread's largest and second largest key (0 for slots without a candidate).
  uint32_t m1 = 0u, m2 = 0u;
#pragma unroll
  for (int u = 0; u < KPT; ++u) {
    const uint32_t x = u < nlive ? key[u] : 0u;
    m2 = max(m2, min(m1, x));
    m1 = max(m1, x);
  }
  // A value that at least k keys reach: each of the nth threads with a key holds one of at least its m1,
  // each of the nth2 threads with two keys another of at least its m2. Beyond 2 * nth2, the least key.
  const int nth = (n + npt - 1) / npt, nth2 = nth - (n % npt == 1 ? 1 : 0);
  uint32_t low = 0xffffffffu;
  if (k <= nth) {  // workgroup-uniform, as below
    if (nlive > 0) low = m1;
  } else if (k <= 2 * nth2) {
    if (nlive > 1) low = m2;
  } else {
#pragma unroll
    for (int u = 0; u < KPT; ++u) low = min(low, u < nlive ? key[u] : 0xffffffffu);
  }
  low = wave_min_u32(low);
  m1 = wave_max_u32(m1);
  if (lane == 0) {
    L.mm[2 * wave] = low;
    L.mm[2 * wave + 1] = m1;
  }
  __syncthreads();
  uint32_t lo = L.mm[0], hi = L.mm[1];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    lo = min(lo, L.mm[2 * w]);
    hi = max(hi, L.mm[2 * w + 1]);
  }

  // The k-th best candidate: taken are the keys above tk, and those equal to it up to index tid.
  uint32_t tk = lo;
  int tid = -1;
  bool found = false;
  int need = k;  // still to take from [lo, hi]; every key above hi is taken
#pragma unroll 1
  for (int pass = 0; pass < kSelPasses; ++pass) {
    if (lo >= hi) break;
    const uint32_t width = hi - lo;
    const int bits = 32 - __clz(width);
    const int shift = bits > 11 ? bits - 11 : 0;
    if (pass > 0) {  // the previous pass read its bins before the barrier that published `info`
      clear_bins<kBpt>(L.hist + threadIdx.x * kBpt);
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < KPT; ++u)
      if (u < nlive && key[u] >= lo && key[u] <= hi) atomicAdd(&L.hist[(key[u] - lo) >> shift], 1u);
    __syncthreads();
    uint32_t cnt[kBpt];
    read_bins<kBpt>(L.hist + threadIdx.x * kBpt, cnt);
    uint32_t local = 0;
#pragma unroll
    for (int b = 0; b < kBpt; ++b) local += cnt[b];
    uint32_t total;
    const uint32_t below = workgroup_exclusive_sum<NT, SCALAR_WAVE>(local, L.scan[0], &total);
    const uint32_t above = total - below - local;  // keys of higher bins (owned by later threads)
    if (above < (uint32_t)need && (uint32_t)need <= above + local) {
      uint32_t acc = above;
#pragma unroll
      for (int b = kBpt - 1; b >= 0; --b) {
        if (acc < (uint32_t)need && (uint32_t)need <= acc + cnt[b]) {
          L.info[0] = (uint32_t)(threadIdx.x * kBpt + b);
          L.info[1] = acc;
          L.info[2] = cnt[b];
          L.info[3] = 0u;
        }
        acc += cnt[b];
      }
    }
    __syncthreads();
    const uint32_t bin = L.info[0];
    need -= (int)L.info[1];
    const uint32_t in_bin = L.info[2];
    const uint32_t new_lo = lo + (bin << shift);
    const uint32_t span = shift ? ((1u << shift) - 1u) : 0u;
    hi = min(hi, new_lo + span);
    lo = new_lo;
    tk = lo;
    if (in_bin == (uint32_t)need) {  // the boundary bin is taken whole
      tid = 0x7fffffff;
      found = true;
      break;
    }
    if (lo < hi && in_bin <= (uint32_t)kSelRank) {
#pragma unroll
      for (int u = 0; u < KPT; ++u) {
        if (u < nlive && key[u] >= lo && key[u] <= hi) {
          const uint32_t slot = atomicAdd(&L.info[3], 1u);
          L.list_key[slot] = key[u];
          L.list_id[slot] = (uint32_t)(i0 + u);
        }
      }
      __syncthreads();
      rank_boundary(L.list_key, L.list_id, (int)in_bin, need, lane, &tk, &tid);
      found = true;
      break;
    }
  }
  if (!found) {
    // Every key left equals tk: the first `need` of them in index order are taken, so tid is the
    // index of the need-th.
    uint32_t tie_m = 0u;
#pragma unroll
    for (int u = 0; u < KPT; ++u) tie_m |= (u < nlive && key[u] == tk ? 1u : 0u) << u;
    uint32_t tot;
    const int before = (int)workgroup_exclusive_sum<NT, SCALAR_WAVE>(__popc(tie_m), L.scan[2], &tot);
    if (before < need && need <= before + (int)__popc(tie_m)) {
      for (int t = before + 1; t < need; ++t) tie_m &= tie_m - 1u;  // drop the ties before it
      L.info[0] = (uint32_t)(i0 + __ffs((int)tie_m) - 1);
    }
    __syncthreads();
    tid = (int)L.info[0];
  }

  // A thread whose run ends by tid takes its keys from tk up, one whose run starts behind it those
  // above tk; only the run that tid cuts looks at indices.
  const bool after = i0 > tid;
  const bool cut = !after && i0 + npt - 1 > tid;
  const uint32_t thr = after ? tk + 1u : tk;
  SelectPick p;
  p.take = 0u;
#pragma unroll
  for (int u = 0; u < KPT; ++u) p.take |= (key[u] >= thr ? 1u : 0u) << u;
  p.take &= (after && tk == 0xffffffffu) ? 0u : live;
  if (cut) {
#pragma unroll
    for (int u = 0; u < KPT; ++u)
      if (key[u] == tk && i0 + u > tid) p.take &= ~(1u << u);
  }
  uint32_t tot;
  p.pos = (int)workgroup_exclusive_sum<NT, SCALAR_WAVE>(__popc(p.take), L.scan[1], &tot);
  p.i0 = i0;
  return p;
}

}  // namespace lkv
