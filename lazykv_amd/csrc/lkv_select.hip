// Quest bound + on-device top-K block selection.
//
// Reference: lazykv/selection.py:38-62 (quest_bound, top_blocks), called per selecting layer at
// lazykv/tiered.py:386 (rank, followed by a host sync) and :500 (gather_zerocopy). There it is two
// batched GEMMs, an add, an amax over the query group and torch.topk; rank() then copies the ids
// to the host. Here two back-to-back kernels stream the block metadata once and leave the ids on
// the device.
//
// bound_kernel: KV head h = blockIdx.x % n_kv, so with 8 KV heads each head's workgroups land on
// one XCD. A workgroup scores a contiguous run of candidate blocks: 16 lanes hold one metadata
// row (head_dim channels), so each wave-wide load covers 4 blocks; every lane keeps q+ and q- for
// its channels of the G query heads in registers. The row sum is a 4-step DPP reduction; the max
// over the group is taken in registers. The float32 bounds go to a scratch row per head.
// bound_kernel_mf: the same on the matrix cores, for a query of the metadata's dtype over aligned rows.
//
// Selection, by range-adaptive radix select: each pass histograms the keys of the current range into
// at most 2048 bins scaled to that range (so the first pass spreads the clustered bounds instead of
// piling them into a few exponent bins) and keeps the bin holding the K-th key; once that bin holds
// few keys they are ranked directly. One 1024-thread workgroup per KV head, with the row in registers
// up to 12,288 candidates (select_block_kernel) and reading it three times beyond
// (select_stream_kernel, select_kernel); beyond 16,384 in parts of 8,192, a workgroup each, and then
// the parts' picks (select_part_kernel, select_block_kernel) where the caller's workspace has room for
// them. The decode and residency launches of a one-call step select inside themselves up to 8,192.
// Scoring and selection are separate launches so that no workgroup has to publish its bounds across
// XCDs inside one launch (a device-scope release writes back the L2); the kernel boundary does that
// once.
#include "lkv_blockselect.h"
#include "lkv_common.h"

namespace {

#ifndef LKV_BOUND_THREADS
#define LKV_BOUND_THREADS 512
#endif
#ifndef LKV_BOUND_ITER
#define LKV_BOUND_ITER 1
#endif
constexpr int kBoundThreads = LKV_BOUND_THREADS;
constexpr int kBoundWaves = kBoundThreads / 64;
constexpr int kIter = LKV_BOUND_ITER;                     // 4-block rows per wave
constexpr int kBlocksPerWG = kBoundWaves * 4 * kIter;     // candidate blocks per workgroup
constexpr int kSelThreads = 1024;
constexpr int kSelWaves = kSelThreads / 64;
constexpr int kMaxSortedK = 2048;

template <int D, int MT, int G>
__global__ __launch_bounds__(kBoundThreads) void bound_kernel(const void* __restrict__ q, int q_dtype,
                                                              const typename lkv::Elem<MT>::T* __restrict__ kmin,
                                                              const typename lkv::Elem<MT>::T* __restrict__ kmax,
                                                              int64_t meta_head_stride, int n_kv, int cand_offset,
                                                              int n_cand, int rank_mode, float* __restrict__ bounds,
                                                              int64_t bound_stride) {
  using E = lkv::Elem<MT>;
  constexpr int EPL = D / 16;
  const int h = blockIdx.x % n_kv;
  const int split = blockIdx.x / n_kv;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane >> 4, c = lane & 15;

  const int wg_begin = split * kBlocksPerWG;
  const int wg_end = min(n_cand, wg_begin + kBlocksPerWG);
  const typename E::T* kmin_h = kmin + (int64_t)h * meta_head_stride + (int64_t)cand_offset * D + c * EPL;
  const typename E::T* kmax_h = kmax + (int64_t)h * meta_head_stride + (int64_t)cand_offset * D + c * EPL;
  float* bound_h = bounds + (int64_t)h * bound_stride;

  // Every metadata load is issued, raw, before anything waits on one: widened as loaded, the
  // first row's conversion sat between the two loads and the second waited for the first.
  lkv::RowWords<MT, EPL> wmax[kIter], wmin[kIter];
#pragma unroll
  for (int it = 0; it < kIter; ++it) {
    const int blk = wg_begin + (it * kBoundWaves + wave) * 4 + r;
    if (blk < wg_end) {
      lkv::load_row_words<MT, EPL>(kmax_h + (int64_t)blk * D, wmax[it]);
      lkv::load_row_words<MT, EPL>(kmin_h + (int64_t)blk * D, wmin[it]);
    } else {
#pragma unroll
      for (int w = 0; w < lkv::RowWords<MT, EPL>::WORDS; ++w) wmax[it].w[w] = wmin[it].w[w] = 0u;
    }
  }
  // The head's G query rows are read once per workgroup into LDS, while the metadata loads above
  // are in flight: every workgroup of a head reads the same rows, and per-wave reads of them were a
  // hot spot on a few L2 lines.
  __shared__ float s_q[G * D];
  for (int i = threadIdx.x; i < G * D; i += kBoundThreads) s_q[i] = lkv::load_any(q, (int64_t)h * G * D + i, q_dtype);
  __syncthreads();
  float qp[G][EPL], qn[G][EPL];
#pragma unroll
  for (int j = 0; j < G; ++j) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float x = s_q[j * D + c * EPL + e];
      qp[j][e] = fmaxf(x, 0.0f);
      qn[j][e] = x - qp[j][e];
    }
  }
#pragma unroll
  for (int it = 0; it < kIter; ++it) {
    const int blk = wg_begin + (it * kBoundWaves + wave) * 4 + r;
    float vmax[EPL], vmin[EPL];
    lkv::widen_row_words<MT, EPL>(wmax[it], vmax);
    lkv::widen_row_words<MT, EPL>(wmin[it], vmin);
    float best = -INFINITY;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      float a = 0.0f, b = 0.0f;
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        a = fmaf(qp[j][e], vmax[e], a);
        b = fmaf(qn[j][e], vmin[e], b);
      }
      float v;
      if (rank_mode == LKV_RANK_MODEL) {
        a = lkv::row16_sum(a);
        b = lkv::row16_sum(b);
        v = lkv::round_through<MT>(lkv::round_through<MT>(a) + lkv::round_through<MT>(b));
      } else {
        v = lkv::row16_sum(a + b);
      }
      best = fmaxf(best, v);
    }
    if (c == 0 && blk < wg_end) bound_h[blk] = best;
  }
}

// ---- the bound on the matrix cores -------------------------------------------------------------
// When the query has the metadata's dtype, the bounds of 16 blocks for the G query heads of a KV
// head are two matrix products, sum_d q+_d kmax_d and sum_d q-_d kmin_d (q+ = max(q, 0) and
// q- = q - q+ are exact in the model dtype): one v_mfma_f32_16x16x32 per 32 channels each, A = the
// 16 blocks' metadata rows (lane l: block l % 16, channels 32s + 8 (l / 16) .. + 7), B = q+ or q-
// (lane l: head l % 16). Products of two model-dtype values are exact in float32 and are summed in
// float32, as in the vector kernel (in another order). The result (lane l: blocks 4 (l / 16) + i,
// i < 4, of head l % 16) is maxed over the G heads across each 16-lane row, and the row's first
// lane writes its 4 bounds. The vector kernel spends ~150 instructions per wave on 4 blocks
// (widening, 16 float32 FMAs per head, DPP row sums); here 16 blocks take 8 MFMAs. Measured in the
// decode step (A/B, same box): the 8B-shaped HBM step 33.9 -> 33.3 us per layer with 4-wave
// workgroups of one 16-block tile per wave, the 1B step unchanged (20.5); two or four tiles per
// wave, or 8- and 16-wave workgroups, were slower at the 1B shape (21.2-22.7). Loading A directly
// in the matrix-core layout puts 16 rows, 16 bytes each, under every quarter-wave of a load; loading
// the tile with contiguous 1 KiB loads and transposing it through LDS took the 8B-shaped step from
// 33.2 to 32.0 us per layer (int8_64k 30.4 -> 30.0, the 1B step 20.3 -> 20.2).
#ifndef LKV_BOUND_MF_THREADS
#define LKV_BOUND_MF_THREADS 256
#endif
// The metadata rows are read once per step, with non-temporal loads (LKV_BOUND_NT 0: ordinary
// loads). Measured per layer, A/B over three rounds on one box: the 8B-shaped step in HBM 31.96 ->
// 31.39 us, the 1B-shaped 32K step 19.51 -> 19.21, int8 records in HBM at 64K 28.82 -> 28.01.
#ifndef LKV_BOUND_NT
#define LKV_BOUND_NT 1
#endif
#ifndef LKV_BOUND_MF_TILES
#define LKV_BOUND_MF_TILES 1
#endif
constexpr int kBoundMfThreads = LKV_BOUND_MF_THREADS;
constexpr int kBoundMfTiles = LKV_BOUND_MF_TILES;       // 16-block tiles per wave, all loads in flight together
constexpr int kBoundMfBlocks = kBoundMfThreads / 64 * 16 * kBoundMfTiles;  // blocks per workgroup

typedef __attribute__((ext_vector_type(4))) float bf32x4;
template <int MT>
struct BoundMma;
template <>
struct BoundMma<LKV_BF16> {
  typedef __attribute__((ext_vector_type(8))) __bf16 V8;
  __device__ __forceinline__ static bf32x4 mma(V8 a, V8 b, bf32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct BoundMma<LKV_F16> {
  typedef __attribute__((ext_vector_type(8))) _Float16 V8;
  __device__ __forceinline__ static bf32x4 mma(V8 a, V8 b, bf32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};

template <int D, int MT, int G>
__global__ __launch_bounds__(kBoundMfThreads) void bound_kernel_mf(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kmin,
                                                                   const uint16_t* __restrict__ kmax, int64_t meta_head_stride, int n_kv,
                                                                   int cand_offset, int n_cand, int rank_mode, float* __restrict__ bounds,
                                                                   int64_t bound_stride) {
  using M = BoundMma<MT>;
  using V8 = typename M::V8;
  constexpr int NS = D / 32;
  constexpr int kWaves = kBoundMfThreads / 64;
  constexpr int T = kBoundMfTiles;
  static_assert(G <= 16, "one MFMA column per query head");
  const int h = blockIdx.x % n_kv;
  const int split = blockIdx.x / n_kv;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, grp = lane >> 4;
  const int b0 = (split * kWaves + wave) * (16 * T);  // this wave's first block
  if (b0 >= n_cand) return;                          // wave-uniform; the kernel has no barrier
  // B: q+ and q- of head r16, split by the sign bit of each 16-bit element. Columns r16 >= G hold
  // head 0's query; their results are masked before the maximum over heads.
  const int j = r16;
  const uint16_t* qrow = q + ((int64_t)h * G + (j < G ? j : 0)) * D + 8 * grp;
  V8 qp[NS], qn[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const uint4 x = *(const uint4*)(qrow + 32 * s);
    const uint4 m = make_uint4(((x.x >> 15) & 0x00010001u) * 0xFFFFu, ((x.y >> 15) & 0x00010001u) * 0xFFFFu,
                               ((x.z >> 15) & 0x00010001u) * 0xFFFFu, ((x.w >> 15) & 0x00010001u) * 0xFFFFu);
    qp[s] = __builtin_bit_cast(V8, make_uint4(x.x & ~m.x, x.y & ~m.y, x.z & ~m.z, x.w & ~m.w));
    qn[s] = __builtin_bit_cast(V8, make_uint4(x.x & m.x, x.y & m.y, x.z & m.z, x.w & m.w));
  }
  // Each wave's 16 x D tile of kmax and of kmin is read with coalesced loads (load s, lane l: the
  // 16 bytes at 1024 s + 16 l of the tile) and handed to the matrix-core layout through the wave's
  // own LDS (lane l: block l % 16, channels 32 s + 8 (l / 16) .. + 7). A row past the candidates
  // reads the last candidate's row instead; its bound is not written. LDS holds 16-byte chunk k of
  // row r at r * D / 8 + (k ^ swz(r)), so that a store of a row and a read of one chunk of 16 rows
  // each touch 64 distinct banks.
  constexpr int kChunks = D / 8;  // 16-byte chunks per row
  constexpr int kRowsPerLoad = 64 / kChunks;
  static_assert(NS * kRowsPerLoad == 16, "NS loads of 64 lanes cover the 16-row tile");
  __shared__ __align__(16) uint4 s_tile[kWaves][T][2][16 * kChunks];
  const int64_t base = (int64_t)h * meta_head_stride + (int64_t)cand_offset * D;
  const auto swz = [](int r) { return kChunks == 16 ? r : (r >> 1) & (kChunks - 1); };
  uint4 amax[T][NS], amin[T][NS];
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int r = kRowsPerLoad * s + lane / kChunks, k = lane % kChunks;
      const int64_t off = base + (int64_t)min(b0 + 16 * t + r, n_cand - 1) * D + 8 * k;
#if LKV_BOUND_NT
      typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
      amax[t][s] = __builtin_bit_cast(uint4, __builtin_nontemporal_load((const u32x4*)(kmax + off)));
      amin[t][s] = __builtin_bit_cast(uint4, __builtin_nontemporal_load((const u32x4*)(kmin + off)));
#else
      amax[t][s] = *(const uint4*)(kmax + off);
      amin[t][s] = *(const uint4*)(kmin + off);
#endif
    }
  }
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int r = kRowsPerLoad * s + lane / kChunks, k = lane % kChunks;
      s_tile[wave][t][0][r * kChunks + (k ^ swz(r))] = amax[t][s];
      s_tile[wave][t][1][r * kChunks + (k ^ swz(r))] = amin[t][s];
    }
  }
  // The tile is this wave's alone: the wave's LDS stores complete before its reads in issue order.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int k = 4 * s + grp;
      amax[t][s] = s_tile[wave][t][0][r16 * kChunks + (k ^ swz(r16))];
      amin[t][s] = s_tile[wave][t][1][r16 * kChunks + (k ^ swz(r16))];
    }
  }
  float* bound_h = bounds + (int64_t)h * bound_stride;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    bf32x4 a = {0.0f, 0.0f, 0.0f, 0.0f}, b = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      a = M::mma(__builtin_bit_cast(V8, amax[t][s]), qp[s], a);
      b = M::mma(__builtin_bit_cast(V8, amin[t][s]), qn[s], b);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = rank_mode == LKV_RANK_MODEL ? lkv::round_through<MT>(lkv::round_through<MT>(a[i]) + lkv::round_through<MT>(b[i]))
                                            : a[i] + b[i];
      v = lkv::row16_max(j < G ? v : -INFINITY);
      const int blk = b0 + 16 * t + 4 * grp + i;
      if (r16 == 0 && blk < n_cand) bound_h[blk] = v;
    }
  }
}

// Rows the in-workgroup top-K may read as 16-byte vectors: aligned, and padded to 4 floats.
static bool rows_vector_readable(const float* bounds, int64_t bstride, int n_cand) {
  return ((uintptr_t)bounds & 15u) == 0 && bstride % 4 == 0 && bstride >= (int64_t)lkv_align_up((size_t)n_cand, 4);
}

// ---- the general selection: any candidate count, any row alignment, either order ------------------
// One 1024-thread workgroup per KV head. Each wave owns a contiguous run of candidates and reads it 256
// at a time, 16 bytes a lane, four reads in flight, on every pass; the row comes from the L2 after the
// first. (Reading a run per thread, a float at a time, the 65,535-candidate selection of a million-token
// context took 155 us, nearly all of it in seven passes of strided 4-byte reads.) The k-th best
// candidate (key, index) is found as block_top_k does (lkv_blockselect.h): a first range that starts at
// the least of the lanes' own largest keys, histograms of the live range, and a boundary bin of at most
// 64 keys ranked directly. The pass that lists that bin also gathers the keys above it, so a selection reads
// the row three times. In ascending mode the picks are bits of a map of the candidates, read in order;
// in sorted mode they are gathered in LDS and sorted, each thread holding one or two in registers:
// only partners in other waves go through LDS, 10 of the 55 steps for 1,024 picks, and the others are lane
// exchanges. With the bound launch, 1,024 of 65,535 in descending order: 176.0 -> 51.1 us (head_dim 64), 2,048
// of 262,144: 654 -> 152. What is left is one CU's vector work per head over three passes.
constexpr int kMaxStreamCand = 1 << 18;  // 262,144 candidates per head: 4M tokens at 16-token blocks

// f(i, keys of candidates i .. i + 3, how many of them exist) over [begin, end), 256 candidates a call.
template <bool VEC, typename F>
__device__ __forceinline__ void for_each_quad(const float* __restrict__ row, int begin, int end, int lane, F&& f) {
  int base = begin;
  if constexpr (VEC) {
#pragma unroll 1
    for (; base + 1024 <= end; base += 1024) {  // whole batches: no bounds to look at
      uint4 x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = *(const uint4*)(row + base + 256 * u + 4 * lane);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t key[4] = {lkv::orderable_bits(x[u].x), lkv::orderable_bits(x[u].y), lkv::orderable_bits(x[u].z), lkv::orderable_bits(x[u].w)};
        f(base + 256 * u + 4 * lane, key, 4);
      }
    }
  }
#pragma unroll 1
  for (; base < end; base += 256) {  // wave-uniform: every lane of the wave calls f
    const int i = base + 4 * lane;
    uint32_t key[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) key[e] = i + e < end ? lkv::orderable_key(row[i + e]) : 0u;
    f(i, key, max(0, min(4, end - i)));
  }
}

// Element of a descending bitonic merge: keeps the larger of its own and its partner's value where
// `larger`, else the smaller.
__device__ __forceinline__ uint64_t keep_one(uint64_t mine, uint64_t theirs, bool larger) {
  return ((mine > theirs) == larger) ? mine : theirs;
}

template <int M>
__device__ __forceinline__ uint64_t lane_xor_u64(uint64_t x) {
  return ((uint64_t)lkv::lane_xor_u32<M>((uint32_t)(x >> 32)) << 32) | lkv::lane_xor_u32<M>((uint32_t)x);
}

// The in-wave steps (stride M, M / 2, .., 1) of a merge.
template <int M>
__device__ __forceinline__ uint64_t merge_in_wave(uint64_t x, int t, bool desc) {
  x = keep_one(x, lane_xor_u64<M>(x), ((t & M) == 0) == desc);
  if constexpr (M > 1) {
    return merge_in_wave<M / 2>(x, t, desc);
  } else {
    return x;
  }
}

struct SortLds {
  uint64_t slot[2][kMaxSortedK];
};

// Sorts the np2 values in L.slot[0] (a power of two, 64 to kMaxSortedK) in descending order. Thread t
// returns elements t and t + 1024.
__device__ __forceinline__ void sort_descending(SortLds& L, int np2, uint64_t (&x)[2]) {
  const int t = threadIdx.x;
  const bool two = np2 > kSelThreads;
  x[0] = t < np2 ? L.slot[0][t] : 0u;
  x[1] = two ? L.slot[0][t + kSelThreads] : 0u;
  int buf = 1;
#pragma unroll 1
  for (int size = 2; size <= np2; size <<= 1) {
    // Element i of a run of `size` merges in descending order where (i & size) == 0. The bit is the same
    // for both elements of a thread but where size is the distance between them.
    const bool d0 = (t & size) == 0, d1 = ((t + kSelThreads) & size) == 0;
#pragma unroll 1
    for (int stride = size >> 1; stride >= 64; stride >>= 1) {
      if (stride == kSelThreads) {  // the thread's own two elements, in the last merge
        const uint64_t a = x[0], b = x[1];
        x[0] = a > b ? a : b;
        x[1] = a > b ? b : a;
        continue;
      }
      // Two buffers in turn: a buffer is written again only after the next step's barrier.
      L.slot[buf][t] = x[0];
      if (two) L.slot[buf][t + kSelThreads] = x[1];
      __syncthreads();
      x[0] = keep_one(x[0], L.slot[buf][t ^ stride], ((t & stride) == 0) == d0);
      if (two) x[1] = keep_one(x[1], L.slot[buf][(t ^ stride) + kSelThreads], ((t & stride) == 0) == d1);
      buf ^= 1;
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (e == 1 && !two) break;
      const bool desc = e == 0 ? d0 : d1;
      switch (min(size >> 1, 32)) {
        case 32: x[e] = merge_in_wave<32>(x[e], t, desc); break;
        case 16: x[e] = merge_in_wave<16>(x[e], t, desc); break;
        case 8: x[e] = merge_in_wave<8>(x[e], t, desc); break;
        case 4: x[e] = merge_in_wave<4>(x[e], t, desc); break;
        case 2: x[e] = merge_in_wave<2>(x[e], t, desc); break;
        default: x[e] = merge_in_wave<1>(x[e], t, desc); break;
      }
    }
  }
}

__device__ __forceinline__ void write_sorted(SortLds& L, int np2, int k, int cand_offset, int32_t* __restrict__ out_h) {
  uint64_t x[2];
  sort_descending(L, np2, x);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int i = (int)threadIdx.x + e * kSelThreads;
    if (i < k) out_h[i] = (int32_t)(0xffffffffu - (uint32_t)x[e]) + cand_offset;
  }
}

struct SelectRowLds {
  alignas(16) uint32_t hist[lkv::kSelBins];
  uint32_t list_key[lkv::kSelRank], list_id[lkv::kSelRank];
  uint32_t mm[2 * kSelWaves];
  uint32_t scan[2][kSelWaves];
  uint32_t info[5];  // boundary bin, keys above it, keys in it, boundary keys listed, picks gathered
  union {
    SortLds sort;                            // sorted mode
    uint32_t picked[kMaxStreamCand / 32];    // ascending mode: one bit per candidate
  };
};

template <bool VEC>
__device__ __forceinline__ void select_row(const float* __restrict__ row, int n, int k, int cand_offset, int sorted,
                                           int32_t* __restrict__ out_h, SelectRowLds& L) {
  constexpr int kBpt = lkv::kSelBins / kSelThreads;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int run = ((n + kSelWaves - 1) / kSelWaves + 255) & ~255;  // candidates a wave owns
  const int begin = min(n, wave * run), end = min(n, begin + run);
  int np2 = 64;  // sorted mode: slots to sort
  while (np2 < k) np2 <<= 1;
  lkv::clear_bins<kBpt>(L.hist + threadIdx.x * kBpt);
  if (sorted) {
    for (int i = k + threadIdx.x; i < np2; i += kSelThreads) L.sort.slot[0][i] = 0u;
  } else {
    for (int i = threadIdx.x; i < (n + 31) / 32; i += kSelThreads) L.picked[i] = 0u;
  }
  if (threadIdx.x == 0) L.info[4] = 0u;

  // ---- the range: what at least k keys reach, and the largest key ---------------------------------
  // n1 lanes hold a key, n2 of them two or more.
  const int tail = n % run;
  const int n1 = n / run * 64 + min(64, (tail + 3) / 4), n2 = n / run * 64 + min(64, (tail + 2) / 4);
  uint32_t m1 = 0u, m2 = 0u, low = 0xffffffffu;
  if (k <= n1) {  // uniform, as below
    for_each_quad<VEC>(row, begin, end, lane, [&](int, const uint32_t (&key)[4], int cnt) {
#pragma unroll
      for (int e = 0; e < 4; ++e) m1 = max(m1, e < cnt ? key[e] : 0u);
    });
    if (begin + 4 * lane < end) low = m1;
  } else if (k <= 2 * n2) {
    for_each_quad<VEC>(row, begin, end, lane, [&](int, const uint32_t (&key)[4], int cnt) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t x = e < cnt ? key[e] : 0u;
        m2 = max(m2, min(m1, x));
        m1 = max(m1, x);
      }
    });
    if (begin + 4 * lane + 1 < end) low = m2;
  } else {
    for_each_quad<VEC>(row, begin, end, lane, [&](int, const uint32_t (&key)[4], int cnt) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        m1 = max(m1, e < cnt ? key[e] : 0u);
        low = min(low, e < cnt ? key[e] : 0xffffffffu);
      }
    });
  }
  low = lkv::wave_min_u32(low);
  m1 = lkv::wave_max_u32(m1);
  if (lane == 0) {
    L.mm[2 * wave] = low;
    L.mm[2 * wave + 1] = m1;
  }
  __syncthreads();
  uint32_t lo = L.mm[0], hi = L.mm[1];
#pragma unroll
  for (int w = 1; w < kSelWaves; ++w) {
    lo = min(lo, L.mm[2 * w]);
    hi = max(hi, L.mm[2 * w + 1]);
  }

  // ---- the range of the k-th best: keys above it are taken, `need` of those in it --------------------
  int need = k;
  bool whole = false, ranked = false;
#pragma unroll 1
  for (int pass = 0; pass < lkv::kSelPasses; ++pass) {
    if (lo >= hi) break;
    const uint32_t width = hi - lo;
    const int bits = 32 - __clz(width);
    const int shift = bits > 11 ? bits - 11 : 0;
    if (pass > 0) {
      lkv::clear_bins<kBpt>(L.hist + threadIdx.x * kBpt);
      __syncthreads();
    }
    for_each_quad<VEC>(row, begin, end, lane, [&](int, const uint32_t (&key)[4], int cnt) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < cnt && key[e] - lo <= width) atomicAdd(&L.hist[(key[e] - lo) >> shift], 1u);
    });
    __syncthreads();
    uint32_t cnt[kBpt];
    lkv::read_bins<kBpt>(L.hist + threadIdx.x * kBpt, cnt);
    uint32_t local = 0;
#pragma unroll
    for (int b = 0; b < kBpt; ++b) local += cnt[b];
    uint32_t total;
    const uint32_t below = lkv::workgroup_exclusive_sum<kSelThreads, true>(local, L.scan[0], &total);
    const uint32_t above = total - below - local;
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
    const uint32_t new_lo = lo + (L.info[0] << shift);
    need -= (int)L.info[1];
    const uint32_t in_bin = L.info[2];
    hi = min(hi, new_lo + (shift ? ((1u << shift) - 1u) : 0u));
    lo = new_lo;
    whole = in_bin == (uint32_t)need;
    ranked = !whole && lo < hi && in_bin <= (uint32_t)lkv::kSelRank;
    if (whole || ranked) break;
  }
  // Taken are the keys above tk, and those equal to it up to index tid; of a boundary bin to be ranked,
  // also the `need` best.
  uint32_t tk = ranked ? hi : lo;
  int tid = whole ? 0x7fffffff : -1;
  if (!whole && !ranked) {
    // Every key left equals tk: the first `need` of them in index order are taken. The wave that holds
    // the need-th looks for its index.
    uint32_t eq = 0;
    for_each_quad<VEC>(row, begin, end, lane, [&](int, const uint32_t (&key)[4], int cnt) {
#pragma unroll
      for (int e = 0; e < 4; ++e) eq += e < cnt && key[e] == tk ? 1u : 0u;
    });
    uint32_t total;
    const uint32_t mine = lkv::workgroup_exclusive_sum<kSelThreads, true>(eq, L.scan[1], &total);
    int before = __builtin_amdgcn_readfirstlane((int)mine);  // ties in the runs of earlier waves
    for_each_quad<VEC>(row, begin, end, lane, [&](int i, const uint32_t (&key)[4], int cnt) {
      uint32_t m = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) m |= (e < cnt && key[e] == tk ? 1u : 0u) << e;
      const uint32_t c = __popc(m), incl = lkv::wave_inclusive_sum(c);
      const int first = before + (int)(incl - c);  // ties before this lane's
      if (first < need && need <= first + (int)c) {
        for (int t = first + 1; t < need; ++t) m &= m - 1u;
        L.info[0] = (uint32_t)(i + __ffs((int)m) - 1);
      }
      before += __builtin_amdgcn_readlane((int)incl, 63);
    });
    __syncthreads();
    tid = (int)L.info[0];
  }

  // ---- the picks --------------------------------------------------------------------------------------
  const auto pick = [&](uint32_t key, int id) {
    if (sorted) {
      const uint32_t slot = atomicAdd(&L.info[4], 1u);
      if (slot < (uint32_t)k) L.sort.slot[0][slot] = ((uint64_t)key << 32) | (uint64_t)(0xffffffffu - (uint32_t)id);
    } else {
      atomicOr(&L.picked[id >> 5], 1u << (id & 31));
    }
  };
  for_each_quad<VEC>(row, begin, end, lane, [&](int i, const uint32_t (&key)[4], int cnt) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (e >= cnt || key[e] < lo) continue;
      if (key[e] > tk || (key[e] == tk && i + e <= tid)) {
        pick(key[e], i + e);
      } else if (ranked) {
        const uint32_t slot = atomicAdd(&L.info[3], 1u);
        L.list_key[slot] = key[e];
        L.list_id[slot] = (uint32_t)(i + e);
      }
    }
  });
  __syncthreads();
  if (ranked) {
    if (wave == 0) {
      const int m = (int)L.info[3];
      lkv::rank_boundary(L.list_key, L.list_id, m, need, lane, &tk, &tid);
      if (lane < m) {
        const uint32_t key = L.list_key[lane];
        const int id = (int)L.list_id[lane];
        if (key > tk || (key == tk && id <= tid)) pick(key, id);
      }
    }
    __syncthreads();
  }

  if (!sorted) {
    const int words = (n + 31) / 32;
    const int per = (words + kSelThreads - 1) / kSelThreads;
    const int w0 = threadIdx.x * per;
    uint32_t mine = 0;
    for (int w = w0; w < min(words, w0 + per); ++w) mine += __popc(L.picked[w]);
    uint32_t total;
    int pos = (int)lkv::workgroup_exclusive_sum<kSelThreads, true>(mine, L.scan[0], &total);
    for (int w = w0; w < min(words, w0 + per); ++w)
      for (uint32_t m = L.picked[w]; m != 0u && pos < k; m &= m - 1u, ++pos) out_h[pos] = 32 * w + __ffs((int)m) - 1 + cand_offset;
    return;
  }
  // Descending key, equal keys by the lower id.
  write_sorted(L.sort, np2, k, cand_offset, out_h);
}

// ---- the selection as one in-workgroup top-K ----------------------------------------------------------
// The rule of select_row, by the routine the decode and residency launches run inside themselves
// (lkv_blockselect.h), which reads the row once into registers: 1,024 threads of 8 keys (8,192 candidates
// per head) or 12 (12,288; every key slot a thread holds costs instructions in each phase: at 8,192
// candidates, against 512 threads of 16, the 128K-token zero-copy step measured 615.23 -> 614.47 us per
// layer), with the wave index scalar in the scans (as lane masks, the scans' wave tests spilled
// scalar registers). VEC: rows that are 16-byte aligned and padded to 4 floats (the workspace's) are read as vectors, a caller's dense
// rows a float at a time. Each thread writes its ids straight to their ascending output positions, or, in sorted mode, to the sort's
// slots. Against select_row, which reads the row three times: 512 of 8,190 in descending order 20.5 -> 16.0 us
// with the bound launch, 768 of 12,286 ascending 19.3 -> 11.9, from dense rows 18.5 -> 13.4.
constexpr int kSelBlockThreads = 1024;
constexpr int kSelBlockCap = kSelBlockThreads * 12;
template <int KPT, bool SORTED, bool VEC>
__global__ __launch_bounds__(kSelBlockThreads) void select_block_kernel(const float* __restrict__ bounds, int64_t bstride,
                                                                        int n_cand, int k, int cand_offset,
                                                                        const int32_t* __restrict__ map,
                                                                        int32_t* __restrict__ out_idx, int64_t idx_stride) {
  static_assert(kSelBlockThreads == kSelThreads, "the sort's thread count");
  __shared__ lkv::SelectLds<kSelBlockThreads, KPT> L;
  const int h = blockIdx.x;
  const float* row = bounds + (int64_t)h * bstride;
  const lkv::SelectPick pk = lkv::block_top_k<kSelBlockThreads, KPT, true>(row, VEC, n_cand, k, L);
  int32_t* out_h = out_idx + (int64_t)h * idx_stride;
  const int32_t* map_h = map != nullptr ? map + (int64_t)h * bstride : nullptr;  // candidates of the parts below
  int pos = pk.pos;
  if constexpr (!SORTED) {
    for (uint32_t take = pk.take; take != 0u && pos < k; take &= take - 1u, ++pos) {
      const int i = pk.i0 + __ffs((int)take) - 1;
      out_h[pos] = (map_h != nullptr ? map_h[i] : i) + cand_offset;
    }
  } else {
    __shared__ SortLds sort;
    int np2 = 64;
    while (np2 < k) np2 <<= 1;
    for (int i = k + threadIdx.x; i < np2; i += kSelThreads) sort.slot[0][i] = 0u;
    for (uint32_t take = pk.take; take != 0u && pos < k; take &= take - 1u, ++pos) {
      const int i = pk.i0 + __ffs((int)take) - 1;
      const uint32_t id = map_h != nullptr ? (uint32_t)map_h[i] : (uint32_t)i;
      sort.slot[0][pos] = ((uint64_t)lkv::orderable_key(row[i]) << 32) | (uint64_t)(0xffffffffu - id);
    }
    __syncthreads();
    write_sorted(sort, np2, k, cand_offset, out_h);
  }
}

// Rows that may be read as 16-byte vectors (the workspace's: aligned, padded to 4 floats).
__global__ __launch_bounds__(kSelThreads) void select_stream_kernel(const float* __restrict__ bounds, int64_t bstride, int n_cand, int k,
                                                                    int cand_offset, int sorted, int32_t* __restrict__ out_idx,
                                                                    int64_t idx_stride) {
  __shared__ SelectRowLds L;
  select_row<true>(bounds + (int64_t)blockIdx.x * bstride, n_cand, k, cand_offset, sorted, out_idx + (int64_t)blockIdx.x * idx_stride, L);
}

// Any row (a caller's dense bounds of more than kSelBlockCap candidates).
__global__ __launch_bounds__(kSelThreads) void select_kernel(const float* __restrict__ bounds, int64_t bstride, int n_cand, int k,
                                                             int cand_offset, int sorted, int32_t* __restrict__ out_idx,
                                                             int64_t idx_stride) {
  __shared__ SelectRowLds L;
  select_row<false>(bounds + (int64_t)blockIdx.x * bstride, n_cand, k, cand_offset, sorted, out_idx + (int64_t)blockIdx.x * idx_stride, L);
}

// ---- long rows in parts -----------------------------------------------------------------------------
// A row of more than kSelBlockCap candidates as parts of kPartCand, one workgroup each: a part's own best k (by the
// same rule, in ascending order) are the only ones of it that can be among the row's, so the row's selection is
// that of the parts' picks, one list in ascending order, of at most kSelBlockCap. One workgroup per head reading the
// whole row three times is bound by that CU's vector work. 1,024 of 65,535 for eight heads, with the bound launch
// at head_dim 64: 42.8 -> 34.7 us ascending, 51.1 -> 41.8 descending. Two parts gain nothing (1,024 of 16,382: 19.7
// and 20.0), so rows of up to two stay whole.
constexpr int kPartCand = kSelBlockThreads * 8;
__global__ __launch_bounds__(kSelBlockThreads) void select_part_kernel(const float* __restrict__ bounds, int64_t bstride, int n_kv, int n_cand,
                                                                       int k, float* __restrict__ part_key, int32_t* __restrict__ part_id,
                                                                       int64_t pstride) {
  __shared__ lkv::SelectLds<kSelBlockThreads, 8> L;
  const int h = blockIdx.x % n_kv, part = blockIdx.x / n_kv;
  const int first = part * kPartCand, m = min(kPartCand, n_cand - first), kk = min(k, m);
  const float* row = bounds + (int64_t)h * bstride + first;
  const lkv::SelectPick pk = lkv::block_top_k<kSelBlockThreads, 8, true>(row, true, m, kk, L);
  const int64_t at = (int64_t)h * pstride + (int64_t)part * k;
  int pos = pk.pos;
  for (uint32_t take = pk.take; take != 0u && pos < kk; take &= take - 1u, ++pos) {
    const int i = pk.i0 + __ffs((int)take) - 1;
    part_key[at + pos] = row[i];
    part_id[at + pos] = first + i;
  }
}

// The parts' picks of one head (0: the row is not selected in parts), and the floats between heads' lists.
static int part_picks(int n_cand, int k) {
  if (n_cand <= 2 * kPartCand || k <= 0) return 0;
  const int64_t picks = (int64_t)((n_cand + kPartCand - 1) / kPartCand) * k;
  return picks <= kSelBlockCap ? (int)picks : 0;
}
static size_t part_stride(int n_cand, int k) { return lkv_align_up((size_t)part_picks(n_cand, k), 4); }

template <int D, int MT, int G>
int launch_bound(hipStream_t stream, const void* q, int q_dtype, const void* kmin, const void* kmax, int64_t mhs, int n_kv,
                 int cand_offset, int n_cand, int rank_mode, float* bounds, int64_t bstride) {
  using T = typename lkv::Elem<MT>::T;
  // A model-dtype query and 16-byte aligned metadata rows: the matrix cores. A row starts at
  // h * mhs + b * D elements; D is 64 or 128, so the rows are aligned when the bases are and the
  // head stride is a multiple of 8 elements. Any other layout takes the vector kernel.
  if (q_dtype == MT && (((uintptr_t)q | (uintptr_t)kmin | (uintptr_t)kmax) & 15u) == 0 && (mhs & 7) == 0) {
    const int splits_mf = (n_cand + kBoundMfBlocks - 1) / kBoundMfBlocks;
    hipLaunchKernelGGL((bound_kernel_mf<D, MT, G>), dim3(splits_mf * n_kv), dim3(kBoundMfThreads), 0, stream, (const uint16_t*)q,
                       (const uint16_t*)kmin, (const uint16_t*)kmax, mhs, n_kv, cand_offset, n_cand, rank_mode, bounds, bstride);
    LKV_CHECK_LAUNCH("bound");
    return LKV_OK;
  }
  const int splits = (n_cand + kBlocksPerWG - 1) / kBlocksPerWG;
  hipLaunchKernelGGL((bound_kernel<D, MT, G>), dim3(splits * n_kv), dim3(kBoundThreads), 0, stream, q, q_dtype,
                     (const T*)kmin, (const T*)kmax, mhs, n_kv, cand_offset, n_cand, rank_mode, bounds, bstride);
  LKV_CHECK_LAUNCH("bound");
  return LKV_OK;
}

template <int D, int MT>
int dispatch_g(int g, hipStream_t s, const void* q, int qd, const void* kmin, const void* kmax, int64_t mhs, int n_kv,
               int co, int nc, int rm, float* b, int64_t bs) {
  switch (g) {
    case 1: return launch_bound<D, MT, 1>(s, q, qd, kmin, kmax, mhs, n_kv, co, nc, rm, b, bs);
    case 2: return launch_bound<D, MT, 2>(s, q, qd, kmin, kmax, mhs, n_kv, co, nc, rm, b, bs);
    case 4: return launch_bound<D, MT, 4>(s, q, qd, kmin, kmax, mhs, n_kv, co, nc, rm, b, bs);
    case 8: return launch_bound<D, MT, 8>(s, q, qd, kmin, kmax, mhs, n_kv, co, nc, rm, b, bs);
    default: lkv_set_error("unsupported GQA group size %d (1, 2, 4 or 8)", g); return LKV_ERR_UNSUPPORTED;
  }
}

}  // namespace

static size_t bound_rows_bytes(int n_kv, int n_cand) { return lkv_align_up((size_t)n_kv * lkv_align_up((size_t)n_cand, 4) * 4, 256); }

// The bound rows, and the parts' picks where a selection of k takes parts.
extern "C" size_t lkv_bound_topk_workspace_bytes(int n_kv, int n_cand, int k) {
  if (n_kv <= 0 || n_cand <= 0) return 0;
  return bound_rows_bytes(n_kv, n_cand) + lkv_align_up(2 * (size_t)n_kv * part_stride(n_cand, k) * 4, 256);
}

int lkv_launch_bounds(hipStream_t s, const void* q, int q_dtype, const void* kmin, const void* kmax, int meta_dtype,
                      int64_t meta_head_stride, int n_kv, int g, int head_dim, int cand_offset, int n_cand, int rank_mode,
                      float* bounds, int64_t bstride) {
  if (head_dim == 128) {
    return meta_dtype == LKV_BF16 ? dispatch_g<128, LKV_BF16>(g, s, q, q_dtype, kmin, kmax, meta_head_stride, n_kv, cand_offset,
                                                               n_cand, rank_mode, bounds, bstride)
                                  : dispatch_g<128, LKV_F16>(g, s, q, q_dtype, kmin, kmax, meta_head_stride, n_kv, cand_offset,
                                                              n_cand, rank_mode, bounds, bstride);
  }
  return meta_dtype == LKV_BF16 ? dispatch_g<64, LKV_BF16>(g, s, q, q_dtype, kmin, kmax, meta_head_stride, n_kv, cand_offset,
                                                            n_cand, rank_mode, bounds, bstride)
                                : dispatch_g<64, LKV_F16>(g, s, q, q_dtype, kmin, kmax, meta_head_stride, n_kv, cand_offset, n_cand,
                                                           rank_mode, bounds, bstride);
}

int lkv_select_max_candidates() { return kMaxStreamCand; }

// Up to kSelBlockCap candidates: the in-workgroup top-K, which reads the row once, as 16-byte vectors where the rows allow (a
// caller's dense rows may not).
// A longer one in parts where `parts` (2 * n_kv * part_stride words) is given and the parts' picks fit the in-workgroup top-K
// (lkv_bound_topk's own rows; the fused calls' workspaces hold no parts). Any other selection reads the row three times.
template <int KPT, bool VEC>
static void launch_select_block(hipStream_t s, const float* bounds, int64_t bstride, int n_kv, int n_cand, int k, int cand_offset, int sorted,
                                const int32_t* map, int32_t* out_idx, int64_t idx_stride) {
  if (sorted) {
    hipLaunchKernelGGL((select_block_kernel<KPT, true, VEC>), dim3(n_kv), dim3(kSelBlockThreads), 0, s, bounds, bstride, n_cand, k, cand_offset,
                       map, out_idx, idx_stride);
  } else {
    hipLaunchKernelGGL((select_block_kernel<KPT, false, VEC>), dim3(n_kv), dim3(kSelBlockThreads), 0, s, bounds, bstride, n_cand, k, cand_offset,
                       map, out_idx, idx_stride);
  }
}

static int launch_select(hipStream_t s, const float* bounds, int64_t bstride, int n_kv, int n_cand, int k, int cand_offset, int sorted,
                         void* parts, int32_t* out_idx, int64_t idx_stride) {
  const bool vec = rows_vector_readable(bounds, bstride, n_cand);
  if (n_cand <= kSelBlockThreads * 8) {
    vec ? launch_select_block<8, true>(s, bounds, bstride, n_kv, n_cand, k, cand_offset, sorted, nullptr, out_idx, idx_stride)
        : launch_select_block<8, false>(s, bounds, bstride, n_kv, n_cand, k, cand_offset, sorted, nullptr, out_idx, idx_stride);
  } else if (n_cand <= kSelBlockCap) {
    vec ? launch_select_block<12, true>(s, bounds, bstride, n_kv, n_cand, k, cand_offset, sorted, nullptr, out_idx, idx_stride)
        : launch_select_block<12, false>(s, bounds, bstride, n_kv, n_cand, k, cand_offset, sorted, nullptr, out_idx, idx_stride);
  } else if (vec && parts != nullptr && part_picks(n_cand, k) > 0) {
    const int n_parts = (n_cand + kPartCand - 1) / kPartCand;
    const int64_t ps = (int64_t)part_stride(n_cand, k);
    float* key = (float*)parts;
    int32_t* id = (int32_t*)(key + n_kv * ps);
    hipLaunchKernelGGL(select_part_kernel, dim3(n_kv * n_parts), dim3(kSelBlockThreads), 0, s, bounds, bstride, n_kv, n_cand, k, key, id, ps);
    // Only the last part can hold fewer than k candidates.
    const int last = n_cand - (n_parts - 1) * kPartCand;
    const int picks = (n_parts - 1) * k + (last < k ? last : k);
    if (picks <= kSelBlockThreads * 8) {
      launch_select_block<8, true>(s, key, ps, n_kv, picks, k, cand_offset, sorted, id, out_idx, idx_stride);
    } else {
      launch_select_block<12, true>(s, key, ps, n_kv, picks, k, cand_offset, sorted, id, out_idx, idx_stride);
    }
  } else if (vec) {
    hipLaunchKernelGGL(select_stream_kernel, dim3(n_kv), dim3(kSelThreads), 0, s, bounds, bstride, n_cand, k, cand_offset, sorted, out_idx,
                       idx_stride);
  } else {
    hipLaunchKernelGGL(select_kernel, dim3(n_kv), dim3(kSelThreads), 0, s, bounds, bstride, n_cand, k, cand_offset, sorted, out_idx,
                       idx_stride);
  }
  LKV_CHECK_LAUNCH("select");
  return LKV_OK;
}

int lkv_launch_select(hipStream_t s, const float* bounds, int64_t bstride, int n_kv, int n_cand, int k, int cand_offset,
                      int32_t* out_idx, int64_t idx_stride) {
  return launch_select(s, bounds, bstride, n_kv, n_cand, k, cand_offset, 0, nullptr, out_idx, idx_stride);
}

extern "C" int lkv_bound_topk(uintptr_t stream, const void* q, int q_dtype, const void* kmin, const void* kmax,
                              int meta_dtype, int64_t meta_head_stride, int n_q, int n_kv, int head_dim,
                              int cand_offset, int n_cand, int k, int rank_mode, int flags, int32_t* out_idx,
                              int64_t idx_stride, float* out_bound, void* ws, size_t ws_bytes) {
  LKV_CHECK_ARG(q && kmin && kmax, "NULL q/kmin/kmax");
  LKV_CHECK_ARG(n_kv > 0 && n_q > 0 && n_q % n_kv == 0, "n_q=%d must be a positive multiple of n_kv=%d", n_q, n_kv);
  LKV_CHECK_ARG(head_dim == 64 || head_dim == 128, "head_dim %d unsupported (64 or 128)", head_dim);
  LKV_CHECK_ARG(meta_dtype == LKV_F16 || meta_dtype == LKV_BF16, "metadata dtype must be f16 or bf16");
  LKV_CHECK_ARG(lkv_is_model_dtype(q_dtype), "bad query dtype");
  LKV_CHECK_ARG(n_cand > 0, "no candidate blocks");
  LKV_CHECK_ARG(cand_offset >= 0, "negative candidate offset");
  LKV_CHECK_ARG(k >= 0 && k <= n_cand, "selected k=%d must be in 0..n_cand=%d", k, n_cand);
  LKV_CHECK_ARG(rank_mode == LKV_RANK_F32 || rank_mode == LKV_RANK_MODEL, "bad rank mode");
  LKV_CHECK_ARG(meta_head_stride >= (int64_t)(cand_offset + n_cand) * head_dim, "metadata head stride too small");
  LKV_CHECK_ARG(k == 0 || (out_idx != nullptr && idx_stride >= k), "out_idx missing or idx_stride < k");
  const int sorted = (flags & LKV_SORTED) ? 1 : 0;
  if (k > 0 && n_cand > kMaxStreamCand) {
    lkv_set_error("%d candidate blocks exceed the per-head select limit %d", n_cand, kMaxStreamCand);
    return LKV_ERR_UNSUPPORTED;
  }
  if (sorted && k > kMaxSortedK) {
    lkv_set_error("sorted selection supports k <= %d", kMaxSortedK);
    return LKV_ERR_UNSUPPORTED;
  }
  // Scratch bound rows are padded to 4 floats so the select can read them as 16-byte vectors;
  // a caller's out_bound is dense [n_kv, n_cand].
  float* bounds = out_bound;
  int64_t bstride = n_cand;
  void* parts = nullptr;
  if (bounds == nullptr) {
    const size_t need = bound_rows_bytes(n_kv, n_cand);
    LKV_CHECK_ARG(ws != nullptr && ws_bytes >= need, "workspace of %zu bytes needed, got %zu", need, ws_bytes);
    LKV_CHECK_ARG(((uintptr_t)ws & 15) == 0, "workspace must be 16-byte aligned");
    bounds = (float*)ws;
    bstride = (int64_t)lkv_align_up((size_t)n_cand, 4);
    // A workspace sized for fewer blocks k than this call's holds no parts: the row is then read whole.
    if (part_picks(n_cand, k) > 0 && ws_bytes >= lkv_bound_topk_workspace_bytes(n_kv, n_cand, k)) parts = (char*)ws + need;
  }
  const int g = n_q / n_kv;
  hipStream_t s = (hipStream_t)stream;
  const int rc = lkv_launch_bounds(s, q, q_dtype, kmin, kmax, meta_dtype, meta_head_stride, n_kv, g, head_dim, cand_offset, n_cand,
                                   rank_mode, bounds, bstride);
  if (rc != LKV_OK || k == 0) return rc;
  return launch_select(s, bounds, bstride, n_kv, n_cand, k, cand_offset, sorted, parts, out_idx, idx_stride);
}
