// Block stores for the tier: int8 pack (bit-exact with lazykv/quant.py), unpack, the seal-time
// copy into the host pool, and per-block key min/max metadata -- fused so a block is read once.
//
// Reference: lazykv/quant.py:59-105 (_affine, pack, unpack), lazykv/tiered.py:162-197 (the
// boundary: host copy or pack, then metadata from the exact or the dequantised keys),
// :353-375 (_seal: one block, blocking D2H, pack + unpack for the int8 metadata), :226-236
// (metadata rebuilt from a stored pool). One wave handles one (block, KV head) pair, or two of 4 tokens at head_dim 64; 16 lanes
// hold one row, so the 4 row groups of the wave see rows r, r+4, r+8, ... of the block.
//
// Bit-exactness. quant.py computes in float32: mn/mx (exact), scale = max((mx-mn)/255, FLT_MIN)
// with an IEEE divide, q = clamp(rint((x-mn)/scale), 0, 255) - 128 (round half to even), and
// stores float16(scale), float16(mn). Dequantisation is ((q+128) * f32(scale16)) + f32(zero16),
// two separately rounded float32 operations, then a round to the model dtype. This file is
// compiled with FP contraction off and the default correctly rounded float32 divide.
#include "lkv_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = 4;

// What a launch does with each pair:
//   MODE_META          metadata of the exact keys only;
//   MODE_COPY          model-dtype pair copied to dst (+ metadata of the exact keys);
//   MODE_INT8          int8 record of the pair written to dst (+ metadata of the dequantised keys);
//   MODE_META_FROM_I8  metadata of an existing record's dequantised keys;
//   MODE_UNPACK        an existing record dequantised into a model-dtype pair of dst (+ metadata of
//                      those keys): quant.py unpack into any block layout.
enum { MODE_META = 0, MODE_COPY = 1, MODE_INT8 = 2, MODE_META_FROM_I8 = 3, MODE_UNPACK = 4 };

struct StoreArgs {
  const void* sk;
  const void* sv;
  int64_t s_bstride, s_hstride;  // elements (bytes for MODE_META_FROM_I8)
  void* dk;
  void* dv;
  int64_t d_bstride, d_hstride;  // elements (bytes for MODE_INT8)
  int n_kv, bs, first_block, n_blocks;
  void* kmin;
  void* kmax;
  int meta_dtype;
  int64_t meta_hstride;
};

__device__ __forceinline__ float f16_round(float x) { return lkv::f16_to_f32(lkv::f32_to_f16(x)); }

template <int MT, int EPL>
__device__ __forceinline__ void store_segment(typename lkv::Elem<MT>::T* p, const float (&x)[EPL]) {
  using T = typename lkv::Elem<MT>::T;
  T t[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) t[e] = lkv::Elem<MT>::store(x[e]);
  constexpr int BYTES = EPL * (int)sizeof(T);
  if constexpr (BYTES == 16) {
    uint4 w;
    __builtin_memcpy(&w, t, 16);
    *(uint4*)p = w;
  } else if constexpr (BYTES == 32) {
    uint4 w[2];
    __builtin_memcpy(w, t, 32);
    ((uint4*)p)[0] = w[0];
    ((uint4*)p)[1] = w[1];
  } else if constexpr (BYTES == 8) {
    uint2 w;
    __builtin_memcpy(&w, t, 8);
    *(uint2*)p = w;
  } else {
#pragma unroll
    for (int e = 0; e < EPL; ++e) p[e] = t[e];
  }
}

template <int EPL>
__device__ __forceinline__ void load_bytes(const int8_t* p, int8_t (&b)[EPL]) {
  if constexpr (EPL == 8) {
    uint2 w = *(const uint2*)p;
    __builtin_memcpy(b, &w, 8);
  } else {
    uint32_t w = *(const uint32_t*)p;
    __builtin_memcpy(b, &w, 4);
  }
}

template <int D, int MT>
__device__ __forceinline__ void write_meta(const StoreArgs& a, int b, int h, int c, const float (&mn)[D / 16],
                                           const float (&mx)[D / 16]) {
  constexpr int EPL = D / 16;
  const int64_t base = (int64_t)h * a.meta_hstride + (int64_t)b * D + c * EPL;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    lkv::store_any(a.kmin, base + e, a.meta_dtype, mn[e]);
    lkv::store_any(a.kmax, base + e, a.meta_dtype, mx[e]);
  }
}

// Sources that are int8 records: 16 lanes hold a row.
template <int D, int MT, int MODE>
__device__ __forceinline__ void store_record(const StoreArgs& a, int64_t pair) {
  static_assert(MODE == MODE_META_FROM_I8 || MODE == MODE_UNPACK, "reads records");
  using T = typename lkv::Elem<MT>::T;
  constexpr int EPL = D / 16;
  const int lane = threadIdx.x & 63;
  const int r = lane >> 4, c = lane & 15;
  const int b = a.first_block + (int)(pair / a.n_kv);
  const int h = (int)(pair % a.n_kv);
  const int bs = a.bs;
  const int rows = bs >> 2;  // rows per row group
  const bool want_meta = a.kmin != nullptr;

  // An existing record: the metadata of its dequantised keys and, for MODE_UNPACK, the pair
  // itself dequantised into dst (quant.py:103-105: ((q + 128) * scale) + zero, two separately
  // rounded float32 operations, then the model dtype).
  const uint8_t* rec = (const uint8_t*)a.sk + (int64_t)b * a.s_bstride + (int64_t)h * a.s_hstride;
  const uint16_t* sc = (const uint16_t*)(rec + 2 * bs * D);
  T* dk = nullptr;
  T* dv = nullptr;
  if constexpr (MODE == MODE_UNPACK) {
    const int64_t doff = (int64_t)b * a.d_bstride + (int64_t)h * a.d_hstride + c * EPL;
    dk = (T*)a.dk + doff;
    dv = (T*)a.dv + doff;
  }
  float ks[EPL], kz[EPL], mn[EPL], mx[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    ks[e] = lkv::f16_to_f32(sc[c * EPL + e]);
    kz[e] = lkv::f16_to_f32(sc[D + c * EPL + e]);
    mn[e] = INFINITY;
    mx[e] = -INFINITY;
  }
  for (int i = 0; i < rows; ++i) {
    const int row = r + 4 * i;
    int8_t q[EPL];
    load_bytes<EPL>((const int8_t*)rec + row * D + c * EPL, q);
    float x[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      x[e] = lkv::round_through<MT>(((float)q[e] + 128.0f) * ks[e] + kz[e]);
      mn[e] = fminf(mn[e], x[e]);
      mx[e] = fmaxf(mx[e], x[e]);
    }
    if constexpr (MODE == MODE_UNPACK) {
      store_segment<MT, EPL>(dk + (int64_t)row * D, x);
      int8_t vq[EPL];
      load_bytes<EPL>((const int8_t*)rec + bs * D + row * D + c * EPL, vq);
      const float vs = lkv::f16_to_f32(sc[2 * D + row]);
      const float vz = lkv::f16_to_f32(sc[2 * D + bs + row]);
      float v[EPL];
#pragma unroll
      for (int e = 0; e < EPL; ++e) v[e] = ((float)vq[e] + 128.0f) * vs + vz;
      store_segment<MT, EPL>(dv + (int64_t)row * D, v);
    }
  }
  if (!want_meta) return;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    mn[e] = lkv::groups4_min(mn[e]);
    mx[e] = lkv::groups4_max(mx[e]);
  }
  if (r == 0) write_meta<D, MT>(a, b, h, c, mn, mx);
}

// ---- sources in the model dtype -----------------------------------------------------------------------
// 8 channels a lane (16 bytes of a 16-bit type): a row is 16 lanes at d 128 and 8 lanes at d 64, and a wave-wide
// load covers 4 or 8 rows. A pair is read once, in chunks of 16 rows: for blocks of up to 16 tokens every load of
// the pair is issued before the first is used (longer blocks read their keys twice to make a record). Read a row
// at a time and the keys twice, with a correctly rounded divide per value, packing 32,768 pairs of 16 x 64 float16
// took 95 us for 134 MB read and 78 MB written; see quantise8 for the divide.
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

template <int D, int MT>
struct Rows {
  static constexpr int LPR = D / 8;       // lanes per row
  static constexpr int RG = 64 / LPR;     // rows per wave-wide load
  static constexpr int W = 2 * (int)sizeof(typename lkv::Elem<MT>::T);  // words of a lane's 8 channels
};

// Whether a lane's 8 channels are two runs of 4, in the row's two halves: float32 rows copied as they are, whose two 16-byte
// accesses a lane each cover the row's lanes without gaps then (256 blocks of 16 tokens, 8 heads, d 64, into a dense cache 7.3 -> 6.1 us; 2,048
// with their metadata 55.7 -> 49.8). Records keep 8 channels together (8 bytes of codes a store).
template <int MT, int MODE>
constexpr bool kSplitRow = MT == LKV_F32 && MODE != MODE_INT8;

// A chunk of 16 rows, or, for blocks of fewer, of NI loads' RG * NI rows. SECOND: words from a lane's first four to its next.
template <int D, int MT, int NI, int SECOND>
struct RowChunk {
  uint32_t w[NI][Rows<D, MT>::W];
  // Rows t0 + r + RG i of the pair at p (this lane's channels); a row past the block reads row 0 instead, which
  // changes no range, and is not stored.
  __device__ __forceinline__ void load(const typename lkv::Elem<MT>::T* p, int t0, int bs, int r) {
    using R = Rows<D, MT>;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = t0 + r + R::RG * i;
      const uint32_t* at = (const uint32_t*)(p + (int64_t)(row < bs ? row : 0) * D);
#pragma unroll
      for (int j = 0; j < R::W; j += 4) {
        const u32x4_a4 x = *(const u32x4_a4*)(at + j / 4 * SECOND);
        w[i][j] = x.x;
        w[i][j + 1] = x.y;
        w[i][j + 2] = x.z;
        w[i][j + 3] = x.w;
      }
    }
  }
  __device__ __forceinline__ void store(typename lkv::Elem<MT>::T* p, int t0, int bs, int r) const {
    using R = Rows<D, MT>;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = t0 + r + R::RG * i;
      if (row < bs) {
        uint32_t* at = (uint32_t*)(p + (int64_t)row * D);
#pragma unroll
        for (int j = 0; j < R::W; j += 4) *(u32x4_a4*)(at + j / 4 * SECOND) = u32x4_a4{w[i][j], w[i][j + 1], w[i][j + 2], w[i][j + 3]};
      }
    }
  }
  __device__ __forceinline__ void widen(int i, float (&x)[8]) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (MT == LKV_F32) {
        x[e] = lkv::bits_to_float(w[i][e]);
      } else {
        x[e] = lkv::Elem<MT>::load((uint16_t)((e & 1) ? w[i][e >> 1] >> 16 : w[i][e >> 1] & 0xffffu));
      }
    }
  }
};

// A lane's 8 channels reduced over the GROUPS row groups of its pair (LPR lanes each): each step keeps one half of the values and
// gives the partner the other, so a lane ends with the totals of its channels own_channel() .. + 8 / GROUPS - 1 in v.
template <int LPR, int GROUPS, typename Op>
__device__ __forceinline__ void reduce_channels(float (&v)[8], int lane, Op op) {
  constexpr int N = LPR == 8 ? 4 : 8;  // values a lane holds after the 8-lane rows' own step
  if constexpr (LPR == 8) {
    const bool odd = (lane & 8) != 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float keep = odd ? v[i + 4] : v[i], give = odd ? v[i] : v[i + 4];
      v[i] = op(keep, lkv::dpp<lkv::kDppRowRor8>(give));
    }
  }
  float x, y;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    lkv::swap_halves<16>(v[i], v[i + N / 2], x, y);
    v[i] = op(x, y);
  }
  if constexpr (LPR * GROUPS == 64) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
      lkv::swap_halves<32>(v[i], v[i + N / 4], x, y);
      v[i] = op(x, y);
    }
  }
}
template <int LPR, int GROUPS>
__device__ __forceinline__ int own_channel(int lane) {
  constexpr int N = LPR == 8 ? 4 : 8;
  return (LPR == 8 && (lane & 8) ? 4 : 0) + ((lane & 16) ? N / 2 : 0) + (LPR * GROUPS == 64 && (lane & 32) ? N / 4 : 0);
}
// The reverse: every lane's 8 channels from the lanes that own them.
template <int LPR, int GROUPS>
__device__ __forceinline__ void gather_channels(float (&v)[8], int lane) {
  constexpr int N = LPR == 8 ? 4 : 8;
  if constexpr (LPR * GROUPS == 64) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) lkv::lane_pair<32>(v[i], v[i], v[i + N / 4]);
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) lkv::lane_pair<16>(v[i], v[i], v[i + N / 2]);
  if constexpr (LPR == 8) {
    const bool odd = (lane & 8) != 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float mine = v[i], theirs = lkv::dpp<lkv::kDppRowRor8>(mine);
      v[i] = odd ? theirs : mine;
      v[i + 4] = odd ? mine : theirs;
    }
  }
}

// range / 255, correctly rounded where it reaches FLT_MIN (the callers take the larger of the two): one corrected
// product with the rounded reciprocal (Markstein's division by a constant; equal to the divide for every
// significand, subnormal to largest exponent). An infinite range stays infinite.
__device__ __forceinline__ float over_255(float range) {
  constexpr float y = 1.0f / 255.0f;
  const float q = range * y;
  const float z = fmaf(fmaf(-q, 255.0f, range), y, q);
  return range == INFINITY ? range : z;
}
__device__ __forceinline__ float scale_of(float mn, float mx) { return fmaxf(over_255(mx - mn), 1.17549435e-38f); }

// The codes clamp(rint((x - mn) / scale), 0, 255) - 128 of 8 values, as 8 bytes. The quotient by the hardware's reciprocal is within
// 1e-4 of the rounded one (at most 255, with relative errors of 2^-23 in the reciprocal and 2^-24 in each of two roundings), so both round
// to the same integer unless it lies that close to a half: then the divide itself decides, for a value in 5,000 of a wide spread, so in
// about one of ten wave-wide steps of 512. (At 1e-3 from a half it was one in 500 and two steps of three: 2,048 blocks of 16 x 128
// float16, 8 heads, packed in 46.0 us, here in 40.3.)
constexpr float kSureRound = 0.4999f;
__device__ __forceinline__ uint2 quantise8(const float (&x)[8], const float (&mn)[8], const float (&scale)[8], const float (&inv)[8]) {
  float q[8], worst = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float t = (x[e] - mn[e]) * inv[e];
    q[e] = rintf(t);
    worst = fmaxf(worst, fabsf(t - q[e]));
  }
  if (worst > kSureRound) {
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = rintf((x[e] - mn[e]) / scale[e]);
  }
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // v_cvt_pk_u8_f32: a whole number of 0..255 into byte e % 4.
    w[e >> 2] = __builtin_amdgcn_cvt_pk_u8_f32(fminf(fmaxf(q[e], 0.0f), 255.0f), e & 3, w[e >> 2]);
  }
  return make_uint2(w[0] ^ 0x80808080u, w[1] ^ 0x80808080u);
}

// The block's key metadata from the lanes that own its channels (SPLIT: kSplitRow's).
template <int D, int LPR, int GROUPS, bool SPLIT>
__device__ __forceinline__ void write_owned(const StoreArgs& a, int b, int h, int c, int lane, const float (&mn)[8], const float (&mx)[8]) {
  const int own = own_channel<LPR, GROUPS>(lane);  // the lane's channels own .. own + 8 / GROUPS - 1 lie in one half
  const int64_t base = (int64_t)h * a.meta_hstride + (int64_t)b * D + (SPLIT ? c * 4 + own % 4 + (own >= 4 ? D / 2 : 0) : c * 8 + own);
#pragma unroll
  for (int i = 0; i < 8 / GROUPS; ++i) {
    lkv::store_any(a.kmin, base + i, a.meta_dtype, mn[i]);
    lkv::store_any(a.kmax, base + i, a.meta_dtype, mx[i]);
  }
}

// PPW: pairs of the wave, each in 64 / PPW lanes (two where one load of the wave has the rows of two blocks). LONG: records of
// blocks of more than one chunk, whose rows are loaded again when the keys' range is known.
template <int D, int MT, int MODE, bool META, int NI, int PPW, bool LONG>
__device__ __forceinline__ void store_rows(const StoreArgs& a, int64_t pair) {
  using T = typename lkv::Elem<MT>::T;
  using R = Rows<D, MT>;
  const int lane = threadIdx.x & 63;
  static_assert(PPW == 1 || (PPW == 2 && NI == 1 && R::RG == 8), "two pairs of at most 4 rows each");
  constexpr int GROUPS = R::RG / PPW;  // row groups of a pair
  const int r = lane / R::LPR % GROUPS, c = lane % R::LPR;
  // A workgroup's four waves take four consecutive blocks of one head, contiguous in a dense cache: a pair per
  // head in turn, they read and wrote at the heads' strides, a power of two apart, at once (a float16 layer of
  // 32K tokens into a pool, dense [h, T, 64] source: 30.2 -> 23.4 us; pool to pool 47.6 -> 46.2).
  static_assert(kWaves == 4, "four blocks of a head per workgroup");
  const int64_t quad = (int64_t)a.n_kv * kWaves;
  int b, h;
  if ((pair / quad + 1) * kWaves <= a.n_blocks) {
    b = a.first_block + (int)(pair / quad) * kWaves + (int)(pair % kWaves);
    h = (int)((pair % quad) / kWaves);
  } else {
    b = a.first_block + (int)(pair / a.n_kv);
    h = (int)(pair % a.n_kv);
  }
  const int bs = a.bs;
  constexpr bool kRange = META || MODE == MODE_INT8;  // the keys' range is wanted
  const auto lower = [](float p, float q) { return fminf(p, q); };
  const auto upper = [](float p, float q) { return fmaxf(p, q); };
  constexpr bool SPLIT = kSplitRow<MT, MODE>;
  const int first = c * (SPLIT ? 4 : 8);  // the lane's first channel
  const int64_t soff = (int64_t)b * a.s_bstride + (int64_t)h * a.s_hstride + first;
  const T* sk = (const T*)a.sk + soff;
  const T* sv = (const T*)a.sv + soff;
  RowChunk<D, MT, NI, SPLIT ? D / 2 : 4> k, v;
  k.load(sk, 0, bs, r);
  if constexpr (MODE == MODE_COPY || (MODE == MODE_INT8 && !LONG)) v.load(sv, 0, bs, r);

  T* dk = nullptr;
  T* dv = nullptr;
  if constexpr (MODE == MODE_COPY) {
    const int64_t doff = (int64_t)b * a.d_bstride + (int64_t)h * a.d_hstride + first;
    dk = (T*)a.dk + doff;
    dv = (T*)a.dv + doff;
  }
  // ---- keys: per-channel range over the block's tokens -----------------------------------------------
  float mn[8], mx[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    mn[e] = INFINITY;
    mx[e] = -INFINITY;
  }
  for (int t0 = 0;;) {
    if constexpr (kRange) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        float x[8];
        k.widen(i, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          mn[e] = fminf(mn[e], x[e]);
          mx[e] = fmaxf(mx[e], x[e]);
        }
      }
    }
    if constexpr (MODE == MODE_COPY) {
      k.store(dk, t0, bs, r);
      v.store(dv, t0, bs, r);
    }
    t0 += 16;
    if (t0 >= bs) break;
    k.load(sk, t0, bs, r);
    if constexpr (MODE == MODE_COPY) v.load(sv, t0, bs, r);
  }
  if constexpr (kRange) {
    reduce_channels<R::LPR, GROUPS>(mn, lane, lower);
    reduce_channels<R::LPR, GROUPS>(mx, lane, upper);
  }
  if constexpr (MODE != MODE_INT8) {
    if constexpr (META) write_owned<D, R::LPR, GROUPS, SPLIT>(a, b, h, c, lane, mn, mx);
  } else {
    uint8_t* rec = (uint8_t*)a.dk + (int64_t)b * a.d_bstride + (int64_t)h * a.d_hstride;
    uint16_t* sc = (uint16_t*)(rec + 2 * bs * D);
    // Each channel's scale is made, and stored, by the lane that owns it.
    float scale[8], inv[8];
#pragma unroll
    for (int i = 0; i < 8 / GROUPS; ++i) {
      scale[i] = scale_of(mn[i], mx[i]);
      sc[c * 8 + own_channel<R::LPR, GROUPS>(lane) + i] = lkv::f32_to_f16(scale[i]);
      sc[D + c * 8 + own_channel<R::LPR, GROUPS>(lane) + i] = lkv::f32_to_f16(mn[i]);
    }
    gather_channels<R::LPR, GROUPS>(scale, lane);
    gather_channels<R::LPR, GROUPS>(mn, lane);
#pragma unroll
    for (int e = 0; e < 8; ++e) inv[e] = __builtin_amdgcn_rcpf(scale[e]);
    float dmn[8], dmx[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      dmn[e] = INFINITY;
      dmx[e] = -INFINITY;
    }
    for (int t0 = 0; t0 < bs; t0 += 16) {
      if constexpr (LONG) {  // one chunk's keys and values are still in their registers
        k.load(sk, t0, bs, r);
        v.load(sv, t0, bs, r);
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int row = t0 + r + R::RG * i;
        float x[8];
        k.widen(i, x);
        const uint2 q = quantise8(x, mn, scale, inv);
        if constexpr (META) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            // The dequantised key (quant.py:103-105), a repeated row 0 included.
            const uint32_t u = (((e < 4 ? q.x : q.y) ^ 0x80808080u) >> (8 * (e & 3))) & 0xffu;
            const float d = lkv::round_through<MT>((float)u * f16_round(scale[e]) + f16_round(mn[e]));
            dmn[e] = fminf(dmn[e], d);
            dmx[e] = fmaxf(dmx[e], d);
          }
        }
        if (row < bs) *(u32x2_a4*)(rec + row * D + c * 8) = u32x2_a4{q.x, q.y};
      }
      // ---- values: per-token range over head_dim -------------------------------------------------------
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int row = t0 + r + R::RG * i;
        float x[8];
        v.widen(i, x);
        float lo = x[0], hi = x[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) {
          lo = fminf(lo, x[e]);
          hi = fmaxf(hi, x[e]);
        }
        lo = lkv::row_min<R::LPR>(lo);
        hi = lkv::row_max<R::LPR>(hi);
        const float vs = scale_of(lo, hi), vi = __builtin_amdgcn_rcpf(vs);
        float lo8[8], vs8[8], vi8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          lo8[e] = lo;
          vs8[e] = vs;
          vi8[e] = vi;
        }
        const uint2 q = quantise8(x, lo8, vs8, vi8);
        if (row < bs) {
          *(u32x2_a4*)(rec + bs * D + row * D + c * 8) = u32x2_a4{q.x, q.y};
          if (c == 0) {
            sc[2 * D + row] = lkv::f32_to_f16(vs);
            sc[2 * D + bs + row] = lkv::f32_to_f16(lo);
          }
        }
      }
    }
    if constexpr (META) {
      reduce_channels<R::LPR, GROUPS>(dmn, lane, lower);
      reduce_channels<R::LPR, GROUPS>(dmx, lane, upper);
      write_owned<D, R::LPR, GROUPS, false>(a, b, h, c, lane, dmn, dmx);
    }
  }
}

// A wave takes PPW (block, head) pairs at a time, the grid striding over the pairs. Waves never synchronise with
// each other, so a grid smaller than the pair count (a host destination) is just a longer loop.
template <int D, int MT, int MODE, bool META, int NI, int PPW, bool LONG>
__global__ __launch_bounds__(kThreads) void store_blocks_kernel(StoreArgs a) {
  const int64_t total = (int64_t)a.n_blocks * a.n_kv;
  constexpr int kLanes = 64 / PPW;
  for (int64_t pair = (int64_t)blockIdx.x * kWaves * PPW + threadIdx.x / kLanes; pair < total; pair += (int64_t)gridDim.x * kWaves * PPW)
    if constexpr (MODE == MODE_META_FROM_I8 || MODE == MODE_UNPACK) {
      store_record<D, MT, MODE>(a, pair);  // `pair` is wave-uniform
    } else {
      store_rows<D, MT, MODE, META, NI, PPW, LONG>(a, pair);  // uniform over kLanes lanes, which exchange with no others
    }
}

template <int D, int MT, int MODE, bool META, int NI, int PPW, bool LONG = false>
void launch_one(hipStream_t s, const StoreArgs& a, int64_t max_wgs) {
  const int64_t pairs = (int64_t)a.n_blocks * a.n_kv;
  int64_t wgs = (pairs + kWaves * PPW - 1) / (kWaves * PPW);
  if (wgs > max_wgs) wgs = max_wgs;
  hipLaunchKernelGGL((store_blocks_kernel<D, MT, MODE, META, NI, PPW, LONG>), dim3((unsigned)wgs), dim3(kThreads), 0, s, a);
}

// The instance for blocks of a.bs tokens: as many loads of RG rows as they fill, up to a 16-row chunk's, and two 4-token blocks in a
// load of 8 rows. (A whole chunk's loads for all: 65,536 pairs of 4 x 64 float16 packed with their metadata in 98 us, of 4 x 128 in 157;
// here in 43 and 82.)
template <int D, int MT, int MODE, bool META>
void launch_rows(hipStream_t s, const StoreArgs& a, int64_t max_wgs) {
  constexpr int RG = Rows<D, MT>::RG;
  if (MODE == MODE_INT8 && a.bs > 16) {
    if constexpr (MODE == MODE_INT8) launch_one<D, MT, MODE, META, 16 / RG, 1, true>(s, a, max_wgs);
  } else if (RG == 8 && a.bs <= 4) {
    if constexpr (RG == 8) launch_one<D, MT, MODE, META, 1, 2>(s, a, max_wgs > 1 ? max_wgs / 2 : 1);  // half the workgroups for a host budget
  } else if (a.bs <= RG) {
    launch_one<D, MT, MODE, META, 1, 1>(s, a, max_wgs);
  } else if (RG == 8 || a.bs <= 2 * RG) {
    launch_one<D, MT, MODE, META, 2, 1>(s, a, max_wgs);
  } else {
    if constexpr (RG == 4) launch_one<D, MT, MODE, META, 4, 1>(s, a, max_wgs);
  }
}

template <int D, int MT>
int launch_store(hipStream_t s, int mode, const StoreArgs& a, int64_t max_wgs) {
  const bool meta = a.kmin != nullptr;
  switch (mode) {
    case MODE_META: launch_rows<D, MT, MODE_META, true>(s, a, max_wgs); break;
    case MODE_COPY: meta ? launch_rows<D, MT, MODE_COPY, true>(s, a, max_wgs) : launch_rows<D, MT, MODE_COPY, false>(s, a, max_wgs); break;
    case MODE_INT8: meta ? launch_rows<D, MT, MODE_INT8, true>(s, a, max_wgs) : launch_rows<D, MT, MODE_INT8, false>(s, a, max_wgs); break;
    case MODE_UNPACK: launch_one<D, MT, MODE_UNPACK, true, 0, 1>(s, a, max_wgs); break;
    default: launch_one<D, MT, MODE_META_FROM_I8, true, 0, 1>(s, a, max_wgs); break;
  }
  LKV_CHECK_LAUNCH("store_blocks");
  return LKV_OK;
}

template <int D>
int launch_store_mt(hipStream_t s, int mt, int mode, const StoreArgs& a, int64_t max_wgs) {
  if (mt == LKV_BF16) return launch_store<D, LKV_BF16>(s, mode, a, max_wgs);
  if (mt == LKV_F16) return launch_store<D, LKV_F16>(s, mode, a, max_wgs);
  return launch_store<D, LKV_F32>(s, mode, a, max_wgs);
}

}  // namespace

extern "C" int lkv_store_blocks(uintptr_t stream, const lkv_kv_source* src, const lkv_kv_source* dst, int n_kv,
                                int head_dim, int block_size, int first_block, int n_blocks, void* kmin, void* kmax,
                                int meta_dtype, int64_t meta_head_stride) {
  LKV_CHECK_ARG(src != nullptr && src->k != nullptr, "source missing");
  LKV_CHECK_ARG(n_kv > 0 && n_blocks >= 0 && first_block >= 0, "bad block range");
  LKV_CHECK_ARG(head_dim == 64 || head_dim == 128, "head_dim %d unsupported (64 or 128)", head_dim);
  LKV_CHECK_ARG(block_size >= 4 && block_size <= 256 && block_size % 4 == 0,
                "block_size %d unsupported (a multiple of 4 up to 256)", block_size);
  LKV_CHECK_ARG((kmin == nullptr) == (kmax == nullptr), "kmin and kmax go together");
  LKV_CHECK_ARG((int64_t)first_block + n_blocks <= src->n_blocks, "blocks %d..%d outside the source (%lld blocks)",
                first_block, first_block + n_blocks, (long long)src->n_blocks);
  LKV_CHECK_ARG(dst == nullptr || (int64_t)first_block + n_blocks <= dst->n_blocks,
                "blocks %d..%d outside the destination", first_block, first_block + n_blocks);
  if (kmin) {
    LKV_CHECK_ARG(lkv_is_model_dtype(meta_dtype), "bad metadata dtype");
    LKV_CHECK_ARG(meta_head_stride >= (int64_t)(first_block + n_blocks) * head_dim, "metadata head stride too small");
  }
  int mode;
  int mt;
  if (src->dtype == LKV_INT8_RECORD) {
    mt = src->deq_dtype;
    if (dst == nullptr) {
      LKV_CHECK_ARG(kmin != nullptr, "nothing to do");
      mode = MODE_META_FROM_I8;
    } else {
      LKV_CHECK_ARG(dst->dtype == mt && dst->k != nullptr && dst->v != nullptr,
                    "int8 records dequantise into a destination of their model dtype");
      mode = MODE_UNPACK;
    }
  } else {
    LKV_CHECK_ARG(lkv_is_model_dtype(src->dtype) && src->v != nullptr, "bad source");
    mt = src->dtype;
    if (dst == nullptr) {
      LKV_CHECK_ARG(kmin != nullptr, "nothing to do");
      mode = MODE_META;
    } else if (dst->dtype == LKV_INT8_RECORD) {
      LKV_CHECK_ARG(dst->k != nullptr, "destination missing");
      mode = MODE_INT8;
    } else {
      LKV_CHECK_ARG(dst->dtype == src->dtype && dst->k && dst->v, "copy destination must match the source dtype");
      mode = MODE_COPY;
    }
  }
  LKV_CHECK_ARG(lkv_is_model_dtype(mt), "bad model dtype");
  if (kmin && mode != MODE_META && mode != MODE_COPY) {
    LKV_CHECK_ARG(meta_dtype == mt, "metadata of dequantised keys must be in the model dtype");
  }
  if (n_blocks == 0) return LKV_OK;
  StoreArgs a{};
  a.sk = src->k;
  a.sv = src->v;
  a.s_bstride = src->block_stride;
  a.s_hstride = src->head_stride;
  if (dst) {
    a.dk = const_cast<void*>(dst->k);
    a.dv = const_cast<void*>(dst->v);
    a.d_bstride = dst->block_stride;
    a.d_hstride = dst->head_stride;
  }
  a.n_kv = n_kv;
  a.bs = block_size;
  a.first_block = first_block;
  a.n_blocks = n_blocks;
  a.kmin = kmin;
  a.kmax = kmax;
  a.meta_dtype = meta_dtype;
  a.meta_hstride = meta_head_stride;
  // A host-memory source or destination: a grid that keeps the host budget in flight, one pair
  // per wave (the kernel strides over the rest).
  int64_t max_wgs = INT64_MAX;
  const lkv_kv_source* host_side = (dst && (dst->flags & LKV_SRC_HOST)) ? dst : ((src->flags & LKV_SRC_HOST) ? src : nullptr);
  if (host_side) {
    const double budget = host_side == dst ? lkv_host_write_inflight() : lkv_host_read_inflight();
    max_wgs = (int64_t)(budget / ((double)kWaves * (double)lkv_pair_bytes(host_side, block_size, head_dim)));
    if (max_wgs < 1) max_wgs = 1;
  }
  hipStream_t s = (hipStream_t)stream;
  return head_dim == 128 ? launch_store_mt<128>(s, mt, mode, a, max_wgs) : launch_store_mt<64>(s, mt, mode, a, max_wgs);
}

// ---- small row copies -----------------------------------------------------------------------------------
// Up to 8 copies in one launch. Small ones are bound by the
// launch: with six separate copies behind its store, a 200-token turn over a 64K-token tier (8 heads, d 128) took
// 120.7 us, with one launch 102.6. (For two copies, torch's cost the host less: appending a token 17.2 us against 18.3.)
namespace {

struct RowCopies {
  lkv_row_copy c[LKV_MAX_ROW_COPIES];
  int32_t end[LKV_MAX_ROW_COPIES];  // workgroups up to and including copy i's
};

// A workgroup per 256 words of its copy, the copies one after another. (As a grid axis of their own, as long as the longest, a turn of
// 65,536 tokens beside the sink and the current block, 8 heads at d 128, launched 131,072 workgroups with nothing to do: 117.0 us by torch's
// copies, 120.6 so, 94.5
// here.)
template <typename W>
__global__ __launch_bounds__(256) void copy_rows_kernel(RowCopies a) {
  const int g = blockIdx.x;
  int n = 0, first = 0;
#pragma unroll
  for (int i = 0; i + 1 < LKV_MAX_ROW_COPIES; ++i) {
    if (g >= a.end[i]) {
      n = i + 1;
      first = a.end[i];
    }
  }
  const lkv_row_copy& c = a.c[n];
  const uint32_t words = (uint32_t)c.row_bytes / (uint32_t)sizeof(W);
  const int64_t i = (int64_t)(g - first) * 256 + threadIdx.x;
  if (i >= (int64_t)c.rows * words) return;
  int64_t row, w;
  if ((int64_t)c.rows * words <= 0xffffffffLL) {  // workgroup-uniform: a 64-bit division costs several of 32
    row = (uint32_t)i / words;
    w = (uint32_t)i % words;
  } else {
    row = i / words;
    w = i % words;
  }
  const char* s = (const char*)c.src + blockIdx.y * c.src_head_stride + row * c.src_row_stride;
  char* d = (char*)c.dst + blockIdx.y * c.dst_head_stride + row * c.dst_row_stride;
  ((W*)d)[w] = ((const W*)s)[w];
}

}  // namespace

extern "C" int lkv_copy_rows(uintptr_t stream, const lkv_row_copy* copies, int n, int heads) {
  LKV_CHECK_ARG(n >= 0 && n <= LKV_MAX_ROW_COPIES, "%d row copies: at most %d", n, LKV_MAX_ROW_COPIES);
  LKV_CHECK_ARG(n == 0 || copies != nullptr, "NULL pointer");
  LKV_CHECK_ARG(heads > 0 && heads <= 65535, "bad head count %d", heads);
  RowCopies a{};
  int used = 0;
  uint64_t mix = 0;  // the low bits set anywhere decide the word
  for (int i = 0; i < n; ++i) {
    const lkv_row_copy& c = copies[i];
    LKV_CHECK_ARG(c.rows >= 0 && c.row_bytes >= 0, "negative size");
    if (c.rows == 0 || c.row_bytes == 0) continue;
    LKV_CHECK_ARG(c.src != nullptr && c.dst != nullptr, "NULL pointer");
    mix |= (uint64_t)(uintptr_t)c.src | (uint64_t)(uintptr_t)c.dst | (uint64_t)c.src_head_stride | (uint64_t)c.src_row_stride |
           (uint64_t)c.dst_head_stride | (uint64_t)c.dst_row_stride | (uint64_t)c.row_bytes;
    a.c[used++] = c;
  }
  LKV_CHECK_ARG((mix & 1) == 0, "row copies move whole 2-byte elements");
  if (used == 0) return LKV_OK;
  const int word = (mix & 15) == 0 ? 16 : (mix & 3) == 0 ? 4 : 2;
  int64_t groups = 0;
  for (int i = 0; i < LKV_MAX_ROW_COPIES; ++i) {
    if (i < used) groups += ((int64_t)a.c[i].rows * (a.c[i].row_bytes / word) + 255) / 256;
    LKV_CHECK_ARG(groups <= 0x7fffffff, "row copy too large");
    a.end[i] = (int32_t)groups;
  }
  const dim3 grid((unsigned)groups, (unsigned)heads);
  hipStream_t s = (hipStream_t)stream;
  if (word == 16) {
    hipLaunchKernelGGL(copy_rows_kernel<uint4>, grid, dim3(256), 0, s, a);
  } else if (word == 4) {
    hipLaunchKernelGGL(copy_rows_kernel<uint32_t>, grid, dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL(copy_rows_kernel<uint16_t>, grid, dim3(256), 0, s, a);
  }
  LKV_CHECK_LAUNCH("copy_rows");
  return LKV_OK;
}

extern "C" int lkv_pack_int8(uintptr_t stream, const void* pairs, int dtype, int64_t m, int block_size, int head_dim,
                             void* records) {
  LKV_CHECK_ARG(pairs != nullptr && records != nullptr, "NULL pointer");
  LKV_CHECK_ARG(m >= 0 && m <= 0x7fffffff, "bad record count");
  LKV_CHECK_ARG(lkv_is_model_dtype(dtype), "bad dtype");
  const int64_t pair_elems = 2LL * block_size * head_dim;
  lkv_kv_source src{pairs, (const char*)pairs + (int64_t)block_size * head_dim * lkv_dtype_size(dtype), pair_elems, 0,
                    m, dtype, dtype};
  lkv_kv_source dst{records, nullptr, lkv_packed_pair_bytes(block_size, head_dim), 0, m, LKV_INT8_RECORD, dtype};
  return lkv_store_blocks(stream, &src, &dst, 1, head_dim, block_size, 0, (int)m, nullptr, nullptr, dtype, 0);
}

extern "C" int lkv_unpack_int8(uintptr_t stream, const void* records, int64_t m, int block_size, int head_dim,
                               int dtype, void* pairs) {
  LKV_CHECK_ARG(pairs != nullptr && records != nullptr, "NULL pointer");
  LKV_CHECK_ARG(m >= 0, "bad record count");
  LKV_CHECK_ARG(head_dim == 64 || head_dim == 128, "head_dim %d unsupported (64 or 128)", head_dim);
  LKV_CHECK_ARG(block_size >= 4 && block_size <= 256 && block_size % 4 == 0,
                "block_size %d unsupported (a multiple of 4 up to 256)", block_size);
  LKV_CHECK_ARG(lkv_is_model_dtype(dtype), "bad dtype");
  LKV_CHECK_ARG(m <= 0x7fffffff, "bad record count");
  // Records [m, P] as m blocks of one head, dequantised into pairs [m, 2, bs, d].
  const int64_t pair_elems = 2LL * block_size * head_dim;
  lkv_kv_source src{records, nullptr, lkv_packed_pair_bytes(block_size, head_dim), 0, m, LKV_INT8_RECORD, dtype, 0};
  lkv_kv_source dst{pairs, (const char*)pairs + (int64_t)block_size * head_dim * lkv_dtype_size(dtype), pair_elems, 0, m,
                    dtype, dtype, 0};
  return lkv_store_blocks(stream, &src, &dst, 1, head_dim, block_size, 0, (int)m, nullptr, nullptr, dtype, 0);
}
