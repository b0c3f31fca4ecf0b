// MiniMax index block scores over the NVFP4 index K: the scores SGLang's top-k selection of KV blocks reads
// (kv_fp4.py:168-222 decode, :407-446 prefill). The index pool holds one key head per slot: payload bytes
// [pages, 128 slots, d/2] (element 2i in the low nibble of byte i) and E4M3 scale bytes [pages, 128, d/16]
// (element j uses scale j / 16), unit global scale; a slot s lives on page s / 128, row s % 128.
//
//   score of key position p for head h = (q_h . k_p) * c with c = (sm_scale * log2(e)) * k_scale in FP32.
//   decode: per request, head and block of block_size positions, the maximum (or log2-sum-exp2) of the scores of the
//     block's positions below seq_len; the last local_blocks blocks read 1e29, else the first init_blocks 1e30.
//   prefill: per query row, head and block, the maximum over the block's positions at or before the row's own
//     position (prefix_len + row), -inf when there are none; a row gets the blocks below
//     min(seq_len, prefix_len + 64 (row / 64 + 1)), the 64-row tile bound of the reference's grid.
//
// Numerics: e2m1 * e4m3 has at most 6 significant bits, so every key value is exact in FP32 and in BF16 (FP16 for an
// FP16 query); v_mfma_f32_32x32x16_{bf16,f16} sums the exact products in FP32. The MFMA takes keys as rows
// (A = 32 keys x 16 dims) and query columns as columns (B = 16 dims x 32 columns); a lane then holds 16 keys of one
// column, so the block maximum is 15 VALU maxima in the lane and one exchange with the lane 32 apart. The dims of a
// lane half h are h d/2 .. h d/2 + d/2 - 1 (k-step kk covers h d/2 + 8 kk .. + 7 in both operands), so a lane reads
// one contiguous run of each key's payload.
#include "xt_common.h"
#include "xt_host.h"

#include <type_traits>

namespace xt {
namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kPoolRows = 128;   // slots per page of the index pool
constexpr int kScoreWaves = 4;

// index arrays given as int32 or int64 (bit i of `wide` set: argument i is int64)
enum : int { kWideR2t = 1, kWideSeq = 2, kWideSlot = 4, kWidePrefix = 8, kWideCu = 16, kOpenEnd = 32 };

__device__ inline int64_t load_index(const void* p, int64_t i, bool wide) {
  return wide ? static_cast<const int64_t*>(p)[i] : (int64_t) static_cast<const int32_t*>(p)[i];
}

// slot -> [0, max_slots): (s + max_slots) % max_slots for the reference's range s >= -max_slots, and kept in range
// for any other value. Slots already in range skip the 64-bit division (about 100 instructions, once per key).
__device__ inline int64_t wrap_slot(int64_t s, int64_t max_slots) {
  if ((uint64_t)s < (uint64_t)max_slots) return s;
  const int64_t r = s % max_slots;
  return r < 0 ? r + max_slots : r;
}

struct ScoreArgs {
  const uint16_t* q;          // decode [batch, heads, d]; prefill [total_q, heads, d] (BF16 / FP16, d contiguous)
  int64_t q_ns, q_hs;         // element strides of a row (request / token) and a head
  const uint8_t* pay;         // index payload
  int64_t pay_ps, pay_rs;     // byte strides of a page and a slot row
  const uint8_t* sc;          // index scale bytes
  int64_t sc_ps, sc_rs;
  int64_t max_slots;          // pages * 128
  const void* r2t;            // req_to_token [reqs, width]
  int64_t r2t_stride;
  const void* seq_lens;
  const void* slot_ids;
  const void* prefix_lens;    // prefill
  const void* cu_seqlens;     // prefill [batch + 1]
  int wide;
  void* score;                // decode [heads, batch, blocks]; prefill [heads, total_q, blocks] (element strides)
  int64_t s_hs, s_ns, s_ks;
  int out_dtype;              // 0 FP32, 1 BF16, 2 FP16
  int batch, heads, block_size;
  float c;
  int init_blocks, local_blocks;
  int skip_topk;              // decode: a request with at most this many blocks gets no scores (-1: none skipped)
  int lse;                    // decode: log2-sum-exp2 instead of the maximum
  int chunks;                 // prefill: block ranges per row tile (grid x = row tiles * chunks)
  int chunk_blocks;           // prefill: blocks per range
};

__device__ inline void store_score(const ScoreArgs& a, int64_t at, float v) {
  if (a.out_dtype == 0)
    static_cast<float*>(a.score)[at] = v;
  else if (a.out_dtype == 1)
    static_cast<uint16_t*>(a.score)[at] = (uint16_t)f32_to_bf16_bits(v);
  else
    static_cast<uint16_t*>(a.score)[at] = (uint16_t)f32_to_f16_bits(v);
}

// Eight E2M1 codes (one dword, low nibble first) times the FP32 scale `sf`, as eight exact 16-bit values.
template <bool BF>
__device__ inline u32x4_t fp4x8_scaled(uint32_t w, float sf) {
  u32x4_t r;
  if constexpr (BF) {
    // the products are exact in FP32 with zero low halves, so their high halves are the BF16 values
#define XT_PAIR(E)                                                                                                 \
  {                                                                                                                \
    const float2_t v = fp4x2_to_f32<E>(w);                                                                         \
    r[E] = __builtin_amdgcn_perm(__float_as_uint(v.y * sf), __float_as_uint(v.x * sf), 0x07060302u);              \
  }
    XT_PAIR(0) XT_PAIR(1) XT_PAIR(2) XT_PAIR(3)
#undef XT_PAIR
  } else {
    const half2_t s2 = {(_Float16)sf, (_Float16)sf};
    r[0] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<0>(w) * s2);
    r[1] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<1>(w) * s2);
    r[2] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<2>(w) * s2);
    r[3] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<3>(w) * s2);
  }
  return r;
}

// The codes alone, without a scale.
template <bool BF>
__device__ inline u32x4_t fp4x8_plain(uint32_t w) {
  u32x4_t r;
  if constexpr (BF) {
    r[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0));
    r[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1));
    r[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2));
    r[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3));
  } else {
    r[0] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<0>(w));
    r[1] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<1>(w));
    r[2] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<2>(w));
    r[3] = __builtin_bit_cast(uint32_t, fp4x2_to_f16<3>(w));
  }
  return r;
}

template <bool BF>
__device__ inline float16_t mfma16(u32x4_t a, u32x4_t b, float16_t c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c,
                                                  0, 0, 0);
}

__device__ inline float scale_of(uint32_t byte) {
  return (float)fp8x2_to_f16<false>(byte)[0];
}

__device__ inline float swap32_max(float x) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ inline float swap32_sum(float x) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// ---------------------------------------------------------------------------------------------------------------
// Decode: grid (x, request b, head group of 32); wavefront w of workgroup x takes blocks x * 4 + w, + 4 gridDim.x,
// ... of its request; T = block_size / 32 key tiles per block, all held until the block's reduction.

template <int NK, int T, bool BF>
__global__ __launch_bounds__(64 * kScoreWaves) void decode_scores_kernel(const ScoreArgs a) {
  constexpr int D = 16 * NK;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int b = blockIdx.y;
  const int64_t seq = load_index(a.seq_lens, b, a.wide & kWideSeq);
  const int64_t nb = (seq + 32 * T - 1) / (32 * T);
  if (a.skip_topk >= 0 && nb <= a.skip_topk) return;
  int64_t blk = (int64_t)blockIdx.x * kScoreWaves + wave;
  if (blk >= nb) return;   // no barrier below
  const int64_t sid = wrap_slot(load_index(a.slot_ids, b, a.wide & kWideSlot), a.max_slots);
  const int head = 32 * blockIdx.z + j;
  const bool live_head = head < a.heads;
  // B = this lane's query column (head), dims h d/2 + 8 kk .. + 7
  u32x4_t qv[NK];
  {
    const uint16_t* qp = a.q + (int64_t)b * a.q_ns + (int64_t)(live_head ? head : 0) * a.q_hs + h * (D / 2);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qv[kk] = live_head ? *reinterpret_cast<const u32x4_t*>(qp + 8 * kk) : u32x4_t{0, 0, 0, 0};
  }
  const int64_t local_start = nb - a.local_blocks > 0 ? nb - a.local_blocks : 0;
  const bool wide_r2t = a.wide & kWideR2t;
  for (; blk < nb; blk += (int64_t)gridDim.x * kScoreWaves) {
    float16_t acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int64_t pos = blk * (32 * T) + 32 * t + j;
      const int64_t slot = pos < seq ? wrap_slot(load_index(a.r2t, sid * a.r2t_stride + pos, wide_r2t), a.max_slots) : 0;
      const uint8_t* pp = a.pay + (slot >> 7) * a.pay_ps + (slot & (kPoolRows - 1)) * a.pay_rs + h * (D / 4);
      const uint8_t* sp = a.sc + (slot >> 7) * a.sc_ps + (slot & (kPoolRows - 1)) * a.sc_rs + h * (D / 32);
      uint32_t pw[NK];
#pragma unroll
      for (int i = 0; i < NK / 4; ++i) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(pp + 16 * i);
        pw[4 * i] = v[0]; pw[4 * i + 1] = v[1]; pw[4 * i + 2] = v[2]; pw[4 * i + 3] = v[3];
      }
      uint64_t sw;
      if constexpr (NK == 4) sw = *reinterpret_cast<const uint16_t*>(sp);
      else if constexpr (NK == 8) sw = *reinterpret_cast<const uint32_t*>(sp);
      else sw = *reinterpret_cast<const uint64_t*>(sp);
      float16_t s = {};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        s = mfma16<BF>(fp4x8_scaled<BF>(pw[kk], scale_of((uint32_t)(sw >> (8 * (kk / 2))) & 0xFFu)), qv[kk], s);
      acc[t] = s;
    }
    // C rows: keys 32 t + 8 (r / 4) + 4 h + r % 4 of the block; scaled, -inf at and past seq_len
    float m = -__builtin_inff();
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t pos = blk * (32 * T) + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
        acc[t][r] = pos < seq ? acc[t][r] * a.c : -__builtin_inff();
        m = fmaxf(m, acc[t][r]);
      }
    m = swap32_max(m);
    float score = m;
    if (a.lse) {
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += exp2f(acc[t][r] - m);
      score = m + log2f(swap32_sum(sum));
      if (score != score) score = -__builtin_inff();
    }
    if (blk >= local_start) score = 1e29f;
    else if (blk < a.init_blocks) score = 1e30f;
    if (h == 0 && live_head) store_score(a, (int64_t)head * a.s_hs + (int64_t)b * a.s_ns + blk * a.s_ks, score);
  }
}

// Decode for at most 32 / NK heads (4 at 128 dims): the 32 rows of the MFMA's A operand are (head, 16-dim scale block)
// pairs, the query block-diagonal: row (head, b) holds the head's query in block b's dims and 0 elsewhere. B is the
// unscaled key tile (one conversion per two values), and C holds, for one key per lane, the partial dot product of
// every head and of the lane half's NK / 2 blocks, so the block scales enter as one FMA per (head, block) in FP32
// (E4M3 values, exact). The kernel above multiplies every key value by its scale and spends its columns past `heads`
// on nothing. Work split as above; the next block's slots are looked up behind the current block's loads. Bound: HBM,
// 76 bytes per key at 128 dims. 32 requests x 32768 keys, 4 heads: 20.8 us (3.8 TB/s) against 28.4 us for the kernel
// above (22.1 us at 152 registers, three wavefronts per SIMD, hence the four in the launch bounds at up to 4 tiles).
// A lane half's NK / 2 scale bytes, as loaded and as FP32.
template <int NK>
using ScaleWord = std::conditional_t<NK == 4, uint16_t, std::conditional_t<NK == 8, uint32_t, uint64_t>>;
template <int NK>
__device__ inline void key_scales(ScaleWord<NK> w, float (&f)[NK / 2]) {
#pragma unroll
  for (int i = 0; i < NK / 4; ++i) {
    const half2_t v = fp8x2_to_f16<false>((uint32_t)(w >> (16 * i)));
    f[2 * i] = (float)v[0];
    f[2 * i + 1] = (float)v[1];
  }
}

template <int CTRL>
__device__ inline float dpp(float x) {   // x of the lane the DPP control names (row rotations: always a live lane)
  return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), CTRL, 0xF, 0xF, true));
}
// Maximum and sum over the 32 lanes of a wavefront half (row rotations by 8, 4, 2, 1, then the row 16 apart).
__device__ inline float half_max(float x) {
  x = fmaxf(x, dpp<0x128>(x)); x = fmaxf(x, dpp<0x124>(x)); x = fmaxf(x, dpp<0x122>(x)); x = fmaxf(x, dpp<0x121>(x));
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ inline float half_sum(float x) {
  x += dpp<0x128>(x); x += dpp<0x124>(x); x += dpp<0x122>(x); x += dpp<0x121>(x);
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

template <int NK, int T>   // wavefronts per SIMD that the registers leave
constexpr int kFewWaves = NK <= 8 && T <= 4 ? 4 : NK * T >= 128 ? 1 : 2;

template <int NK, int T, bool BF>
__global__ __launch_bounds__(64 * kScoreWaves, (kFewWaves<NK, T>)) void decode_scores_few_kernel(const ScoreArgs a) {
  constexpr int D = 16 * NK, NB = NK / 2, H = 16 / NB;   // scale blocks of a lane half; heads
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int b = blockIdx.y;
  const int64_t seq = load_index(a.seq_lens, b, a.wide & kWideSeq);
  const int64_t nb = (seq + 32 * T - 1) / (32 * T);
  if (a.skip_topk >= 0 && nb <= a.skip_topk) return;
  int64_t blk = (int64_t)blockIdx.x * kScoreWaves + wave;
  if (blk >= nb) return;   // no barrier below
  const int64_t sid = wrap_slot(load_index(a.slot_ids, b, a.wide & kWideSlot), a.max_slots);
  const int64_t r2t_row = sid * a.r2t_stride;
  const bool wide_r2t = a.wide & kWideR2t;
  int64_t slot[T];
  auto load_slots = [&](int64_t at) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int64_t pos = at * (32 * T) + 32 * t + j;
      slot[t] = pos < seq ? load_index(a.r2t, r2t_row + pos, wide_r2t) : 0;
    }
  };
  load_slots(blk);
  // A: C row 8 (r / 4) + 4 half + r % 4 (r = 0 .. 15) is head r / NB, block NB half + r % NB, so that a lane's C rows
  // are the blocks of its own half. k-step kk covers dims h d/2 + 8 kk .. + 7 (block NB h + kk / 2) in both operands.
  const int r_row = 4 * (j >> 3) + (j & 3), q_head = r_row / NB, q_blk = r_row % NB;
  const bool own = ((j >> 2) & 1) == h && q_head < a.heads;
  u32x4_t qv[NK];
  {
    const uint16_t* qp = a.q + (int64_t)b * a.q_ns + (int64_t)(own ? q_head : 0) * a.q_hs + h * (D / 2) + 16 * q_blk;
    const u32x4_t q0 = *reinterpret_cast<const u32x4_t*>(qp), q1 = *reinterpret_cast<const u32x4_t*>(qp + 8);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) qv[kk] = own && kk / 2 == q_blk ? (kk & 1 ? q1 : q0) : u32x4_t{0, 0, 0, 0};
  }
  const int64_t local_start = nb - a.local_blocks > 0 ? nb - a.local_blocks : 0;
  for (; blk < nb; blk += (int64_t)gridDim.x * kScoreWaves) {
    // every load of the block first, then the next block's slots
    u32x4_t pw[T][NK / 4];
    ScaleWord<NK> sw[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int64_t s = wrap_slot(slot[t], a.max_slots);
      const uint8_t* pp = a.pay + (s >> 7) * a.pay_ps + (s & (kPoolRows - 1)) * a.pay_rs + h * (D / 4);
      sw[t] = *reinterpret_cast<const ScaleWord<NK>*>(a.sc + (s >> 7) * a.sc_ps + (s & (kPoolRows - 1)) * a.sc_rs +
                                                      h * (D / 32));
#pragma unroll
      for (int i = 0; i < NK / 4; ++i) pw[t][i] = *reinterpret_cast<const u32x4_t*>(pp + 16 * i);
    }
    const int64_t next = blk + (int64_t)gridDim.x * kScoreWaves;
    if (next < nb) load_slots(next);
    const int64_t left = seq - blk * (32 * T);   // live keys of the block
    float v[T][H], m[H];
#pragma unroll
    for (int i = 0; i < H; ++i) m[i] = -__builtin_inff();
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float sc[NB];
      key_scales<NK>(sw[t], sc);
      float16_t s = {};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) s = mfma16<BF>(qv[kk], fp4x8_plain<BF>(pw[t][kk / 4][kk % 4]), s);
#pragma unroll
      for (int i = 0; i < H; ++i) {
        float x = s[NB * i] * sc[0];
#pragma unroll
        for (int k = 1; k < NB; ++k) x = __builtin_fmaf(s[NB * i + k], sc[k], x);
        x = swap32_sum(x);
        v[t][i] = 32 * t + j < left ? x * a.c : -__builtin_inff();
        m[i] = fmaxf(m[i], v[t][i]);
      }
    }
    float score = 0.0f;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      float r = half_max(m[i]);
      if (a.lse) {
        float sum = 0.0f;
#pragma unroll
        for (int t = 0; t < T; ++t) sum += exp2f(v[t][i] - r);
        r += log2f(half_sum(sum));
        if (r != r) r = -__builtin_inff();
      }
      score = j == i ? r : score;
    }
    if (blk >= local_start) score = 1e29f;
    else if (blk < a.init_blocks) score = 1e30f;
    if (lane < min(H, a.heads)) store_score(a, (int64_t)lane * a.s_hs + (int64_t)b * a.s_ns + blk * a.s_ks, score);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Prefill: grid (row tile x block range, request b, head group of HPW heads); a workgroup covers R = 128 G / HPW query
// rows of request b and one range of chunk_blocks blocks (the per-block results are independent, so ranges split a
// long prompt's work over many workgroups). Column j of wavefront w's column group g is (row (32 / HPW)(G w + g) +
// j / HPW, head j % HPW). Key chunks of SK = kStageKeys positions are staged as 16-bit values in LDS by the whole
// workgroup (two threads per key, once for its 128 G columns), then each wavefront runs its G column groups over them.
// SHORT: blocks shorter than a chunk, which ends them tile by tile; a chunk per block, 32 keys, had left three quarters
// of the threads idle while staging and made 64 dims slower than one LDS stage (4 heads x 8192 rows against 38192 keys
// in blocks of 32: 466 us, 352 us now; 128 dims 510 us, 446 us).
// Two LDS stages: while one is computed on, the next chunk's payload and scales are in flight to registers and the
// slots of the one after are being looked up, and one barrier per chunk suffices. Chunks wholly at or below every row's
// position skip the causal test and scale once after the maximum (c > 0: the maximum commutes with the rounding of the
// product).
// Bound: the matrix cores, with the staging's conversions and LDS reads beside them, so G = 4 shares each staged key
// and each LDS read among twice the columns. 4096 rows x 4 heads against 65536 keys at 128 dims (266 GFLOP): 235 us
// (1130 TFLOP/s) against 400 us for one LDS stage, G = 2 and a 64-bit division per staged piece.

template <int NK>
constexpr int kStageKeys = NK <= 8 ? 128 : 64;

template <int NK, int HPW, int G, bool BF, bool SHORT>
__global__ __launch_bounds__(64 * kScoreWaves, 2) void prefill_scores_kernel(const ScoreArgs a) {
  constexpr int D = 16 * NK;
  constexpr int ROW_U32 = D / 2 + 4;          // LDS row: D 16-bit values + 16 bytes of padding
  constexpr int R = 128 * G / HPW;            // rows per workgroup
  constexpr int RG = 32 / HPW;                // rows per column group
  constexpr int SK = kStageKeys<NK>;
  __shared__ uint32_t lds[2][SK * ROW_U32];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5, tid = threadIdx.x;
  const int b = blockIdx.y;
  const int64_t q0 = load_index(a.cu_seqlens, b, a.wide & kWideCu);
  const int64_t q_len = load_index(a.cu_seqlens, b + 1, a.wide & kWideCu) - q0;
  const int tiles = (int)gridDim.x / a.chunks, chunk = (int)blockIdx.x % a.chunks;
  const int64_t row0 = (int64_t)(tiles - 1 - (int)blockIdx.x / a.chunks) * R;   // the longest rows first
  if (row0 >= q_len) return;   // uniform over the workgroup: before every barrier
  const int64_t seq = load_index(a.seq_lens, b, a.wide & kWideSeq);
  const int64_t pre = load_index(a.prefix_lens, b, a.wide & kWidePrefix);
  const int64_t sid = wrap_slot(load_index(a.slot_ids, b, a.wide & kWideSlot), a.max_slots);
  const int bs = a.block_size;
  // the workgroup's block count: that of its last live row (block counts grow with the row)
  const int64_t last = min(q_len, row0 + R) - 1;
  const int64_t wg_blocks = (min(seq, pre + 64 * (last / 64 + 1)) + bs - 1) / bs;
  const int64_t blk_lo = (int64_t)chunk * a.chunk_blocks, blk_hi = min(wg_blocks, blk_lo + a.chunk_blocks);
  if (blk_lo >= wg_blocks) return;   // uniform: before every barrier
  const bool wide_r2t = a.wide & kWideR2t;
  const int S = SHORT ? SK : bs < SK ? bs : SK;
  const int parts = bs / (SHORT ? 32 : S);                // 32-key tiles or chunks per block
  const int keys = (int)(blk_hi - blk_lo) * bs;
  const int n_chunks = SHORT ? (keys + S - 1) / S : (int)(blk_hi - blk_lo) * parts;
  const int64_t pos_lo = blk_lo * bs;                     // first position of the range
  const int64_t r2t_row = sid * a.r2t_stride;
  // staging: thread 2 key + half takes that half of the key's dims
  const int s_key = tid >> 1, s_half = tid & 1;
  const bool stager = s_key < S;
  auto slot_at = [&](int n) -> int64_t {   // of this thread's key in chunk n; positions past the row read slot 0
    const int64_t pos = pos_lo + (int64_t)n * S + s_key;
    return stager && n < n_chunks && pos < seq ? load_index(a.r2t, r2t_row + pos, wide_r2t) : 0;
  };
  u32x4_t raw[NK / 4];
  ScaleWord<NK> raw_sc;
  auto load_raw = [&](int64_t slot) {
    const int64_t s = wrap_slot(slot, a.max_slots);
    const uint8_t* pp = a.pay + (s >> 7) * a.pay_ps + (s & (kPoolRows - 1)) * a.pay_rs + s_half * (D / 4);
    const uint8_t* sp = a.sc + (s >> 7) * a.sc_ps + (s & (kPoolRows - 1)) * a.sc_rs + s_half * (D / 32);
#pragma unroll
    for (int i = 0; i < NK / 4; ++i) raw[i] = *reinterpret_cast<const u32x4_t*>(pp + 16 * i);
    raw_sc = *reinterpret_cast<const ScaleWord<NK>*>(sp);
  };
  int64_t slot_next = slot_at(0);
  // rows of this lane's columns, their block counts, and last visible position relative to pos_lo
  int nblk[G], vis[G];
  u32x4_t qv[G][NK];
  const int head = HPW * blockIdx.z + (j % HPW);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t row = row0 + RG * (G * wave + g) + j / HPW;
    const bool live = row < q_len && head < a.heads;
    const int64_t hi = min(seq, pre + 64 * (row / 64 + 1));
    nblk[g] = live ? (int)(min((hi + bs - 1) / bs, blk_hi) - blk_lo) : 0;
    vis[g] = (int)max((int64_t)-1, min(min(pre + row, seq - 1) - pos_lo, (int64_t)0x7FFFFFFF));
    const uint16_t* qp = a.q + (q0 + (live ? row : 0)) * a.q_ns + (int64_t)(live ? head : 0) * a.q_hs + h * (D / 2);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qv[g][kk] = live ? *reinterpret_cast<const u32x4_t*>(qp + 8 * kk) : u32x4_t{0, 0, 0, 0};
  }
  // chunks (SHORT: tiles) before this one are at or below every row's position and below seq_len, whole
  const int64_t whole = a.c > 0.0f ? max((int64_t)0, min(pre + row0 + 1, seq) - pos_lo) / (SHORT ? 32 : S) : 0;
  load_raw(slot_next);
  slot_next = slot_at(1);
  // scaled maxima of masked chunks, raw maxima of unmasked ones (with c <= 0 there are none: c times none is -inf, or
  // NaN)
  float m[G], mr[G];
  const float none = a.c > 0.0f ? -__builtin_inff() : __builtin_inff();
#pragma unroll
  for (int g = 0; g < G; ++g) m[g] = -__builtin_inff(), mr[g] = none;
  // The block is complete: max(round(c x)) = round(c max(x)) for c > 0. (As a lambda it took registers from the long
  // form's loop, 1 %.)
#define XT_BLOCK_DONE                                                                                                \
  do {                                                                                                               \
    _Pragma("unroll") for (int g = 0; g < G; ++g) {                                                                  \
      const float v = swap32_max(fmaxf(m[g], mr[g] * a.c));                                                          \
      const int64_t row = row0 + RG * (G * wave + g) + j / HPW;                                                      \
      if (h == 0 && bi < nblk[g])                                                                                    \
        store_score(a, (int64_t)head * a.s_hs + (q0 + row) * a.s_ns + (blk_lo + bi) * a.s_ks, v);                    \
      m[g] = -__builtin_inff(), mr[g] = none;                                                                        \
    }                                                                                                                \
    sub = 0;                                                                                                         \
    ++bi;                                                                                                            \
  } while (0)
  for (int n = 0, sub = 0, bi = 0; n < n_chunks; ++n) {
    uint32_t* buf = lds[n & 1];
    if (stager) {
      uint32_t* dst = &buf[s_key * ROW_U32 + s_half * (D / 4)];
      float scf[NK / 2];
      key_scales<NK>(raw_sc, scf);
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        *reinterpret_cast<u32x4_t*>(dst + 4 * kk) = fp4x8_scaled<BF>(raw[kk / 4][kk % 4], scf[kk / 2]);
    }
    if (n + 1 < n_chunks) {
      load_raw(slot_next);
      slot_next = slot_at(n + 2);
    }
    __syncthreads();   // chunk n is staged; every wavefront is past chunk n - 1, whose buffer chunk n + 1 takes
    const int tiles32 = (SHORT ? min(S, keys - n * S) : S) / 32;
    bool unmasked = n < whole;
    for (int t = 0; t < tiles32; ++t) {
      if (SHORT) unmasked = n * (SK / 32) + t < whole;
      float16_t s[G];
#pragma unroll
      for (int g = 0; g < G; ++g) s[g] = float16_t{};
      const uint32_t* kp = &buf[(32 * t + j) * ROW_U32 + h * (D / 4)];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const u32x4_t kv = *reinterpret_cast<const u32x4_t*>(kp + 4 * kk);
#pragma unroll
        for (int g = 0; g < G; ++g) s[g] = mfma16<BF>(kv, qv[g][kk], s[g]);
      }
      if (unmasked) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int r = 0; r < 16; ++r) mr[g] = fmaxf(mr[g], s[g][r]);
      } else {
        // a key counts for a row at or after it, below seq_len
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int lim = vis[g] - (n * S + 32 * t + 4 * h);
#pragma unroll
          for (int r = 0; r < 16; ++r)
            m[g] = fmaxf(m[g], 8 * (r >> 2) + (r & 3) <= lim ? s[g][r] * a.c : -__builtin_inff());
        }
      }
      if (SHORT && ++sub == parts) XT_BLOCK_DONE;
    }
    if (!SHORT && ++sub == parts) XT_BLOCK_DONE;
  }
#undef XT_BLOCK_DONE
}

// ---------------------------------------------------------------------------------------------------------------
// The per-row arguments of a ragged block-sparse prefill (kv_fp4.py:384-400 derives them per program): thread = row. A
// row at or past cu_seqlens[batch] is no request's and gets no keys, unless the last request's end is open.

struct RowArgs {
  const void *cu_seqlens, *slot_ids, *prefix_lens, *seq_lens;   // [batch + 1] ([batch], open end), [batch] ...
  const int64_t* cu_blocks;   // [batch] query blocks before each request, or NULL: from cu_seqlens
  int wide;
  int batch, rows, block_q;
  int64_t max_slots;
  int reqs, width, list_rows;   // req_to_token rows and columns, list rows: upper bounds
  int64_t* row_req;
  int32_t *row_seq, *row_qpos, *row_idx;
};

__global__ __launch_bounds__(256) void prefill_rows_kernel(const RowArgs a) {
  const int r = (int)blockIdx.x * 256 + (int)threadIdx.x;
  if (r >= a.rows) return;
  const bool wide_cu = a.wide & kWideCu;
  // the request: how many of the ends cu[1 .. ends] are at or below r; without cu_blocks the walk counts the blocks on
  // its way
  const int ends = a.batch - (a.wide & kOpenEnd ? 1 : 0);
  int b = 0;
  int64_t start = load_index(a.cu_seqlens, 0, wide_cu), blocks = 0;
  if (a.cu_blocks) {
    int n = ends;
    while (n > 0) {
      const int half = n / 2;
      if (load_index(a.cu_seqlens, b + half + 1, wide_cu) <= r) {
        b += half + 1;
        n -= half + 1;
      } else {
        n = half;
      }
    }
    if (b < a.batch) {
      start = load_index(a.cu_seqlens, b, wide_cu);
      blocks = a.cu_blocks[b];
    }
  } else {
    while (b < ends) {
      const int64_t end = load_index(a.cu_seqlens, b + 1, wide_cu);
      if (end > r) break;
      blocks += (end - start + a.block_q - 1) / a.block_q;
      start = end;
      ++b;
    }
  }
  if (b >= a.batch) {
    a.row_req[r] = 0;
    a.row_seq[r] = a.row_idx[r] = 0;
    a.row_qpos[r] = -1;
    return;
  }
  const int64_t local = r - start;
  a.row_req[r] = min(wrap_slot(load_index(a.slot_ids, b, a.wide & kWideSlot), a.max_slots), (int64_t)a.reqs - 1);
  a.row_seq[r] = min((int32_t)load_index(a.seq_lens, b, a.wide & kWideSeq), a.width);
  a.row_qpos[r] = (int32_t)(load_index(a.prefix_lens, b, a.wide & kWidePrefix) + local);
  a.row_idx[r] = (int32_t)min(blocks + local / a.block_q, (int64_t)a.list_rows - 1);
}

}  // namespace
}  // namespace xt

using namespace xt;

namespace {

int score_common(const char* what, ScoreArgs& a, int dim, int q_dtype, const void* q, const void* pay,
                 const void* sc, const void* r2t, int64_t pay_ps, int64_t pay_rs, int64_t sc_ps, int64_t sc_rs,
                 void* scores, int score_dtype) {
  if (!q || !pay || !sc || !r2t || !scores || !a.seq_lens || !a.slot_ids)
    return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (dim != 64 && dim != 128 && dim != 256) return fail(XT_EUNSUPPORTED, "%s: head dim %d (64, 128 or 256)", what, dim);
  if (q_dtype != XT_DTYPE_BF16 && q_dtype != XT_DTYPE_F16) return fail(XT_EUNSUPPORTED, "%s: queries must be BF16 or FP16", what);
  if (score_dtype < 0 || score_dtype > 2) return fail(XT_EINVAL, "%s: score dtype %d (0 FP32, 1 BF16, 2 FP16)", what,
                                                      score_dtype);
  // powers of two only, as the reference's tl.arange(0, block_size) requires: the prefill stages 128 keys at a time
  // and masks keys by causality and length, not by the block's end
  if (a.block_size != 32 && a.block_size != 64 && a.block_size != 128 && a.block_size != 256)
    return fail(XT_EUNSUPPORTED, "%s: block size %d (32, 64, 128 or 256)", what, a.block_size);
  if (a.max_slots < kPoolRows || a.max_slots % kPoolRows)
    return fail(XT_EINVAL, "%s: the index pool holds %lld slots (whole pages of 128)", what, (long long)a.max_slots);
  if (!aligned(pay, 16) || pay_ps % 16 || pay_rs % 16 || pay_rs < dim / 2 || !aligned(sc, 8) || sc_rs < dim / 16 ||
      sc_rs % (dim / 32) || sc_ps % (dim / 32) || !aligned(q, 16))
    return fail(XT_EINVAL, "%s: index pool rows must be 16-byte (payload) and %d-byte (scales) aligned", what, dim / 32);
  a.q = static_cast<const uint16_t*>(q);
  a.pay = static_cast<const uint8_t*>(pay);
  a.pay_ps = pay_ps;
  a.pay_rs = pay_rs;
  a.sc = static_cast<const uint8_t*>(sc);
  a.sc_ps = sc_ps;
  a.sc_rs = sc_rs;
  a.r2t = r2t;
  a.score = scores;
  a.out_dtype = score_dtype;
  return XT_OK;
}

template <int NK, bool BF>
int decode_dispatch(int T, const ScoreArgs& a, dim3 grid, hipStream_t st) {
  // The block-diagonal query fits the MFMA's rows. At 64 dims a block of 32 or 64 keys has fewer products than its
  // reductions over the lanes, one per head, cost (heads x requests x keys, block size: this kernel / the other): 4 x
  // 64 x 32768, 32: 41.9 / 36.2 us; 4 x 16 x 4096, 64: 4.5 / 4.2; but 4 x 64 x 32768, 128: 36.2 / 44.4. At 128 dims it
  // is ahead from 32 keys on (4 x 64 x 32768, 32: 49.8 / 50.1 us, 64: 48.4 / 49.3, 128: 52.8 / 60.0).
  if (a.heads <= 32 / NK) {
    const dim3 block(64 * kScoreWaves);
    if constexpr (NK > 4) {
      if (T == 1) {
        hipLaunchKernelGGL((decode_scores_few_kernel<NK, 1, BF>), grid, block, 0, st, a);
        return XT_OK;
      }
      if (T == 2) {
        hipLaunchKernelGGL((decode_scores_few_kernel<NK, 2, BF>), grid, block, 0, st, a);
        return XT_OK;
      }
    }
    if (T == 4) {
      hipLaunchKernelGGL((decode_scores_few_kernel<NK, 4, BF>), grid, block, 0, st, a);
      return XT_OK;
    }
    if (T == 8) {
      hipLaunchKernelGGL((decode_scores_few_kernel<NK, 8, BF>), grid, block, 0, st, a);
      return XT_OK;
    }
  }
  switch (T) {
    case 1: hipLaunchKernelGGL((decode_scores_kernel<NK, 1, BF>), grid, dim3(64 * kScoreWaves), 0, st, a); break;
    case 2: hipLaunchKernelGGL((decode_scores_kernel<NK, 2, BF>), grid, dim3(64 * kScoreWaves), 0, st, a); break;
    case 4: hipLaunchKernelGGL((decode_scores_kernel<NK, 4, BF>), grid, dim3(64 * kScoreWaves), 0, st, a); break;
    case 8: hipLaunchKernelGGL((decode_scores_kernel<NK, 8, BF>), grid, dim3(64 * kScoreWaves), 0, st, a); break;
    default: return XT_EUNSUPPORTED;
  }
  return XT_OK;
}

template <int NK, int G, bool BF, bool SHORT>
void prefill_launch(int hpw, const ScoreArgs& a, dim3 grid, hipStream_t st) {
  const dim3 block(64 * kScoreWaves);
  if (hpw == 1)
    hipLaunchKernelGGL((prefill_scores_kernel<NK, 1, G, BF, SHORT>), grid, block, 0, st, a);
  else if (hpw == 2)
    hipLaunchKernelGGL((prefill_scores_kernel<NK, 2, G, BF, SHORT>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((prefill_scores_kernel<NK, 4, G, BF, SHORT>), grid, block, 0, st, a);
}

template <int NK, int G, bool BF>
void prefill_dispatch(int hpw, const ScoreArgs& a, dim3 grid, hipStream_t st) {
  // From 128 dims on, blocks of 64 keys stay chunks of their own: in chunks of 128 most calls gain (4 heads x 2048 rows
  // against 2048 keys 20.3 us -> 17.9 us), some lose (8 x 4096 rows against 8192 keys 84 us -> 88 us).
  if (a.block_size < (NK == 4 ? kStageKeys<NK> : 64))
    prefill_launch<NK, G, BF, true>(hpw, a, grid, st);
  else
    prefill_launch<NK, G, BF, false>(hpw, a, grid, st);
}

}  // namespace

extern "C" int xt_minimax_decode_scores(const void* q, int64_t q_batch_stride, int64_t q_head_stride, int batch,
                                        int heads, int dim, int q_dtype, const void* index_payload,
                                        int64_t pay_page_stride, int64_t pay_slot_stride, const void* index_scales,
                                        int64_t sc_page_stride, int64_t sc_slot_stride, int64_t max_slots,
                                        const void* req_to_token, int64_t r2t_stride, const void* seq_lens,
                                        const void* slot_ids, int index_int64, int block_size, float score_factor,
                                        int init_blocks, int local_blocks, int skip_topk, int lse, void* scores,
                                        int score_dtype, int64_t s_head_stride, int64_t s_batch_stride,
                                        int64_t s_block_stride, int max_blocks_hint, xt_stream_t stream) {
  const char* what = "xt_minimax_decode_scores";
  if (batch < 0 || heads < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (batch == 0 || heads == 0) return ok();
  ScoreArgs a = {};
  a.seq_lens = seq_lens;
  a.slot_ids = slot_ids;
  a.block_size = block_size;
  a.max_slots = max_slots;
  int rc = score_common(what, a, dim, q_dtype, q, index_payload, index_scales, req_to_token, pay_page_stride,
                        pay_slot_stride, sc_page_stride, sc_slot_stride, scores, score_dtype);
  if (rc != XT_OK) return rc;
  a.q_ns = q_batch_stride;
  a.q_hs = q_head_stride;
  a.r2t_stride = r2t_stride;
  a.wide = index_int64;
  a.s_hs = s_head_stride;
  a.s_ns = s_batch_stride;
  a.s_ks = s_block_stride;
  a.batch = batch;
  a.heads = heads;
  a.c = score_factor;
  a.init_blocks = init_blocks;
  a.local_blocks = local_blocks;
  a.skip_topk = skip_topk;
  a.lse = lse;
  // workgroups per request: enough to cover max_blocks_hint blocks with one per wavefront, at most what fills the
  // device about four times over; the kernel strides over any blocks beyond
  const int cus = device_cus();
  int per_req = (max(1, max_blocks_hint) + kScoreWaves - 1) / kScoreWaves;
  per_req = min(per_req, max(1, 4 * cus / batch));
  const dim3 grid((unsigned)per_req, (unsigned)batch, (unsigned)((heads + 31) / 32));
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int T = block_size / 32;
  const bool bf = q_dtype == XT_DTYPE_BF16;
  switch (dim) {
    case 64: rc = bf ? decode_dispatch<4, true>(T, a, grid, st) : decode_dispatch<4, false>(T, a, grid, st); break;
    case 128: rc = bf ? decode_dispatch<8, true>(T, a, grid, st) : decode_dispatch<8, false>(T, a, grid, st); break;
    default: rc = bf ? decode_dispatch<16, true>(T, a, grid, st) : decode_dispatch<16, false>(T, a, grid, st); break;
  }
  if (rc != XT_OK) return fail(rc, "%s: block size %d (32, 64, 128 or 256)", what, block_size);
  return check_launch(what);
}

extern "C" int xt_minimax_prefill_scores(const void* q, int64_t q_token_stride, int64_t q_head_stride, int batch,
                                         int heads, int dim, int q_dtype, int max_q_len, const void* index_payload,
                                         int64_t pay_page_stride, int64_t pay_slot_stride, const void* index_scales,
                                         int64_t sc_page_stride, int64_t sc_slot_stride, int64_t max_slots,
                                         const void* req_to_token, int64_t r2t_stride, const void* cu_seqlens,
                                         const void* seq_lens, const void* prefix_lens, const void* slot_ids,
                                         int index_int64, int block_size, float score_factor, void* scores,
                                         int score_dtype, int64_t s_head_stride, int64_t s_token_stride,
                                         int64_t s_block_stride, xt_stream_t stream) {
  const char* what = "xt_minimax_prefill_scores";
  if (batch < 0 || heads < 0 || max_q_len < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (batch == 0 || heads == 0 || max_q_len == 0) return ok();
  if (!cu_seqlens || !prefix_lens) return fail(XT_EINVAL, "%s: a required pointer is null", what);
  ScoreArgs a = {};
  a.seq_lens = seq_lens;
  a.slot_ids = slot_ids;
  a.block_size = block_size;
  a.max_slots = max_slots;
  int rc = score_common(what, a, dim, q_dtype, q, index_payload, index_scales, req_to_token, pay_page_stride,
                        pay_slot_stride, sc_page_stride, sc_slot_stride, scores, score_dtype);
  if (rc != XT_OK) return rc;
  a.q_ns = q_token_stride;
  a.q_hs = q_head_stride;
  a.r2t_stride = r2t_stride;
  a.prefix_lens = prefix_lens;
  a.cu_seqlens = cu_seqlens;
  a.wide = index_int64;
  a.s_hs = s_head_stride;
  a.s_ns = s_token_stride;
  a.s_ks = s_block_stride;
  a.batch = batch;
  a.heads = heads;
  a.c = score_factor;
  const int hpw = heads >= 4 ? 4 : heads >= 2 ? 2 : 1;   // heads per workgroup: 256 / hpw rows each
  // block ranges: the request's blocks are at most ceil(r2t_stride / block_size) (its positions index a row of
  // req_to_token); ranges of at least 8 blocks, at most 64 ranges
  const int64_t max_blocks = (r2t_stride + block_size - 1) / block_size;
  const int64_t want_chunks = (max_blocks + 7) / 8;
  a.chunks = want_chunks < 1 ? 1 : want_chunks > 64 ? 64 : (int)want_chunks;
  a.chunk_blocks = max_blocks > 0 ? (int)((max_blocks + a.chunks - 1) / a.chunks) : 0x7FFFFFFF;
  // Four column groups per wavefront share each staged key where the query fits the registers and the row tiles still
  // give every CU its two workgroups. At 64 dims a short block's products are fewer than what ends it, and two groups
  // leave registers for twice the wavefronts (4 heads x 8192 rows against 38192 keys, blocks of 32, four / two: 352 /
  // 299 us, 64: 247 / 225, against 8292 keys, 32: 63 / 47; 128: about even).
  const int64_t tiles4 = ((int64_t)max_q_len * hpw + 511) / 512;
  const bool wide = dim == 128 || (dim == 64 && block_size >= 128);
  const int G = wide && tiles4 * a.chunks * batch >= 2 * device_cus() ? 4 : 2;
  const int rows = 128 * G / hpw;
  const int64_t tiles = (max_q_len + rows - 1) / rows;
  if (tiles * a.chunks > 0x7FFFFFFF) return fail(XT_EUNSUPPORTED, "%s: %lld query tiles", what, (long long)tiles);
  const dim3 grid((unsigned)(tiles * a.chunks), (unsigned)batch, (unsigned)((heads + hpw - 1) / hpw));
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool bf = q_dtype == XT_DTYPE_BF16;
#define XT_PREFILL(NK, G)                                                                                           \
  bf ? prefill_dispatch<NK, G, true>(hpw, a, grid, st) : prefill_dispatch<NK, G, false>(hpw, a, grid, st)
  if (dim == 64) {
    if (G == 4) XT_PREFILL(4, 4); else XT_PREFILL(4, 2);
  } else if (dim == 128) {
    if (G == 4) XT_PREFILL(8, 4); else XT_PREFILL(8, 2);
  } else {
    XT_PREFILL(16, 2);
  }
#undef XT_PREFILL
  return check_launch(what);
}

extern "C" int xt_block_prefill_rows(const void* cu_seqlens, const void* slot_ids, const void* prefix_lens,
                                     const void* seq_lens, const int64_t* cu_seqblocks, int index_int64, int batch,
                                     int rows, int block_q, int64_t max_slots, int reqs, int width, int list_rows,
                                     int64_t* row_req, int32_t* row_seq, int32_t* row_qpos, int32_t* row_idx,
                                     xt_stream_t stream) {
  const char* what = "xt_block_prefill_rows";
  if (batch < 0 || rows < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (batch == 0 || rows == 0) return ok();
  if (!cu_seqlens || !slot_ids || !prefix_lens || !seq_lens || !row_req || !row_seq || !row_qpos || !row_idx)
    return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (block_q <= 0 || max_slots <= 0 || reqs <= 0 || width < 0 || list_rows <= 0)
    return fail(XT_EINVAL, "%s: block size, slots, table and list rows must be positive", what);
  const RowArgs a = {cu_seqlens, slot_ids, prefix_lens, seq_lens, cu_seqblocks, index_int64, batch, rows, block_q,
                     max_slots, reqs, width, list_rows, row_req, row_seq, row_qpos, row_idx};
  hipLaunchKernelGGL(prefill_rows_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  return check_launch(what);
}
