// The step before the sparse attention: the indexer logits that score every key for each query, and the top-k
// selection that turns them into the int32 [rows, topk] position lists the attention kernels read.
//
//   QSA indexer logits (BF16 / FP16 q and k): logits[r, n] = sum_h ReLU(q[r, h] . k[n]) / score_scale, -inf outside
//     the row's [start, end). v_mfma_f32_32x32x16_{bf16,f16}: A = (32 / H rows x H heads) x 16 dims, B = 16 dims x 32
//     keys staged in LDS; a lane holds one key and 16 (row, head) pairs, so ReLU and the head sum run on its
//     accumulators (from 8 heads on with one exchange with the lane 32 apart); the division as a multiplication by
//     1 / score_scale. Logit rows too far apart for 31-bit offsets take a kernel that reads the keys straight from L2.
//   DSA logits (FP8 E4M3 q and k, an FP32 scale per key, FP32 head weights): logits[q, n] = sum_h w[q, h] ReLU(q_h .
//     k_n) * k_scale[n], outside [ks, ke) 0 or -inf. v_mfma_f32_32x32x16_f16 on the E4M3 values converted exactly to
//     FP16, with the heads as rows (A = 32 heads x 16 dims of one query, B = 16 dims x 32 keys): a lane then holds 16
//     heads of one key, so the weighted head sum is 16 FMAs in the lane and one exchange with the lane 32 apart. (The
//     FP8 MFMA rounds inside its 16-product sum, to about 2^-16 of the sum of magnitudes; the FP16 one sums the exact
//     products to FP32 accuracy.) Keys come from a flat array or, for decode, from the paged cache (page = block x D
//     E4M3 values, then block FP32 scales) through the block table.
//   Top-k rows: per row the positions of the topk largest finite values, ascending (ties toward the lower position),
//     -1 padded. One workgroup per row: a three-pass radix select over an order-preserving key finds the topk-th
//     largest key T and how many keys equal to T are taken. Rows up to 196608 columns live in registers: the first
//     pass (13 bits) leaves a small candidate bucket whose keys go to LDS for the other two passes, and bitmaps of the
//     taken columns are turned into positions with one block scan. Longer rows are streamed three times (11, 11, 10
//     bits), and one pass in position order writes the positions, each 1024-position chunk placed by a block-wide
//     prefix count.
#include "xt_common.h"
#include "xt_host.h"

#include <algorithm>
#include <atomic>

namespace xt {
namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef short short8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------------------------------------------
// Block-wide prefix counts (1024 threads = 16 wavefronts).

__device__ inline uint32_t wave_exclusive_count(bool flag, uint32_t& wave_total) {
  const uint64_t bits = __builtin_amdgcn_ballot_w64(flag);
  wave_total = (uint32_t)__builtin_popcountll(bits);
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(bits >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bits, 0u));
}

// Exclusive prefix of `flag` over the workgroup in thread order, and the total; `scratch` holds 16 words. Two barriers.
__device__ inline uint32_t block_exclusive_count(bool flag, uint32_t* scratch, uint32_t& total) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t wt;
  const uint32_t in_wave = wave_exclusive_count(flag, wt);
  if (lane == 0) scratch[wave] = wt;
  __syncthreads();
  uint32_t before = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const uint32_t c = scratch[w];
    before += w < wave ? c : 0u;
    sum += c;
  }
  __syncthreads();   // scratch is reused by the next call
  total = sum;
  return before + in_wave;
}

// ---------------------------------------------------------------------------------------------------------------
// Top-k rows

__device__ inline bool finite_f32(float f) { return (__float_as_uint(f) & 0x7F800000u) != 0x7F800000u; }
// Order-preserving key: a larger float has a larger key, and -0 has the key of +0 (they compare equal, so they tie).
__device__ inline uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return u == 0x80000000u ? 0x80000000u : (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int kTopkThreads = 1024;

__global__ __launch_bounds__(kTopkThreads) void topk_rows_kernel(const float* x, int64_t ld, int cols, int topk,
                                                                   int32_t* out, int64_t out_ld) {
  __shared__ uint32_t hist[2048];
  __shared__ uint32_t scratch[16];
  __shared__ uint32_t sel[2];   // the chosen digit's bucket, the rank left inside it
  const int tid = threadIdx.x;
  const float* xr = x + (int64_t)blockIdx.x * ld;
  int32_t* o = out + (int64_t)blockIdx.x * out_ld;

  uint32_t prefix = 0, pmask = 0, remaining = 0, k = 0;
  for (int pass = 0; pass < 3; ++pass) {
    const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
    const uint32_t dmask = pass == 2 ? 0x3FFu : 0x7FFu;
    for (int i = tid; i < 2048; i += kTopkThreads) hist[i] = 0;
    __syncthreads();
    for (int c = tid; c < cols; c += kTopkThreads) {
      const float f = xr[c];
      const uint32_t key = order_key(f);
      if (finite_f32(f) && (key & pmask) == prefix) atomicAdd(&hist[(key >> shift) & dmask], 1u);
    }
    __syncthreads();
    // thread t owns buckets 2047 - 2t and 2046 - 2t (from the top); the exclusive prefix of their counts in thread
    // order is the number of keys in higher buckets
    const uint32_t hi = 2047 - 2 * tid, lo = hi - 1;
    const uint32_t chi = hist[hi], clo = hist[lo];
    // a block prefix sum of the pair counts (counts up to 2^31: the same wave / block structure with sums)
    const int wave = tid >> 6, lane = tid & 63;
    uint32_t v = chi + clo, incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
      if (lane >= d) incl += y;
    }
    if (lane == 63) scratch[wave] = incl;
    __syncthreads();
    uint32_t above = incl - v, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const uint32_t c = scratch[w];
      above += w < wave ? c : 0u;
      all += c;
    }
    if (pass == 0) {
      k = min((uint32_t)topk, all);   // the finite keys bound how many can be taken
      remaining = k;
    }
    if (k != 0) {
      if (above < remaining && remaining <= above + chi) {
        sel[0] = hi;
        sel[1] = remaining - above;
      } else if (above + chi < remaining && remaining <= above + chi + clo) {
        sel[0] = lo;
        sel[1] = remaining - above - chi;
      }
    }
    __syncthreads();
    if (k == 0) break;
    prefix |= sel[0] << shift;
    pmask |= dmask << shift;
    remaining = sel[1];
    __syncthreads();   // sel and scratch are rewritten by the next pass
  }
  // positions in order: keys above T, then the first `remaining` keys equal to T
  uint32_t placed = 0, eq_seen = 0;
  for (int base = 0; k != 0 && base < cols && placed < k; base += kTopkThreads) {
    const int c = base + tid;
    const float f = c < cols ? xr[c] : -__builtin_inff();
    const bool fin = finite_f32(f);
    const uint32_t key = order_key(f);
    const bool eq = fin && key == prefix;
    uint32_t n_eq, n_take;
    const uint32_t eq_before = eq_seen + block_exclusive_count(eq, scratch, n_eq);
    const bool take = fin && (key > prefix || (eq && eq_before < remaining));
    const uint32_t at = placed + block_exclusive_count(take, scratch, n_take);
    if (take) o[at] = c;
    placed += n_take;
    eq_seen += n_eq;
  }
  for (int i = (int)k + tid; i < topk; i += kTopkThreads) o[i] = -1;
}

// Rows of at most kTopkRegMax columns: the row is read once into registers as order keys (a non-finite value as key 0,
// which no finite value has; the smallest finite key is 0x00800000). Chunk i of thread t holds columns 4 (TH i + t) ..
// + 3.
//   1. A histogram of the top 13 bits finds the bucket b0 that holds the topk-th largest key (counted as the row
//      arrives).
//   2. One pass over the registers classifies every key: one of a bucket above b0 is taken (bit e of byte TH i + t of
//      the map, so byte j covers columns 4 j .. 4 j + 3), one of b0 is a candidate, appended with its column to its
//      wavefront's list in LDS.
//   3. Two histograms over the candidates (bits 18..9, then 8..0, both over 1024 buckets) find the topk-th largest key
//      T and how many keys equal to T are taken; the candidates above T join the taken bits, those equal to T are ties
//      (bits 4-7 of the map's bytes). When a wavefront's list overflows, the two histograms run over the whole row
//      instead and the map is rewritten against T.
//   4. Thread t turns bytes CH t .. CH (t + 1) - 1 of the map (columns 4 CH t ..) into positions in column order: one
//      block scan places them, and a key equal to T is written only while fewer than `remaining` of them come before
//      it.
//
// A workgroup of TH threads holds CH chunks, 4 TH CH columns, and every chunk costs its share of each pass whether the
// row fills it or not, so a row takes the smallest form that holds it (xt_topk_rows). Measured per call at 512 keys,
// the form of 98304 columns -> the smallest: 4096 columns 26.7 us -> 8.4 us (1 row), 54.4 us -> 9.7 us (352 rows,
// several workgroups to a CU); 32768 columns 26.4 us -> 14.6 us (32 rows). Bound: LDS atomics of the histogram, then
// the classification and two block scans in a row, on as many CUs as there are rows.
// A 16-byte load of dword alignment is all that these loads need: rows of any stride take the register forms (32 rows x
// 32767 columns 59.6 us -> 14.6 us, 352 x 95087 254 us -> 46 us, against streaming them).
typedef float4_t float4_dw_t __attribute__((aligned(4)));
constexpr int kTopkRegMax = 4 * 1024 * 48;   // columns of the largest form

template <int NW>
__device__ inline uint32_t block_exclusive_sum(uint32_t v, uint32_t* scratch, uint32_t& total) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
    if (lane >= d) incl += y;
  }
  if (lane == 63) scratch[wave] = incl;
  __syncthreads();
  uint32_t before = incl - v, sum = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const uint32_t c = scratch[w];
    before += w < wave ? c : 0u;
    sum += c;
  }
  __syncthreads();   // scratch is reused by the next call
  total = sum;
  return before;
}

// The bucket of histogram h (NBK buckets) that holds the remaining-th largest key, and how many keys of that bucket
// are then taken. Thread t owns buckets NBK - 1 - NB t down to NBK - NB (t + 1); the exclusive prefix of their counts
// in thread order is the number of keys in higher buckets. With first_topk >= 0, remaining starts as min(first_topk,
// keys counted), returned in k. remaining is 0 afterwards when there is nothing to take (the bucket is then
// meaningless).
template <int TH, int NBK>
__device__ inline uint32_t pick_bucket(const uint32_t* h, uint32_t& remaining, uint32_t* scratch, uint32_t* sel,
                                       int first_topk = -1, uint32_t* k = nullptr) {
  constexpr int NB = NBK / TH, NW = TH / 64;
  const int top = NBK - 1 - NB * (int)threadIdx.x;
  uint32_t cnt[NB], sum = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    cnt[b] = h[top - b];
    sum += cnt[b];
  }
  uint32_t all;
  uint32_t above = block_exclusive_sum<NW>(sum, scratch, all);
  if (first_topk >= 0) {
    remaining = min((uint32_t)first_topk, all);
    *k = remaining;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (above < remaining && remaining <= above + cnt[b]) {
      sel[0] = top - b;
      sel[1] = remaining - above;
    }
    above += cnt[b];
  }
  __syncthreads();
  const uint32_t bucket = sel[0];
  remaining = remaining == 0 ? 0u : sel[1];
  __syncthreads();   // sel is rewritten by the next call
  return bucket;
}

// Sets the bit of column `col` (plus `shift`: 4 for the ties) in the byte map (byte col / 4): a word-wide LDS atomic.
__device__ inline void map_set(uint32_t* map, uint32_t col, uint32_t shift) {
  const uint32_t byte = col >> 2;
  atomicOr(&map[byte >> 2], 1u << (8u * (byte & 3u) + (col & 3u) + shift));
}

// ALIGNED4: cols % 4 == 0, so every chunk row loads as float4 from an address clamped into the row (columns past the
// end are masked when converted) and the loads have no branches, which lets the histogram of the first chunk rows run
// while the later ones are still in flight. Otherwise the last chunk rows load per element behind uniform branches,
// and the histogram starts after the whole row has arrived.
// PACK: only the top 16 bits of a key stay in registers, two keys to one, so a CU holds two rows of 98304 columns (one
// loads while the other computes) or one of 196608; the candidates' keys are read from the row again, and a list
// overflow reads the row for each of its three passes, four chunks in flight. 352 rows x 95088 columns: 46.9 us (2.9
// TB/s) against 63.4 us for one row of whole keys per CU; 32 rows x 131072 columns 40.6 us against 205.7 us for the
// streaming kernel. The price is the overflow: 352 rows x 95088 values within a sixteenth of each other take 255 us
// (280 us one chunk at a time) against 237 us with whole keys. Up to one row per CU whole keys are as fast where the
// lists hold (95088 columns, 1 row 25.4 us, packed 25.5) and faster where they overflow (111 us, packed 127).
template <int TH, int CH, bool ALIGNED4, bool PACK>
__global__ __launch_bounds__(TH, TH > 256 && CH <= 8 ? 8 : 4) void topk_rows_reg_kernel(
    const float* x, int64_t ld, int cols, int topk, int32_t* out, int64_t out_ld) {
  constexpr int NW = TH / 64;
  constexpr int MAPW = TH * CH / 4;         // words per map
  // one list of keys and one of columns per wavefront fill the 32 KB histogram
  constexpr int kTopkCandPerWave = 8192 / 2 / NW;
  __shared__ __align__(16) uint32_t hist[8192];   // the 13-bit histogram, then the candidate lists
  __shared__ uint32_t hist2[1024];
  __shared__ __align__(16) uint32_t map[MAPW];   // per byte: bits 0-3 the taken columns, bits 4-7 the ties
  __shared__ uint32_t scratch[NW], sel[2], wcount[NW];
  const int tid = threadIdx.x, wave = tid >> 6;
  const float* xr = x + (int64_t)blockIdx.x * ld;
  int32_t* o = out + (int64_t)blockIdx.x * out_ld;
  // 1. the top 13 bits, counted as the row arrives: each chunk row's atomics run while the later chunk rows' loads
  // are still in flight, so the histogram's LDS time hides under the HBM stream
#pragma unroll
  for (int j = 0; j < 2048 / TH; ++j)
    reinterpret_cast<uint4*>(hist)[tid + TH * j] = uint4{0, 0, 0, 0};
  __syncthreads();
  // chunk row i is loaded in step i and converted and counted in step i + kTopkAhead, so kTopkAhead chunk rows of
  // loads stay in flight while the histogram's atomics run
  constexpr int kTopkAhead = 2;
  uint32_t key[CH][PACK ? 2 : 4];   // PACK: the top halves of elements 0, 1 and 2, 3
  uint32_t in[kTopkAhead + 1][4];   // the chunk rows in flight
  const auto load = [&](int i, uint32_t (&v4)[4]) {   // chunk i of the row, as bits
    const int c = 4 * (TH * i + tid);
    if (ALIGNED4 || 4 * TH * (i + 1) <= cols) {   // uniform: the whole chunk row is inside the row, or clamped into it
      const float4_dw_t v = *reinterpret_cast<const float4_dw_t*>(xr + (ALIGNED4 ? min(c, cols - 4) : c));
      v4[0] = __float_as_uint(v[0]); v4[1] = __float_as_uint(v[1]);
      v4[2] = __float_as_uint(v[2]); v4[3] = __float_as_uint(v[3]);
    } else {   // an address inside the row; columns past the end are masked when converted
#pragma unroll
      for (int e = 0; e < 4; ++e) v4[e] = __float_as_uint(xr[min(c + e, cols - 1)]);
    }
  };
  const auto convert = [&](int i, int e, uint32_t bits) {
    const float f = __uint_as_float(bits);
    return finite_f32(f) && 4 * (TH * i + tid) + e < cols ? order_key(f) : 0u;
  };
#pragma unroll
  for (int step = 0; step < CH + kTopkAhead; ++step) {
    if (step < CH) load(step, in[step % (kTopkAhead + 1)]);
    if (step >= kTopkAhead) {
      const int i = step - kTopkAhead;
      uint32_t k4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k4[e] = convert(i, e, in[i % (kTopkAhead + 1)][e]);
        if (k4[e] != 0u) atomicAdd(&hist[k4[e] >> 19], 1u);
        if constexpr (!PACK) key[i][e] = k4[e];
      }
      if constexpr (PACK) {
        key[i][0] = __builtin_amdgcn_perm(k4[1], k4[0], 0x07060302u);
        key[i][1] = __builtin_amdgcn_perm(k4[3], k4[2], 0x07060302u);
        asm volatile("" : "+v"(key[i][0]), "+v"(key[i][1]));   // packed here: else the four keys stay to their uses
      }
    }
  }
  const auto bucket_of = [&](int i, int e) {   // the top 13 bits
    if constexpr (PACK) return e & 1 ? key[i][e >> 1] >> 19 : (key[i][e >> 1] & 0xFFFFu) >> 3;
    else return key[i][e] >> 19;
  };
  __syncthreads();
  uint32_t remaining = 0, k = 0;
  const uint32_t b0 = pick_bucket<TH, 8192>(hist, remaining, scratch, sel, topk, &k);
  if (k == 0) {   // uniform: no finite value
    for (int i = tid; i < topk; i += TH) o[i] = -1;
    return;
  }

  // 2. classify: buckets above b0 taken, b0 appended to the wavefront's candidate list (the count stays uniform)
  uint32_t* cand_key = hist + wave * kTopkCandPerWave;
  uint32_t* cand_col = hist + (NW + wave) * kTopkCandPerWave;
  uint8_t* mapb = reinterpret_cast<uint8_t*>(map);
  uint32_t wc = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    uint32_t nib = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t d = bucket_of(i, e);
      nib |= d > b0 ? 1u << e : 0u;
      const bool c = d == b0;
      const uint64_t m = __builtin_amdgcn_ballot_w64(c);
      if (m != 0) {
        const uint32_t pos =
            wc + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (c && pos < (uint32_t)kTopkCandPerWave) {
          if constexpr (!PACK) cand_key[pos] = key[i][e];
          cand_col[pos] = (uint32_t)(4 * (TH * i + tid) + e);
        }
        wc += (uint32_t)__builtin_popcountll(m);
      }
    }
    mapb[TH * i + tid] = (uint8_t)nib;
  }
  // Whole keys must be in registers here: left to itself the compiler keeps the loads' comparison masks for them, which
  // spills registers between the row's loads and waits for all of them there (95088 columns: 1 row 28.1 us -> 25.4 us,
  // 256 rows 37.3 us -> 31.0 us; 49152: 17.2 us -> 16.1 us).
  if constexpr (!PACK) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(key[i][e]));
  }
  if ((tid & 63) == 0) wcount[wave] = wc;
  __syncthreads();
  bool fits = true;
#pragma unroll
  for (int w = 0; w < NW; ++w) fits = fits && wcount[w] <= (uint32_t)kTopkCandPerWave;

  // 3. bits 18..9 and 8..0 of the keys in b0
  uint32_t t_key;
  if (fits) {   // uniform
    const int n = (int)wc;
    if constexpr (PACK)
      for (int j = tid & 63; j < n; j += 64) cand_key[j] = order_key(xr[cand_col[j]]);
    for (int j = tid; j < 1024; j += TH) hist2[j] = 0;
    __syncthreads();
    for (int j = tid & 63; j < n; j += 64) atomicAdd(&hist2[(cand_key[j] >> 9) & 1023u], 1u);
    __syncthreads();
    const uint32_t b1 = pick_bucket<TH, 1024>(hist2, remaining, scratch, sel);
    for (int j = tid; j < 1024; j += TH) hist2[j] = 0;
    __syncthreads();
    const uint32_t hi1 = (b0 << 10) | b1;
    for (int j = tid & 63; j < n; j += 64)
      if ((cand_key[j] >> 9) == hi1) atomicAdd(&hist2[cand_key[j] & 511u], 1u);
    __syncthreads();
    const uint32_t b2 = pick_bucket<TH, 1024>(hist2, remaining, scratch, sel);
    t_key = (hi1 << 9) | b2;
    for (int j = tid & 63; j < n; j += 64) {
      const uint32_t c = cand_key[j];
      if (c > t_key) map_set(map, cand_col[j], 0u);
      else if (c == t_key) map_set(map, cand_col[j], 4u);
    }
  } else {
    // f(i, the whole keys of chunk i): from the registers, or (PACK, not unrolled) from the row again
    const auto for_chunks = [&](auto f) {
      if constexpr (PACK) {
        // chunks in flight (rows of other lengths load their last chunks element by element: one, since four cost the
        // whole form 1 %)
        constexpr int kOnce = ALIGNED4 ? 4 : 1;
#pragma unroll 1
        for (int i = 0; i < CH; i += kOnce) {
          uint32_t k4[kOnce][4];
#pragma unroll
          for (int u = 0; u < kOnce; ++u) load(i + u, k4[u]);
#pragma unroll
          for (int u = 0; u < kOnce; ++u) {
#pragma unroll
            for (int e = 0; e < 4; ++e) k4[u][e] = convert(i + u, e, k4[u][e]);
            f(i + u, k4[u]);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < CH; ++i) f(i, key[i]);
      }
    };
    for (int j = tid; j < 1024; j += TH) hist2[j] = 0;
    __syncthreads();
    for_chunks([&](int, const uint32_t* k4) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((k4[e] >> 19) == b0) atomicAdd(&hist2[(k4[e] >> 9) & 1023u], 1u);
    });
    __syncthreads();
    const uint32_t b1 = pick_bucket<TH, 1024>(hist2, remaining, scratch, sel);
    for (int j = tid; j < 1024; j += TH) hist2[j] = 0;
    __syncthreads();
    const uint32_t hi1 = (b0 << 10) | b1;
    for_chunks([&](int, const uint32_t* k4) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((k4[e] >> 9) == hi1) atomicAdd(&hist2[k4[e] & 511u], 1u);
    });
    __syncthreads();
    const uint32_t b2 = pick_bucket<TH, 1024>(hist2, remaining, scratch, sel);
    t_key = (hi1 << 9) | b2;
    for_chunks([&](int i, const uint32_t* k4) {
      uint32_t n = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) n |= k4[e] > t_key ? 1u << e : k4[e] == t_key ? 16u << e : 0u;
      mapb[TH * i + tid] = (uint8_t)n;
    });
  }
  __syncthreads();

  // 4. positions in column order
  constexpr int TW = MAPW / TH;   // words of each map per thread
  uint32_t gw[TW], ew[TW], ng = 0, ne = 0;
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    const uint32_t w = map[TW * tid + j];
    gw[j] = w & 0x0F0F0F0Fu;
    ew[j] = (w >> 4) & 0x0F0F0F0Fu;
  }
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    ng += (uint32_t)__builtin_popcount(gw[j]);
    ne += (uint32_t)__builtin_popcount(ew[j]);
  }
  uint32_t tot;
  uint32_t gt_b = block_exclusive_sum<NW>(ng, scratch, tot);
  uint32_t eq_b = block_exclusive_sum<NW>(ne, scratch, tot);
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    uint32_t m = gw[j] | ew[j];
    while (m != 0u) {
      const uint32_t b = (uint32_t)__builtin_ctz(m);
      m &= m - 1u;
      const int col = 4 * (4 * (TW * tid + j) + (int)(b >> 3)) + (int)(b & 7u);
      if ((gw[j] >> b) & 1u) {
        o[gt_b + min(eq_b, remaining)] = col;
        ++gt_b;
      } else {
        if (eq_b < remaining) o[gt_b + eq_b] = col;
        ++eq_b;
      }
    }
  }
  for (int i = (int)k + tid; i < topk; i += TH) o[i] = -1;
}

// ---------------------------------------------------------------------------------------------------------------
// QSA indexer logits

template <bool BF>
__device__ inline float16_t mfma_qk(short8_t a, short8_t b, float16_t c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c,
                                                  0, 0, 0);
}

struct QsaArgs {
  const uint16_t* q;
  int64_t q_rs, q_hs;
  const uint16_t* k;
  int64_t k_rs;
  const int32_t* starts;
  const int32_t* ends;
  float score_scale;
  float* logits;
  int64_t ld;
  int rows, keys;
  int keys_per_wg;
  int vec_store;             // logits rows are 16-byte aligned: stores of 4 floats
};

constexpr int kQsaWaves = 4;

// Workgroup = (4 wavefronts x 2 column groups of 32 / H rows, keys_per_wg keys): every wavefront sweeps the whole key
// range for its own 2 x 32 / H rows, so the four wavefronts read the same K blocks (from L1 after the first) and each
// K block leaves L2 once per 8 x 32 / H rows. Lane layouts (32x32x16): A = keys, lane (key l % 32, dims
// 16kk + 8 (l / 32) .. +7) read straight from k; B = queries, lane (column j = l % 32: row j / H, head j % H; same
// dims) kept in registers, one set per column group; C = S^T, lane (column j, keys 8 (r / 4) + 4 (l / 32) + r % 4).
constexpr int kQsaGroups = 2;   // column groups per wavefront

template <int H, int NK, bool BF>
__global__ __launch_bounds__(64 * kQsaWaves) void qsa_logits_kernel(const QsaArgs a) {
  constexpr int kRowsG = 32 / H, kRowsW = kQsaGroups * kRowsG;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int rw = (blockIdx.x * kQsaWaves + wave) * kRowsW;   // this wavefront's first row
  const int head = j % H;
  int my_row[kQsaGroups], start[kQsaGroups], end[kQsaGroups];
  bool row_ok[kQsaGroups];
  short8_t qb[kQsaGroups][NK];
#pragma unroll
  for (int g = 0; g < kQsaGroups; ++g) {
    my_row[g] = rw + g * kRowsG + j / H;
    row_ok[g] = my_row[g] < a.rows;
    start[g] = row_ok[g] ? a.starts[my_row[g]] : 0;
    end[g] = row_ok[g] ? a.ends[my_row[g]] : 0;
    const uint16_t* qp = a.q + (int64_t)(row_ok[g] ? my_row[g] : 0) * a.q_rs + (int64_t)head * a.q_hs + 8 * h;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const uint4 w = row_ok[g] ? *reinterpret_cast<const uint4*>(qp + 16 * kk) : uint4{0u, 0u, 0u, 0u};
      qb[g][kk] = __builtin_bit_cast(short8_t, w);
    }
  }
  // the wavefront's key range: a 32-key block outside every one of its rows' [start, end) is written as -inf
  // without the product
  int lo = 0x7FFFFFFF, hi = 0;
  for (int r = 0; r < kRowsW; ++r) {
    if (rw + r < a.rows) {
      lo = min(lo, max(0, a.starts[rw + r]));
      hi = max(hi, min(a.keys, a.ends[rw + r]));
    }
  }
  // x / score_scale as x * (1 / score_scale): one more rounding, at most 2^-24 relative
  const float inv = 1.0f / a.score_scale;
  const int k_begin = blockIdx.y * a.keys_per_wg, k_end = min(a.keys, k_begin + a.keys_per_wg);
  if constexpr (H <= 4) {
    // Queries as rows: S = Q . K^T with A = the query columns above, B = K; C lane (key kb + j, column-group rows
    // i = 8 (r / 4) + 4 h + r % 4: row i / H, head i % H). A row's H heads are H consecutive r of one lane, so the
    // head sum stays in the lane, and lane j writes key kb + j of 16 / H rows (each row: 32 consecutive keys across
    // the lanes).
    constexpr int kOut = 16 / H;
    int orow[kQsaGroups][kOut], ost[kQsaGroups][kOut], oen[kQsaGroups][kOut];
    int max_start = 0, min_end = 0x7FFFFFFF;
#pragma unroll
    for (int g = 0; g < kQsaGroups; ++g)
#pragma unroll
      for (int o = 0; o < kOut; ++o) {
        const int r = o * H;
        orow[g][o] = rw + g * kRowsG + (8 * (r >> 2) + 4 * h + (r & 3)) / H;
        const bool ok = orow[g][o] < a.rows;
        ost[g][o] = ok ? a.starts[orow[g][o]] : 0;
        oen[g][o] = ok ? a.ends[orow[g][o]] : 0;
        if (ok) {
          max_start = max(max_start, ost[g][o]);
          min_end = min(min_end, oen[g][o]);
        }
      }
    // over the wavefront: a block inside every row's range needs no per-key test
    for (int d = 1; d < 64; d <<= 1) {
      max_start = max(max_start, __shfl_xor(max_start, d));
      min_end = min(min_end, __shfl_xor(min_end, d));
    }
    for (int kb = k_begin; kb < k_end; kb += 32) {
      const int key = kb + j;
      if (kb + 32 <= lo || kb >= hi) {   // uniform over the wavefront
#pragma unroll
        for (int g = 0; g < kQsaGroups; ++g)
#pragma unroll
          for (int o = 0; o < kOut; ++o)
            if (orow[g][o] < a.rows && key < a.keys) a.logits[(int64_t)orow[g][o] * a.ld + key] = -__builtin_inff();
        continue;
      }
      const bool inside = kb >= max_start && kb + 32 <= min_end;
      const uint16_t* kp = a.k + (int64_t)min(key, a.keys - 1) * a.k_rs + 8 * h;
      short8_t kf[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) kf[kk] = __builtin_bit_cast(short8_t, *reinterpret_cast<const uint4*>(kp + 16 * kk));
#pragma unroll
      for (int g = 0; g < kQsaGroups; ++g) {
        float16_t sc = {};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) sc = mfma_qk<BF>(qb[g][kk], kf[kk], sc);
#pragma unroll
        for (int o = 0; o < kOut; ++o) {
          float x = fmaxf(sc[o * H], 0.0f);
#pragma unroll
          for (int e = 1; e < H; ++e) x += fmaxf(sc[o * H + e], 0.0f);
          const bool in_range = inside || (key >= ost[g][o] && key < oen[g][o]);
          if (orow[g][o] < a.rows && key < a.keys)
            a.logits[(int64_t)orow[g][o] * a.ld + key] = in_range ? x * inv : -__builtin_inff();
        }
      }
    }
    return;
  }
  for (int kb = k_begin; kb < k_end; kb += 32) {
    float v[kQsaGroups][16];
    if (kb + 32 <= lo || kb >= hi) {   // uniform over the wavefront
#pragma unroll
      for (int g = 0; g < kQsaGroups; ++g)
#pragma unroll
        for (int r = 0; r < 16; ++r) v[g][r] = -__builtin_inff();
    } else {
      const int key = min(kb + j, a.keys - 1);
      const uint16_t* kp = a.k + (int64_t)key * a.k_rs + 8 * h;
      short8_t kf[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) kf[kk] = __builtin_bit_cast(short8_t, *reinterpret_cast<const uint4*>(kp + 16 * kk));
#pragma unroll
      for (int g = 0; g < kQsaGroups; ++g) {
        float16_t s = {};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) s = mfma_qk<BF>(kf[kk], qb[g][kk], s);
        // ReLU, then the sum over the H heads of a row (H consecutive lanes), in the order lane ^ 1, ^ 2, ...
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float x = fmaxf(s[r], 0.0f);
          if constexpr (H >= 2) x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false));
          if constexpr (H >= 4) x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, false));
          if constexpr (H >= 8) x += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), (4 << 10) | 0x1F));
          if constexpr (H >= 16) x += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), (8 << 10) | 0x1F));
          if constexpr (H >= 32) x += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), (16 << 10) | 0x1F));
          const int kr = kb + 8 * (r >> 2) + 4 * h + (r & 3);
          v[g][r] = (kr >= start[g] && kr < end[g]) ? x * inv : -__builtin_inff();
        }
      }
    }
    // the lane of head 0 of each row writes its 16 keys: 4 runs of 4 consecutive keys
#pragma unroll
    for (int g = 0; g < kQsaGroups; ++g) {
      if (row_ok[g] && head == 0) {
        float* op = a.logits + (int64_t)my_row[g] * a.ld;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int key = kb + 8 * q4 + 4 * h;
          if (key + 4 <= a.keys && a.vec_store) {
            *reinterpret_cast<float4_t*>(op + key) =
                float4_t{v[g][4 * q4], v[g][4 * q4 + 1], v[g][4 * q4 + 2], v[g][4 * q4 + 3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (key + e < a.keys) op[key + e] = v[g][4 * q4 + e];
          }
        }
      }
    }
  }
}

// Keys through LDS: a workgroup is 4 wavefronts x G column groups of 32 / H rows over keys_per_wg keys, S keys at a
// time staged once for all its 128 G (row, head) columns. Queries are the MFMA rows (A: column j of a group; B: keys),
// so C lane (key kb + j, columns 8 (r / 4) + 4 h + r % 4) holds whole rows for H <= 4 and half rows, exchanged with the
// lane 32 apart, for H >= 8. The next stage's loads are issued before this stage's stores and the stores carry no
// branch (rows and keys past the end have offsets past the buffer's range, which drops them), so the wait for those
// loads does not wait for the stores behind them. Bound: HBM, the FP32 logits written, with the matrix product and the
// head sum beside it (from 8 heads on they are the larger part). 352 rows x 95088 keys, 4 heads x 128: 50.4 us (3.1
// TB/s) against 91.8 us for the kernel above, whose wavefronts each read the keys from L2 and wait for their stores
// with them; 352 x 65536: 8 heads 128 -> 61 us, 16 heads 261 -> 99, 32 heads 590 -> 188.
// With four column groups (32 MB of logits and more at 4 heads) the stores are non-temporal: the logits alone take
// 50.4 us in place of 60.5 at 352 x 95088. With the selection of 2048 positions behind them 352 x 32768 takes 48.3 ->
// 47.5 us, but from about 60 MB on the selection, which then reads them from HBM, loses more than the stores gain (352
// x 65536 78.3 -> 79.4, x 95088 104.5 -> 109.5; 512 x 95088 129 -> 137). With fewer groups they are of device scope,
// which passes them on without waiting for the end of the kernel and leaves them to the selection (4 heads, plain /
// non-temporal / device scope, alone 32 x 4100 4.7 / 5.1 / 4.6 us, 352 x 4100 10.2 / 10.0 / 9.3; with the selection 32
// x 4100 13.9 / 14.4 / 13.8, 352 x 4100 23.0 / 21.6 / 21.0, 32 x 65536 29.7 / 29.3 / 28.9).
template <int NK, int G>
constexpr int kQsaStage = (NK <= 8 ? 64 : 32) * (G == 4 ? 2 : 1);   // keys per stage

template <int H, int NK, int G, bool BF>
__global__ __launch_bounds__(64 * kQsaWaves, 2) void qsa_logits_lds_kernel(const QsaArgs a) {
  constexpr int D = 16 * NK, S = kQsaStage<NK, G>;
  constexpr int ROW = D + 8;                       // 16-bit values per LDS row: conflict-free 16-byte reads
  constexpr int kRowsG = 32 / H, kRowsW = G * kRowsG, kRowsWg = kQsaWaves * kRowsW;
  constexpr int kPieces = S * 2 * NK / (64 * kQsaWaves);   // 16-byte pieces a thread stages
  constexpr int kOut = H <= 4 ? 16 / H : H == 32 ? 1 : 16 / H;   // logits per lane and column group
  constexpr int kStorePolicy = G == 4 ? 2 : 16;    // non-temporal; device scope
  __shared__ __align__(16) uint16_t lds[2][S * ROW];
  __shared__ int2 range[kRowsWg];   // [start, end) of the rows (read behind the loop's first barrier)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const int row0 = blockIdx.x * kRowsWg, rw = row0 + wave * kRowsW;   // the workgroup's and the wavefront's first row
  const int k_begin = blockIdx.y * a.keys_per_wg, k_end = min(a.keys, k_begin + a.keys_per_wg);
  const int n_stages = (k_end - k_begin + S - 1) / S;
  xt_u32x4_t raw[kPieces];
  auto load_raw = [&](int n) {   // piece i of a thread: key (i 256 + tid) / (2 NK) of the stage
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = i * 64 * kQsaWaves + tid;
      const int key = min(k_begin + n * S + c / (2 * NK), a.keys - 1);
      raw[i] = *reinterpret_cast<const xt_u32x4_t*>(a.k + (int64_t)key * a.k_rs + 8 * (c % (2 * NK)));
    }
  };
  load_raw(0);
  for (int r = tid; r < kRowsWg; r += 64 * kQsaWaves)
    range[r] = row0 + r < a.rows ? int2{a.starts[row0 + r], a.ends[row0 + r]} : int2{0, 0};
  short8_t qb[G][NK];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int row = min(rw + g * kRowsG + j / H, a.rows - 1);   // rows past the end repeat the last and store nothing
    const uint16_t* qp = a.q + (int64_t)row * a.q_rs + (int64_t)(j % H) * a.q_hs + 8 * h;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qb[g][kk] = __builtin_bit_cast(short8_t, *reinterpret_cast<const xt_u32x4_t*>(qp + 16 * kk));
  }
  // Logit (g, o) of a lane is that of row rw + g kRowsG + first(o) + h half: for H <= 4 a row's heads are H consecutive
  // C elements of one lane, for H >= 8 the halves split pairs of rows (32 heads: one row, which the lower half stores).
  constexpr int half = H <= 4 ? 4 / H : H == 32 ? 0 : 1;
  const auto first = [](int o) constexpr { return H <= 4 ? (8 * (o * H >> 2) + (o * H & 3)) / H : 2 * o; };
  static_assert((kQsaWaves - 1) * kRowsW + (G - 1) * kRowsG + first(kOut - 1) + half < kRowsWg,
                "the last lane's last row is one of the workgroup's (an entry of range)");
  int max_start = 0, min_end = 0x7FFFFFFF, lo = 0x7FFFFFFF, hi = 0;
  for (int r = rw + lane; r < min(rw + kRowsW, a.rows); r += 64) {
    const int st = a.starts[r], en = a.ends[r];
    max_start = max(max_start, st);
    min_end = min(min_end, en);
    lo = min(lo, max(0, st));
    hi = max(hi, min(a.keys, en));
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    max_start = max(max_start, __shfl_xor(max_start, d));
    min_end = min(min_end, __shfl_xor(min_end, d));
    lo = min(lo, __shfl_xor(lo, d));
    hi = max(hi, __shfl_xor(hi, d));
  }
  // uniform over the wavefront: a 32-key block outside [lo, hi) is in no row's range, one inside [max_start, min_end)
  // in every row's
  max_start = __builtin_amdgcn_readfirstlane(max_start);
  min_end = __builtin_amdgcn_readfirstlane(min_end);
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  const int live_rows = min(a.rows - row0, kRowsWg);
  float* const base = a.logits + (int64_t)row0 * a.ld;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      base, 0, (int)((int64_t)(live_rows - 1) * a.ld * 4 + (int64_t)a.keys * 4), 0x00020000);
  const uint32_t ld4 = (uint32_t)a.ld * 4u;   // every offset of a live row is below 2^31 (host)
  const uint32_t lane_off = (uint32_t)(wave * kRowsW + h * half) * ld4;
  const float inv = 1.0f / a.score_scale;   // as in the kernel above
  // the query arrives before the loop: waited for inside, its loads' counts would make every pass wait for stores
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) asm volatile("" : "+v"(qb[g][kk]));
  for (int n = 0; n < n_stages; ++n) {
    uint16_t* const buf = lds[n & 1];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = i * 64 * kQsaWaves + tid;
      *reinterpret_cast<xt_u32x4_t*>(buf + (c / (2 * NK)) * ROW + 8 * (c % (2 * NK))) = raw[i];
    }
    load_raw(min(n + 1, n_stages - 1));
    __syncthreads();   // stage n is written; every wavefront is past stage n - 1, whose buffer stage n + 1 takes
#pragma unroll
    for (int t = 0; t < S / 32; ++t) {
      const int kb = k_begin + n * S + 32 * t, key = kb + j;
      const bool any = kb + 32 > lo && kb < hi && kb < k_end, inside = kb >= max_start && kb + 32 <= min_end;
      const uint32_t koff = key < k_end && (H < 32 || h == 0) ? lane_off + 4u * (uint32_t)key : 0x80000000u;
      short8_t kf[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        kf[kk] = __builtin_bit_cast(short8_t, *reinterpret_cast<const uint4*>(buf + (32 * t + j) * ROW + 16 * kk + 8 * h));
#pragma unroll
      for (int g = 0; g < G; ++g) {
        // formed anew for each group: kept across the loop, the store offsets would take the query's registers
        uint32_t row_step = ld4;
        asm volatile("" : "+s"(row_step));
        float x[kOut];
        if (any) {
          float16_t sc = {};
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) sc = mfma_qk<BF>(qb[g][kk], kf[kk], sc);
          if constexpr (H <= 4) {
#pragma unroll
            for (int o = 0; o < kOut; ++o) {
              x[o] = fmaxf(sc[o * H], 0.0f);
#pragma unroll
              for (int e = 1; e < H; ++e) x[o] += fmaxf(sc[o * H + e], 0.0f);
            }
          } else {
            float part[32 / H];   // this half's heads of each row
#pragma unroll
            for (int o = 0; o < 32 / H; ++o) {
              float quad[H / 8];
#pragma unroll
              for (int e = 0; e < H / 8; ++e) {
                const int r = o * (H / 2) + 4 * e;
                quad[e] = (fmaxf(sc[r], 0.0f) + fmaxf(sc[r + 1], 0.0f)) + (fmaxf(sc[r + 2], 0.0f) + fmaxf(sc[r + 3], 0.0f));
              }
              part[o] = quad[0];
#pragma unroll
              for (int e = 1; e < H / 8; ++e) part[o] += quad[e];
            }
#pragma unroll
            for (int o = 0; o < kOut; ++o) {   // the lower half ends up with row 2 o, the upper with row 2 o + 1
              const float p0 = part[H == 32 ? 0 : 2 * o], p1 = part[H == 32 ? 0 : 2 * o + 1];
              const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(p0), __float_as_uint(p1), false, false);
              x[o] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
            }
          }
#pragma unroll
          for (int o = 0; o < kOut; ++o) x[o] *= inv;
          if (!inside) {
            // from LDS: a global load here would make the wait for the next stage's loads one for the stores as well
            const int2* rp = range + wave * kRowsW + g * kRowsG + h * half;
#pragma unroll
            for (int o = 0; o < kOut; ++o) {
              const int2 se = rp[first(o)];
              x[o] = key >= se.x && key < se.y ? x[o] : -__builtin_inff();
            }
          }
        } else {
#pragma unroll
          for (int o = 0; o < kOut; ++o) x[o] = -__builtin_inff();
        }
#pragma unroll
        for (int o = 0; o < kOut; ++o)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[o]), rsrc,
                                              (int)(koff + (uint32_t)(g * kRowsG + first(o)) * row_step), 0, kStorePolicy);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// DSA logits (FP8)

struct DsaArgs {
  const uint8_t* q;          // [num_q, heads, D] E4M3
  int64_t q_rs, q_hs;
  const uint8_t* k;          // flat: [num_kv, D] E4M3 with k_rs bytes per key; paged: the page buffer
  int64_t k_rs;
  const float* k_scale;      // flat: [num_kv]
  int64_t page_bytes;        // paged: bytes from one page to the next (block x (D + 4))
  int64_t num_pages;         // paged: pages in the cache (table entries past it read as no key)
  int block;                 // paged: keys per page (0: flat keys)
  const int32_t* block_table;
  int64_t bt_stride;
  int bt_width;
  const float* w;            // [num_q, heads]
  int64_t w_rs;
  const int32_t* ks;         // flat: [num_q] (inclusive) start, or NULL
  const int32_t* ke;         // flat: end (exclusive); paged: context length per row
  int clean;
  float* logits;
  int64_t ld;
  int num_q, num_kv, heads;
  int keys_per_wg;
  int out_cols;              // columns written per row (paged: max_seq_len)
};

constexpr int kDsaWaves = 4;

// The shapes the two kernels below do not take (query and weights past their registers, pages off the 32-key grid, rows
// off 16-byte alignment). Workgroup = (4 query rows, one per wavefront, keys_per_wg keys); the wavefronts walk the same
// 32-key blocks, so a block's key bytes are fetched once for the four rows. Per block and 32-head group, S = Q . K^T on
// 32x32x16 FP16 MFMAs of the converted E4M3 values (A = Q: lane (head l % 32, dims 16kk + 8 (l / 32) .. +7); B = K^T:
// lane (key l % 32, same dims); C: lane (key column l % 32, heads 8 (r / 4) + 4 (l / 32) + r % 4)).
template <int NK>
__global__ __launch_bounds__(64 * kDsaWaves) void dsa_logits_kernel(const DsaArgs a) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int qrow = blockIdx.x * kDsaWaves + wave;
  if (qrow >= a.num_q) return;   // no barrier below
  const int groups = a.heads / 32;
  const int k_begin = blockIdx.y * a.keys_per_wg, k_end = min(a.out_cols, k_begin + a.keys_per_wg);
  const bool paged = a.block > 0;
  const int lim_lo = (!paged && a.ks) ? a.ks[qrow] : 0;
  const int lim_hi = paged ? a.ke[qrow] : (a.ke ? a.ke[qrow] : a.num_kv);
  const float fill = a.clean ? -__builtin_inff() : 0.0f;
  for (int kb = k_begin; kb < k_end; kb += 32) {
    const int key = kb + j;
    bool live = key >= lim_lo && key < lim_hi && key < (paged ? a.bt_width * a.block : a.num_kv);
    int32_t page = 0;
    if (paged) {
      // a negative entry reads page 0, as the reference's clamp does (indexer_torch.py:61); an entry past the cache
      // reads as no key
      page = live ? max(a.block_table[(int64_t)qrow * a.bt_stride + key / a.block], 0) : 0;
      live = live && page < a.num_pages;
      page = live ? page : 0;
    }
    float total = 0.0f;
    if (__builtin_amdgcn_ballot_w64(live)) {
      // this lane's key row and scale
      const uint8_t* kp;
      float ksc;
      if (paged) {
        const int kk = live ? key : 0;
        const uint8_t* pg = a.k + (int64_t)page * a.page_bytes;
        kp = pg + (int64_t)(kk % a.block) * (16 * NK);
        ksc = *reinterpret_cast<const float*>(pg + (int64_t)a.block * (16 * NK) + 4 * (kk % a.block));
      } else {
        const int kk = live ? key : 0;
        kp = a.k + (int64_t)kk * a.k_rs;
        ksc = a.k_scale[kk];
      }
      uint64_t kf[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) kf[kk] = *reinterpret_cast<const uint64_t*>(kp + 16 * kk + 8 * h);
      float acc = 0.0f;
      for (int g = 0; g < groups; ++g) {
        const uint8_t* qp = a.q + (int64_t)qrow * a.q_rs + (int64_t)(32 * g + j) * a.q_hs + 8 * h;
        float16_t s = {};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
          s = __builtin_amdgcn_mfma_f32_32x32x16_f16(fp8x8_to_f16(*reinterpret_cast<const uint64_t*>(qp + 16 * kk)),
                                                     fp8x8_to_f16(kf[kk]), s, 0, 0, 0);
        const float* wp = a.w + (int64_t)qrow * a.w_rs + 32 * g + 4 * h;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc += fmaxf(s[r], 0.0f) * wp[8 * (r >> 2) + (r & 3)];
      }
      // the other 16 heads of each group are in the lane 32 apart
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
      total = (__uint_as_float(sw[0]) + __uint_as_float(sw[1])) * ksc;
    }
    if (h == 0 && key < k_end) a.logits[(int64_t)qrow * a.ld + key] = live ? total : fill;
  }
}

// Flat keys, heads x dim within registers (G head groups of 32, G * NK <= 16): the four rows of a workgroup read the
// same keys, so the workgroup stages them once per 128 keys in LDS (E4M3 bytes, double-buffered, one barrier per
// stage), each wavefront keeps its row's query (as FP16) and head weights in registers for the whole key range, and
// converts each 32-key block's K once for all its head groups.
constexpr int kDsaStageKeys = 128;

template <int NK, int G>
__global__ __launch_bounds__(64 * kDsaWaves) void dsa_flat_kernel(const DsaArgs a) {
  // LDS bytes per key: D + 8, so the 32 keys a half-wavefront reads sit on 32 distinct bank pairs ((D + 8) / 4 is
  // twice an odd number)
  constexpr int D = 16 * NK, ROW = D + 8;
  constexpr int PIECES = kDsaStageKeys * D / 16;           // 16-byte pieces per stage
  constexpr int PER_THREAD = PIECES / (64 * kDsaWaves);
  __shared__ __align__(16) uint8_t kt[2][kDsaStageKeys * ROW];   // ROW * 128 is a multiple of 16
  __shared__ float kst[2][kDsaStageKeys];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5, tid = threadIdx.x;
  const int qrow = blockIdx.x * kDsaWaves + wave;
  const bool row_ok = qrow < a.num_q;   // every thread takes every barrier below
  const int k_begin = blockIdx.y * a.keys_per_wg, k_end = min(a.num_kv, k_begin + a.keys_per_wg);
  const int lim_lo = (row_ok && a.ks) ? a.ks[qrow] : 0;
  const int lim_hi = row_ok ? (a.ke ? a.ke[qrow] : a.num_kv) : 0;
  const float fill = a.clean ? -__builtin_inff() : 0.0f;
  // this row's query (A operand: head 32 g + j, dims 16 kk + 8 h .. + 7) and weights (C rows of lane half h)
  half8_t qf[G][NK];
  float wv[G][16];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint8_t* qp = a.q + (int64_t)(row_ok ? qrow : 0) * a.q_rs + (int64_t)(32 * g + j) * a.q_hs + 8 * h;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qf[g][kk] = fp8x8_to_f16(row_ok ? *reinterpret_cast<const uint64_t*>(qp + 16 * kk) : 0ull);
    const float* wp = a.w + (int64_t)(row_ok ? qrow : 0) * a.w_rs + 32 * g + 4 * h;
#pragma unroll
    for (int r = 0; r < 16; ++r) wv[g][r] = row_ok ? wp[8 * (r >> 2) + (r & 3)] : 0.0f;
  }
  uint4 reg[PER_THREAD];
  float sreg = 0.0f;
  auto load_stage = [&](int k0) {   // keys past the end read the last key (never written out)
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int c = tid + 64 * kDsaWaves * i, key = min(k0 + c / (D / 16), a.num_kv - 1);
      reg[i] = *reinterpret_cast<const uint4*>(a.k + (int64_t)key * a.k_rs + 16 * (c % (D / 16)));
    }
    if (tid < kDsaStageKeys) sreg = a.k_scale[min(k0 + tid, a.num_kv - 1)];
  };
  auto store_stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int c = tid + 64 * kDsaWaves * i;
      uint2* dst = reinterpret_cast<uint2*>(&kt[buf][(c / (D / 16)) * ROW + 16 * (c % (D / 16))]);
      dst[0] = uint2{reg[i].x, reg[i].y};   // 8-byte aligned rows: two 8-byte stores
      dst[1] = uint2{reg[i].z, reg[i].w};
    }
    if (tid < kDsaStageKeys) kst[buf][tid] = sreg;
  };
  const int stages = k_end > k_begin ? (k_end - k_begin + kDsaStageKeys - 1) / kDsaStageKeys : 0;
  if (stages > 0) {
    load_stage(k_begin);
    store_stage(0);
  }
  __syncthreads();
  for (int st = 0; st < stages; ++st) {
    const int k0 = k_begin + st * kDsaStageKeys, buf = st & 1;
    if (st + 1 < stages) load_stage(k0 + kDsaStageKeys);   // in flight during this stage's MFMAs
#pragma unroll 1
    for (int t = 0; t < kDsaStageKeys / 32; ++t) {
      const uint8_t* kr = &kt[buf][(32 * t + j) * ROW + 8 * h];
      half8_t kv[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) kv[kk] = fp8x8_to_f16(*reinterpret_cast<const uint64_t*>(kr + 16 * kk));
      float acc = 0.0f;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float16_t sc = {};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(qf[g][kk], kv[kk], sc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc += fmaxf(sc[r], 0.0f) * wv[g][r];
      }
      // the other 16 heads of each group are in the lane 32 apart
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
      const float total = (__uint_as_float(sw[0]) + __uint_as_float(sw[1])) * kst[buf][32 * t + j];
      const int key = k0 + 32 * t + j;
      const bool live = key >= lim_lo && key < lim_hi;
      if (row_ok && h == 0 && key < k_end) a.logits[(int64_t)qrow * a.ld + key] = live ? total : fill;
    }
    if (st + 1 < stages) store_stage(buf ^ 1);   // its readers finished the stage before the last barrier
    __syncthreads();
  }
}

// Paged keys whose pages hold a multiple of 32 keys (decode): one row per workgroup, `bpw` consecutive 32-key blocks
// per wavefront, so a batch of a few rows still spreads over every CU. The row's query (as FP16) and head weights stay
// in registers for the wavefront's whole range; a block's page is uniform, so the wavefront's table entries are one
// vector load before the loop and a block's address is scalar. k-step kk covers dims h D/2 + 8 kk .. + 7 in both
// operands (not 16 kk + 8 h), so a lane reads its half of a key's row as 16-byte pieces. Bound: HBM, D + 4 bytes per
// key; a wavefront keeps one block's loads in flight beyond the one it computes (two or three measured 21.3 us against
// 20.8). 32 rows x 32 heads x 128, up to 32768 keys each (16.6K in the mean, 69 MB): 20.8 us = 3.3 TB/s against 352 us
// for dsa_logits_kernel, which puts four rows in a workgroup and 4096 keys in a wavefront's serial walk.
constexpr int kDsaAhead = 1;

template <int NK, int G>
__global__ __launch_bounds__(64 * kDsaWaves) void dsa_paged_kernel(const DsaArgs a, int bpw) {
  constexpr int D = 16 * NK, PIECES = D / 32;   // 16-byte pieces of a lane's half row
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int row = blockIdx.y;
  const int b0 = __builtin_amdgcn_readfirstlane(((int)blockIdx.x * kDsaWaves + wave) * bpw);   // first 32-key block
  const int cols = a.out_cols, n_blocks = min(bpw, (cols + 31) / 32 - b0);
  if (n_blocks <= 0) return;   // no barrier below
  const int len = uniform_load(a.ke + row), width = a.bt_width * (a.block / 32);
  const int lim = min(len, width <= 0x3FFFFFF ? width * 32 : 0x7FFFFFFF);
  const int live_blocks = min(n_blocks, (max(lim, 0) + 31) / 32 - b0);
  const float fill = a.clean ? -__builtin_inff() : 0.0f;
  float* out = a.logits + (int64_t)row * a.ld;
  // table entries of this range: lane i holds that of block b0 + i; a negative one reads page 0, as the reference's
  // clamp does (indexer_torch.py:61), and one past the cache reads as no key
  const int bpp = a.block / 32;   // 32-key blocks per page
  int page = 0;
  if (lane < live_blocks) page = max(a.block_table[(int64_t)row * a.bt_stride + (b0 + lane) / bpp], 0);
  half8_t qf[G][NK];
  float wv[G][16];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint8_t* qp = a.q + (int64_t)row * a.q_rs + (int64_t)(32 * g + j) * a.q_hs + h * (D / 2);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) qf[g][kk] = fp8x8_to_f16(*reinterpret_cast<const uint64_t*>(qp + 8 * kk));
    const float* wp = a.w + (int64_t)row * a.w_rs + 32 * g + 4 * h;
#pragma unroll
    for (int r = 0; r < 16; ++r) wv[g][r] = wp[8 * (r >> 2) + (r & 3)];
  }
  uint4 raw[kDsaAhead + 1][PIECES];
  float ksc[kDsaAhead + 1];
  auto load = [&](int i, int slot) {   // block i of the range
    const int pg_i = __builtin_amdgcn_readlane(page, i);
    const int in = (b0 + i) % bpp * 32;   // first key within the page
    const uint8_t* pg = a.k + (int64_t)(pg_i < a.num_pages ? pg_i : 0) * a.page_bytes;
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
      raw[slot][p] = *reinterpret_cast<const uint4*>(pg + (uint32_t)((in + j) * D + h * (D / 2) + 16 * p));
    ksc[slot] = *reinterpret_cast<const float*>(pg + (uint32_t)(a.block * D + 4 * (in + j)));
  };
  auto compute = [&](int i, int slot) {
    float acc = 0.0f;
    half8_t kv[NK];
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      kv[2 * p] = fp8x8_to_f16((uint64_t)raw[slot][p].x | ((uint64_t)raw[slot][p].y << 32));
      kv[2 * p + 1] = fp8x8_to_f16((uint64_t)raw[slot][p].z | ((uint64_t)raw[slot][p].w << 32));
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float16_t s = {};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(qf[g][kk], kv[kk], s, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; ++r) acc += fmaxf(s[r], 0.0f) * wv[g][r];
    }
    // the other 16 heads of each group are in the lane 32 apart
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
    const float total = (__uint_as_float(sw[0]) + __uint_as_float(sw[1])) * ksc[slot];
    const int key = 32 * (b0 + i) + j;
    const bool live = key < lim && __builtin_amdgcn_readlane(page, i) < a.num_pages;
    if (h == 0 && key < cols) out[key] = live ? total : fill;
  };
  if (live_blocks > 0) {
#pragma unroll
    for (int s = 0; s < kDsaAhead; ++s)
      if (s < live_blocks) load(s, s);
    // kDsaAhead + 1 blocks per trip, so every register slot is a constant; the trips before the last blocks test
    // nothing
    constexpr int S = kDsaAhead + 1;
    int i = 0;
    for (; i + S + kDsaAhead <= live_blocks; i += S) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        load(i + s + kDsaAhead, (s + kDsaAhead) % S);
        compute(i + s, s);
      }
    }
#pragma unroll
    for (int s = 0; s < S + kDsaAhead - 1; ++s) {   // the rest (fewer than S + kDsaAhead blocks)
      if (i + s + kDsaAhead < live_blocks) load(i + s + kDsaAhead, (s + kDsaAhead) % S);
      if (i + s < live_blocks) compute(i + s, s % S);
    }
  }
  for (int i = max(live_blocks, 0); i < n_blocks; ++i) {
    const int key = 32 * (b0 + i) + j;
    if (h == 0 && key < cols) out[key] = fill;
  }
}

}  // namespace
}  // namespace xt

using namespace xt;

extern "C" int xt_topk_rows(const float* x, int64_t ld, int rows, int cols, int topk, int32_t* out, int64_t out_ld,
                            xt_stream_t stream) {
  const char* what = "xt_topk_rows";
  if (rows < 0 || cols < 0 || topk < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (rows == 0 || topk == 0) return ok();
  if (!out || (!x && cols > 0)) return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (ld < cols || out_ld < topk) return fail(XT_EINVAL, "%s: row strides shorter than the rows", what);
  // empty rows stream, reading nothing, and come out all -1
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // Short rows stream while every row is on the CUs at once (two workgroups to a CU): the 8192-bucket histogram costs
  // more than the passes it saves. 512 keys, streamed / in registers: up to 2048 columns with at most a row per CU (32
  // rows x 1000 columns 6.4 / 8.8 us, x 2048 8.0 / 8.8 us), up to 1024 with two (512 x 1000 9.3 / 9.8 us; 257 x 1300
  // 9.4 / 9.4 us). Past that the register form's four workgroups to a CU win at any length (513 rows x 400 11.5 / 10.3
  // us, 1024 x 1000 16.6 / 12.4 us).
  const int streamed = rows <= device_cus() ? 2048 : rows <= 2 * device_cus() ? 1024 : 0;
  if (cols > streamed && cols <= kTopkRegMax) {
    const auto go = [&](auto kernel, int threads) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3((unsigned)threads), 0, st, x, ld, cols, topk, out, out_ld);
    };
    const bool al = cols % 4 == 0;
    // past one round at one workgroup per CU two packed rows share a CU (whole / packed: 257 rows x 20000 columns 22.5
    // / 19.8 us, x 98304 53.7 / 44.1; 520 x 65536 59.2 / 55.9; 2048 x 32768 105 / 81; up to 16384 columns whole keys
    // fit twice or more often as they are)
    const bool many = rows > device_cus();
#define XT_TOPK(TH, CH, PACK, RULE)                                                                                  \
  if (cols <= 4 * TH * CH && (RULE)) {                                                                               \
    al ? go(topk_rows_reg_kernel<TH, CH, true, PACK>, TH) : go(topk_rows_reg_kernel<TH, CH, false, PACK>, TH);       \
    return check_launch(what);                                                                                       \
  }
    XT_TOPK(256, 4, false, true) XT_TOPK(512, 4, false, true) XT_TOPK(1024, 4, false, true)
    XT_TOPK(512, 16, true, many) XT_TOPK(1024, 8, false, true) XT_TOPK(512, 24, true, many)
    XT_TOPK(1024, 12, false, true)
    XT_TOPK(512, 32, true, many) XT_TOPK(1024, 16, false, true) XT_TOPK(512, 48, true, many)
    XT_TOPK(1024, 24, false, true) XT_TOPK(1024, 48, true, true)
#undef XT_TOPK
  }
  hipLaunchKernelGGL(topk_rows_kernel, dim3((unsigned)rows), dim3(kTopkThreads), 0, st, x, ld, cols, topk, out, out_ld);
  return check_launch(what);
}

// Workgroups of one instantiation that fit a CU at once (its register use sets it), read once per process.
template <int H, int NK, bool BF>
static int qsa_per_cu() {
  static std::atomic<int> cached{0};
  int n = cached.load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, qsa_logits_kernel<H, NK, BF>, 64 * kQsaWaves, 0) !=
            hipSuccess || n <= 0)
      n = 1;
    cached.store(n, std::memory_order_relaxed);
  }
  return n;
}

// Rows too far apart for the LDS kernel's 31-bit offsets. The grid: row tiles x key chunks, the chunks sized so that
// the workgroups fit one round on the CUs (a second round of a few workgroups would take as long as the first: 558
// workgroups at 512 per round measured 116 us).
template <int H, int NK, bool BF>
static void qsa_go(QsaArgs a, int row_tiles, hipStream_t st) {
  const int64_t slots = (int64_t)device_cus() * qsa_per_cu<H, NK, BF>();
  const int64_t chunks = std::max<int64_t>(1, slots / row_tiles);
  a.keys_per_wg = (int)std::max<int64_t>(32, ((a.keys + chunks - 1) / chunks + 31) / 32 * 32);
  const dim3 grid((unsigned)row_tiles, (unsigned)((a.keys + a.keys_per_wg - 1) / a.keys_per_wg));
  hipLaunchKernelGGL((qsa_logits_kernel<H, NK, BF>), grid, dim3(64 * kQsaWaves), 0, st, a);
}

// As qsa_go, with the workgroups that fit a CU at two (the LDS and registers of the kernel); whole stages per chunk.
template <int H, int NK, int G, bool BF>
static void qsa_lds_go(QsaArgs a, hipStream_t st) {
  constexpr int rows_wg = kQsaWaves * G * (32 / H);
  const int tiles = (a.rows + rows_wg - 1) / rows_wg;
  const int64_t chunks = std::max<int64_t>(1, 2 * device_cus() / tiles);
  constexpr int S = kQsaStage<NK, G>;
  a.keys_per_wg = (int)std::max<int64_t>(S, ((a.keys + chunks - 1) / chunks + S - 1) / S * S);
  const dim3 grid((unsigned)tiles, (unsigned)((a.keys + a.keys_per_wg - 1) / a.keys_per_wg));
  hipLaunchKernelGGL((qsa_logits_lds_kernel<H, NK, G, BF>), grid, dim3(64 * kQsaWaves), 0, st, a);
}

template <int H>
static int qsa_lds_launch(int nk, bool bf, const QsaArgs& a, hipStream_t st) {
  // the fewest column groups whose rows one workgroup holds, else as many as the registers do, except where four (and
  // their longer stages) would leave a CU without its two workgroups
  const int64_t wgs4 = ((int64_t)a.rows * H + 511) / 512 * ((a.keys + 127) / 128);
#define XT_QSA(NK, G)                                                                                                \
  if (nk == NK && (a.rows <= kQsaWaves * G * (32 / H) || G == (NK <= 8 ? 4 : 2) ||                                   \
                   (G == 2 && wgs4 < 2 * device_cus()))) {                                                           \
    bf ? qsa_lds_go<H, NK, G, true>(a, st) : qsa_lds_go<H, NK, G, false>(a, st);                                     \
    return XT_OK;                                                                                                    \
  }
  XT_QSA(4, 1) XT_QSA(4, 2) XT_QSA(4, 4) XT_QSA(8, 1) XT_QSA(8, 2) XT_QSA(8, 4) XT_QSA(16, 1) XT_QSA(16, 2)
#undef XT_QSA
  return XT_EUNSUPPORTED;
}

template <int H>
static int qsa_launch(int nk, bool bf, const QsaArgs& a, int row_tiles, hipStream_t st) {
#define XT_QSA(NK)                                                                                                    \
  if (nk == NK) {                                                                                                    \
    if (bf)                                                                                                          \
      qsa_go<H, NK, true>(a, row_tiles, st);                                                                         \
    else                                                                                                             \
      qsa_go<H, NK, false>(a, row_tiles, st);                                                                        \
    return XT_OK;                                                                                                    \
  }
  XT_QSA(4)
  XT_QSA(8)
  XT_QSA(16)
#undef XT_QSA
  return XT_EUNSUPPORTED;
}

extern "C" int xt_qsa_indexer_logits(const void* q, int64_t q_row_stride, int64_t q_head_stride, int rows, int heads,
                                     int dim, const void* k, int64_t k_row_stride, int keys, const int32_t* starts,
                                     const int32_t* ends, float score_scale, int dtype, float* logits, int64_t ld,
                                     xt_stream_t stream) {
  const char* what = "xt_qsa_indexer_logits";
  if (rows < 0 || keys < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (rows == 0 || keys == 0) return ok();
  if (!q || !k || !starts || !ends || !logits) return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (heads != 1 && heads != 2 && heads != 4 && heads != 8 && heads != 16 && heads != 32)
    return fail(XT_EUNSUPPORTED, "%s: %d heads (supported: powers of 2 up to 32)", what, heads);
  if (dim != 64 && dim != 128 && dim != 256) return fail(XT_EUNSUPPORTED, "%s: head size %d (64, 128, 256)", what, dim);
  if (dtype != XT_DTYPE_BF16 && dtype != XT_DTYPE_F16) return fail(XT_EINVAL, "%s: q / k must be BF16 or FP16", what);
  if (!aligned(q, 16) || !aligned(k, 16) || q_row_stride % 8 || q_head_stride % 8 || k_row_stride % 8 ||
      ld < keys || !(score_scale > 0.0f))
    return fail(XT_EINVAL, "%s: rows must be 16-byte aligned, ld >= keys, score_scale > 0", what);
  QsaArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.q_rs = q_row_stride;
  a.q_hs = q_head_stride;
  a.k = static_cast<const uint16_t*>(k);
  a.k_rs = k_row_stride;
  a.starts = starts;
  a.ends = ends;
  a.score_scale = score_scale;
  a.logits = logits;
  a.ld = ld;
  a.rows = rows;
  a.keys = keys;
  a.keys_per_wg = 1024;   // set with the grid in qsa_go
  a.vec_store = (ld % 4 == 0) && aligned(logits, 16);
  const int rows_per_wg = kQsaWaves * kQsaGroups * (32 / heads);
  const int row_tiles = (rows + rows_per_wg - 1) / rows_per_wg;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool bf = dtype == XT_DTYPE_BF16;
  const int nk = dim / 16;
  int e = XT_EUNSUPPORTED;
  // the LDS kernel's store offsets are 31-bit: its rows per workgroup (512 / heads, 256 / heads at 256 dims) times ld
  if ((int64_t)(512 / heads) * ld * 4 + 4 * (int64_t)keys < 0x7FFFFFFF) {
    switch (heads) {
      case 1: e = qsa_lds_launch<1>(nk, bf, a, st); break;
      case 2: e = qsa_lds_launch<2>(nk, bf, a, st); break;
      case 4: e = qsa_lds_launch<4>(nk, bf, a, st); break;
      case 8: e = qsa_lds_launch<8>(nk, bf, a, st); break;
      case 16: e = qsa_lds_launch<16>(nk, bf, a, st); break;
      case 32: e = qsa_lds_launch<32>(nk, bf, a, st); break;
    }
    if (e != XT_OK) return fail(e, "%s: no kernel for %d heads x %d", what, heads, dim);
    return check_launch(what);
  }
  switch (heads) {
    case 1: e = qsa_launch<1>(nk, bf, a, row_tiles, st); break;
    case 2: e = qsa_launch<2>(nk, bf, a, row_tiles, st); break;
    case 4: e = qsa_launch<4>(nk, bf, a, row_tiles, st); break;
    case 8: e = qsa_launch<8>(nk, bf, a, row_tiles, st); break;
    case 16: e = qsa_launch<16>(nk, bf, a, row_tiles, st); break;
    case 32: e = qsa_launch<32>(nk, bf, a, row_tiles, st); break;
  }
  if (e != XT_OK) return fail(e, "%s: no kernel for %d heads x %d", what, heads, dim);
  return check_launch(what);
}

static int dsa_common(const char* what, DsaArgs& a, int dim, xt_stream_t stream) {
  if (a.heads % 32 || a.heads <= 0 || a.heads > 128)
    return fail(XT_EUNSUPPORTED, "%s: %d heads (supported: 32, 64, 96, 128)", what, a.heads);
  if (dim != 64 && dim != 128 && dim != 256) return fail(XT_EUNSUPPORTED, "%s: head size %d (64, 128, 256)", what, dim);
  if (!aligned(a.q, 8) || a.q_rs % 8 || a.q_hs % 8 || !aligned(a.w, 4) || a.ld < a.out_cols)
    return fail(XT_EINVAL, "%s: q rows must be 8-byte aligned and ld >= the columns written", what);
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int nk = dim / 16, groups = a.heads / 32;
  if (a.block > 0 && a.block % 32 == 0 && groups * nk <= 16 && aligned(a.k, 16) && a.page_bytes % 16 == 0 &&
      a.num_q <= 65535) {
    // blocks per wavefront: about 8 wavefronts per CU over the whole [rows, columns] area, at most 64 (one table
    // entry per lane). Rows end early at their lengths, and the workgroups behind write the fill and leave. More
    // wavefronts repeat the query's load and conversion (16 per CU: 22.8 us, 32: 23.3), fewer leave CUs short of loads
    // (6: 25.9 us).
    const int64_t blocks = ((int64_t)a.out_cols + 31) / 32;
    const int64_t per = (blocks * a.num_q + 8 * device_cus() - 1) / (8 * device_cus());
    const int bpw = (int)std::min<int64_t>(64, std::max<int64_t>(1, per));
    const dim3 grid((unsigned)((blocks + (int64_t)bpw * kDsaWaves - 1) / (bpw * kDsaWaves)), (unsigned)a.num_q);
#define XT_DSA_PAGED(NK, G)                                                                                          \
  if (nk == NK && groups == G) {                                                                                     \
    hipLaunchKernelGGL((dsa_paged_kernel<NK, G>), grid, dim3(64 * kDsaWaves), 0, st, a, bpw);                       \
    return check_launch(what);                                                                                       \
  }
    XT_DSA_PAGED(4, 1) XT_DSA_PAGED(4, 2) XT_DSA_PAGED(4, 3) XT_DSA_PAGED(4, 4) XT_DSA_PAGED(8, 1) XT_DSA_PAGED(8, 2)
    XT_DSA_PAGED(16, 1)
#undef XT_DSA_PAGED
  }
  a.keys_per_wg = 4096;
  const dim3 grid((unsigned)((a.num_q + kDsaWaves - 1) / kDsaWaves), (unsigned)((a.out_cols + 4095) / 4096));
  if (a.block == 0 && groups * nk <= 16 && aligned(a.k, 16) && a.k_rs % 16 == 0) {
#define XT_DSA_FLAT(NK, G)                                                                                           \
  if (nk == NK && groups == G) {                                                                                     \
    hipLaunchKernelGGL((dsa_flat_kernel<NK, G>), grid, dim3(64 * kDsaWaves), 0, st, a);                             \
    return check_launch(what);                                                                                       \
  }
    XT_DSA_FLAT(4, 1) XT_DSA_FLAT(4, 2) XT_DSA_FLAT(4, 3) XT_DSA_FLAT(4, 4) XT_DSA_FLAT(8, 1) XT_DSA_FLAT(8, 2)
    XT_DSA_FLAT(16, 1)
#undef XT_DSA_FLAT
  }
  switch (dim / 16) {
    case 4: hipLaunchKernelGGL(dsa_logits_kernel<4>, grid, dim3(64 * kDsaWaves), 0, st, a); break;
    case 8: hipLaunchKernelGGL(dsa_logits_kernel<8>, grid, dim3(64 * kDsaWaves), 0, st, a); break;
    default: hipLaunchKernelGGL(dsa_logits_kernel<16>, grid, dim3(64 * kDsaWaves), 0, st, a); break;
  }
  return check_launch(what);
}

extern "C" int xt_dsa_mqa_logits(const void* q, int64_t q_row_stride, int64_t q_head_stride, int num_q, int heads,
                                 int dim, const void* k, int64_t k_row_stride, const float* k_scale, int num_kv,
                                 const float* weights, int64_t w_row_stride, const int32_t* ks, const int32_t* ke,
                                 int clean_logits, float* logits, int64_t ld, xt_stream_t stream) {
  const char* what = "xt_dsa_mqa_logits";
  if (num_q < 0 || num_kv < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (num_q == 0 || num_kv == 0) return ok();
  if (!q || !k || !k_scale || !weights || !logits) return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (!aligned(k, 8) || k_row_stride % 8 || k_row_stride < dim)
    return fail(XT_EINVAL, "%s: key rows must be 8-byte aligned", what);
  DsaArgs a = {};
  a.q = static_cast<const uint8_t*>(q);
  a.q_rs = q_row_stride;
  a.q_hs = q_head_stride;
  a.k = static_cast<const uint8_t*>(k);
  a.k_rs = k_row_stride;
  a.k_scale = k_scale;
  a.block = 0;
  a.w = weights;
  a.w_rs = w_row_stride;
  a.ks = ks;
  a.ke = ke;
  a.clean = clean_logits;
  a.logits = logits;
  a.ld = ld;
  a.num_q = num_q;
  a.num_kv = num_kv;
  a.heads = heads;
  a.out_cols = num_kv;
  return dsa_common(what, a, dim, stream);
}

extern "C" int xt_dsa_paged_mqa_logits(const void* q, int64_t q_row_stride, int64_t q_head_stride, int batch,
                                       int heads, int dim, const void* kvcache, int64_t num_pages, int64_t page_bytes,
                                       int block,
                                       const int32_t* block_table, int64_t bt_stride, int bt_width,
                                       const int32_t* context_lens, const float* weights, int64_t w_row_stride,
                                       int max_seq_len, int clean_logits, float* logits, int64_t ld,
                                       xt_stream_t stream) {
  const char* what = "xt_dsa_paged_mqa_logits";
  if (batch < 0 || max_seq_len < 0) return fail(XT_EINVAL, "%s: negative size", what);
  if (batch == 0 || max_seq_len == 0) return ok();
  if (!q || !kvcache || !block_table || !context_lens || !weights || !logits)
    return fail(XT_EINVAL, "%s: a required pointer is null", what);
  if (block <= 0 || num_pages <= 0 || page_bytes < (int64_t)block * (dim + 4) || page_bytes % 8 ||
      !aligned(kvcache, 8) || bt_width <= 0 || bt_stride < bt_width)
    return fail(XT_EINVAL, "%s: pages of %d keys need %d bytes each (8-byte aligned)", what, block, block * (dim + 4));
  DsaArgs a = {};
  a.q = static_cast<const uint8_t*>(q);
  a.q_rs = q_row_stride;
  a.q_hs = q_head_stride;
  a.k = static_cast<const uint8_t*>(kvcache);
  a.page_bytes = page_bytes;
  a.num_pages = num_pages;
  a.block = block;
  a.block_table = block_table;
  a.bt_stride = bt_stride;
  a.bt_width = bt_width;
  a.w = weights;
  a.w_rs = w_row_stride;
  a.ks = nullptr;
  a.ke = context_lens;
  a.clean = clean_logits;
  a.logits = logits;
  a.ld = ld;
  a.num_q = batch;
  a.num_kv = bt_width * block;
  a.heads = heads;
  a.out_cols = max_seq_len;
  return dsa_common(what, a, dim, stream);
}
