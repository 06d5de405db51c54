// Quantize-on-flush, hot-ring append and group reconstruction (gfx950).
//
// Bit-exactness contract (this file is compiled with -ffp-contract=off and
// uses explicitly rounded __f*_rn operations): every code, scale, mean, norm
// and outlier entry equals what the reference's NumPy encoder produces for the
// same fp16 inputs.  NumPy's operation order is restated exactly:
//   keys   (turboquant_pro/per_channel_kv.py:269-401, nf4_asym)
//     mean  = token-order sequential fp32 sum / G ("calibrated"; "sparse"
//             multiplies it by the DC-channel mask, "bias" takes it given)
//     amax  = max(max_s |x_s - mean|, 1e-8)            (NaN propagates)
//     cent  = mean + amax * NF4[l]
//     code  = first argmin_l |x - cent_l|               (NaN counts as minimal)
//     outlier threshold = k-th largest |x| (ties kept), flat (s, j) order
//   values (turboquant_pro/core.py:569-606, CPU full-QR branch)
//     norm  = sqrt(pairwise sum of squares)              (numpy pairwise_sum, n = D)
//     u     = v / max(norm, 1e-30)
//     y_e   = sequential over d of (u_d * PiT[d][e]), separately rounded
//     code  = #{ boundaries < y_e }                      (searchsorted, side="left";
//                                                         a NaN y_e takes the last code)
#include "tqk_common.h"

namespace {

constexpr int kThreads = 256;
// The group encodes by the largest group they take (MG tokens).  256: eight
// waves; the LDS (under 80 KiB at head_dim 128) lets two workgroups share a CU,
// four waves per SIMD.  64 (and 128, fp16 at head_dim 64): four waves and a
// smaller key tile, so that four workgroups do: a short group is a chain of latencies, in which eight
// waves wait no shorter than four.  8 sequences x 2000 tokens x 8 heads, NF4 keys
// with a side-list, us by eight waves / by four: groups of 8 tokens at head_dim 64
// 598 / 365, of 32 at 64 183 / 129, at 128 in fp32 300 / 265, at 256 850 / 502.
constexpr int enc_threads(int MG) { return MG > 128 ? 512 : 256; }
// tokens of a batch of PolarQuant rows: four threads each
constexpr int enc_batch(int MG) { return enc_threads(MG) / 4; }

// the order of stored codes, as PolarStage has it
struct TokenRows { static constexpr bool value = false; };
struct TiledRows { static constexpr bool value = true; };

// What an append of a few sequences passes with the launch instead of in device
// memory: a copy to the device and its launch cost more than the append itself.
constexpr int kInlineSeqs = 64, kInlineItems = 128;
struct InlineItems {
  int32_t prev[kInlineSeqs];
  int32_t item[2 * kInlineItems];
};

struct EncodeArgs {
  tqk_cache_desc d;
  tqk_cache_ptrs p;
  const int32_t* items;     // nullptr: in.item, in.prev
  const int32_t* prev_len;
  const void* chunk_k;  // fp16, or fp32 (input_f32)
  const void* chunk_v;
  int chunk_tokens;
  int n_items;
  int unit0;  // first (item, kv head) of the launch, a multiple of 8
  int32_t* overflow;
  InlineItems in;
};
__device__ __forceinline__ int item_word(const EncodeArgs& a, int i) { return a.items ? a.items[i] : a.in.item[i]; }

// Source row (D values of type T: fp16 bits or fp32) of token t of sequence
// b, kv head h: the hot ring for tokens already in the cache, the appended
// chunk for new ones.
template <int D, typename T = uint16_t>
__device__ __forceinline__ const T* token_src(const EncodeArgs& a, const void* ring,
                                              const void* chunk, int b, int h, int t) {
  const tqk_cache_desc& d = a.d;
  const int prev = a.items ? a.prev_len[b] : a.in.prev[b];
  if (t < prev)
    return static_cast<const T*>(ring) +
           (((size_t)b * d.n_kv_heads + h) * d.hot_ring + (t % d.hot_ring)) * D;
  return static_cast<const T*>(chunk) + (((size_t)b * d.n_kv_heads + h) * a.chunk_tokens + (t - prev)) * D;
}

__device__ __forceinline__ uint32_t abs_h(uint16_t x) { return x & 0x7FFFu; }

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

// v into the K-long descending lists held in the two halves of t (one
// packed 16-bit max and min per list entry)
template <int K>
__device__ __forceinline__ void topk_insert(u16x2_t (&t)[K], u16x2_t v) {
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const u16x2_t hi = __builtin_elementwise_max(t[i], v);
    v = __builtin_elementwise_min(t[i], v);
    t[i] = hi;
  }
}

// The k-th largest (1 <= k <= K) of a channel's magnitude patterns, held two
// per register in m by the four lanes l, l ^ 16, l ^ 32, l ^ 48: each lane
// keeps the K largest of each half of its registers, the halves' lists are
// merged, then the lanes' lists over the two permlane swaps.  The largest T
// with #{m >= T} >= k is exactly this k-th largest value (with multiplicity),
// so it equals the bitwise threshold search's result.
template <int K, int N>
__device__ __forceinline__ uint32_t kth_largest(const u16x2_t (&m)[N], int k, int G) {
  u16x2_t t[K];
#pragma unroll
  for (int i = 0; i < K; ++i) t[i] = u16x2_t{0, 0};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    topk_insert<K>(t, m[i]);
  }
  {
    u16x2_t sw[K];
#pragma unroll
    for (int i = 0; i < K; ++i) sw[i] = t[i].yx;
#pragma unroll
    for (int i = 0; i < K; ++i) topk_insert<K>(t, sw[i]);
  }
  // a permlane swap returns this lane's list and its partner's, in an order
  // that depends on the lane; the merge is symmetric in the two
#pragma unroll
  for (int step = 0; step < 2; ++step) {
    u16x2_t other[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const uint32_t x = __builtin_bit_cast(uint32_t, t[i]);
      const auto r = step == 0 ? __builtin_amdgcn_permlane32_swap(x, x, false, false)
                               : __builtin_amdgcn_permlane16_swap(x, x, false, false);
      t[i] = __builtin_bit_cast(u16x2_t, (uint32_t)r[0]);
      other[i] = __builtin_bit_cast(u16x2_t, (uint32_t)r[1]);
    }
#pragma unroll
    for (int i = 0; i < K; ++i) topk_insert<K>(t, other[i]);
  }
  uint32_t T = t[0].x;
#pragma unroll
  for (int i = 1; i < K; ++i)
    if (i == k - 1) T = t[i].x;
  return T;
}

// Sum over lanes l, l ^ 16, l ^ 32, l ^ 48 (the four 16-lane rows).
__device__ __forceinline__ int sum_quarters(int x) {
  auto a = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
  x = (int)(a[0] + a[1]);
  auto b = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
  return (int)(b[0] + b[1]);
}


// ---- asym-NF4 codes by bucket -----------------------------------------------
// With the normalised key t = (x - mean) / amax cut into 32 buckets of 1/16 on
// [-1, 1], every bucket widened by 0.004 on both sides holds at most one
// midpoint of two NF4 levels (they are at least 0.080 apart), so a bucket's
// codes are those of its pair k (kNf4From[k] <= bucket < kNf4From[k + 1]), k and
// k + 1, and one comparison of x decides:
// code = pair + (x >= X), X the smallest fp16 number that argmin puts on the
// pair's upper level.  kNf4From[k] is the first bucket of pair k.
__constant__ static const int kNf4From[16] = {0, 3, 7, 9, 11, 13, 14, 16, 17, 18, 20, 21, 23, 25, 27, 32};

// the smallest fp16 number x (as bits; 0x7C00 when there is none) with
// fl|x - c1| < fl|x - c0|, for levels c0 < c1 far enough apart that the two
// rounded distances order like the real ones away from the midpoint: nearly
// always next to the rounded midpoint, else searched for
__device__ __forceinline__ uint16_t nf4_threshold(float c0, float c1) {
  auto bits = [](int o) { return (uint16_t)(o < 0 ? 0x8000 - o : o); };
  auto upper = [&](int o) {
    const float x = h2f(bits(o));
    return x >= c1 || (x > c0 && fabsf(__fsub_rn(x, c1)) < fabsf(__fsub_rn(x, c0)));
  };
  const uint16_t mb = f2h(0.5f * c0 + 0.5f * c1);
  const int m = (mb & 0x8000) ? -(int)(mb & 0x7FFF) : (int)mb;
  if (m > -0x7BFF && m < 0x7BFF && !upper(m - 1) && upper(m + 1)) return bits(upper(m) ? m : m + 1);
  int lo = -0x7C00, hi = 0x7C00;  // not upper, upper (neither is evaluated)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (upper(mid)) hi = mid;
    else lo = mid;
  }
  return bits(hi);
}

// One workgroup per (group, kv head) and side: eight consecutive key
// workgroups, then the eight value workgroups of the same groups, so that
// every XCD and CU gets both kinds and a flush of one group runs them side by
// side.  What bounds it: the keys' VALU work and LDS traffic (statistics,
// thresholds, side-list, codes): 32 sequences x 4096 tokens x 8 heads, NF4 keys
// with a side-list, VALU 65 % busy at four waves per SIMD, LDS 22 %, a quarter of
// that bank conflicts, matrix cores 5 %.  16 sequences x 8192 tokens x 8 heads at
// head_dim 128, appended in 4096-token chunks: 868 us with both sides in one
// 256-thread workgroup and the argmin over 16 levels, 629 us like this.
template <int VB, int D, int MG>
__global__ __launch_bounds__(enc_threads(MG), D <= 128 ? 4 : 2) void tqk_encode_group(EncodeArgs a) {
  constexpr int kEncThreads = enc_threads(MG), kEncWaves = kEncThreads / 64, kVBatch = enc_batch(MG);
  using Stage = PolarStage<D, kVBatch>;
  const int unit = a.unit0 + (int)(blockIdx.x >> 4) * 8 + (int)(blockIdx.x & 7u);
  const bool key_side = ((blockIdx.x >> 3) & 1u) == 0u;
  if (unit >= a.n_items * a.d.n_kv_heads) return;
  const int item = unit % a.n_items, h = unit / a.n_items, tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const tqk_cache_desc& d = a.d;
  const int b = item_word(a, 2 * item), g = item_word(a, 2 * item + 1);
  const int G = d.group_tokens, P = d.page_tokens, Hkv = d.n_kv_heads;
  const int slot = a.p.group_table[(size_t)b * d.max_groups_per_seq + g];
  const int kout = d.outliers_per_channel;
  const size_t mbase = ((size_t)slot * Hkv + h) * D;
  const size_t obase = (size_t)slot * Hkv + h;

  // Key tile (fp16 bits, rows padded against bank conflicts).  Its rows also
  // take the key codes: the codes of token t overwrite the first D / 2 bytes of
  // row t once the wave that owns the row has read it (kc_row).  On the value
  // side the area holds the rows and stage of a value batch.
  constexpr size_t kBatchBytes = sizeof(uint16_t) * kVBatch * (D + 8);
  constexpr size_t kTileBytes = sizeof(uint16_t) * MG * (D + 8);
  static_assert(kBatchBytes % 16 == 0, "the stage follows the batch's rows");
  __shared__ __align__(16) uint8_t area_s[kTileBytes > kBatchBytes + sizeof(Stage) ? kTileBytes : kBatchBytes + sizeof(Stage)];
  uint16_t (*kt_s)[D + 8] = reinterpret_cast<uint16_t (*)[D + 8]>(area_s);
  __shared__ float stat_s[D][2];             // per channel: (mean, amax) or (min, scale)
  // per channel: 0x8000 - the fp16 magnitude threshold T (so m + it has bit 15
  // set exactly when m >= T; 0 for a NaN T), read eight channels at a time by
  // the side-list scan
  __shared__ __align__(16) uint16_t tbias_s[D];
  // channels of each token stored in the side-list: in the tile rows' padding
  // where it fits
  __shared__ uint32_t omx_s[D > 128 ? MG : 1][D / 32];
  // per bucket and channel (of 64 channels): X | rev4(code) << 16 | rev4(code +
  // 1) << 20; row 32: the stored outliers' code.  Channel c at column (c >> 1) +
  // 32 (c & 1): the two half-waves read columns of different halves at a time,
  // so a wave's reads never share a bank.
  __shared__ uint32_t nf_s[33][64];
  __shared__ uint32_t crowded_s;  // bit of every 64 channels with levels too close for the buckets
  __shared__ int32_t wsum_s[kEncWaves];
  auto kc_row = [&](int t) { return reinterpret_cast<uint8_t*>(&kt_s[t][0]); };
  auto om_row = [&](int t) {
    if constexpr (D > 128) return &omx_s[t][0];
    else return reinterpret_cast<uint32_t*>(&kt_s[t][D]);
  };

  if (d.key_grid != 2 && key_side) {
    // ---- stage the key tile ----------------------------------------------
    for (int idx = tid; idx < G * (D / 8); idx += kEncThreads) {
      const int t = idx / (D / 8), c = idx % (D / 8);
      const uint4* src =
          reinterpret_cast<const uint4*>(token_src<D>(a, a.p.hot_k, a.chunk_k, b, h, g * G + t));
      reinterpret_cast<uint4*>(&kt_s[t][0])[c] = src[c];
    }
    if (tid == 0) crowded_s = 0u;
    __syncthreads();

    // ---- the zero point (turboquant_pro/per_channel_kv.py:327-345), thread j:
    // channel j, a sum in token order
    if (tid < D && d.key_grid != 1) {
      const int j = tid;
      float mu;
      if (d.zero_point == 2) {
        // "bias": the RoPE-averaged k_proj bias of the group's positions
        mu = a.p.zp_mean[((size_t)g * Hkv + h) * D + j];
      } else {
        float acc = 0.0f;
        int s = 0;
        for (; s + 16 <= G; s += 16) {
          uint16_t x[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) x[u] = kt_s[s + u][j];
#pragma unroll
          for (int u = 0; u < 16; ++u) acc = __fadd_rn(acc, h2f(x[u]));
        }
        for (; s < G; ++s) acc = __fadd_rn(acc, h2f(kt_s[s][j]));
        // np.mean divides the fp32 sum by an intp count: a float64 division, then fp32
        mu = (float)((double)acc / (double)G);
        // "sparse": the mean times the DC-channel mask (a float product, so a
        // non-DC channel gets a signed zero, or NaN from a NaN mean)
        if (d.zero_point == 1) mu = __fmul_rn(mu, ((d.dc_mask[j >> 5] >> (j & 31)) & 1u) ? 1.0f : 0.0f);
      }
      stat_s[j][0] = mu;
    }
    __syncthreads();
    // ---- the other statistics and the outlier thresholds, 16 channels per
    // wave and pass: lanes l, l ^ 16, l ^ 32, l ^ 48 hold a quarter of the
    // tokens each, two per register.
    // Thresholds: the k-th largest |x| of each channel as the largest fp16
    // magnitude pattern T with #{ |x_s| >= T } >= k (NaN patterns order above
    // inf, as np.partition does).  For k <= 8 the k largest are kept directly
    // (packed 16-bit max/min insertion); otherwise a bitwise search, a
    // candidate's count the carry bit of a packed 16-bit add, summed over the
    // four lanes.
    {
      const int part = lane >> 4;
      for (int j = 16 * wv + (lane & 15); j < D; j += 16 * kEncWaves) {
        // lane quarter `part` takes token pairs 8i + 2 part (rows 4 apart fall on
        // LDS banks 8 apart, so the four quarters never conflict); eight pairs
        // at a time, pairs past G repeat the last token
        auto for_quarter = [&](auto f) {
#pragma unroll 1
          for (int i0 = 0; 8 * i0 < G; i0 += 8) {
            uint16_t x[16];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int s = 8 * (i0 + i) + 2 * part;
              x[2 * i] = kt_s[min(s, G - 1)][j];
              x[2 * i + 1] = kt_s[min(s + 1, G - 1)][j];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) f(x[2 * i], x[2 * i + 1]);
          }
        };
        // NaN propagates into scale and zero point
        uint32_t top = 0;  // the largest magnitude pattern
        if (d.key_grid == 1) {
          // uniform (turboquant_pro/per_channel_kv.py:303-306): channel min and
          // max, scale = max(max - min, 1e-8) / (2^bits - 1)
          float mn = __builtin_inff(), mx = -__builtin_inff();
          for_quarter([&](uint16_t ya, uint16_t yb) {
            top = max(top, max(abs_h(ya), abs_h(yb)));
            const float x0 = h2f(ya), x1 = h2f(yb);
            mn = fminf(mn, fminf(x0, x1));
            mx = fmaxf(mx, fmaxf(x0, x1));
          });
#pragma unroll
          for (int o = 16; o < 64; o <<= 1) {
            mn = fminf(mn, __shfl_xor(mn, o, 64));
            mx = fmaxf(mx, __shfl_xor(mx, o, 64));
            top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
          }
          if (part == 0) {
            const bool nan = top > 0x7C00u;
            const float sc = nan ? __builtin_nanf("")
                                 : __fdiv_rn(fmaxf(__fsub_rn(mx, mn), 1e-8f), (float)((1 << d.key_bits) - 1));
            if (nan) mn = __builtin_nanf("");
            stat_s[j][0] = mn;
            stat_s[j][1] = sc;
            a.p.gscale[mbase + j] = sc;
            a.p.gmean[mbase + j] = mn;
          }
        } else {
          // amax = max |x - mean|, as magnitude patterns (a NaN is the largest)
          const float mu = stat_s[j][0];
          for_quarter([&](uint16_t ya, uint16_t yb) {
            const uint32_t d0 = __float_as_uint(fabsf(__fsub_rn(h2f(ya), mu)));
            const uint32_t d1 = __float_as_uint(fabsf(__fsub_rn(h2f(yb), mu)));
            top = max(top, max(d0, d1));
          });
#pragma unroll
          for (int o = 16; o < 64; o <<= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
          if (part == 0) {
            const float amax = top > 0x7F800000u ? __builtin_nanf("") : fmaxf(__uint_as_float(top), 1e-8f);
            stat_s[j][1] = amax;
            a.p.gscale[mbase + j] = amax;
            a.p.gmean[mbase + j] = mu;
            // sorted levels far enough apart for the rounded distances to order
            // as the real ones: every token has |x - mean| <= amax, so a
            // distance is below R = 2 (|mean| + amax), and gaps of at least
            // R * 2^-19 (16 ulps of R) cannot round away
            const float r = __fmul_rn(__fadd_rn(fabsf(mu), amax), 0x1p-18f);
            bool ok = true;
            float c = __fadd_rn(mu, __fmul_rn(amax, kNF4[0]));
#pragma unroll
            for (int l = 1; l < 16; ++l) {
              const float n = __fadd_rn(mu, __fmul_rn(amax, kNF4[l]));
              ok &= __fsub_rn(n, c) >= r;  // (false for any level that is not finite)
              c = n;
            }
            if (!(ok && __builtin_isfinite(c))) atomicOr(&crowded_s, 1u << (j >> 6));
          }
        }
        if (kout > 0 && kout < G) {
          u16x2_t m2[MG / 8];
#pragma unroll
          for (int i = 0; i < MG / 8; ++i) {
            const int s = 8 * i + 2 * part;  // tokens past G count as magnitude 0
            m2[i] = u16x2_t{(uint16_t)(s < G ? abs_h(kt_s[s][j]) : 0u),
                            (uint16_t)(s + 1 < G ? abs_h(kt_s[s + 1][j]) : 0u)};
            if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);  // (the gathered halves are packed as they come)
          }
          uint32_t T = 0;
          if (kout <= 5) {
            T = kth_largest<5>(m2, kout, G);
          } else if (kout <= 8) {
            T = kth_largest<8>(m2, kout, G);
          } else {
            for (int bit = 14; bit >= 0; --bit) {
              const uint32_t cand = T | (1u << bit);
              // m + (0x8000 - cand) has bit 15 set exactly when m >= cand (m, cand < 2^15)
              const uint16_t bias = (uint16_t)(0x8000u - cand);
              const u16x2_t bv = {bias, bias};
              uint32_t acc = 0;  // two 16-bit counts
#pragma unroll
              for (int i = 0; i < MG / 8; ++i)
                acc += (__builtin_bit_cast(uint32_t, (u16x2_t)(m2[i] + bv)) >> 15) & 0x00010001u;
              const int cnt = sum_quarters((int)((acc & 0xFFFFu) + (acc >> 16)));
              if (cnt >= kout) T = cand;
            }
          }
          // the scan compares magnitudes as floats, as the reference's mask
          // |x| >= t does: a NaN threshold selects nothing (bias 0)
          if (part == 0) tbias_s[j] = (uint16_t)(T > 0x7C00u ? 0u : 0x8000u - T);
        }
      }
    }
    __syncthreads();

    // ---- outlier side-list in flat (token, channel) order, two threads per
    // token, half of the channels each.  ocount holds cumulative counts at
    // every TQK_OBLK-token boundary of the group (entry TQK_NOB-1 = total), so a
    // decode block finds its entries without searching; om_row records the
    // stored (token, channel) positions, whose codes become the grid's zero
    // level below.
    if (kout > 0) {
      static_assert(kEncThreads >= 2 * MG, "two threads per token");
      const bool all = kout >= G;
      constexpr int NW = D / 64;  // mask words per thread
      const int tt = tid >> 1, w0 = NW * (tid & 1);
      // the token's outlier channels, eight at a time: magnitudes and biases
      // as packed 16-bit pairs, bit 15 of each half of m + bias is the test
      // m >= T; NaN magnitudes (m > 0x7C00, where m + 0x03FF reaches bit 15)
      // are never selected, as |x| >= t is false for them
      uint32_t om[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) om[k] = 0u;
      if (tt < G) {
#pragma unroll
        for (int c8 = 0; c8 < D / 16; ++c8) {
          const uint4 xw = *reinterpret_cast<const uint4*>(&kt_s[tt][32 * w0 + 8 * c8]);
          const uint4 bw = *reinterpret_cast<const uint4*>(&tbias_s[32 * w0 + 8 * c8]);
          const uint32_t xs[4] = {xw.x, xw.y, xw.z, xw.w}, bs[4] = {bw.x, bw.y, bw.z, bw.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const u16x2_t m = __builtin_bit_cast(u16x2_t, xs[i] & 0x7FFF7FFFu);
            const uint32_t t = __builtin_bit_cast(uint32_t, (u16x2_t)(m + __builtin_bit_cast(u16x2_t, bs[i])));
            const uint32_t tn = __builtin_bit_cast(uint32_t, (u16x2_t)(m + u16x2_t{0x03FF, 0x03FF}));
            const uint32_t sel = t & ~tn;
            const uint32_t two = ((sel >> 15) & 1u) | ((sel >> 30) & 2u);  // channels 8c8 + 2i, + 1
            om[c8 >> 2] |= two << (8 * (c8 & 3) + 2 * i);
          }
        }
        if (all) {
#pragma unroll
          for (int k = 0; k < NW; ++k) om[k] = 0xFFFFFFFFu;
        }
      }
      int cnt = 0;
#pragma unroll
      for (int k = 0; k < NW; ++k) cnt += __builtin_popcount(om[k]);
      // block exclusive scan of cnt
      int incl = cnt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      if (lane == 63) wsum_s[wv] = incl;
      __syncthreads();
      int wofs = 0, total = 0;
#pragma unroll
      for (int w = 0; w < kEncWaves; ++w) {
        wofs += w < wv ? wsum_s[w] : 0;
        total += wsum_s[w];
      }
      int off = wofs + incl - cnt;
      // token s = TQK_OBLK*k - 1 closes block k-1: its inclusive offset is the bound
      if (tt < G && (tid & 1) && ((tt + 1) % TQK_OBLK) == 0 && (tt + 1) / TQK_OBLK <= TQK_NOB)
        a.p.ocount[obase * TQK_NOB + (tt + 1) / TQK_OBLK - 1] = off + cnt;
      if (tid < TQK_NOB && TQK_OBLK * (tid + 1) > G) a.p.ocount[obase * TQK_NOB + tid] = total;
      if (tt < G) {
        // entries in channel order; those past the side-list's capacity are
        // dropped (and leave their codes alone).  A stored position's key gives
        // way to +inf, the last bucket of the codes below.
#pragma unroll
        for (int k = 0; k < NW; ++k) {
          uint32_t w = om[k];
          while (w) {
            const int j = 32 * (w0 + k) + __builtin_ctz(w);
            w &= w - 1u;
            if (off < d.outlier_cap) {
              a.p.oent[obase * d.outlier_cap + off] = (uint32_t)(tt * D + j) | ((uint32_t)kt_s[tt][j] << 16);
              kt_s[tt][j] = 0x7C00u;
            } else {
              om[k] &= ~(1u << (j & 31));
            }
            ++off;
          }
        }
#pragma unroll
        for (int k = 0; k < NW; ++k) om_row(tt)[w0 + k] = om[k];
      }
      if (tid == 0 && total > d.outlier_cap && a.overflow) atomicOr(a.overflow, TQK_OVF_OUTLIERS);
    } else if (tid < TQK_NOB) {
      a.p.ocount[obase * TQK_NOB + tid] = 0;
    }
    __syncthreads();

    // ---- codes, 64 channels at a time: a wave takes two tokens, a half-wave
    // the 32 channel pairs of one.  The rows belong to their wave alone and
    // 64 channels' codes are 32 bytes at or before the channels' own place, so
    // a row's codes replace keys that have been read.  A stored outlier takes
    // the grid level whose value is gmean -- NF4's zero level (code 7), or
    // code 0 of a uniform grid -- so the dense part of a decode contributes
    // gmean there and the side-list adds val - gmean; export restores the
    // reference's code.
    const int kb = d.key_bits, half = lane >> 5, pr = lane & 31;
    const uint32_t crowded = crowded_s;
    for (int c0 = 0; c0 < D; c0 += 64) {
      const int ja = c0 + 2 * pr;  // the lane's channels ja, ja + 1
      const float st00 = stat_s[ja][0], st01 = stat_s[ja][1];
      const float st10 = stat_s[ja + 1][0], st11 = stat_s[ja + 1][1];
      // the wave's token pairs: t and t + 8 of a 16-token stretch (LDS rows 8
      // apart fall on the other 32 banks)
      auto for_pairs = [&](auto f) {
        for (int s = wv; s < (G + 15) / 16 * 8; s += kEncWaves) {
          const int t = (s >> 3) * 16 + (s & 7) + 8 * half;
          f(t, t < G);
        }
      };
      if (d.key_grid == 1) {
        // uniform: clip(round_half_even((x - min) / scale), 0, 2^bits - 1)
        const float qmax = (float)((1 << kb) - 1);
        for_pairs([&](int t, bool in) {
          if (!in) return;
          const uint32_t xx = *reinterpret_cast<const uint32_t*>(&kt_s[t][ja]);
          const float r0 = __builtin_rintf(__fdiv_rn(__fsub_rn(h2f((uint16_t)xx), st00), st01));
          const float r1 = __builtin_rintf(__fdiv_rn(__fsub_rn(h2f((uint16_t)(xx >> 16)), st10), st11));
          uint32_t b0 = (uint32_t)fminf(fmaxf(r0, 0.0f), qmax);
          uint32_t b1 = (uint32_t)fminf(fmaxf(r1, 0.0f), qmax);
          if (kout > 0) {
            const uint32_t om = om_row(t)[ja >> 5] >> (ja & 31);
            if (om & 1u) b0 = 0u;
            if (om & 2u) b1 = 0u;
          }
          // one table index per channel pair (the key row layout of tqk_common.h)
          kc_row(t)[ja >> 1] = (uint8_t)(kb == 4 ? ((rev4(b0) << 4) | rev4(b1)) : (b0 | (b1 << kb)));
        });
      } else if (!((crowded >> (c0 >> 6)) & 1u)) {
        // asym-NF4 by bucket (above): the 15 thresholds of every channel, then
        // about 11 VALU and one LDS read a key (the argmin over 16 levels took
        // 45: the codes were half of the keys' work)
        __syncthreads();
        {
          const int c = tid & 63;
          const float mu = stat_s[c0 + c][0], amax = stat_s[c0 + c][1];
          const int col = (c >> 1) + 32 * (c & 1);
          for (int k = wv; k < 15; k += kEncWaves) {
            const uint32_t X = nf4_threshold(__fadd_rn(mu, __fmul_rn(amax, kNF4[k])),
                                             __fadd_rn(mu, __fmul_rn(amax, kNF4[k + 1])));
            const uint32_t e = X | (rev4((uint32_t)k) << 16) | (rev4((uint32_t)k + 1u) << 20);
            for (int i = kNf4From[k]; i < kNf4From[k + 1]; ++i) nf_s[i][col] = e;
          }
          if (wv == kEncWaves - 1) nf_s[32][col] = rev4(7u) << 16 | rev4(7u) << 20;
        }
        __syncthreads();
        // (a hair under 16: |x - mean| = amax stays short of bucket 32)
        const float inv0 = 15.9995f * __builtin_amdgcn_rcpf(st01), inv1 = 15.9995f * __builtin_amdgcn_rcpf(st11);
        // first read and second read: channel ja + half, then the other one
        const float muA = half ? st10 : st00, invA = half ? inv1 : inv0;
        const float muB = half ? st00 : st10, invB = half ? inv0 : inv1;
        const uint32_t* tabA = &nf_s[0][pr + 32 * half];
        const uint32_t* tabB = &nf_s[0][pr + 32 * (half ^ 1)];
        for_pairs([&](int t, bool in) {
          const uint32_t xx = *reinterpret_cast<const uint32_t*>(&kt_s[min(t, G - 1)][ja]);
          const float x0 = h2f((uint16_t)xx), x1 = h2f((uint16_t)(xx >> 16));
          const float xA = half ? x1 : x0, xB = half ? x0 : x1;
          const uint32_t iA = min((uint32_t)fmaf(__fsub_rn(xA, muA), invA, 16.0f), 32u);
          const uint32_t iB = min((uint32_t)fmaf(__fsub_rn(xB, muB), invB, 16.0f), 32u);
          const uint32_t eA = tabA[64 * iA], eB = tabB[64 * iB];
          const uint32_t nA = (eA >> (xA >= h2f((uint16_t)eA) ? 20 : 16)) & 15u;
          const uint32_t nB = (eB >> (xB >= h2f((uint16_t)eB) ? 20 : 16)) & 15u;
          if (in) kc_row(t)[ja >> 1] = (uint8_t)(half ? (nB << 4) | nA : (nA << 4) | nB);
        });
      } else {
        // levels too close together, or not finite: the argmin over all levels
        // cent_l = mean + amax * NF4[l]
        float l0[16], l1[16];
#pragma unroll
        for (int l = 0; l < 16; ++l) {
          l0[l] = __fadd_rn(st00, __fmul_rn(st01, kNF4[l]));
          l1[l] = __fadd_rn(st10, __fmul_rn(st11, kNF4[l]));
        }
        bool lv_finite = true;
#pragma unroll
        for (int l = 0; l < 16; ++l) lv_finite &= __builtin_isfinite(l0[l]) && __builtin_isfinite(l1[l]);
        for_pairs([&](int t, bool in) {
          const uint32_t xx = *reinterpret_cast<const uint32_t*>(&kt_s[min(t, G - 1)][ja]);
          const float x0 = h2f((uint16_t)xx), x1 = h2f((uint16_t)(xx >> 16));
          uint32_t b0 = 0, b1 = 0;
          float d0 = fabsf(__fsub_rn(x0, l0[0])), d1 = fabsf(__fsub_rn(x1, l1[0]));
          // with finite levels and a finite x no distance is NaN, and the
          // strict comparison is all that argmin needs
          const bool fin = lv_finite && (xx & 0x7C00u) != 0x7C00u && (xx & 0x7C000000u) != 0x7C000000u;
          if (__all(fin)) {
#pragma unroll
            for (int l = 1; l < 16; ++l) {
              const float e0 = fabsf(__fsub_rn(x0, l0[l])), e1 = fabsf(__fsub_rn(x1, l1[l]));
              if (e0 < d0) { d0 = e0; b0 = l; }
              if (e1 < d1) { d1 = e1; b1 = l; }
            }
          } else {
#pragma unroll
            for (int l = 1; l < 16; ++l) {
              const float e0 = fabsf(__fsub_rn(x0, l0[l])), e1 = fabsf(__fsub_rn(x1, l1[l]));
              // np.argmin: strictly smaller wins; the first NaN wins over any number
              if (e0 < d0 || (e0 != e0 && d0 == d0)) { d0 = e0; b0 = l; }
              if (e1 < d1 || (e1 != e1 && d1 == d1)) { d1 = e1; b1 = l; }
            }
          }
          if (!in) return;
          if (kout > 0) {
            const uint32_t om = om_row(t)[ja >> 5] >> (ja & 31);
            if (om & 1u) b0 = 7u;
            if (om & 2u) b1 = 7u;
          }
          kc_row(t)[ja >> 1] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
        });
      }
    }

    __syncthreads();
    // key code rows, one 32-channel chunk (16 pair indices) per thread
    const int KROW = k_row_bytes(d.key_bits, D);
    for (int idx = tid; idx < G * (D / 32); idx += kEncThreads) {
      const int t = idx / (D / 32), ch = idx % (D / 32);
      const size_t row = page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t, P, d.n_pages, h);
      const uint4 f16 = *reinterpret_cast<const uint4*>(kc_row(t) + 16 * ch);
      if (d.key_bits == 4) {
        *reinterpret_cast<uint4*>(a.p.kcodes + row * KROW + 16 * ch) = f16;
      } else {
        // 16 fields of 2*kb bits, little-endian, into kb dwords
        const int kb = d.key_bits;
        const uint32_t fw[4] = {f16.x, f16.y, f16.z, f16.w};
        uint32_t o[3] = {0u, 0u, 0u};
        for (int i = 0; i < 16; ++i) {
          const uint32_t f = (fw[i >> 2] >> (8 * (i & 3))) & 0xFFu;
          const int bo = 2 * kb * i, w = bo >> 5, sh = bo & 31;
          o[w] |= f << sh;
          if (sh + 2 * kb > 32) o[w + 1] |= f >> (32 - sh);
        }
        uint32_t* dst = reinterpret_cast<uint32_t*>(a.p.kcodes + row * KROW + 4 * kb * ch);
        for (int w = 0; w < kb; ++w) dst[w] = o[w];
      }
    }
    __syncthreads();
  }

  // ---- values (and PolarQuant keys) ----------------------------------------
  // kVBatch tokens at a time: their rows staged in the key tile's area, norms
  // (four threads per token, the reference's pairwise order), estimated codes
  // (wave w: channels [16 w, 16 w + 16), then as many waves further on), the
  // flagged ones recomputed, then the rows: LE bit streams of VB-bit codes per
  // token, or 4-token x 8-channel units (the same eight fields a thread either way)
  constexpr int VROW = D * VB / 8, NT = 1;
  Stage& st = *reinterpret_cast<Stage*>(area_s + kBatchBytes);
  float bnd[15];
#pragma unroll
  for (int k = 0; k < 15; ++k) bnd[k] = k < (1 << VB) - 1 ? a.p.vbnd[k] : 0.f;
  auto polar_phase = [&](const void* ring, const void* chunk, float* nout, bool vcheck, auto trows,
                         auto put) {
    constexpr bool TROWS = decltype(trows)::value;
    for (int t0 = 0; t0 < G; t0 += kVBatch) {
      const int nb = min(kVBatch, G - t0);
      for (int idx = tid; idx < nb * (D / 8); idx += kEncThreads) {
        const int t = idx / (D / 8), c = idx % (D / 8);
        reinterpret_cast<uint4*>(&kt_s[t][0])[c] =
            reinterpret_cast<const uint4*>(token_src<D>(a, ring, chunk, b, h, g * G + t0 + t))[c];
      }
      if (tid == 0) st.nlist = 0;
      __syncthreads();
      for (int t4 = tid; t4 < 4 * nb; t4 += kEncThreads) {
        const int t = t4 >> 2, q = t4 & 3;
        const uint32_t* src = reinterpret_cast<const uint32_t*>(&kt_s[t][0]);
        float x0[D / 8], x1[D / 8];
        uint32_t any = 0;
#pragma unroll
        for (int m = 0; m < D / 8; ++m) {
          const uint32_t w2 = src[4 * m + q];  // channels 8m + 2q, 8m + 2q + 1
          any |= w2;
          x0[m] = h2f((uint16_t)(w2 & 0xFFFFu));
          x1[m] = h2f((uint16_t)(w2 >> 16));
        }
        any |= __shfl_xor(any, 1, 4);
        any |= __shfl_xor(any, 2, 4);
        const float ss = pairwise_sumsq<D>(x0, x1, q);
        const float nrm = __builtin_sqrtf(ss);  // correctly rounded (-fhip-fp32-correctly-rounded-divide-sqrt)
        if (q == 0) {
          polar_token(st, t, ss, nrm, (any & 0x7FFF7FFFu) == 0u, __builtin_amdgcn_rcpf(nrm) * (1.0f / kPiScale));
          nout[page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t0 + t, P, d.n_pages, h)] = nrm;
          if (vcheck && nrm > TQK_MAX_VNORM && a.overflow) atomicOr(a.overflow, TQK_OVF_VNORM);
        }
      }
      __syncthreads();
      for (int e0 = 16 * wv; e0 < D; e0 += 16 * kEncWaves) {
        PiFrags<D, NT> pf;
        load_pi(pf, a.p.pi, e0, lane, bnd, (1 << VB) - 1);
        polar_codes<D, NT, VB, false, TROWS>(st, pf, &kt_s[0][0], D + 8, nb, e0, lane, bnd);
      }
      __syncthreads();
      if (st.nlist > 0) {
        polar_fix<D, VB, TROWS, kEncThreads>(st, a.p.pi, nb, tid, bnd, [&](int t, int dd) {
          const uint2 w = *reinterpret_cast<const uint2*>(&kt_s[t][dd]);
          return make_float4(h2f((uint16_t)w.x), h2f((uint16_t)(w.x >> 16)), h2f((uint16_t)w.y),
                             h2f((uint16_t)(w.y >> 16)));
        });
        __syncthreads();
      }
      for (int f8 = tid; f8 < nb * (D / 32); f8 += kEncThreads) {
        uint32_t w[VB];
        pack_fields<VB>(st, f8, w);
        put(t0, f8, w);
      }
      // (the next batch's rows may replace these: the fields are written again
      // only two barriers later)
    }
    __syncthreads();
  };
  auto put_row = [&](uint8_t* base, int t0, int f8, const uint32_t (&w)[VB]) {
    const size_t row = page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t0 + f8 / (D / 32), P,
                                d.n_pages, h);
    uint32_t* dst = reinterpret_cast<uint32_t*>(base + row * VROW) + VB * (f8 % (D / 32));
#pragma unroll
    for (int k = 0; k < VB; ++k) dst[k] = w[k];
  };
  if (key_side) {
    if (d.key_grid != 2) return;
    // PolarQuant keys (turboquant_pro/core.py:542-617 with kind="key"; key_bits
    // == value_bits): the value encode on the key tokens, norms to knorm; 2-
    // and 3-bit key rows are the same bit stream, 4-bit ones its bytes with
    // their bits reversed.  The per-channel stats are the identity (scale 1,
    // mean 0) and there is no side-list.
    polar_phase(a.p.hot_k, a.chunk_k, a.p.knorm, false, TokenRows{}, [&](int t0, int f8, uint32_t (&w)[VB]) {
      if constexpr (VB == 4) {
#pragma unroll
        for (int k = 0; k < VB; ++k) w[k] = __builtin_bswap32(__builtin_bitreverse32(w[k]));
      }
      put_row(a.p.kcodes, t0, f8, w);
    });
    if (tid < D) {
      a.p.gscale[mbase + tid] = 1.0f;
      a.p.gmean[mbase + tid] = 0.0f;
    }
    if (tid < TQK_NOB) a.p.ocount[obase * TQK_NOB + tid] = 0;
    return;
  }
  if (D == TQK_D && v_tiled(G, P, D, d.input_f32)) {
    polar_phase(a.p.hot_v, a.chunk_v, a.p.vnorm, true, TiledRows{}, [&](int t0, int f8, uint32_t (&w)[VB]) {
      // unit (lg, c): tokens [4 lg, +4) of tile T, channels [8c, +8)
      const int T = f8 >> 6, lg = (f8 >> 4) & 3, c = f8 & 15;
      const size_t row0 = page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t0 + 16 * T, P, d.n_pages, h);
      uint32_t* dst = reinterpret_cast<uint32_t*>(a.p.vcodes + row0 * VROW + v_unit_offset(lg, c, VROW));
#pragma unroll
      for (int k = 0; k < VB; ++k) dst[k] = w[k];
    });
  } else {
    polar_phase(a.p.hot_v, a.chunk_v, a.p.vnorm, true, TokenRows{},
                [&](int t0, int f8, uint32_t (&w)[VB]) { put_row(a.p.vcodes, t0, f8, w); });
  }
}


// ---------------------------------------------------------------------------
// Quantize-on-flush of an fp32 cache (input_f32): the same codes, stats and
// side-list as the fp16 encode, in the same NumPy operation order, with key and
// value workgroups as there.  The keys go 64 channels at a time through an LDS
// tile; a token's side-list bits are collected over the 64-channel pieces and its
// entries written at the end.  The side-list positions keep the reference's
// codes (argmin on the fp32 value); value codes are per-token rows.  Value norms
// are not bounded: the VALU decode, the one that serves fp32 caches, keeps its
// weights in fp32.  4 sequences x 5000 tokens x 8 heads x 128: 607 us with one
// 256-thread workgroup per (group, head) reading the keys through L1 and L2 in
// every phase, 226 us like this.
template <int VB, int D, int MG>
__global__ __launch_bounds__(enc_threads(MG), D <= 128 ? 4 : 2) void tqk_encode_group_f32(EncodeArgs a) {
  constexpr int kEncThreads = enc_threads(MG), kEncWaves = kEncThreads / 64;
  constexpr int kVBatch = enc_batch(MG);  // tokens per value batch
  const int unit = a.unit0 + (int)(blockIdx.x >> 4) * 8 + (int)(blockIdx.x & 7u);
  const bool key_side = ((blockIdx.x >> 3) & 1u) == 0u;
  if (unit >= a.n_items * a.d.n_kv_heads) return;
  const int item = unit % a.n_items, h = unit / a.n_items, tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const tqk_cache_desc& d = a.d;
  const int b = item_word(a, 2 * item), g = item_word(a, 2 * item + 1);
  const int G = d.group_tokens, P = d.page_tokens, Hkv = d.n_kv_heads;
  const int slot = a.p.group_table[(size_t)b * d.max_groups_per_seq + g];
  const int kout = d.outliers_per_channel;
  const size_t mbase = ((size_t)slot * Hkv + h) * D;
  const size_t obase = (size_t)slot * Hkv + h;
  constexpr int VROW = D * VB / 8;
  constexpr int LD = 68;        // key tile row stride: eight tokens x eight channels nearly on 64 banks

  struct KeyLds {
    float tile[MG][LD];      // 64 channels; then a row's 32 code bytes at its start
    uint32_t om[MG][D / 32]; // side-list bits of every token
    float lev[16][64];              // NF4 levels of the channels, (channel / 2) + 32 (channel % 2)
    float stat[64][2];              // (mean, amax) or (min, scale)
    float thr[64];
    uint32_t crowded;
    int32_t wsum[kEncWaves];
    uint8_t pair[32];
  };
  struct ValueLds {
    uint16_t uv[kVBatch][2 * D + 8];  // scaled rows as fp16 pairs (high halves, then low ones)
    PolarStage<D, kVBatch> st;
    const float* row[kVBatch];
  };
  union Lds {
    KeyLds k;
    ValueLds v;
  };
  __shared__ __align__(16) uint8_t lds_s[sizeof(Lds)];

  if (key_side && d.key_grid != 2) {
    KeyLds& L = reinterpret_cast<Lds*>(lds_s)->k;
    const int kb = d.key_bits;
    const bool all = kout >= G;
    if (tid < 15)
      for (int i = kNf4From[tid]; i < kNf4From[tid + 1]; ++i) L.pair[i] = (uint8_t)tid;
    for (int c0 = 0; c0 < D; c0 += 64) {
      // ---- 64 channels of the group's keys
      if (tid == 0) L.crowded = 0u;
      for (int idx = tid; idx < G * 16; idx += kEncThreads) {
        const int t = idx >> 4, c = idx & 15;
        *reinterpret_cast<float4*>(&L.tile[t][4 * c]) =
            reinterpret_cast<const float4*>(token_src<D, float>(a, a.p.hot_k, a.chunk_k, b, h, g * G + t) + c0)[c];
      }
      __syncthreads();
      // the zero point, a sum in token order
      if (tid < 64 && d.key_grid != 1) {
        const int j = c0 + tid;
        float mu;
        if (d.zero_point == 2) {
          mu = a.p.zp_mean[((size_t)g * Hkv + h) * D + j];
        } else {
          float acc = 0.0f;
          int s = 0;
          for (; s + 16 <= G; s += 16) {
            float x[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) x[u] = L.tile[s + u][tid];
#pragma unroll
            for (int u = 0; u < 16; ++u) acc = __fadd_rn(acc, x[u]);
          }
          for (; s < G; ++s) acc = __fadd_rn(acc, L.tile[s][tid]);
          mu = (float)((double)acc / (double)G);
          if (d.zero_point == 1) mu = __fmul_rn(mu, ((d.dc_mask[j >> 5] >> (j & 31)) & 1u) ? 1.0f : 0.0f);
        }
        L.stat[tid][0] = mu;
      }
      // Channel ends and outlier thresholds, eight channels a wave, eight lanes
      // a channel with every eighth token.  amax = max |x - mean| is taken at
      // the ends (rounding is monotone).  The threshold is the k-th largest |x|
      // as the largest fp32 magnitude pattern T with #{ |x_s| >= T } >= k (NaN
      // patterns order above inf, as np.partition places NaN last): for k <= 8
      // every lane's eight largest, merged; otherwise a bitwise search.
      for (int cw = 8 * wv; cw < 64; cw += 8 * kEncWaves) {
        const int cl = cw + (lane & 7), part = lane >> 3;
        float mn = __builtin_inff(), mx = -__builtin_inff();
        uint32_t top[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) top[i] = 0u;
        auto insert = [&](uint32_t v) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const uint32_t hi = max(top[i], v);
            v = min(top[i], v);
            top[i] = hi;
          }
        };
        for (int s = part; s < G; s += 8) {
          const float x = L.tile[s][cl];
          mn = fminf(mn, x);
          mx = fmaxf(mx, x);
          insert(__float_as_uint(fabsf(x)));
        }
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) {
          mn = fminf(mn, __shfl_xor(mn, o, 64));
          mx = fmaxf(mx, __shfl_xor(mx, o, 64));
          uint32_t other[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) other[i] = (uint32_t)__shfl_xor((int)top[i], o, 64);
#pragma unroll
          for (int i = 0; i < 8; ++i) insert(other[i]);
        }
        const bool xnan = top[0] > 0x7F800000u;
        uint32_t T = 0;
        if (kout > 0 && kout <= 8) {
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (i == kout - 1) T = top[i];
        } else if (kout > 8 && kout < G) {
          for (int bit = 30; bit >= 0; --bit) {
            const uint32_t cand = T | (1u << bit);
            int cnt = 0;
            for (int s = part; s < G; s += 8) cnt += __float_as_uint(fabsf(L.tile[s][cl])) >= cand ? 1 : 0;
            cnt += __shfl_xor(cnt, 8, 64);
            cnt += __shfl_xor(cnt, 16, 64);
            cnt += __shfl_xor(cnt, 32, 64);
            if (cnt >= kout) T = cand;
          }
        }
        __syncthreads();  // the means
        if (part == 0) {
          L.thr[cl] = __uint_as_float(T);  // a NaN threshold selects nothing, as |x| >= NaN
          float st0, st1;
          if (d.key_grid == 1) {
            st0 = xnan ? __builtin_nanf("") : mn;
            st1 = xnan ? __builtin_nanf("")
                       : __fdiv_rn(fmaxf(__fsub_rn(mx, mn), 1e-8f), (float)((1 << d.key_bits) - 1));
          } else {
            st0 = L.stat[cl][0];
            const float lo = fabsf(__fsub_rn(mn, st0)), hi = fabsf(__fsub_rn(mx, st0));
            st1 = xnan || lo != lo || hi != hi ? __builtin_nanf("") : fmaxf(fmaxf(lo, hi), 1e-8f);
            // levels finite and far enough apart, as in the fp16 encode
            const float r = __fmul_rn(__fadd_rn(fabsf(st0), st1), 0x1p-18f);
            bool ok = true;
            float c = __fadd_rn(st0, __fmul_rn(st1, kNF4[0]));
            L.lev[0][(cl >> 1) + 32 * (cl & 1)] = c;
#pragma unroll
            for (int l = 1; l < 16; ++l) {
              const float n = __fadd_rn(st0, __fmul_rn(st1, kNF4[l]));
              ok &= __fsub_rn(n, c) >= r;
              c = n;
              L.lev[l][(cl >> 1) + 32 * (cl & 1)] = c;
            }
            // (normalised keys must not overflow: amax well inside fp32's range)
            if (!(ok && __builtin_isfinite(c) && st1 < 0x1p100f && fabsf(st0) < 0x1p100f)) atomicOr(&L.crowded, 1u);
          }
          L.stat[cl][0] = st0;
          L.stat[cl][1] = st1;
          a.p.gscale[mbase + c0 + cl] = st1;
          a.p.gmean[mbase + c0 + cl] = st0;
        }
      }
      __syncthreads();
      // side-list bits, two threads per token, 32 channels each
      if (kout > 0 && (tid >> 1) < G) {
        const int t = tid >> 1, hf = tid & 1;
        uint32_t m = 0;
#pragma unroll
        for (int c4 = 0; c4 < 8; ++c4) {
          const float4 x = *reinterpret_cast<const float4*>(&L.tile[t][32 * hf + 4 * c4]);
          const float4 th = *reinterpret_cast<const float4*>(&L.thr[32 * hf + 4 * c4]);
          m |= (fabsf(x.x) >= th.x ? 1u : 0u) << (4 * c4);
          m |= (fabsf(x.y) >= th.y ? 2u : 0u) << (4 * c4);
          m |= (fabsf(x.z) >= th.z ? 4u : 0u) << (4 * c4);
          m |= (fabsf(x.w) >= th.w ? 8u : 0u) << (4 * c4);
        }
        L.om[t][c0 / 32 + hf] = all ? 0xFFFFFFFFu : m;
      }
      __syncthreads();
      // codes: a wave takes two tokens, a half-wave the 32 channel pairs of
      // one; a row's 32 code bytes replace its first keys once they are read
      const int half = lane >> 5, pr = lane & 31;
      const float st00 = L.stat[2 * pr][0], st01 = L.stat[2 * pr][1];
      const float st10 = L.stat[2 * pr + 1][0], st11 = L.stat[2 * pr + 1][1];
      auto for_pairs = [&](auto code) {
        for (int s = wv; s < (G + 1) / 2; s += kEncWaves) {
          const int t = 2 * s + half;
          const float2 xx = *reinterpret_cast<const float2*>(&L.tile[min(t, G - 1)][2 * pr]);
          const uint32_t byte = code(xx.x, xx.y);
          if (t < G) reinterpret_cast<uint8_t*>(&L.tile[t][0])[pr] = (uint8_t)byte;
        }
      };
      if (d.key_grid == 1) {
        const float qmax = (float)((1 << kb) - 1);
        for_pairs([&](float x0, float x1) {
          const float r0 = __builtin_rintf(__fdiv_rn(__fsub_rn(x0, st00), st01));
          const float r1 = __builtin_rintf(__fdiv_rn(__fsub_rn(x1, st10), st11));
          const uint32_t b0 = (uint32_t)fminf(fmaxf(r0, 0.0f), qmax);
          const uint32_t b1 = (uint32_t)fminf(fmaxf(r1, 0.0f), qmax);
          return kb == 4 ? ((rev4(b0) << 4) | rev4(b1)) : (b0 | (b1 << kb));
        });
      } else if (L.crowded == 0u) {
        // by bucket: two neighbouring levels, the nearer one (the first on a tie)
        const float inv0 = 15.9995f / st01, inv1 = 15.9995f / st11;
        auto nearer = [&](float x, float mu, float inv, int col) {
          const uint32_t i = min((uint32_t)fmaf(__fsub_rn(x, mu), inv, 16.0f), 31u);
          const uint32_t k = L.pair[i];
          const float lo = L.lev[k][col], hi = L.lev[k + 1][col];
          return k + (fabsf(__fsub_rn(x, hi)) < fabsf(__fsub_rn(x, lo)) ? 1u : 0u);
        };
        for_pairs([&](float x0, float x1) {
          const uint32_t b0 = nearer(x0, st00, inv0, pr), b1 = nearer(x1, st10, inv1, pr + 32);
          return (rev4(b0) << 4) | rev4(b1);
        });
      } else {
        for_pairs([&](float x0, float x1) {
          uint32_t b0 = 0, b1 = 0;
          float d0 = fabsf(__fsub_rn(x0, L.lev[0][pr])), d1 = fabsf(__fsub_rn(x1, L.lev[0][pr + 32]));
#pragma unroll
          for (int l = 1; l < 16; ++l) {
            const float e0 = fabsf(__fsub_rn(x0, L.lev[l][pr])), e1 = fabsf(__fsub_rn(x1, L.lev[l][pr + 32]));
            // np.argmin: strictly smaller wins; the first NaN wins over any number
            if (e0 < d0 || (e0 != e0 && d0 == d0)) { d0 = e0; b0 = l; }
            if (e1 < d1 || (e1 != e1 && d1 == d1)) { d1 = e1; b1 = l; }
          }
          return (rev4(b0) << 4) | rev4(b1);
        });
      }
      __syncthreads();
      // key code rows, one 32-channel chunk (16 table indices) per thread
      const int KROW = k_row_bytes(kb, D);
      for (int idx = tid; idx < G * 2; idx += kEncThreads) {
        const int t = idx >> 1, ch = c0 / 32 + (idx & 1);
        const size_t row = page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t, P, d.n_pages, h);
        const uint4 f16 = *reinterpret_cast<const uint4*>(&L.tile[t][4 * (idx & 1)]);
        if (kb == 4) {
          *reinterpret_cast<uint4*>(a.p.kcodes + row * KROW + 16 * ch) = f16;
        } else {
          const uint32_t fw[4] = {f16.x, f16.y, f16.z, f16.w};
          uint32_t o[3] = {0u, 0u, 0u};
          for (int i = 0; i < 16; ++i) {
            const uint32_t f = (fw[i >> 2] >> (8 * (i & 3))) & 0xFFu;
            const int bo = 2 * kb * i, w = bo >> 5, sh = bo & 31;
            o[w] |= f << sh;
            if (sh + 2 * kb > 32) o[w + 1] |= f >> (32 - sh);
          }
          uint32_t* dst = reinterpret_cast<uint32_t*>(a.p.kcodes + row * KROW + 4 * kb * ch);
          for (int w = 0; w < kb; ++w) dst[w] = o[w];
        }
      }
      __syncthreads();  // the tile is the next channels'
    }
    // ---- the side-list in flat (token, channel) order, two threads per token
    // (cumulative counts at every TQK_OBLK-token boundary as the fp16 encode)
    if (kout > 0) {
      constexpr int NW = D / 64;
      const int tt = tid >> 1, w0 = NW * (tid & 1);
      uint32_t om[NW];
      int cnt = 0;
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        om[k] = tt < G ? L.om[tt][w0 + k] : 0u;
        cnt += __builtin_popcount(om[k]);
      }
      int incl = cnt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      if (lane == 63) L.wsum[wv] = incl;
      __syncthreads();
      int wofs = 0, total = 0;
#pragma unroll
      for (int w = 0; w < kEncWaves; ++w) {
        wofs += w < wv ? L.wsum[w] : 0;
        total += L.wsum[w];
      }
      int off = wofs + incl - cnt;
      if (tt < G && (tid & 1) && ((tt + 1) % TQK_OBLK) == 0 && (tt + 1) / TQK_OBLK <= TQK_NOB)
        a.p.ocount[obase * TQK_NOB + (tt + 1) / TQK_OBLK - 1] = off + cnt;
      if (tid < TQK_NOB && TQK_OBLK * (tid + 1) > G) a.p.ocount[obase * TQK_NOB + tid] = total;
      if (cnt > 0) {
        const float* row = token_src<D, float>(a, a.p.hot_k, a.chunk_k, b, h, g * G + tt);
#pragma unroll
        for (int k = 0; k < NW; ++k) {
          while (om[k] && off < d.outlier_cap) {
            const int j = 32 * (w0 + k) + __builtin_ctz(om[k]);
            om[k] &= om[k] - 1u;
            a.p.oent[obase * d.outlier_cap + off] = (uint32_t)(tt * D + j) | ((uint32_t)f2h(row[j]) << 16);
            ++off;
          }
        }
      }
      if (tid == 0 && total > d.outlier_cap && a.overflow) atomicOr(a.overflow, TQK_OVF_OUTLIERS);
    } else if (tid < TQK_NOB) {
      a.p.ocount[obase * TQK_NOB + tid] = 0;
    }
    return;
  }

  ValueLds& L = reinterpret_cast<Lds*>(lds_s)->v;
  PolarStage<D, kVBatch>& st = L.st;
  float bnd[15];
#pragma unroll
  for (int k = 0; k < 15; ++k) bnd[k] = k < (1 << VB) - 1 ? a.p.vbnd[k] : 0.f;
  // PolarQuant of the group's tokens, kVBatch at a time: norms (four threads
  // per token, pairwise_sumsq) and the scaled rows' fp16 pairs, estimated
  // codes, the flagged ones recomputed from the fp32 rows, the bit streams
  const void* ring = key_side ? a.p.hot_k : a.p.hot_v;
  const void* chunk = key_side ? a.chunk_k : a.chunk_v;
  float* nout = key_side ? a.p.knorm : a.p.vnorm;
  uint8_t* rows = key_side ? a.p.kcodes : a.p.vcodes;
  const bool reversed = key_side && VB == 4;  // PolarQuant key rows, as the fp16 encode writes them
  if (key_side) {
    if (tid < D) {
      a.p.gscale[mbase + tid] = 1.0f;
      a.p.gmean[mbase + tid] = 0.0f;
    }
    if (tid < TQK_NOB) a.p.ocount[obase * TQK_NOB + tid] = 0;
  }
  for (int t0 = 0; t0 < G; t0 += kVBatch) {
    const int nb = min(kVBatch, G - t0);
    if (tid == 0) st.nlist = 0;
    const int tt = tid >> 2, q = tid & 3;
    if (tt < nb) {
      const int t = g * G + t0 + tt;
      const float* sp = token_src<D, float>(a, ring, chunk, b, h, t);
      if (q == 0) L.row[tt] = sp;
      const float2* src = reinterpret_cast<const float2*>(sp);
      float x0[D / 8], x1[D / 8];
      uint32_t any = 0;
#pragma unroll
      for (int m = 0; m < D / 8; ++m) {
        const float2 w2 = src[4 * m + q];  // channels 8m + 2q, 8m + 2q + 1
        x0[m] = w2.x;
        x1[m] = w2.y;
        any |= __float_as_uint(w2.x) | __float_as_uint(w2.y);
      }
      any |= __shfl_xor(any, 1, 4);
      any |= __shfl_xor(any, 2, 4);
      const float ss = pairwise_sumsq<D>(x0, x1, q);
      const float nrm = __builtin_sqrtf(ss);
      const bool zero = (any & 0x7FFFFFFFu) == 0u;
      polar_stage_row<D>(&L.uv[tt][0], x0, x1, q, zero ? 0.f : kPiScale * __builtin_amdgcn_rcpf(nrm));
      if (q == 0) {
        polar_token(st, tt, ss, nrm, zero, 1.0f / (kPiScale * kPiScale));
        nout[page_row(a.p.block_table, d.max_pages_per_seq, b, t, P, d.n_pages, h)] = nrm;
      }
    }
    __syncthreads();
    for (int e0 = 16 * wv; e0 < D; e0 += 16 * kEncWaves) {
      PiFrags<D, 1> pf;
      load_pi(pf, a.p.pi, e0, lane, bnd, (1 << VB) - 1);
      polar_codes<D, 1, VB, true, false>(st, pf, &L.uv[0][0], 2 * D + 8, nb, e0, lane, bnd);
    }
    __syncthreads();
    if (st.nlist > 0) {
      polar_fix<D, VB, false, kEncThreads>(st, a.p.pi, nb, tid, bnd, [&](int t, int dd) {
        return *reinterpret_cast<const float4*>(L.row[t] + dd);
      });
      __syncthreads();
    }
    for (int f8 = tid; f8 < nb * (D / 32); f8 += kEncThreads) {
      uint32_t w[VB];
      pack_fields<VB>(st, f8, w);
      const size_t row = page_row(a.p.block_table, d.max_pages_per_seq, b, g * G + t0 + f8 / (D / 32), P,
                                  d.n_pages, h);
      uint32_t* dst = reinterpret_cast<uint32_t*>(rows + row * VROW) + VB * (f8 % (D / 32));
#pragma unroll
      for (int k = 0; k < VB; ++k) dst[k] = reversed ? __builtin_bswap32(__builtin_bitreverse32(w[k])) : w[k];
    }
    __syncthreads();
  }
}


struct HotArgs {
  tqk_cache_desc d;
  uint8_t* hot_k;
  uint8_t* hot_v;
  const int32_t* prev_len;  // nullptr: the inline lengths
  const int32_t* n_new;
  const int32_t* hot_start;
  const uint8_t* chunk_k;
  const uint8_t* chunk_v;
  int chunk_tokens;
  int32_t* seq_lens;        // with inline lengths: the new lengths are written here
  int32_t in_prev[kInlineSeqs];
  int32_t in_new[kInlineSeqs];
};

constexpr int kHotSlice = 64;  // tokens per workgroup of the ring copy

// grid (batch, Hkv, slices): copies the surviving new tokens into the ring,
// kHotSlice tokens per workgroup and round (slices stride by gridDim.z), so a
// chunk's copy spreads over the whole chip instead of one workgroup per
// (sequence, kv head).
__global__ __launch_bounds__(kThreads) void tqk_append_hot_kernel(HotArgs a) {
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const tqk_cache_desc& d = a.d;
  int prev, nn, start;
  if (a.prev_len) {
    prev = a.prev_len[b];
    nn = a.n_new[b];
    start = a.hot_start[b];
  } else {
    prev = a.in_prev[b];
    nn = a.in_new[b];
    start = n_groups_of(prev + nn, d.hot_window, d.group_tokens) * d.group_tokens;
    if (h == 0 && blockIdx.z == 0 && tid == 0) a.seq_lens[b] = prev + nn;
  }
  const int t0 = max(prev, start), t1 = prev + nn;
  const int R = d.hot_ring;
  const size_t rb = ((size_t)b * d.n_kv_heads + h) * R;
  const size_t cb = ((size_t)b * d.n_kv_heads + h) * a.chunk_tokens;
  const int rowb = d.head_dim * (d.input_f32 ? 4 : 2), nc = rowb / 16;  // 16-byte pieces per row
  for (int s0 = t0 + (int)blockIdx.z * kHotSlice; s0 < t1; s0 += (int)gridDim.z * kHotSlice) {
    const int n = min(kHotSlice, t1 - s0);
    for (int idx = tid; idx < n * nc; idx += kThreads) {
      const int t = s0 + idx / nc, c = idx % nc;
      const size_t src = (cb + (t - prev)) * rowb;
      const size_t dst = (rb + (t % R)) * rowb;
      reinterpret_cast<uint4*>(a.hot_k + dst)[c] = reinterpret_cast<const uint4*>(a.chunk_k + src)[c];
      reinterpret_cast<uint4*>(a.hot_v + dst)[c] = reinterpret_cast<const uint4*>(a.chunk_v + src)[c];
    }
  }
}

constexpr int kDqTokens = 64;  // tokens per reconstruction workgroup

struct DequantArgs {
  tqk_cache_desc d;
  tqk_cache_ptrs p;
  const int32_t* items;     // (b, g) pairs of the groups, or nullptr: every token of every sequence
  const int32_t* seq_lens;  // without items: [batch] lengths
  int chunks;               // kDqTokens-token chunks of a group; without items, of a sequence
  int max_len;              // without items: rows of a sequence in kout / vout
  void* kout;
  void* vout;
};

// a reconstructed fp32 value in the output's type, rounded to nearest even (the
// barrier keeps a product before it from being rounded to fp16 directly)
__device__ __forceinline__ void put_as(float* o, float x) { *o = x; }
__device__ __forceinline__ void put_as(_Float16* o, float x) {
  asm volatile("" : "+v"(x));
  *o = (_Float16)x;
}
__device__ __forceinline__ void put_as(__bf16* o, float x) { *o = (__bf16)x; }

// Keys and values of 64 tokens of one kv head: keys as grid value, then the fp16
// outlier overwrite; values ((cent[code] @ Pi) * norm, NumPy order), PolarQuant
// keys likewise; hot tokens (without items) converted.  Bound: the 2 D VALU
// operations of every rotated value (rotate_rows).  One token per thread with Pi
// from memory, a workgroup per group, took 260 us for 224 group-heads of 256
// tokens (head_dim 128), and a dense prefill of 2 x 4000 tokens x 8 heads (encode,
// this, and torch's transposes, concatenation and conversion) 503 us; written
// in place in the output's type it takes 191 us.
template <int VB, int D, typename T>
__global__ __launch_bounds__(kThreads, 2) void tqk_dequant_tokens(DequantArgs a) {
  constexpr int VROW = D * VB / 8;
  const tqk_cache_desc& d = a.d;
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int u = blockIdx.x / a.chunks, c = blockIdx.x % a.chunks;
  const int G = d.group_tokens, P = d.page_tokens, Hkv = d.n_kv_heads;
  const int cpg = (G + kDqTokens - 1) / kDqTokens;  // chunks per group
  int b, g, t0;        // t0: first token of the chunk in its group
  T *ko, *vo;          // the chunk's first output rows
  if (a.items) {
    b = a.items[2 * u];
    g = a.items[2 * u + 1];
    t0 = c * kDqTokens;
    const size_t row = ((size_t)u * Hkv + h) * G + t0;
    ko = static_cast<T*>(a.kout) + row * D;
    vo = static_cast<T*>(a.vout) + row * D;
  } else {
    b = u;
    g = c / cpg;
    t0 = (c % cpg) * kDqTokens;
    const int L = a.seq_lens[b], ng = n_groups_of(L, d.hot_window, G);
    const size_t base = ((size_t)b * Hkv + h) * a.max_len;
    const int max_cold = n_groups_of(a.max_len, d.hot_window, G) * cpg;
    if (c >= max_cold) {
      // the hot window
      const int s0 = ng * G + (c - max_cold) * kDqTokens, n = min(kDqTokens, L - s0);
      const size_t ring = ((size_t)b * Hkv + h) * d.hot_ring;
      for (int i = tid; i < n * D; i += kThreads) {
        const int s = s0 + i / D, j = i % D;
        const size_t src = (ring + s % d.hot_ring) * D + j, dst = (base + s) * D + j;
        if (d.input_f32) {
          put_as(static_cast<T*>(a.kout) + dst, static_cast<const float*>(a.p.hot_k)[src]);
          put_as(static_cast<T*>(a.vout) + dst, static_cast<const float*>(a.p.hot_v)[src]);
        } else {
          put_as(static_cast<T*>(a.kout) + dst, h2f(static_cast<const uint16_t*>(a.p.hot_k)[src]));
          put_as(static_cast<T*>(a.vout) + dst, h2f(static_cast<const uint16_t*>(a.p.hot_v)[src]));
        }
      }
      return;
    }
    if (g >= ng) return;
    ko = static_cast<T*>(a.kout) + (base + g * G + t0) * D;
    vo = static_cast<T*>(a.vout) + (base + g * G + t0) * D;
  }
  const int nb = min(kDqTokens, G - t0);
  const int slot = a.p.group_table[(size_t)b * d.max_groups_per_seq + g];
  const size_t mbase = ((size_t)slot * Hkv + h) * D, obase = (size_t)slot * Hkv + h;

  __shared__ __align__(16) float y_s[kDqTokens][D];
  __shared__ float nrm_s[2][kDqTokens];  // key norms (PolarQuant), value norms
  __shared__ int row_s[kDqTokens];       // row of every token in the head's pages
  __shared__ float cent_s[16];
  if (tid < nb) {
    const int t = g * G + t0 + tid;
    const int phys = a.p.block_table[(size_t)b * d.max_pages_per_seq + t / P];
    row_s[tid] = phys * P + t % P;
    const size_t row = (size_t)h * d.n_pages * P + row_s[tid];
    nrm_s[0][tid] = d.key_grid == 2 ? a.p.knorm[row] : 0.f;
    nrm_s[1][tid] = a.p.vnorm[row];
  }
  if (tid >= 64 && tid < 64 + (1 << VB)) cent_s[tid - 64] = a.p.vcent[tid - 64];
  __syncthreads();
  const size_t head = (size_t)h * d.n_pages * P;

  // centroids of the chunk's rows: a thread takes 32 codes (VB dwords), 32
  // channels of a token
  auto rows_to_lds = [&](const uint8_t* rows, bool reversed) {
    for (int i = tid; i < nb * (D / 32); i += kThreads) {
      const int t = i / (D / 32), c32 = i % (D / 32);
      const uint32_t* src = reinterpret_cast<const uint32_t*>(rows + (head + row_s[t]) * VROW) + VB * c32;
      uint32_t w[VB];
#pragma unroll
      for (int k = 0; k < VB; ++k) w[k] = reversed ? __builtin_bswap32(__builtin_bitreverse32(src[k])) : src[k];
#pragma unroll
      for (int k = 0; k < 32; k += 4)
        *reinterpret_cast<float4*>(&y_s[t][32 * c32 + k]) =
            make_float4(cent_s[stream_code<VB>(w, k)], cent_s[stream_code<VB>(w, k + 1)],
                        cent_s[stream_code<VB>(w, k + 2)], cent_s[stream_code<VB>(w, k + 3)]);
    }
  };
  auto rotate_out = [&](T* out, const float* nrm) {
    for (int e0 = 16 * wv; e0 < D; e0 += 16 * (kThreads / 64)) {
      const int e = e0 + (lane & 15);
      rotate_rows<D>(a.p.pi, y_s, nb, e, lane, [&](int t, float x) {
        put_as(out + (size_t)t * D + e, __fmul_rn(x, nrm[t]));
      });
    }
  };

  if (d.key_grid == 2) {
    // PolarQuant keys (key_bits == value_bits): (cent[code] @ Pi) * norm
    rows_to_lds(a.p.kcodes, VB == 4);
    __syncthreads();
    rotate_out(ko, nrm_s[0]);
    __syncthreads();
  } else {
    // four channels (two table indices) a thread
    const int kb = d.key_bits, KROW = k_row_bytes(kb, D);
    for (int i = tid; i < nb * (D / 4); i += kThreads) {
      const int t = i / (D / 4), j = 4 * (i % (D / 4));
      const uint8_t* src = a.p.kcodes + (head + row_s[t]) * KROW;
      uint32_t f[2];
      if (kb == 4) {
        const uint32_t two = *reinterpret_cast<const uint16_t*>(src + j / 2);
        f[0] = two & 0xFFu;
        f[1] = two >> 8;
      } else {
        // bits kb * j .. of the row's stream (the 32-channel chunks follow on)
        const int bit = kb * j;
        const uint32_t v = ((uint32_t)src[bit >> 3] | (uint32_t)src[min((bit >> 3) + 1, KROW - 1)] << 8) >> (bit & 7);
        f[0] = v & ((1u << (2 * kb)) - 1u);
        f[1] = (v >> (2 * kb)) & ((1u << (2 * kb)) - 1u);
      }
      const float4 sc = *reinterpret_cast<const float4*>(a.p.gscale + mbase + j);
      const float4 mu = *reinterpret_cast<const float4*>(a.p.gmean + mbase + j);
      T* o = ko + (size_t)t * D + j;
      put_as(o, __fadd_rn(__fmul_rn(sc.x, key_level(d.key_grid, k_code_even(f[0], kb))), mu.x));
      put_as(o + 1, __fadd_rn(__fmul_rn(sc.y, key_level(d.key_grid, k_code_odd(f[0], kb))), mu.y));
      put_as(o + 2, __fadd_rn(__fmul_rn(sc.z, key_level(d.key_grid, k_code_even(f[1], kb))), mu.z));
      put_as(o + 3, __fadd_rn(__fmul_rn(sc.w, key_level(d.key_grid, k_code_odd(f[1], kb))), mu.w));
    }
  }
  if (D == TQK_D && v_tiled(G, P, D, d.input_f32)) {
    // unit (lg, c8) of a 16-token tile: tokens 4 lg .. + 3 x channels 8 c8 .. + 7
    for (int i = tid; i < nb * (D / 32); i += kThreads) {
      const int tile = i >> 6, lg = (i >> 4) & 3, c8 = i & 15;
      const uint32_t* src = reinterpret_cast<const uint32_t*>(
          a.p.vcodes + (head + row_s[16 * tile]) * VROW + v_unit_offset(lg, c8, VROW));
      uint32_t w[VB];
#pragma unroll
      for (int k = 0; k < VB; ++k) w[k] = src[k];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int n = 0; n < 8; n += 4)
          *reinterpret_cast<float4*>(&y_s[16 * tile + 4 * lg + t][8 * c8 + n]) =
              make_float4(cent_s[stream_code<VB>(w, 4 * n + t)], cent_s[stream_code<VB>(w, 4 * n + 4 + t)],
                          cent_s[stream_code<VB>(w, 4 * n + 8 + t)], cent_s[stream_code<VB>(w, 4 * n + 12 + t)]);
      }
    }
  } else {
    rows_to_lds(a.p.vcodes, false);
  }
  __syncthreads();
  if (d.key_grid != 2 && d.outliers_per_channel > 0) {
    // the chunk's side-list entries (its bounds are 32-token blocks)
    const int32_t* oc = a.p.ocount + obase * TQK_NOB;
    const int cap = d.outlier_cap, q = t0 / TQK_OBLK;
    const int lo = min(q > 0 ? oc[q - 1] : 0, cap);
    const int hi = min(oc[min(q + kDqTokens / TQK_OBLK, TQK_NOB) - 1], cap);
    for (int e = lo + tid; e < hi; e += kThreads) {
      const uint32_t ent = a.p.oent[obase * cap + e];
      put_as(ko + (int)(ent & 0xFFFFu) - t0 * D, h2f((uint16_t)(ent >> 16)));
    }
  }
  rotate_out(vo, nrm_s[1]);
}

// one kernel instance per (value bits, head_dim, group size); a key and a value workgroup per
// (item, kv head), see tqk_encode_group, as many as fewer than 2^32 threads allow
// at a time
template <int D, int MG>
void launch_by_vb(int vb, hipStream_t st, EncodeArgs a) {
  constexpr int kMost = 1 << 21;
  const dim3 threads(enc_threads(MG));
  const int units = a.n_items * a.d.n_kv_heads;
  for (; a.unit0 < units; a.unit0 += kMost) {
    const dim3 grid(16 * ((min(kMost, units - a.unit0) + 7) / 8));
    if (a.d.input_f32) {
      if constexpr (MG != 128) {
        if (vb == 2)
          hipLaunchKernelGGL((tqk_encode_group_f32<2, D, MG>), grid, threads, 0, st, a);
        else if (vb == 3)
          hipLaunchKernelGGL((tqk_encode_group_f32<3, D, MG>), grid, threads, 0, st, a);
        else
          hipLaunchKernelGGL((tqk_encode_group_f32<4, D, MG>), grid, threads, 0, st, a);
      }
    } else if (vb == 2) {
      hipLaunchKernelGGL((tqk_encode_group<2, D, MG>), grid, threads, 0, st, a);
    } else if (vb == 3) {
      hipLaunchKernelGGL((tqk_encode_group<3, D, MG>), grid, threads, 0, st, a);
    } else {
      hipLaunchKernelGGL((tqk_encode_group<4, D, MG>), grid, threads, 0, st, a);
    }
  }
}
// the smallest instance that takes the groups (at 128 tokens only where its key
// tile lets four workgroups share a CU: fp16 at head_dim 64)
template <int D>
void launch_by_group(hipStream_t st, const EncodeArgs& a) {
  const int G = a.d.group_tokens;
  if (G <= 64) return launch_by_vb<D, 64>(a.d.value_bits, st, a);
  if constexpr (D == 64) {
    if (G <= 128 && !a.d.input_f32) return launch_by_vb<D, 128>(a.d.value_bits, st, a);
  }
  launch_by_vb<D, TQK_MAX_G>(a.d.value_bits, st, a);
}
template <int D, typename T>
void launch_dequant(int vb, dim3 grid, hipStream_t st, const DequantArgs& a) {
  if (vb == 2)
    hipLaunchKernelGGL((tqk_dequant_tokens<2, D, T>), grid, dim3(kThreads), 0, st, a);
  else if (vb == 3)
    hipLaunchKernelGGL((tqk_dequant_tokens<3, D, T>), grid, dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((tqk_dequant_tokens<4, D, T>), grid, dim3(kThreads), 0, st, a);
}
template <typename T>
int launch_dequant(dim3 grid, void* stream, const DequantArgs& a) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (a.d.head_dim == 64)
    launch_dequant<64, T>(a.d.value_bits, grid, st, a);
  else if (a.d.head_dim == 128)
    launch_dequant<128, T>(a.d.value_bits, grid, st, a);
  else
    launch_dequant<256, T>(a.d.value_bits, grid, st, a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

int launch_encode(const EncodeArgs& a, void* stream) {
  const tqk_cache_desc& d = a.d;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (d.key_grid == 0 && d.zero_point == 2 && !a.p.zp_mean) return TQK_EINVAL;
  if (d.key_grid == 2 && !a.p.knorm) return TQK_EINVAL;
  if (d.head_dim == 64)
    launch_by_group<64>(st, a);
  else if (d.head_dim == 128)
    launch_by_group<128>(st, a);
  else
    launch_by_group<256>(st, a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

int launch_hot(const HotArgs& a, int batch, void* stream) {
  // the surviving tokens of a sequence number at most min(chunk, ring)
  const int span = min(a.chunk_tokens, a.d.hot_ring);
  const int slices = max(1, (span + kHotSlice - 1) / kHotSlice);
  hipLaunchKernelGGL(tqk_append_hot_kernel, dim3(batch, a.d.n_kv_heads, slices), dim3(kThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

}  // namespace

extern "C" {

int tqk_encode_groups(const tqk_cache_desc* d, const tqk_cache_ptrs* p, int32_t batch,
                      int32_t n_items, const int32_t* items, const int32_t* prev_len,
                      const void* chunk_k, const void* chunk_v, int32_t chunk_tokens,
                      int32_t* overflow, void* stream) {
  int rc = tqk_check_desc(d);
  if (rc != TQK_OK) return rc;
  if (!p || batch <= 0 || n_items < 0 || chunk_tokens < 0) return TQK_EINVAL;
  if (n_items == 0) return TQK_OK;
  if (!items || !prev_len) return TQK_EINVAL;
  EncodeArgs a{};
  a.d = *d;
  a.p = *p;
  a.items = items;
  a.prev_len = prev_len;
  a.chunk_k = chunk_k;
  a.chunk_v = chunk_v;
  a.chunk_tokens = chunk_tokens;
  a.n_items = n_items;
  a.overflow = overflow;
  return launch_encode(a, stream);
}

int tqk_append_hot(const tqk_cache_desc* d, const tqk_cache_ptrs* p, int32_t batch,
                   const int32_t* prev_len, const int32_t* n_new, const int32_t* hot_start,
                   const void* chunk_k, const void* chunk_v, int32_t chunk_tokens,
                   void* stream) {
  int rc = tqk_check_desc(d);
  if (rc != TQK_OK) return rc;
  if (!p || batch <= 0 || !prev_len || !n_new || !hot_start || !chunk_k || !chunk_v ||
      chunk_tokens <= 0)
    return TQK_EINVAL;
  HotArgs a{};
  a.d = *d;
  a.hot_k = static_cast<uint8_t*>(p->hot_k);
  a.hot_v = static_cast<uint8_t*>(p->hot_v);
  a.prev_len = prev_len;
  a.n_new = n_new;
  a.hot_start = hot_start;
  a.chunk_k = static_cast<const uint8_t*>(chunk_k);
  a.chunk_v = static_cast<const uint8_t*>(chunk_v);
  a.chunk_tokens = chunk_tokens;
  return launch_hot(a, batch, stream);
}

int tqk_append_tokens(const tqk_cache_desc* d, const tqk_cache_ptrs* p, int32_t batch,
                      const int32_t* prev_len, const int32_t* n_new, const void* chunk_k,
                      const void* chunk_v, int32_t chunk_tokens, int32_t* seq_lens,
                      int32_t* overflow, void* stream) {
  int rc = tqk_check_desc(d);
  if (rc != TQK_OK) return rc;
  if (!p || !prev_len || !n_new || !chunk_k || !chunk_v || !seq_lens || chunk_tokens <= 0 || batch <= 0 ||
      batch > kInlineSeqs)
    return TQK_EINVAL;
  EncodeArgs e{};
  HotArgs a{};
  for (int b = 0; b < batch; ++b) {
    if (prev_len[b] < 0 || n_new[b] < 0 || n_new[b] > chunk_tokens) return TQK_EINVAL;
    e.in.prev[b] = a.in_prev[b] = prev_len[b];
    a.in_new[b] = n_new[b];
    if (n_new[b] > INT32_MAX - prev_len[b]) return TQK_EINVAL;
    const int g1 = n_groups_of(prev_len[b] + n_new[b], d->hot_window, d->group_tokens);
    int g = n_groups_of(prev_len[b], d->hot_window, d->group_tokens);
    // the new groups' slots and pages are in the tables
    if (g < g1 && (g1 > d->max_groups_per_seq ||
                   (long long)g1 * d->group_tokens > (long long)d->max_pages_per_seq * d->page_tokens))
      return TQK_EINVAL;
    for (; g < g1; ++g) {
      if (e.n_items == kInlineItems) return TQK_EINVAL;
      e.in.item[2 * e.n_items] = b;
      e.in.item[2 * e.n_items + 1] = g;
      ++e.n_items;
    }
  }
  if (e.n_items > 0) {
    e.d = *d;
    e.p = *p;
    e.chunk_k = chunk_k;
    e.chunk_v = chunk_v;
    e.chunk_tokens = chunk_tokens;
    e.overflow = overflow;
    rc = launch_encode(e, stream);
    if (rc != TQK_OK) return rc;
  }
  a.d = *d;
  a.hot_k = static_cast<uint8_t*>(p->hot_k);
  a.hot_v = static_cast<uint8_t*>(p->hot_v);
  a.chunk_k = static_cast<const uint8_t*>(chunk_k);
  a.chunk_v = static_cast<const uint8_t*>(chunk_v);
  a.chunk_tokens = chunk_tokens;
  a.seq_lens = seq_lens;
  return launch_hot(a, batch, stream);
}

int tqk_dequant_groups(const tqk_cache_desc* d, const tqk_cache_ptrs* p, int32_t n_items,
                       const int32_t* items, float* kout, float* vout, void* stream) {
  int rc = tqk_check_desc(d);
  if (rc != TQK_OK) return rc;
  if (!p || n_items < 0 || (n_items > 0 && (!items || !kout || !vout))) return TQK_EINVAL;
  if (n_items == 0) return TQK_OK;
  if (d->key_grid == 2 && !p->knorm) return TQK_EINVAL;
  const int chunks = (d->group_tokens + kDqTokens - 1) / kDqTokens;
  const DequantArgs a{*d, *p, items, nullptr, chunks, 0, kout, vout};
  return launch_dequant<float>(dim3((unsigned)n_items * (unsigned)chunks, d->n_kv_heads), stream, a);
}

int tqk_dequant_dense(const tqk_cache_desc* d, const tqk_cache_ptrs* p, int32_t batch,
                      const int32_t* seq_lens, int32_t max_len, int32_t out_type, void* kout,
                      void* vout, void* stream) {
  int rc = tqk_check_desc(d);
  if (rc != TQK_OK) return rc;
  if (!p || batch <= 0 || max_len <= 0 || !seq_lens || !kout || !vout) return TQK_EINVAL;
  if (d->key_grid == 2 && !p->knorm) return TQK_EINVAL;
  if (out_type < 0 || out_type > 2) return TQK_EINVAL;
  const int G = d->group_tokens, cpg = (G + kDqTokens - 1) / kDqTokens;
  const long long chunks = (long long)n_groups_of(max_len, d->hot_window, G) * cpg +
                           (min(max_len, d->hot_window) + kDqTokens - 1) / kDqTokens;
  if (chunks * batch >= (1LL << 31)) return TQK_EINVAL;
  const DequantArgs a{*d, *p, nullptr, seq_lens, (int)chunks, max_len, kout, vout};
  const dim3 grid((unsigned)(chunks * batch), d->n_kv_heads);
  if (out_type == 0) return launch_dequant<float>(grid, stream, a);
  if (out_type == 1) return launch_dequant<_Float16>(grid, stream, a);
  return launch_dequant<__bf16>(grid, stream, a);
}

}  // extern "C"
