// Stateless block quantizers and their reconstruction (gfx950).
//
// One (B, H, S, D) block per call, every (b, h) pair one quantization group of
// S tokens (any S >= 1), fp16 or fp32 input, outputs in the reference
// containers' layouts: the whole-layer records of the plugin / block-store
// path, which the cache's 256-token group encode does not cover.
//
// Bit-exactness contract (compiled with -ffp-contract=off, explicitly rounded
// __f*_rn operations), the same NumPy operation order as the group encode:
//   keys   (turboquant_pro/per_channel_kv.py:269-401)
//     asym-NF4: mu = token-order sequential fp32 sum / S (a float64 division,
//               then fp32), times the DC mask ("sparse") or given ("bias");
//               amax = max(max_s |x_s - mu|, 1e-8); cent = mu + amax * NF4[l];
//               code = first argmin_l |x - cent_l|
//     uniform:  scale = max(max - min, 1e-8) / (2^bits - 1);
//               code = clip(rint((x - min) / scale), 0, 2^bits - 1)
//   key packing (per_channel_kv.py:87-100): each code's bits LSB first, in
//   MSB-first bytes, codes in (b, h, s, j) order (4-bit: byte n =
//   rev4(code[2n]) << 4 | rev4(code[2n+1]); a token row is D * bits / 8 bytes)
//     outliers: threshold = k-th largest |x| over s; every |x| >= it, (s, j) order
//   values (turboquant_pro/core.py:569-606): pairwise norm, u = x / max(norm, 1e-30),
//     y_e = sequential over d of u_d * Pi[e][d], code = #{ boundaries < y_e }
#include "tqk_common.h"

namespace {

constexpr int kKbThreads = 256;  // key dequant kernels
constexpr int kVbThreads = 512;  // value block: 64 tokens per workgroup
constexpr int kVbTokens = 64;

__device__ __forceinline__ float load_x(const void* x, int f32, size_t i) {
  return f32 ? reinterpret_cast<const float*>(x)[i] : h2f(reinterpret_cast<const uint16_t*>(x)[i]);
}
// N values of x at i0, i0 + stride, ..., every load issued before any is used
template <int N>
__device__ __forceinline__ void load_xn(const void* x, int f32, size_t i0, size_t stride, float (&v)[N]) {
  if (f32) {
    const float* p = reinterpret_cast<const float*>(x) + i0;
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = p[u * stride];
  } else {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(x) + i0;
    uint16_t r[N];
#pragma unroll
    for (int u = 0; u < N; ++u) r[u] = p[u * stride];
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = h2f(r[u]);
  }
}
// f(s, x[s, col]) for s = s0, s0 + st, ... < s1, in that order, the loads of
// 32 tokens at a time in flight (rows of D elements; one or two waves per SIMD
// run these loops, so each batch waits one memory latency)
template <int D, typename F>
__device__ __forceinline__ void for_tokens(const void* x, int f32, size_t col, int s0, int s1, int st, F f) {
  constexpr int N = 32;
  int s = s0;
  for (; s + (N - 1) * st < s1; s += N * st) {
    float v[N];
    load_xn<N>(x, f32, col + (size_t)s * D, (size_t)st * D, v);
#pragma unroll
    for (int u = 0; u < N; ++u) f(s + u * st, v[u]);
  }
  for (; s < s1; s += st) f(s, load_x(x, f32, col + (size_t)s * D));
}
// f(s, x[s, col], x[s, col + 1]) in token order, 16 tokens' loads in flight
template <int D, typename F>
__device__ __forceinline__ void for_token_pairs(const void* x, int f32, size_t col, int s0, int s1, F f) {
  constexpr int N = 16;
  int s = s0;
  for (; s + N - 1 < s1; s += N) {
    float v0[N], v1[N];
    load_xn<N>(x, f32, col + (size_t)s * D, D, v0);
    load_xn<N>(x, f32, col + 1 + (size_t)s * D, D, v1);
#pragma unroll
    for (int u = 0; u < N; ++u) f(s + u, v0[u], v1[u]);
  }
  for (; s < s1; ++s) f(s, load_x(x, f32, col + (size_t)s * D), load_x(x, f32, col + 1 + (size_t)s * D));
}
__device__ __forceinline__ bool dc_channel(const tqk_block_desc& d, int j) {
  return (d.dc_mask[j >> 5] >> (j & 31)) & 1u;
}
// code c of channel j into a token row of little-endian dwords, in the
// reference's bit order (bit k of c at stream position j * bits + k, streams
// filling bytes from their most significant bit)
__device__ __forceinline__ void put_code_ref(uint32_t* rw, int j, int bits, uint32_t c) {
  for (int k = 0; k < bits; ++k) {
    const int p = j * bits + k;
    rw[p >> 5] |= ((c >> k) & 1u) << (8 * ((p >> 3) & 3) + 7 - (p & 7));
  }
}
// code n of a packed key stream (the reference's bit order)
__device__ __forceinline__ uint32_t get_code_ref(const uint8_t* packed, size_t n, int bits, size_t nbytes) {
  const size_t p = n * (size_t)bits, b0 = p >> 3;
  const uint32_t win = ((uint32_t)packed[b0] << 8) | (b0 + 1 < nbytes ? packed[b0 + 1] : 0u);
  const int o = (int)(p & 7);
  uint32_t c = 0;
  for (int k = 0; k < bits; ++k) c |= ((win >> (15 - o - k)) & 1u) << k;
  return c;
}

struct KeyBlockArgs {
  tqk_block_desc d;
  const void* x;
  const float* zp;
  uint8_t* packed;
  float* scale;
  float* zero;
  uint32_t* out_pos;
  uint16_t* out_val;
  int32_t* out_count;
  int n_chunks;  // kKbChunk-token chunks of a (b, h)
  int bh0;       // first (b, h) of the launch
};

// ---- key blocks over the chip -------------------------------------------------
// Four kernels: tqk_key_block_stats (a workgroup per (b, h) and 16 channels:
// zero point, scale, outlier threshold), tqk_key_block_masks (a workgroup per
// (b, h) and 256 tokens: the outlier bits of every token and the chunk's
// count), tqk_key_block_list (the same grid: the side-list, each chunk at the
// offset that the counts before it give) and tqk_key_block_codes (the same
// grid).  Until the codes are written, the (b, h)'s part of the packed output
// holds what the first kernels hand on, from its first dword boundary: D
// thresholds, n_chunks counts, and D bits a token (KbScratch).  Neither the
// side-list's capacity nor the alignment of x and packed matters.  Bound: the stats kernel's ordered sum, 16000 tokens
// one after another at about five cycles each, and its passes over the block.
// One 1 x 8 x 16000 x 128 fp32 block: 3147 us with the thresholds on a workgroup
// per 64 channels (16 passes) and statistics and side-list on one per (b, h),
// 251 us like this.
constexpr int kKbChunk = 256;
constexpr int kKbTile = 512;           // tokens per LDS tile of the ordered sum
constexpr int kKbLd = kKbTile + 4;     // tile row stride: 16 channels x 4 tokens on 64 banks
constexpr int kKbStatThreads = 1024;

struct KbScratch {
  uint32_t* thr;     // [D]
  uint32_t* count;   // [n_chunks]
  uint32_t* mask;    // [S][D / 32]
};
__device__ __forceinline__ KbScratch kb_scratch(const KeyBlockArgs& a, int bh) {
  const int D = a.d.head_dim;
  uint8_t* p = a.packed + (size_t)bh * ((size_t)a.d.tokens * D * a.d.bits / 8);
  uint32_t* base = reinterpret_cast<uint32_t*>(p + (-reinterpret_cast<uintptr_t>(p) & 3u));
  return {base, base + D, base + D + a.n_chunks};
}

template <bool F32>
__device__ __forceinline__ float kb_load(const void* x, size_t i) {
  if constexpr (F32) return reinterpret_cast<const float*>(x)[i];
  else return h2f(reinterpret_cast<const uint16_t*>(x)[i]);
}

// Statistics and thresholds of 16 channels.  A wave's load is four tokens x 16
// channels (lane: token lane / 16, channel lane % 16).
// Pass 1 reads the block tile by tile: minimum, maximum, a histogram of the top
// eight magnitude bits (LDS columns of the lane's own, so atomics never share a
// bank), and the tile transposed for wave 0, which sums it in token order (its
// lane c: channel c) while the others read on.
// amax = max |x - mu| is taken at the channel's two ends: rounding is monotone.
// Passes 2 .. 4 refine the threshold by 8, 8 and 7 bits: the largest magnitude
// pattern T with #{ |x| >= T } >= k is the k-th largest, so each pass picks the
// bin, counted from the top, in which the k-th falls.  Up to 128 tokens a wave
// counts for its channel, a lane two tokens, how many are above them instead
// (clearing and scanning the histograms took most of such a block: 1 x 8 x 64 x
// 128 fp32 at 2 bits 78 us, with the codes of short blocks over all threads 31).
template <int D, bool F32>
__global__ __launch_bounds__(kKbStatThreads) void tqk_key_block_stats(KeyBlockArgs a) {
  constexpr int NW = kKbStatThreads / 64, PER = kKbTile / (4 * NW);  // loads per thread and tile
  const tqk_block_desc& d = a.d;
  const int bh = a.bh0 + blockIdx.x / (D / 16), c0 = 16 * (blockIdx.x % (D / 16));
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, ch = lane & 15, sub = lane >> 4;
  const int S = d.tokens, kout = d.outliers_per_channel;
  const bool small = S <= 128, select = kout > 0 && kout < S, radix = select && !small, sum = d.key_grid == 0 && d.zero_point != 2;
  const size_t base = (size_t)bh * S * D + c0 + ch;

  __shared__ __align__(16) float tile_s[2][16][kKbLd];
  __shared__ uint32_t hist_s[256][64];
  __shared__ float red_s[3][NW][16];
  __shared__ float mean_s[16];
  __shared__ uint32_t pre_s[16];  // the threshold's bits found so far
  __shared__ int rem_s[16];       // the rank left within them

  auto clear = [&]() {
    for (int i = tid; i < 256 * 64; i += kKbStatThreads) (&hist_s[0][0])[i] = 0u;
  };
  // channel wv: the bin in which the rem-th value from the top falls
  auto pick = [&](int shift) {
    int n[4], tot = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t* row = hist_s[255 - (4 * lane + i)];
      n[i] = (int)(row[wv] + row[16 + wv] + row[32 + wv] + row[48 + wv]);
      tot += n[i];
    }
    int incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    int left = rem_s[wv] - (incl - tot);
    if (left > 0 && left <= tot) {
      int i = 0;
      while (left > n[i]) left -= n[i++];
      pre_s[wv] |= (uint32_t)(255 - (4 * lane + i)) << shift;
      rem_s[wv] = left;
    }
  };

  if (tid < 16) {
    pre_s[tid] = 0u;
    rem_s[tid] = kout;
  }
  if (radix) clear();
  __syncthreads();

  // ---- pass 1
  float mn = __builtin_inff(), mx = -__builtin_inff(), acc = 0.0f;
  uint32_t top = 0;
  const int n_tiles = (S + kKbTile - 1) / kKbTile;
  float x[PER], nx[PER];
  auto load_tile = [&](int t0, float (&v)[PER]) {
#pragma unroll
    for (int u = 0; u < PER; ++u)
      v[u] = kb_load<F32>(a.x, base + (size_t)min(S - 1, t0 + 4 * (PER * wv + u) + sub) * D);
  };
  load_tile(0, x);
  for (int ti = 0; ti < n_tiles; ++ti) {
    const int t0 = ti * kKbTile;
    if (ti + 1 < n_tiles) load_tile(t0 + kKbTile, nx);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int s = 4 * (PER * wv + u) + sub;
      const uint32_t m = __float_as_uint(fabsf(x[u]));
      mn = fminf(mn, x[u]);  // (tokens past the end repeat the last one)
      mx = fmaxf(mx, x[u]);
      top = max(top, m);
      if (sum || small) tile_s[ti & 1][ch][s] = x[u];
      if (radix && t0 + s < S) atomicAdd(&hist_s[m >> 23][lane], 1u);
    }
    __syncthreads();
    // (the other buffer is written next; this one only after the next barrier)
    if (sum && wv == 0) {
      const float* row = tile_s[ti & 1][ch];
      const int n = min(kKbTile, S - t0);
      int s = 0;
      for (; s + 32 <= n; s += 32) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const float4*>(row + s + 4 * u);
#pragma unroll
        for (int u = 0; u < 8; ++u)
          acc = __fadd_rn(__fadd_rn(__fadd_rn(__fadd_rn(acc, v[u].x), v[u].y), v[u].z), v[u].w);
      }
      for (; s < n; ++s) acc = __fadd_rn(acc, row[s]);
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) x[u] = nx[u];
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
  }
  if (sub == 0) {
    red_s[0][wv][ch] = mn;
    red_s[1][wv][ch] = mx;
    red_s[2][wv][ch] = __uint_as_float(top);
  }
  if (wv == 0 && sub == 0) mean_s[ch] = acc;
  if (radix) pick(23);
  if (select && small) {
    uint32_t m[2];
    int above[2] = {0, 0}, from[2] = {0, 0};  // tokens above the lane's, and not below it
#pragma unroll
    for (int u = 0; u < 2; ++u) m[u] = __float_as_uint(fabsf(tile_s[0][wv][lane + 64 * u]));
    auto count = [&](uint32_t src, int n) {
      for (int s = 0; s < n; ++s) {
        const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)src, s);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          above[u] += v > m[u] ? 1 : 0;
          from[u] += v >= m[u] ? 1 : 0;
        }
      }
    };
    count(m[0], min(S, 64));
    count(m[1], S - 64);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (lane + 64 * u < S && above[u] < kout && kout <= from[u]) pre_s[wv] = m[u];  // (ties: the same value)
  }
  __syncthreads();
  if (tid < 16) {
    for (int w = 0; w < NW; ++w) {
      mn = fminf(mn, red_s[0][w][tid]);
      mx = fmaxf(mx, red_s[1][w][tid]);
      top = max(top, __float_as_uint(red_s[2][w][tid]));
    }
    const int j = c0 + tid;
    const bool xnan = top > 0x7F800000u;
    float z, sc;
    if (d.key_grid == 1) {
      z = xnan ? __builtin_nanf("") : mn;
      sc = xnan ? __builtin_nanf("") : __fdiv_rn(fmaxf(__fsub_rn(mx, mn), 1e-8f), (float)((1 << d.bits) - 1));
    } else {
      if (d.zero_point == 2) {
        z = a.zp[(size_t)(bh % d.n_heads) * D + j];
      } else {
        z = (float)((double)mean_s[tid] / (double)S);
        if (d.zero_point == 1) z = __fmul_rn(z, dc_channel(d, j) ? 1.0f : 0.0f);
      }
      const float lo = fabsf(__fsub_rn(mn, z)), hi = fabsf(__fsub_rn(mx, z));
      const bool nan = xnan || lo != lo || hi != hi;
      sc = nan ? __builtin_nanf("") : fmaxf(fmaxf(lo, hi), 1e-8f);
    }
    a.scale[(size_t)bh * D + j] = sc;
    a.zero[(size_t)bh * D + j] = z;
    if (kout == 0 && j == 0) a.out_count[bh] = 0;
  }
  if (!select) return;

  // ---- passes 2 .. 4 (fp16 values have no bits below the third)
  for (int lv = 1; radix && lv < (F32 ? 4 : 3); ++lv) {
    const int above = 31 - 8 * lv, shift = lv == 3 ? 0 : above - 8, mask = lv == 3 ? 127 : 255;
    __syncthreads();
    clear();
    const uint32_t pre = pre_s[ch] >> above;
    __syncthreads();
    for (int s0 = 0; s0 < S; s0 += kKbTile) {
      float v[PER];
      load_tile(s0, v);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const uint32_t m = __float_as_uint(fabsf(v[u]));
        if ((m >> above) == pre && s0 + 4 * (PER * wv + u) + sub < S)
          atomicAdd(&hist_s[(m >> shift) & mask][lane], 1u);
      }
    }
    __syncthreads();
    pick(shift);
  }
  __syncthreads();
  if (tid < 16) kb_scratch(a, bh).thr[c0 + tid] = pre_s[tid];
}

// The outlier bits of 256 tokens: a lane per channel of each 64-channel piece,
// a ballot a token; a wave takes 64 tokens and lane t keeps token t's bits.
template <int D, bool F32>
__global__ __launch_bounds__(kKbChunk) void tqk_key_block_masks(KeyBlockArgs a) {
  constexpr int NC = D / 64, N = 16;
  const int bh = a.bh0 + blockIdx.x / a.n_chunks, c = blockIdx.x % a.n_chunks;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, S = a.d.tokens;
  const KbScratch sc = kb_scratch(a, bh);
  const int s0 = c * kKbChunk + 64 * wv, n = min(64, S - s0);
  __shared__ int n_s[kKbChunk / 64];
  int cnt = 0;
  if (n > 0) {
#pragma unroll
    for (int p = 0; p < NC; ++p) {
      const float th = __uint_as_float(sc.thr[64 * p + lane]);  // (a NaN threshold selects nothing)
      const size_t base = ((size_t)bh * S + s0) * D + 64 * p + lane;
      uint64_t mine = 0;
      for (int t = 0; t < n; t += N) {
        float v[N];
#pragma unroll
        for (int u = 0; u < N; ++u) v[u] = kb_load<F32>(a.x, base + (size_t)min(t + u, n - 1) * D);
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const uint64_t m = __ballot(fabsf(v[u]) >= th);
          mine = lane == t + u ? m : mine;
        }
      }
      if (lane < n) {
        uint32_t* dst = sc.mask + (size_t)(s0 + lane) * (D / 32) + 2 * p;
        dst[0] = (uint32_t)mine;
        dst[1] = (uint32_t)(mine >> 32);
        cnt += __popcll(mine);
      }
    }
  }
  cnt = wave_sum(cnt);
  if (lane == 0) n_s[wv] = cnt;
  __syncthreads();
  if (tid == 0) sc.count[c] = (uint32_t)(n_s[0] + n_s[1] + n_s[2] + n_s[3]);
}

// The side-list entries of 256 tokens in (s, j) order, one token per thread;
// every element is one when k >= S.
template <int D, bool F32>
__global__ __launch_bounds__(kKbChunk) void tqk_key_block_list(KeyBlockArgs a) {
  const tqk_block_desc& d = a.d;
  const int bh = a.bh0 + blockIdx.x / a.n_chunks, c = blockIdx.x % a.n_chunks;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, S = d.tokens;
  const bool all = d.outliers_per_channel >= S;
  const KbScratch sc = kb_scratch(a, bh);
  const int s = c * kKbChunk + tid;
  __shared__ uint32_t sum_s[2][kKbChunk / 64];
  // entries in the chunks before this one, and in all of them (S * D < 2^32)
  uint32_t before = 0, total = 0;
  if (all) {
    before = (uint32_t)c * kKbChunk * D;
    total = (uint32_t)S * D;
  } else {
    for (int i = tid; i < a.n_chunks; i += kKbChunk) {
      const uint32_t n = sc.count[i];
      total += n;
      before += i < c ? n : 0u;
    }
    before = wave_sum(before);
    total = wave_sum(total);
    if (lane == 0) {
      sum_s[0][wv] = before;
      sum_s[1][wv] = total;
    }
    __syncthreads();
    before = sum_s[0][0] + sum_s[0][1] + sum_s[0][2] + sum_s[0][3];
    total = sum_s[1][0] + sum_s[1][1] + sum_s[1][2] + sum_s[1][3];
    __syncthreads();
  }
  if (c == 0 && tid == 0) a.out_count[bh] = (int32_t)total;
  uint32_t w[D / 32];
  uint32_t cnt = 0;
#pragma unroll
  for (int k = 0; k < D / 32; ++k) {
    w[k] = s < S ? (all ? 0xFFFFFFFFu : sc.mask[(size_t)s * (D / 32) + k]) : 0u;
    cnt += (uint32_t)__builtin_popcount(w[k]);
  }
  uint32_t incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) sum_s[0][wv] = incl;
  __syncthreads();
  uint32_t off = before + incl - cnt;
  for (int i = 0; i < wv; ++i) off += sum_s[0][i];
  const size_t lb = (size_t)bh * d.outlier_cap, row = ((size_t)bh * S + s) * D;
#pragma unroll
  for (int k = 0; k < D / 32; ++k) {
    while (w[k] && off < (uint32_t)d.outlier_cap) {
      const int j = 32 * k + __builtin_ctz(w[k]);
      w[k] &= w[k] - 1u;
      a.out_pos[lb + off] = (uint32_t)s * D + (uint32_t)j;
      a.out_val[lb + off] = f2h(kb_load<F32>(a.x, row + j));  // fp16, round to nearest even
      ++off;
    }
  }
}

// The codes of 256 tokens.  4-bit: thread = (channel pair, token slice), the
// levels rebuilt from the stored scale and zero point with the same arithmetic.
// Levels that are finite and far enough apart for the rounded distances to
// order as the real ones (gaps of at least 16 ulps of the largest distance, 2
// (|mean| + amax)) make the first argmin the number of strict decreases from
// level to level; the others take the comparison that also orders NaN.  2- and
// 3-bit (uniform): a token row, or 32 channels of it, per thread.
template <int D, bool F32>
__global__ __launch_bounds__(kKbChunk) void tqk_key_block_codes(KeyBlockArgs a) {
  constexpr int NPR = D / 2, NS = kKbChunk / NPR, PER = kKbChunk / NS;
  const tqk_block_desc& d = a.d;
  const int bh = a.bh0 + blockIdx.x / a.n_chunks, c = blockIdx.x % a.n_chunks;
  const int tid = threadIdx.x, S = d.tokens;
  const size_t base = (size_t)bh * S * D;
  const int t0 = c * kKbChunk, t1 = min(S, t0 + kKbChunk);
  if (d.bits != 4) {
    // a token row per thread, or for up to 128 tokens 32 channels of it (whole
    // dwords), so that a short block's threads all have work
    const int bits = d.bits;
    const float qmax = (float)((1 << bits) - 1);
    auto code = [&](size_t i, size_t j) {
      const float r = __builtin_rintf(__fdiv_rn(__fsub_rn(kb_load<F32>(a.x, i), a.zero[j]), a.scale[j]));
      return (uint32_t)fminf(fmaxf(r, 0.0f), qmax);
    };
    if (t1 - t0 <= 128) {
      for (int i = tid; i < (t1 - t0) * (D / 32); i += kKbChunk) {
        const int s = t0 + i / (D / 32), c32 = i % (D / 32);
        uint32_t rw[4] = {0u, 0u, 0u, 0u};
        for (int j = 0; j < 32; ++j)
          put_code_ref(rw, j, bits, code(base + (size_t)s * D + 32 * c32 + j, (size_t)bh * D + 32 * c32 + j));
        uint8_t* dst = a.packed + ((size_t)bh * S + s) * (size_t)(D * bits / 8) + 4 * bits * c32;  // (at any byte)
        for (int w = 0; w < bits; ++w) __builtin_memcpy(dst + 4 * w, &rw[w], 4);
      }
      return;
    }
    const int s = t0 + tid;
    if (s >= S) return;
    uint32_t rw[D / 8] = {0u};
    for (int j = 0; j < D; ++j) put_code_ref(rw, j, bits, code(base + (size_t)s * D + j, (size_t)bh * D + j));
    uint8_t* dst = a.packed + ((size_t)bh * S + s) * (size_t)(D * bits / 8);
    for (int w = 0; w < D * bits / 32; ++w) __builtin_memcpy(dst + 4 * w, &rw[w], 4);
    return;
  }
  const int jp = tid % NPR, sq = tid / NPR;
  const int s0 = min(t1, t0 + sq * PER), s1 = min(t1, s0 + PER);
  uint8_t* out = a.packed + base / 2 + jp;
  const size_t cj = (size_t)bh * D + 2 * jp;
  const float sc0 = a.scale[cj], z0 = a.zero[cj], sc1 = a.scale[cj + 1], z1 = a.zero[cj + 1];
  auto for_pairs = [&](auto f) {
    constexpr int N = 8;
    for (int s = s0; s < s1; s += N) {
      float v0[N], v1[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const size_t i = base + (size_t)min(s + u, s1 - 1) * D + 2 * jp;
        // (the pair may start at any element's boundary)
        if constexpr (F32) {
          float p[2];
          __builtin_memcpy(p, reinterpret_cast<const float*>(a.x) + i, sizeof(p));
          v0[u] = p[0];
          v1[u] = p[1];
        } else {
          uint32_t p;
          __builtin_memcpy(&p, reinterpret_cast<const uint16_t*>(a.x) + i, sizeof(p));
          v0[u] = h2f((uint16_t)p);
          v1[u] = h2f((uint16_t)(p >> 16));
        }
      }
#pragma unroll
      for (int u = 0; u < N; ++u)
        if (s + u < s1) f(s + u, v0[u], v1[u]);
    }
  };
  if (d.key_grid == 1) {
    for_pairs([&](int s, float x0, float x1) {
      const float r0 = __builtin_rintf(__fdiv_rn(__fsub_rn(x0, z0), sc0));
      const float r1 = __builtin_rintf(__fdiv_rn(__fsub_rn(x1, z1), sc1));
      const uint32_t b0 = (uint32_t)fminf(fmaxf(r0, 0.0f), 15.0f);
      const uint32_t b1 = (uint32_t)fminf(fmaxf(r1, 0.0f), 15.0f);
      out[(size_t)s * (D / 2)] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
    });
    return;
  }
  float c0[16], c1[16];
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    c0[l] = __fadd_rn(z0, __fmul_rn(sc0, kNF4[l]));
    c1[l] = __fadd_rn(z1, __fmul_rn(sc1, kNF4[l]));
  }
  const float r0 = __fmul_rn(__fadd_rn(fabsf(z0), sc0), 0x1p-18f);
  const float r1 = __fmul_rn(__fadd_rn(fabsf(z1), sc1), 0x1p-18f);
  // (false for levels that are not finite; every |x - mean| <= amax, so finite
  // levels mean finite keys)
  bool spread = __builtin_isfinite(c0[15]) && __builtin_isfinite(c1[15]);
#pragma unroll
  for (int l = 1; l < 16; ++l)
    spread &= __fsub_rn(c0[l], c0[l - 1]) >= r0 && __fsub_rn(c1[l], c1[l - 1]) >= r1;
  if (__all(spread)) {
    for_pairs([&](int s, float x0, float x1) {
      uint32_t b0 = 0, b1 = 0;
      float d0 = fabsf(__fsub_rn(x0, c0[0])), d1 = fabsf(__fsub_rn(x1, c1[0]));
#pragma unroll
      for (int l = 1; l < 16; ++l) {
        const float e0 = fabsf(__fsub_rn(x0, c0[l])), e1 = fabsf(__fsub_rn(x1, c1[l]));
        b0 += (e0 < d0) ? 1u : 0u;
        b1 += (e1 < d1) ? 1u : 0u;
        d0 = e0;
        d1 = e1;
      }
      out[(size_t)s * (D / 2)] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
    });
  } else {
    for_pairs([&](int s, float x0, float x1) {
      uint32_t b0 = 0, b1 = 0;
      float d0 = fabsf(__fsub_rn(x0, c0[0])), d1 = fabsf(__fsub_rn(x1, c1[0]));
#pragma unroll
      for (int l = 1; l < 16; ++l) {
        const float e0 = fabsf(__fsub_rn(x0, c0[l])), e1 = fabsf(__fsub_rn(x1, c1[l]));
        // np.argmin: strictly smaller wins; the first NaN wins over any number
        if (e0 < d0 || (e0 != e0 && d0 == d0)) { d0 = e0; b0 = l; }
        if (e1 < d1 || (e1 != e1 && d1 == d1)) { d1 = e1; b1 = l; }
      }
      out[(size_t)s * (D / 2)] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
    });
  }
}

// The same in one workgroup of 2 * D threads per (b, h): blocks with outliers
// whose packed output cannot hold KbScratch: S D bits / 32 dwords below D + 2 + S
// D / 32, fewer than 34 tokens at 2 bits and head_dim 64.
constexpr int kKbFew = 36;
template <int D>
__global__ __launch_bounds__(2 * D) void tqk_key_block(KeyBlockArgs a) {
  constexpr int T = 2 * D;  // threads
  const tqk_block_desc& d = a.d;
  const int bh = blockIdx.x, h = bh % d.n_heads, tid = threadIdx.x;
  const int S = d.tokens, f32 = d.input_f32, kout = d.outliers_per_channel;
  const size_t base = (size_t)bh * S * D;
  auto X = [&](int s, int j) { return load_x(a.x, f32, base + (size_t)s * D + j); };

  __shared__ float cent_s[D][17];  // per-channel grid (uniform: min, scale)
  __shared__ float thr_s[D];       // outlier threshold magnitude per channel
  __shared__ int32_t wsum_s[T / 64];

  // ---- per-channel statistics (threads 0..D-1) and thresholds (D..2D-1)
  if (tid < D) {
    const int j = tid;
    if (d.key_grid == 1) {
      float mn = X(0, j), mx = mn;
      bool nan = (mn != mn);
      for_tokens<D>(a.x, f32, base + j, 1, S, 1, [&](int, float xv) {
        nan |= (xv != xv);
        mn = fminf(mn, xv);
        mx = fmaxf(mx, xv);
      });
      const float sc = nan ? __builtin_nanf("") : __fdiv_rn(fmaxf(__fsub_rn(mx, mn), 1e-8f),
                                                            (float)((1 << d.bits) - 1));
      if (nan) mn = __builtin_nanf("");
      cent_s[j][0] = mn;
      cent_s[j][1] = sc;
      a.scale[(size_t)bh * D + j] = sc;
      a.zero[(size_t)bh * D + j] = mn;
    } else {
      float mu;
      if (d.zero_point == 2) {
        mu = a.zp[(size_t)h * D + j];
      } else {
        float acc = 0.0f;  // in token order
        for_tokens<D>(a.x, f32, base + j, 0, S, 1, [&](int, float xv) { acc = __fadd_rn(acc, xv); });
        mu = (float)((double)acc / (double)S);
        if (d.zero_point == 1) mu = __fmul_rn(mu, dc_channel(d, j) ? 1.0f : 0.0f);
      }
      float amax = 0.0f;
      bool nan = (mu != mu);
      for_tokens<D>(a.x, f32, base + j, 0, S, 1, [&](int, float xv) {
        const float dv = fabsf(__fsub_rn(xv, mu));
        nan |= (dv != dv);
        amax = fmaxf(amax, dv);
      });
      amax = nan ? __builtin_nanf("") : fmaxf(amax, 1e-8f);
#pragma unroll
      for (int l = 0; l < 16; ++l) cent_s[j][l] = __fadd_rn(mu, __fmul_rn(amax, kNF4[l]));
      a.scale[(size_t)bh * D + j] = amax;
      a.zero[(size_t)bh * D + j] = mu;
    }
  } else if (tid < 2 * D && kout > 0 && kout < S) {
    // k-th largest |x| as the largest fp32 magnitude pattern T with
    // #{ |x_s| >= T } >= k (NaN patterns order above inf, as np.partition does)
    const int j = tid - D;
    uint32_t m[kKbFew];  // (no tokens: magnitude 0)
#pragma unroll
    for (int s = 0; s < kKbFew; ++s) m[s] = s < S ? __float_as_uint(fabsf(X(s, j))) : 0u;
    uint32_t T = 0;
    for (int bit = 30; bit >= 0; --bit) {
      const uint32_t cand = T | (1u << bit);
      int cnt = 0;
#pragma unroll
      for (int s = 0; s < kKbFew; ++s) cnt += m[s] >= cand ? 1 : 0;
      if (cnt >= kout) T = cand;
    }
    thr_s[j] = __uint_as_float(T);
  }
  __syncthreads();

  // ---- codes of 3- and 2-bit (uniform) keys: one token row per thread
  if (d.bits != 4) {
    const int bits = d.bits, rwords = D * bits / 32;  // D * bits / 8 bytes per token
    const float qmax = (float)((1 << bits) - 1);
    for (int s = tid; s < S; s += T) {
      uint32_t rw[D / 8] = {0u};
      for (int j = 0; j < D; ++j) {
        const float r = __builtin_rintf(__fdiv_rn(__fsub_rn(X(s, j), cent_s[j][0]), cent_s[j][1]));
        put_code_ref(rw, j, bits, (uint32_t)fminf(fmaxf(r, 0.0f), qmax));
      }
      uint32_t* dst = reinterpret_cast<uint32_t*>(a.packed + ((size_t)bh * S + s) * (size_t)(D * bits / 8));
      for (int w = 0; w < rwords; ++w) dst[w] = rw[w];
    }
  }
  // ---- 4-bit codes: thread = (channel pair, token slice), one byte per (token, pair)
  else {
    const int jp = tid % (D / 2), sq = tid / (D / 2);  // four token slices
    const int per = (S + 3) / 4, s0 = sq * per, s1 = min(S, s0 + per);
    uint8_t* out = a.packed + base / 2 + jp;
    if (d.key_grid == 1) {
      const float mn0 = cent_s[2 * jp][0], sc0 = cent_s[2 * jp][1];
      const float mn1 = cent_s[2 * jp + 1][0], sc1 = cent_s[2 * jp + 1][1];
      for_token_pairs<D>(a.x, f32, base + 2 * jp, s0, s1, [&](int s, float x0, float x1) {
        const float r0 = __builtin_rintf(__fdiv_rn(__fsub_rn(x0, mn0), sc0));
        const float r1 = __builtin_rintf(__fdiv_rn(__fsub_rn(x1, mn1), sc1));
        const uint32_t b0 = (uint32_t)fminf(fmaxf(r0, 0.0f), 15.0f);
        const uint32_t b1 = (uint32_t)fminf(fmaxf(r1, 0.0f), 15.0f);
        out[(size_t)s * (D / 2)] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
      });
    } else {
      float c0[16], c1[16];
#pragma unroll
      for (int l = 0; l < 16; ++l) {
        c0[l] = cent_s[2 * jp][l];
        c1[l] = cent_s[2 * jp + 1][l];
      }
      for_token_pairs<D>(a.x, f32, base + 2 * jp, s0, s1, [&](int s, float x0, float x1) {
        int b0 = 0, b1 = 0;
        float d0 = fabsf(__fsub_rn(x0, c0[0])), d1 = fabsf(__fsub_rn(x1, c1[0]));
#pragma unroll
        for (int l = 1; l < 16; ++l) {
          const float e0 = fabsf(__fsub_rn(x0, c0[l])), e1 = fabsf(__fsub_rn(x1, c1[l]));
          // np.argmin: strictly smaller wins; the first NaN wins over any number
          if (e0 < d0 || (e0 != e0 && d0 == d0)) { d0 = e0; b0 = l; }
          if (e1 < d1 || (e1 != e1 && d1 == d1)) { d1 = e1; b1 = l; }
        }
        out[(size_t)s * (D / 2)] = (uint8_t)((rev4(b0) << 4) | rev4(b1));
      });
    }
  }

  // ---- outlier side-list in (s, j) order: wave w owns a contiguous token
  // range and a lane one channel of each 64-channel piece of a token row (one
  // coalesced row piece per load); the pieces' ballots count the wave's
  // entries, its offset comes from the waves before it, and the entries are
  // written at offset + the lanes before them in the ballot
  if (kout > 0) {
    const bool all = kout >= S;
    constexpr int NWV = T / 64, NC = D / 64;
    const int wv = tid >> 6, ln = tid & 63;
    const int chunk = (S + NWV - 1) / NWV;
    const int s0 = min(S, wv * chunk), s1 = min(S, s0 + chunk);
    float th[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) th[c] = thr_s[c * 64 + ln];
    int cnt = 0;  // the same in every lane of the wave
#pragma unroll
    for (int c = 0; c < NC; ++c)
      for_tokens<D>(a.x, f32, base + c * 64 + ln, s0, s1, 1, [&](int, float xv) {
        cnt += __popcll(__ballot(all || fabsf(xv) >= th[c]));
      });
    if (ln == 0) wsum_s[wv] = cnt;
    __syncthreads();
    int off = 0, total = 0;
    for (int w = 0; w < NWV; ++w) {
      if (w < wv) off += wsum_s[w];
      total += wsum_s[w];
    }
    if (tid == 0) a.out_count[bh] = total;
    const size_t lb = (size_t)bh * d.outlier_cap;
    const uint64_t before = (1ull << ln) - 1ull;  // the lanes ahead of this one
    for (int s4 = s0; s4 < s1 && off < d.outlier_cap; s4 += 4) {
      float xr[4][NC];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int c = 0; c < NC; ++c) xr[u][c] = X(min(s4 + u, s1 - 1), c * 64 + ln);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = s4 + u;
        if (s >= s1) break;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int j = c * 64 + ln;
          const float xv = xr[u][c];
          const bool hit = all || fabsf(xv) >= th[c];
          const uint64_t m = __ballot(hit);
          const int at = off + __popcll(m & before);
          if (hit && at < d.outlier_cap) {
            a.out_pos[lb + at] = (uint32_t)s * D + (uint32_t)j;
            a.out_val[lb + at] = f2h(xv);  // fp16, round to nearest even
          }
          off += __popcll(m);
        }
      }
    }
  } else if (tid == 0) {
    a.out_count[bh] = 0;
  }
}

struct ValueBlockArgs {
  tqk_block_desc d;
  const void* x;
  const float* pi;
  const float* vbnd;
  uint8_t* packed;
  float* norms;
};

// 64 tokens of one (b, h) per workgroup.  Four threads per token compute the
// norm in the reference's pairwise order and stage the scaled row as fp16
// pairs; then every wave estimates the codes of its channels on the matrix
// cores, the flagged ones are recomputed, and the bit streams written.
template <int VB, int D>
__global__ __launch_bounds__(kVbThreads) void tqk_value_block(ValueBlockArgs a) {
  constexpr int VROW = D * VB / 8, NT = D / 16 > kVbThreads / 64 ? 2 : 1;
  const tqk_block_desc& d = a.d;
  const int S = d.tokens, bh = blockIdx.y, t0 = blockIdx.x * kVbTokens, tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const int nb = min(kVbTokens, S - t0);
  const size_t tok0 = (size_t)bh * S + t0;  // flat token index of the first token
  __shared__ __align__(16) uint16_t uv_s[kVbTokens][2 * D + 8];
  __shared__ __align__(16) PolarStage<D, kVbTokens> st;

  if (tid == 0) st.nlist = 0;
  {
    const int tt = tid >> 2, q = tid & 3;
    if (tt < nb) {
      const size_t row = (tok0 + tt) * D;
      float x0[D / 8], x1[D / 8];
      uint32_t any = 0;
#pragma unroll
      for (int m = 0; m < D / 8; ++m) {  // channels 8m + 2q, 8m + 2q + 1
        x0[m] = load_x(a.x, d.input_f32, row + 8 * m + 2 * q);
        x1[m] = load_x(a.x, d.input_f32, row + 8 * m + 2 * q + 1);
        any |= __float_as_uint(x0[m]) | __float_as_uint(x1[m]);
      }
      any |= __shfl_xor(any, 1, 4);
      any |= __shfl_xor(any, 2, 4);
      const float ss = pairwise_sumsq<D>(x0, x1, q);
      const float nrm = __builtin_sqrtf(ss);  // correctly rounded (-fhip-fp32-correctly-rounded-divide-sqrt)
      const bool zero = (any & 0x7FFFFFFFu) == 0u;
      polar_stage_row<D>(&uv_s[tt][0], x0, x1, q, zero ? 0.f : kPiScale * __builtin_amdgcn_rcpf(nrm));
      if (q == 0) {
        polar_token(st, tt, ss, nrm, zero, 1.0f / (kPiScale * kPiScale));
        a.norms[tok0 + tt] = nrm;
      }
    }
  }
  float bnd[15];
#pragma unroll
  for (int k = 0; k < 15; ++k) bnd[k] = k < (1 << VB) - 1 ? a.vbnd[k] : 0.f;
  __syncthreads();
  const int e0 = 16 * NT * wv;
  if (e0 < D) {
    PiFrags<D, NT> pf;
    load_pi(pf, a.pi, e0, lane, bnd, (1 << VB) - 1);
    polar_codes<D, NT, VB, true, false>(st, pf, &uv_s[0][0], 2 * D + 8, nb, e0, lane, bnd);
  }
  __syncthreads();
  if (st.nlist > 0) {
    polar_fix<D, VB, false, kVbThreads>(st, a.pi, nb, tid, bnd, [&](int t, int dd) {
      const size_t i = (tok0 + t) * D + dd;
      return make_float4(load_x(a.x, d.input_f32, i), load_x(a.x, d.input_f32, i + 1),
                         load_x(a.x, d.input_f32, i + 2), load_x(a.x, d.input_f32, i + 3));
    });
    __syncthreads();
  }
  for (int f8 = tid; f8 < nb * (D / 32); f8 += kVbThreads) {
    uint32_t w[VB];
    pack_fields<VB>(st, f8, w);
    uint32_t* dst = reinterpret_cast<uint32_t*>(a.packed + (tok0 + f8 / (D / 32)) * VROW) + VB * (f8 % (D / 32));
#pragma unroll
    for (int k = 0; k < VB; ++k) dst[k] = w[k];
  }
}

struct KeyDequantArgs {
  tqk_block_desc d;
  const uint8_t* packed;
  const float* scale;
  const float* zero;
  float* out;
};

// one thread per code byte (two channels): zero + scale * level[code]; 3- and
// 2-bit keys one thread per code
__global__ __launch_bounds__(kKbThreads) void tqk_key_block_dequant(KeyDequantArgs a) {
  const tqk_block_desc& d = a.d;
  const int D = d.head_dim;
  if (d.bits != 4) {
    const size_t n = (size_t)d.batch * d.n_heads * d.tokens * D;
    const size_t i = (size_t)blockIdx.x * kKbThreads + threadIdx.x;
    if (i >= n) return;
    const size_t bh = i / ((size_t)d.tokens * D);
    const int j = (int)(i % D);
    const uint32_t c = get_code_ref(a.packed, i, d.bits, (n * d.bits + 7) / 8);
    a.out[i] = __fadd_rn(__fmul_rn(a.scale[bh * D + j], (float)c), a.zero[bh * D + j]);
    return;
  }
  const size_t n = (size_t)d.batch * d.n_heads * d.tokens * (D / 2);
  const size_t i = (size_t)blockIdx.x * kKbThreads + threadIdx.x;
  if (i >= n) return;
  const size_t bh = i / ((size_t)d.tokens * (D / 2));
  const int j0 = 2 * (int)(i % (D / 2));
  const uint32_t byte = a.packed[i];
  const float* sc = a.scale + bh * D;
  const float* zr = a.zero + bh * D;
  a.out[2 * i] = __fadd_rn(__fmul_rn(sc[j0], key_level(d.key_grid, rev4(byte >> 4))), zr[j0]);
  a.out[2 * i + 1] = __fadd_rn(__fmul_rn(sc[j0 + 1], key_level(d.key_grid, rev4(byte & 15u))), zr[j0 + 1]);
}

// the side-list overwrite (after the dense pass on the same stream); an index
// outside [0, total) is skipped here and reported by the host-side check
__global__ __launch_bounds__(kKbThreads) void tqk_key_block_outliers(float* out, int n,
                                                                   int64_t total,
                                                                   const int32_t* idx,
                                                                   const uint16_t* val) {
  const int i = blockIdx.x * kKbThreads + threadIdx.x;
  if (i < n) {
    const int64_t p = idx[i];
    if (p >= 0 && p < total) out[p] = h2f(val[i]);
  }
}

struct ValueDequantArgs {
  tqk_block_desc d;
  const uint8_t* packed;
  const float* norms;
  const float* pi;
  const float* vcent;
  float* out;
};

// 64 tokens per workgroup: y = vcent[code] staged in LDS (a thread takes 32 codes),
// x_e = sequential over j of y_j * Pi[j][e] (rotate_rows), times the norm
template <int VB, int D>
__global__ __launch_bounds__(kKbThreads, 2) void tqk_value_block_dequant(ValueDequantArgs a) {
  constexpr int VROW = D * VB / 8;
  const tqk_block_desc& d = a.d;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const size_t n = (size_t)d.batch * d.n_heads * d.tokens, tok0 = (size_t)blockIdx.x * kVbTokens;
  const int nb = (int)(n - tok0 < (size_t)kVbTokens ? n - tok0 : (size_t)kVbTokens);
  __shared__ __align__(16) float y_s[kVbTokens][D];
  __shared__ float nrm_s[kVbTokens];
  __shared__ float cent_s[16];
  if (tid < nb) nrm_s[tid] = a.norms[tok0 + tid];
  if (tid >= 64 && tid < 64 + (1 << VB)) cent_s[tid - 64] = a.vcent[tid - 64];
  __syncthreads();
  for (int i = tid; i < nb * (D / 32); i += kKbThreads) {
    const int t = i / (D / 32), c32 = i % (D / 32);
    const uint8_t* src = a.packed + (tok0 + t) * VROW + 4 * VB * c32;
    uint32_t w[VB];
    __builtin_memcpy(w, src, sizeof(w));  // (a row may start at any byte)
#pragma unroll
    for (int k = 0; k < 32; k += 4)
      *reinterpret_cast<float4*>(&y_s[t][32 * c32 + k]) =
          make_float4(cent_s[stream_code<VB>(w, k)], cent_s[stream_code<VB>(w, k + 1)],
                      cent_s[stream_code<VB>(w, k + 2)], cent_s[stream_code<VB>(w, k + 3)]);
  }
  __syncthreads();
  for (int e0 = 16 * wv; e0 < D; e0 += 16 * (kKbThreads / 64)) {
    const int e = e0 + (lane & 15);
    rotate_rows<D>(a.pi, y_s, nb, e, lane, [&](int t, float x) {
      a.out[(tok0 + t) * D + e] = __fmul_rn(x, nrm_s[t]);
    });
  }
}

int check_block(const tqk_block_desc* d, bool key) {
  if (!d) return TQK_EINVAL;
  if (!head_dim_ok(d->head_dim)) return TQK_EUNSUPPORTED;
  if (d->batch <= 0 || d->n_heads <= 0 || d->tokens <= 0) return TQK_EINVAL;
  if ((long long)d->batch * d->n_heads * d->tokens * d->head_dim >= (1LL << 40)) return TQK_EINVAL;
  if (key) {
    if (d->bits < 2 || d->bits > 4) return TQK_EUNSUPPORTED;
    if (d->key_grid != 0 && d->key_grid != 1) return TQK_EINVAL;
    if (d->bits != 4 && d->key_grid != 1) return TQK_EUNSUPPORTED;  // NF4 is 4-bit
    if (d->zero_point < 0 || d->zero_point > 2 || (d->zero_point != 0 && d->key_grid != 0))
      return TQK_EINVAL;
    if (d->outliers_per_channel < 0 || d->outlier_cap < 0) return TQK_EINVAL;
    // side-list positions s * D + j are 32-bit
    if ((long long)d->tokens * d->head_dim >= (1LL << 32)) return TQK_EUNSUPPORTED;
  } else if (d->bits < 2 || d->bits > 4) {
    return TQK_EUNSUPPORTED;
  }
  return TQK_OK;
}

// Key blocks go over the chip where the packed output has room for KbScratch
// (with no outliers nothing is handed on): 1 x 8 x 33 x 128 fp32 at 2 bits takes
// 27 us, at 4 bits 29; 16 tokens at 2 bits, in one workgroup per (b, h), 40.
// A launch takes fewer than 2^32 threads: as many (b, h) at a time as that allows
// (131072 at head_dim 256).
template <int D, bool F32>
void launch_key_chip(hipStream_t st, KeyBlockArgs a) {
  const int n_bh = a.d.batch * a.d.n_heads;
  const int most = min((1 << 21) / (D / 16), max(1, (1 << 23) / a.n_chunks));
  for (; a.bh0 < n_bh; a.bh0 += most) {
    const unsigned bh = (unsigned)min(most, n_bh - a.bh0), n = bh * (unsigned)a.n_chunks;
    hipLaunchKernelGGL((tqk_key_block_stats<D, F32>), dim3(bh * (D / 16)), dim3(kKbStatThreads), 0, st, a);
    if (a.d.outliers_per_channel > 0) {
      if (a.d.outliers_per_channel < a.d.tokens)
        hipLaunchKernelGGL((tqk_key_block_masks<D, F32>), dim3(n), dim3(kKbChunk), 0, st, a);
      hipLaunchKernelGGL((tqk_key_block_list<D, F32>), dim3(n), dim3(kKbChunk), 0, st, a);
    }
    hipLaunchKernelGGL((tqk_key_block_codes<D, F32>), dim3(n), dim3(kKbChunk), 0, st, a);
  }
}
template <int D>
void launch_key(hipStream_t st, const KeyBlockArgs& a) {
  const long long words = (long long)a.d.tokens * D * a.d.bits / 32;
  const long long pad = (reinterpret_cast<uintptr_t>(a.packed) & 3u) ? 1 : 0;  // to the first dword boundary
  const long long need = pad + D + a.n_chunks + (long long)a.d.tokens * (D / 32);
  const bool chip = a.d.outliers_per_channel == 0 || need <= words;
  if (!chip)
    hipLaunchKernelGGL(tqk_key_block<D>, dim3(a.d.batch * a.d.n_heads), dim3(2 * D), 0, st, a);
  else if (a.d.input_f32)
    launch_key_chip<D, true>(st, a);
  else
    launch_key_chip<D, false>(st, a);
}

// one kernel instance per (bits, head_dim)
template <int D>
void launch_value(int vb, dim3 grid, hipStream_t st, const ValueBlockArgs& a) {
  if (vb == 2)
    hipLaunchKernelGGL((tqk_value_block<2, D>), grid, dim3(kVbThreads), 0, st, a);
  else if (vb == 3)
    hipLaunchKernelGGL((tqk_value_block<3, D>), grid, dim3(kVbThreads), 0, st, a);
  else
    hipLaunchKernelGGL((tqk_value_block<4, D>), grid, dim3(kVbThreads), 0, st, a);
}
template <int D>
void launch_value(int vb, dim3 grid, hipStream_t st, const ValueDequantArgs& a) {
  if (vb == 2)
    hipLaunchKernelGGL((tqk_value_block_dequant<2, D>), grid, dim3(kKbThreads), 0, st, a);
  else if (vb == 3)
    hipLaunchKernelGGL((tqk_value_block_dequant<3, D>), grid, dim3(kKbThreads), 0, st, a);
  else
    hipLaunchKernelGGL((tqk_value_block_dequant<4, D>), grid, dim3(kKbThreads), 0, st, a);
}

}  // namespace

extern "C" {

int tqk_encode_key_block(const tqk_block_desc* d, const void* x, const float* zp, uint8_t* packed,
                         float* scale, float* zero, uint32_t* out_pos, uint16_t* out_val,
                         int32_t* out_count, void* stream) {
  int rc = check_block(d, true);
  if (rc != TQK_OK) return rc;
  if (!x || !packed || !scale || !zero || !out_count) return TQK_EINVAL;
  if (d->key_grid == 0 && d->zero_point == 2 && !zp) return TQK_EINVAL;
  if (d->outliers_per_channel > 0 && d->outlier_cap > 0 && (!out_pos || !out_val)) return TQK_EINVAL;
  const int n_chunks = (d->tokens + kKbChunk - 1) / kKbChunk;
  KeyBlockArgs a{*d, x, zp, packed, scale, zero, out_pos, out_val, out_count, n_chunks, 0};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (d->head_dim == 64)
    launch_key<64>(st, a);
  else if (d->head_dim == 128)
    launch_key<128>(st, a);
  else
    launch_key<256>(st, a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

int tqk_encode_value_block(const tqk_block_desc* d, const void* x, const float* pi,
                           const float* vbnd, uint8_t* packed, float* norms, void* stream) {
  int rc = check_block(d, false);
  if (rc != TQK_OK) return rc;
  if (!x || !pi || !vbnd || !packed || !norms) return TQK_EINVAL;
  ValueBlockArgs a{*d, x, pi, vbnd, packed, norms};
  const dim3 grid((d->tokens + kVbTokens - 1) / kVbTokens, d->batch * d->n_heads);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (d->head_dim == 64)
    launch_value<64>(d->bits, grid, st, a);
  else if (d->head_dim == 128)
    launch_value<128>(d->bits, grid, st, a);
  else
    launch_value<256>(d->bits, grid, st, a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

int tqk_dequant_key_block(const tqk_block_desc* d, const uint8_t* packed, const float* scale,
                          const float* zero, int32_t n_out, const int32_t* out_idx,
                          const uint16_t* out_val, float* out, void* stream) {
  int rc = check_block(d, true);
  if (rc != TQK_OK) return rc;
  if (!packed || !scale || !zero || !out || n_out < 0 || (n_out > 0 && (!out_idx || !out_val)))
    return TQK_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const size_t total = (size_t)d->batch * d->n_heads * d->tokens * d->head_dim;
  const size_t n = d->bits == 4 ? total / 2 : total;  // threads: code bytes, or codes
  KeyDequantArgs a{*d, packed, scale, zero, out};
  hipLaunchKernelGGL(tqk_key_block_dequant, dim3((unsigned)((n + kKbThreads - 1) / kKbThreads)),
                     dim3(kKbThreads), 0, st, a);
  if (n_out > 0)
    hipLaunchKernelGGL(tqk_key_block_outliers, dim3((n_out + kKbThreads - 1) / kKbThreads),
                       dim3(kKbThreads), 0, st, out, n_out, (int64_t)total, out_idx, out_val);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

int tqk_dequant_value_block(const tqk_block_desc* d, const uint8_t* packed, const float* norms,
                            const float* pi, const float* vcent, float* out, void* stream) {
  int rc = check_block(d, false);
  if (rc != TQK_OK) return rc;
  if (!packed || !norms || !pi || !vcent || !out) return TQK_EINVAL;
  const size_t n = (size_t)d->batch * d->n_heads * d->tokens;
  ValueDequantArgs a{*d, packed, norms, pi, vcent, out};
  const dim3 grid((unsigned)((n + kVbTokens - 1) / kVbTokens));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (d->head_dim == 64)
    launch_value<64>(d->bits, grid, st, a);
  else if (d->head_dim == 128)
    launch_value<128>(d->bits, grid, st, a);
  else
    launch_value<256>(d->bits, grid, st, a);
  return hipGetLastError() == hipSuccess ? TQK_OK : TQK_EHIP;
}

}  // extern "C"
