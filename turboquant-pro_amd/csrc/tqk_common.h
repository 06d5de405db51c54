// Shared device helpers and tables for the gfx950 TurboQuant KV kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tqk.h"

#define TQK_D 128          // head_dim of the MFMA decode (other head dims run the VALU decode)
#define TQK_MAX_G 256      // largest group (flush) size
#define TQK_OBLK 32        // outlier side-list bound granularity (tokens)
#define TQK_NOB 8          // cumulative outlier counts kept per (group slot, head)
// Largest value norm the decode's fp16 PV weights carry: the online softmax
// keeps every weight p <= 4, and p * norm must stay below fp16's 65504.
#define TQK_MAX_VNORM 16376.0f
// Bits of tqk_encode_groups' overflow word
#define TQK_OVF_OUTLIERS 1  // a (group, head) side-list exceeded outlier_cap
#define TQK_OVF_VNORM 2     // a value norm exceeded TQK_MAX_VNORM

// head dims the kernels are built for
__host__ __device__ __forceinline__ bool head_dim_ok(int D) { return D == 64 || D == 128 || D == 256; }

// Value codes use the MFMA-tiled byte order when the MFMA decode serves the
// cache (head_dim 128, fp16 inputs), every 16-token tile lies in one page and
// groups are whole 32-token blocks; otherwise per-token rows.
__host__ __device__ __forceinline__ bool v_tiled(int G, int P, int D, int f32) {
  return D == TQK_D && !f32 && (P % 16 == 0) && (G % 32 == 0);
}

// Byte offset of the value-code unit holding tokens [4*lg, 4*lg+4) of a
// 16-token tile and channels [8*c, 8*c+8), relative to the tile start.
// A unit is vrow/4 bytes (12 for 3-bit, 16 for 4-bit codes).
__host__ __device__ __forceinline__ int v_unit_offset(int lg, int c, int vrow) {
  return (16 * lg + c) * (vrow / 4);
}
// Bit position, inside a unit, of the code of token u (0..3 within the unit)
// and channel nt (0..7 within the unit): codes of the token pairs (0,1) and
// (2,3) of one channel sit next to each other as one 2*vb-bit field.
__host__ __device__ __forceinline__ int v_unit_bit(int u, int nt, int vb) {
  return (2 * nt + (u >> 1)) * (2 * vb) + (u & 1) * vb;
}

// NormalFloat-4 levels, turboquant_pro/per_channel_kv.py:64-84.
// Key level of code c: NF4 for key_grid 0, the code itself for uniform keys
__device__ __forceinline__ float key_level(int grid, uint32_t c);
__constant__ static const float kNF4[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.44070982933044434f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f};
__device__ __forceinline__ float key_level(int grid, uint32_t c) {
  return grid ? (float)c : kNF4[c];
}

__device__ __forceinline__ float h2f(uint16_t x) {
  return (float)__builtin_bit_cast(_Float16, x);
}
__device__ __forceinline__ uint16_t f2h(float x) {  // round to nearest even
  return __builtin_bit_cast(uint16_t, (_Float16)x);
}

// 4-bit nibble bit reversal: the key stream stores each code LSB-first inside
// MSB-first bytes (turboquant_pro/per_channel_kv.py:87-93), so byte n holds
// rev4(code[2n]) << 4 | rev4(code[2n+1]).
__host__ __device__ __forceinline__ uint32_t rev4(uint32_t x) {
  return ((x & 1u) << 3) | ((x & 2u) << 1) | ((x & 4u) >> 1) | ((x & 8u) >> 3);
}

// Key code rows: k_row_bytes(kb, D) bytes per token.  4-bit keys are the
// reference's byte stream (byte n = rev4(code[2n]) << 4 | rev4(code[2n+1])).
// 3- and 2-bit keys (uniform grid) are D / 32 chunks of 32 channels, 4 * kb
// bytes each; in chunk c the little-endian field i (2*kb bits at bit 2*kb*i)
// is code(32c + 2i) | code(32c + 2i + 1) << kb.  Either way a channel pair has
// one table index: the byte, or the field.
__host__ __device__ __forceinline__ int k_row_bytes(int kb, int D) { return D * kb / 8; }
// table index of channel pair `pair` (channels 2*pair, 2*pair + 1) of a row
// given as little-endian dwords
__device__ __forceinline__ uint32_t k_pair_index(const uint32_t* rw, int kb, int pair) {
  if (kb == 4) return (rw[pair >> 2] >> (8 * (pair & 3))) & 0xFFu;
  const int o = (pair >> 4) * (32 * kb) + 2 * kb * (pair & 15);  // bit offset in the row (32 channels a chunk)
  const int w = o >> 5, sh = o & 31;
  uint32_t v = rw[w] >> sh;
  if (sh + 2 * kb > 32) v |= rw[w + 1] << (32 - sh);
  return v & ((1u << (2 * kb)) - 1u);
}
// the two codes of a table index
__host__ __device__ __forceinline__ uint32_t k_code_even(uint32_t f, int kb) {
  return kb == 4 ? rev4(f >> 4) : (f & ((1u << kb) - 1u));
}
__host__ __device__ __forceinline__ uint32_t k_code_odd(uint32_t f, int kb) {
  return kb == 4 ? rev4(f & 15u) : (f >> kb);
}

// Number of flushed groups after `len` appends: the first flush fires at
// hot_window + 1 tokens, then every G tokens (turboquant_pro/core.py:1006-1016).
__host__ __device__ __forceinline__ int n_groups_of(int len, int hot_window, int G) {
  return (len <= hot_window) ? 0 : (len - (hot_window + 1)) / G + 1;
}

// Row index of token t (absolute position in its sequence) for kv head h in
// the page pool.
__device__ __forceinline__ size_t page_row(const int32_t* __restrict__ block_table, int max_pages,
                                           int b, int t, int P, int n_pages, int h) {
  // head-major pages: row of token t of sequence b in head h's region
  const int phys = block_table[(size_t)b * max_pages + t / P];
  return ((size_t)h * n_pages + phys) * P + (t % P);
}

// Lane I of each 16-lane row, broadcast to the row (DPP row_newbcast).
template <int I>
__device__ __forceinline__ float dpp_row_bcast(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + I, 0xF, 0xF, true));
}
// y += the eight values of lane K of the 16-lane row, in order, then those of
// the lanes after it up to NL - 1 (plain operators, so that the broadcast
// folds into the addition; every lane of the row gets the sum)
template <int K, int NL>
__device__ __forceinline__ void add_row_dpp(float& y, const float (&f)[8]) {
#pragma unroll
  for (int r = 0; r < 8; ++r) y = y + dpp_row_bcast<K>(f[r]);
  if constexpr (K + 1 < NL) add_row_dpp<K + 1, NL>(y, f);
}

// y0 += u_a[d] * col[d], y1 += u_b[d] * col[d] for d = 8K .. 8K + 7 and on to d =
// 8 NL - 1, each product and sum separately rounded, in d order; u_a[d] lives in
// register d % 8 of lane d / 8 of the 16-lane row.  Plain operators, so that the
// broadcast folds into the multiply as its DPP operand: only for units built
// with -ffp-contract=off.
template <int K, int NL, int N>
__device__ __forceinline__ void rotate_row_dpp(float& y0, float& y1, const float (&ua)[8], const float (&ub)[8],
                                               const float (&col)[N]) {
  static_assert(NL <= 16 && 8 * NL <= N, "a chunk spans at most one 16-lane row");
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float p0 = dpp_row_bcast<K>(ua[r]) * col[8 * K + r];
    const float p1 = dpp_row_bcast<K>(ub[r]) * col[8 * K + r];
    y0 = y0 + p0;
    y1 = y1 + p1;
  }
  if constexpr (K + 1 < NL) rotate_row_dpp<K + 1, NL>(y0, y1, ua, ub, col);
}

// PolarQuant reconstruction before the norm: x_e = sum over j, in order, of
// y_j * pi[j][e], every product and sum separately rounded (turboquant_pro/
// core.py:619-654), of nb <= 64 rows in LDS for the channel e of this lane;
// store(token, x_e) takes the results.  Bound by its 2 D VALU operations a
// value: a lane keeps column e of pi, a 16-lane row takes one token of a step
// and broadcasts its values by DPP.  Rows longer than 128 channels go in
// 128-channel chunks, every step's sums carried on.  All 64 lanes run it.
template <int D, typename Store>
__device__ __forceinline__ void rotate_rows(const float* __restrict__ pi, const float (*y_s)[D], int nb, int e,
                                            int lane, Store store) {
  constexpr int CH = D < 128 ? D : 128;
  const int rt = lane >> 4, lc = (lane & 15) % (CH / 8);
  auto load_y = [&](int t, int c, float (&u)[8]) {
    const float4* r = reinterpret_cast<const float4*>(&y_s[min(t, nb - 1)][CH * c + 8 * lc]);
    const float4 a = r[0], b = r[1];
    u[0] = a.x; u[1] = a.y; u[2] = a.z; u[3] = a.w;
    u[4] = b.x; u[5] = b.y; u[6] = b.z; u[7] = b.w;
  };
  auto load_col = [&](int c, float (&col)[CH]) {
#pragma unroll
    for (int k = 0; k < CH; ++k) col[k] = pi[(size_t)(CH * c + k) * D + e];
  };
  if constexpr (D <= 128) {
    float col[CH];
    load_col(0, col);
    for (int j0 = 0; j0 < nb; j0 += 8) {
      float ua[8], ub[8];
      load_y(j0 + rt, 0, ua);
      load_y(j0 + 4 + rt, 0, ub);
      float y0 = 0.f, y1 = 0.f;
      rotate_row_dpp<0, CH / 8>(y0, y1, ua, ub, col);
      // keeps the sums out of the conditional stores: sunk into them, the
      // multiplies would leave their broadcasts behind as separate moves
      asm volatile("" : "+v"(y0), "+v"(y1));
      if (j0 + rt < nb) store(j0 + rt, y0);
      if (j0 + 4 + rt < nb) store(j0 + 4 + rt, y1);
    }
  } else {
    float ya[8], yb[8];
#pragma unroll
    for (int st = 0; st < 8; ++st) ya[st] = yb[st] = 0.f;
    for (int c = 0; c < D / CH; ++c) {
      float col[CH];
      load_col(c, col);
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        if (8 * st < nb) {
          float ua[8], ub[8];
          load_y(8 * st + rt, c, ua);
          load_y(8 * st + 4 + rt, c, ub);
          rotate_row_dpp<0, CH / 8>(ya[st], yb[st], ua, ub, col);
          asm volatile("" : "+v"(ya[st]), "+v"(yb[st]));
        }
      }
    }
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      if (8 * st + rt < nb) store(8 * st + rt, ya[st]);
      if (8 * st + 4 + rt < nb) store(8 * st + 4 + rt, yb[st]);
    }
  }
}

// code i of VB dwords holding a 32-code bit stream
template <int VB>
__device__ __forceinline__ uint32_t stream_code(const uint32_t (&w)[VB], int i) {
  const int bit = VB * i;
  uint32_t c = w[bit >> 5] >> (bit & 31);
  if ((bit & 31) + VB > 32) c |= w[(bit >> 5) + 1] << (32 - (bit & 31));
  return c & ((1u << VB) - 1u);
}

// ---------------------------------------------------------------------------
// PolarQuant codes.  The code of a rotated channel is #{ boundaries < y_e } for
// the reference's y_e: the sum over d, in order, of u_d * pi[e][d], every
// product and sum separately rounded (a NaN y_e takes the last code, as
// searchsorted does).  Only the code is stored, so y_e itself is needed only
// where it lies close to a boundary: the matrix cores give an estimate whose
// error has a bound, every estimate further than the bound from all boundaries
// has the reference's code, and the others (about 1 in 780 at 3
// bits and head_dim 128) are listed and recomputed in the reference's order.
// (Evaluating the ordered sum everywhere took 256 VALU instructions per channel
// and bounded the whole encode: 16 sequences x 8192 tokens x 8 heads appended
// in 1584 us, with the estimate, about 20 instructions, in 868 us.)
//
// The estimate: x (fp16 as it is, or the fp32 row scaled to |u| <= 256 and
// split into an fp16 pair) times 256 * pi split into an fp16 pair, summed in
// fp32 by MFMA, all products of low halves before those of high ones (among
// them each of those MFMAs would truncate at full scale too: twice the bound
// for fp16 rows and three times for fp32 ones), scaled back by 1 / norm.  Against the real sum sum_d u_d pi[e][d], with |u| <= 1 and N =
// |pi[e]| in [2^-8, 50]:
//   the ordered sum errs by at most D 2^-24 N            (D roundings)
//   the MFMA sums by at most (D / 32) 33 2^-23 N         (every one of a step's
//                            32 products and its sum truncated at full scale)
//   the low halves' sum before, at most 2^-10 N, by twice as much of that
//   the dropped low x low products and the pairs' own rounding 3 2^-22 N, the
//   scaling by 1 / norm and u's own rounding 2^-22 N, low halves of pi below
//   fp16's normal range sqrt(D) 2^-33
// together below 0.86 D 2^-22 N for D = 64, 128 and 256.
// ---------------------------------------------------------------------------
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr float kPiScale = 256.0f;  // fp16 pairs of pi (and of u): far from fp16's subnormals
constexpr float kEstimateBound = 0.9f;  // on an estimate's distance from the ordered sum, in D 2^-22 N

// The 16 * NT rows of pi from e0 on as MFMA operands (lane: row e0 + 16 nt +
// lane % 16, channels 32 ks + 8 (lane / 16) .. + 7), and the bound on an
// estimate's distance from the ordered sum: infinite (every code recomputed)
// for rows that are not finite, longer than 50 or shorter than 2^-8 (the fp16
// pairs of a short row's channels are subnormal: they err by 2^-33 a channel,
// sqrt(D) 2^-33 in all, however short the row is, while the bound shrinks with
// it), and for boundaries that do not ascend (the code's search needs them to).
template <int D, int NT>
struct PiFrags {
  h8_t hi[D / 32][NT], lo[D / 32][NT];
  float delta;
};
template <int D, int NT, int NB>
__device__ __forceinline__ void load_pi(PiFrags<D, NT>& f, const float* __restrict__ pi, int e0, int lane,
                                        const float (&bnd)[NB], int nbnd) {
  float most = 0.f;
  bool bad = false;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float* row = pi + (size_t)(e0 + 16 * nt + (lane & 15)) * D + 8 * (lane >> 4);
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      const float4 a = *reinterpret_cast<const float4*>(row + 32 * ks);
      const float4 b = *reinterpret_cast<const float4*>(row + 32 * ks + 4);
      const float p[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float s = p[i] * kPiScale;
        const _Float16 h = (_Float16)s;
        f.hi[ks][nt][i] = h;
        f.lo[ks][nt][i] = (_Float16)(s - (float)h);
        ss += p[i] * p[i];
      }
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    bad |= !(ss >= 0x1p-16f && ss <= 2500.0f);
    most = fmaxf(most, ss);
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) most = fmaxf(most, __shfl_xor(most, o, 64));
  for (int k = 1; k < nbnd; ++k) bad |= !(bnd[k - 1] < bnd[k]);
  f.delta = __any(bad) ? __builtin_inff() : kEstimateBound * (float)D * 0x1p-22f * __builtin_sqrtf(most);
}

// #{ b < y } by binary search, and the distance m to the nearest boundary:
// both neighbours of the final interval are on the search's path
template <int VB>
__device__ __forceinline__ uint32_t code_margin(float y, const float (&b)[15], float& m) {
  if constexpr (VB == 2) {
    const bool c1 = b[1] < y;
    const float q = c1 ? b[2] : b[0];
    m = fminf(fabsf(y - b[1]), fabsf(y - q));
    return (c1 ? 2u : 0u) + (q < y ? 1u : 0u);
  } else if constexpr (VB == 3) {
    const bool c1 = b[3] < y;
    const float p = c1 ? b[5] : b[1], r0 = c1 ? b[4] : b[0], r1 = c1 ? b[6] : b[2];
    const bool c2 = p < y;
    const float r = c2 ? r1 : r0;
    m = fminf(fminf(fabsf(y - b[3]), fabsf(y - p)), fabsf(y - r));
    return (c1 ? 4u : 0u) + (c2 ? 2u : 0u) + (r < y ? 1u : 0u);
  } else {
    const bool c1 = b[7] < y;
    float t[7];
#pragma unroll
    for (int i = 0; i < 7; ++i) t[i] = c1 ? b[8 + i] : b[i];
    const bool c2 = t[3] < y;
    const float p = c2 ? t[5] : t[1], r0 = c2 ? t[4] : t[0], r1 = c2 ? t[6] : t[2];
    const bool c3 = p < y;
    const float r = c3 ? r1 : r0;
    m = fminf(fminf(fabsf(y - b[7]), fabsf(y - t[3])), fminf(fabsf(y - p), fabsf(y - r)));
    return (c1 ? 8u : 0u) + (c2 ? 4u : 0u) + (c3 ? 2u : 0u) + (r < y ? 1u : 0u);
  }
}
template <int VB>
__device__ __forceinline__ uint32_t code_exact(float y, const float (&b)[15]) {
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < (1 << VB) - 1; ++k) c += (b[k] < y) ? 1u : 0u;
  return y != y ? (1u << VB) - 1u : c;
}

// A batch's staging in LDS.  Codes sit in 16-bit fields of four codes: four
// tokens of one channel (TROWS, the MFMA-tiled value order: field (t / 4) * D +
// e) or four channels of one token (field t * (D / 4) + e / 4), in either case
// the order in which eight consecutive fields' bits make up VB whole dwords of
// the stored row.
template <int D, int NTOK>
struct PolarStage {
  uint16_t fld[NTOK * D / 4];
  float2 tk[NTOK];   // (estimate scale, factor of the bound)
  float nrm[NTOK];
  uint16_t list[1024];  // flagged codes, t * D + e
  int nlist;
};

// The token's entry of the stage from its sum of squares.  Zero rows need no
// bound (their y is exactly 0, as the estimate); rows whose sum of squares is
// not finite or so small that u may be longer than 1 get a NaN scale, which
// flags every code of theirs.
template <int D, int NTOK>
__device__ __forceinline__ void polar_token(PolarStage<D, NTOK>& st, int t, float ss, float nrm, bool zero,
                                            float scale) {
  st.nrm[t] = nrm;
  const bool plain = ss >= 0x1p-60f && ss <= 0x1p100f;
  st.tk[t] = zero ? make_float2(0.f, -1.f)
                  : make_float2(plain ? scale : __builtin_nanf(""), 1.f);
}

// Estimated codes of the stage's nb tokens for the wave's 16 * NT channels from
// e0 on; xs: the tokens' rows, fp16 (hi, and at column D the low halves when
// LO), `stride` halves apart.  All 64 lanes run it.
template <int D, int NT, int VB, bool LO, bool TROWS, int NTOK>
__device__ __forceinline__ void polar_codes(PolarStage<D, NTOK>& st, const PiFrags<D, NT>& pf,
                                            const uint16_t* xs, int stride, int nb, int e0, int lane,
                                            const float (&bnd)[15]) {
  const int c16 = lane & 15, lg = lane >> 4;
  for (int t0 = 0; t0 < nb; t0 += 16) {
    const uint16_t* row = xs + (size_t)min(t0 + c16, nb - 1) * stride + 8 * lg;
    f4_t acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f4_t{0.f, 0.f, 0.f, 0.f};
    auto add = [&](const uint16_t* x, const h8_t (&p)[NT]) {
      const h8_t xv = *reinterpret_cast<const h8_t*>(x);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[nt] = TROWS ? __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, p[nt], acc[nt], 0, 0, 0)
                        : __builtin_amdgcn_mfma_f32_16x16x32_f16(p[nt], xv, acc[nt], 0, 0, 0);
    };
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      add(row + 32 * ks, pf.lo[ks]);
      if constexpr (LO) add(row + D + 32 * ks, pf.hi[ks]);
    }
    // (the rows are read again: at head_dim 128 no registers are left to hold them)
    if constexpr (D <= 128) asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) add(row + 32 * ks, pf.hi[ks]);
    // the lane's four results of a tile: tokens t0 + 4 lg + r of channel e0 +
    // 16 nt + c16 (TROWS), else channels e0 + 16 nt + 4 lg + r of token t0 + c16
    float2 tk[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) tk[r] = st.tk[min(TROWS ? t0 + 4 * lg + r : t0 + c16, nb - 1)];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      uint32_t f = 0;
      uint32_t near = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = acc[nt][r] * tk[r].x;
        float m;
        f |= code_margin<VB>(y, bnd, m) << (VB * r);
        near |= (m > tk[r].y * pf.delta) ? 0u : (1u << r);
      }
      const int t = TROWS ? t0 + 4 * lg : t0 + c16, e = e0 + 16 * nt + (TROWS ? c16 : 4 * lg);
      if (t < nb) st.fld[TROWS ? (t >> 2) * D + e : t * (D / 4) + (e >> 2)] = (uint16_t)f;
      while (near) {
        const int r = __builtin_ctz(near);
        near &= near - 1u;
        const int tt = TROWS ? t + r : t, ee = TROWS ? e : e + r;
        if (tt < nb) {
          const int at = atomicAdd(&st.nlist, 1);
          if (at < 1024) st.list[at] = (uint16_t)(tt * D + ee);
        }
      }
    }
  }
}

// code of (token t, channel e) in the stage (other codes of the word may
// change at the same time)
template <int D, int VB, bool TROWS, int NTOK>
__device__ __forceinline__ void set_code(PolarStage<D, NTOK>& st, int t, int e, uint32_t code) {
  const int idx = TROWS ? (t >> 2) * D + e : t * (D / 4) + (e >> 2);
  const int sh = 16 * (idx & 1) + VB * (TROWS ? t & 3 : e & 3);
  uint32_t* w = reinterpret_cast<uint32_t*>(st.fld) + (idx >> 1);
  const uint32_t old = (*reinterpret_cast<volatile uint32_t*>(w) >> sh) & ((1u << VB) - 1u);
  if (old != code) atomicXor(w, (old ^ code) << sh);
}

// The flagged codes in the reference's order; x4(t, d) gives channels d .. d + 3
// of token t as they came.  A list that overflowed (rows of NaN, infinities or
// vanishing norms, a rotation that puts whole channels on a boundary) has
// every code recomputed, a wave per token and a lane per channel.  All NTH
// threads run it, between barriers.
template <int D, int VB, bool TROWS, int NTH, int NTOK, typename X4>
__device__ __forceinline__ void polar_fix(PolarStage<D, NTOK>& st, const float* __restrict__ pi, int nb, int tid,
                                          const float (&bnd)[15], X4 x4) {
  const int n = st.nlist;
  if (n <= 1024) {
    // sixteen lanes per code: each holds eight products of a 128-channel chunk,
    // and all add them up in order, one lane's after another (DPP)
    constexpr int CH = D < 128 ? D : 128;
    const int li = tid & 15;
    for (int i0 = 0; i0 + 4 * (tid >> 6) < n; i0 += NTH / 16) {  // (waves without a code stop)
      const int i = i0 + (tid >> 4), at = st.list[min(i, n - 1)], t = at / D, e = at % D;
      const float safe = fmaxf(st.nrm[t], 1e-30f);
      float y = 0.f;
#pragma unroll
      for (int c = 0; c < D / CH; ++c) {
        const int d = CH * c + 8 * (li % (CH / 8));
        const float4 xa = x4(t, d), xb = x4(t, d + 4);
        const float4* pr = reinterpret_cast<const float4*>(pi + (size_t)e * D + d);
        const float4 pa = pr[0], pb = pr[1];
        const float f[8] = {__fmul_rn(__fdiv_rn(xa.x, safe), pa.x), __fmul_rn(__fdiv_rn(xa.y, safe), pa.y),
                            __fmul_rn(__fdiv_rn(xa.z, safe), pa.z), __fmul_rn(__fdiv_rn(xa.w, safe), pa.w),
                            __fmul_rn(__fdiv_rn(xb.x, safe), pb.x), __fmul_rn(__fdiv_rn(xb.y, safe), pb.y),
                            __fmul_rn(__fdiv_rn(xb.z, safe), pb.z), __fmul_rn(__fdiv_rn(xb.w, safe), pb.w)};
        add_row_dpp<0, CH / 8>(y, f);
      }
      // keeps the sum out of the conditional store: sunk into it, the additions
      // would leave their broadcasts behind as separate moves
      asm volatile("" : "+v"(y));
      if (i < n && li == 0)  // (a NaN norm makes u, and so y, NaN)
        set_code<D, VB, TROWS>(st, t, e, code_exact<VB>(st.nrm[t] != st.nrm[t] ? st.nrm[t] : y, bnd));
    }
    return;
  }
  const int lane = tid & 63;
  for (int t = tid >> 6; t < nb; t += NTH / 64) {
    const float safe = fmaxf(st.nrm[t], 1e-30f);
    float y[D / 64];
#pragma unroll
    for (int k = 0; k < D / 64; ++k) y[k] = st.nrm[t] != st.nrm[t] ? st.nrm[t] : 0.f;
#pragma unroll 1
    for (int d = st.nrm[t] != st.nrm[t] ? D : 0; d < D; d += 4) {
      const float4 x = x4(t, d);
      const float u[4] = {__fdiv_rn(x.x, safe), __fdiv_rn(x.y, safe), __fdiv_rn(x.z, safe), __fdiv_rn(x.w, safe)};
#pragma unroll
      for (int k = 0; k < D / 64; ++k) {
        const float4 p = *reinterpret_cast<const float4*>(pi + (size_t)(lane + 64 * k) * D + d);
        y[k] = __fadd_rn(y[k], __fmul_rn(u[0], p.x));
        y[k] = __fadd_rn(y[k], __fmul_rn(u[1], p.y));
        y[k] = __fadd_rn(y[k], __fmul_rn(u[2], p.z));
        y[k] = __fadd_rn(y[k], __fmul_rn(u[3], p.w));
      }
    }
#pragma unroll
    for (int k = 0; k < D / 64; ++k) set_code<D, VB, TROWS>(st, t, lane + 64 * k, code_exact<VB>(y[k], bnd));
  }
}

// Eight fields (field f8 * 8 on) as VB dwords of the stored bits.
template <int VB, int D, int NTOK>
__device__ __forceinline__ void pack_fields(const PolarStage<D, NTOK>& st, int f8, uint32_t (&w)[VB]) {
  const uint4 v = *reinterpret_cast<const uint4*>(&st.fld[8 * f8]);
  const uint32_t two[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < VB; ++k) w[k] = 0u;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t f = (i & 1) ? two[i >> 1] >> 16 : two[i >> 1] & 0xFFFFu;
    const int bit = 4 * VB * i;
    w[bit >> 5] |= f << (bit & 31);
    if ((bit & 31) + 4 * VB > 32) w[(bit >> 5) + 1] |= f >> (32 - (bit & 31));
  }
}

// Sum of squares of a D-channel row in NumPy's pairwise order (the L2 norm of
// np.linalg.norm over a contiguous row), four threads per row: thread q
// (= lane & 3, the four consecutive lanes of the row) holds x0[m], x1[m] =
// channels 8m + 2q, 8m + 2q + 1.  NumPy sums a run of n <= 128 values with
// eight strided accumulators r[k] (channels = k mod 8, in order) combined as
// ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7)); a longer run is split into
// halves (at a multiple of 8) summed apart and added, so D = 256 is the two
// 128-channel halves.  Every product and sum is separately rounded.
template <int D>
__device__ __forceinline__ float pairwise_sumsq(const float (&x0)[D / 8], const float (&x1)[D / 8],
                                                int q) {
  constexpr int M = D > 128 ? 16 : D / 8;  // 8-channel steps per pairwise block
  float ss = 0.f;
#pragma unroll
  for (int blk = 0; blk < D / 8 / M; ++blk) {
    float r0 = __fmul_rn(x0[M * blk], x0[M * blk]), r1 = __fmul_rn(x1[M * blk], x1[M * blk]);
#pragma unroll
    for (int m = 1; m < M; ++m) {
      r0 = __fadd_rn(r0, __fmul_rn(x0[M * blk + m], x0[M * blk + m]));
      r1 = __fadd_rn(r1, __fmul_rn(x1[M * blk + m], x1[M * blk + m]));
    }
    // pairwise tree ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7))
    const float pa = __fadd_rn(r0, r1);
    const float po = __shfl_xor(pa, 1, 4);
    const float pb = (q & 1) ? __fadd_rn(po, pa) : __fadd_rn(pa, po);
    const float pbo = __shfl_xor(pb, 2, 4);
    const float bs = (q & 2) ? __fadd_rn(pbo, pb) : __fadd_rn(pb, pbo);
    ss = blk == 0 ? bs : __fadd_rn(ss, bs);
  }
  return ss;
}

// The thread's channels (8m + 2q, 8m + 2q + 1) of a row times `scale`, as fp16
// pairs: high halves to row[0..D), low ones to row[D..2D).
template <int D>
__device__ __forceinline__ void polar_stage_row(uint16_t* row, const float (&x0)[D / 8], const float (&x1)[D / 8],
                                                int q, float scale) {
#pragma unroll
  for (int m = 0; m < D / 8; ++m) {
    const float s0 = x0[m] * scale, s1 = x1[m] * scale;
    const uint16_t h0 = f2h(s0), h1 = f2h(s1);
    const uint16_t l0 = f2h(s0 - h2f(h0)), l1 = f2h(s1 - h2f(h1));
    *reinterpret_cast<uint32_t*>(row + 8 * m + 2 * q) = (uint32_t)h0 | ((uint32_t)h1 << 16);
    *reinterpret_cast<uint32_t*>(row + D + 8 * m + 2 * q) = (uint32_t)l0 | ((uint32_t)l1 << 16);
  }
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
