// encode_rows.hpp -- the codec of a wave per one or several rows: the append
// above padded 128 (append.hip) and the decode step over the fp32 mirror, whose
// token it appends (mirror_step.hip).
#pragma once

#include "encode_one.hpp"

namespace aq {

// Codes, packs and stores the nr rows of a wide wave: the codes of all rows go
// to LDS (s_code, R * P bytes), then the lanes take the rows' words in order.
// Row r goes to slot (slot0 + r) % cap, and nowhere if r + age < 0 (the call
// itself evicts it).  nan_rows: bit r, row r takes the NaN code throughout.
// xmask: the K rows' XOR byte order (kperm_mask; 0: none).
template <int P, int R, int B>
__device__ __forceinline__ void store_wide_rows(const float (&v)[R][P / 64], uint32_t nan_rows,
                                                uint8_t *codes, int slot0, int cap, int nr,
                                                int age, int lane, uint32_t xmask,
                                                const Q4Cell *s_q4, uint8_t *s_code) {
  constexpr int NW = P * B / 32;  // words of a row
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool nan = (nan_rows >> r) & 1u;  // (a NaN is no index into the cell table)
#pragma unroll
    for (int e = 0; e < P / 64; ++e) {
      const uint32_t q = B == 4   ? quantize_g4(nan ? 0.0f : v[r][e], s_q4)
                         : B == 3 ? quantize_ss3(v[r][e])
                                  : quantize_ss2(v[r][e]);
      s_code[r * P + lane + 64 * e] = (uint8_t)q;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const uint32_t *s_word = reinterpret_cast<const uint32_t *>(s_code);
#pragma unroll 2
  for (int i = lane; i < nr * NW; i += 64) {
    const int r = i / NW, k = i % NW;
    const uint32_t *cw = s_word + r * (P / 4);
    uint32_t w = 0u;
    if constexpr (B == 4) {
      // four bytes of two codes, high nibble first: eight codes from two words
      const uint32_t lo = cw[2 * k], hi = cw[2 * k + 1];
      const uint32_t a = (lo << 4 | lo >> 8) & 0x00FF00FFu, b = (hi << 4 | hi >> 8) & 0x00FF00FFu;
      w = __builtin_amdgcn_perm(b, a, 0x06040200u);
    } else if constexpr (B == 2) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t c = cw[4 * k + j];  // four codes: one byte, the first on top
        w |= (((c << 6) | (c >> 4) | (c >> 14) | (c >> 24)) & 255u) << (8 * j);
      }
    } else {
      // word k holds bytes 4 k .. 4 k + 3 of the row's 24-bit big-endian groups
      // of 8 codes: two groups at most, g = 4 k / 3 and the next
      const int g = 4 * k / 3;
      uint32_t grp[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int at = min(g + h, P / 8 - 1);
        const uint32_t lo = cw[2 * at], hi = cw[2 * at + 1];
        auto four = [](uint32_t c) {  // c0 << 9 | c1 << 6 | c2 << 3 | c3
          return ((c & 7u) << 9) | ((c >> 2) & 0x1C0u) | ((c >> 13) & 0x38u) | (c >> 24);
        };
        grp[h] = four(lo) << 12 | four(hi);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = 4 * k + j - 3 * g;  // byte of the two groups, 0 .. 5
        const uint32_t x = b < 3 ? grp[0] : grp[1];
        w |= ((x >> (16 - 8 * (b < 3 ? b : b - 3))) & 255u) << (8 * j);
      }
    }
    if ((nan_rows >> r) & 1u) w = nan_word<B>(k);
    int slot = slot0 + r;
    if (slot >= cap) slot %= cap;
    const uint32_t x = (uint32_t)slot & xmask;
    if (kperm_mask(P, B) != 0) w = __builtin_amdgcn_perm(0u, w, 0x03020100u ^ ((x & 3u) * 0x01010101u));
    if (r + age >= 0)
      reinterpret_cast<uint32_t *>(codes + (size_t)slot * (P * B / 8))[(uint32_t)k ^ (x >> 2)] = w;
  }
}

// A wave encodes R rows of one side of one head (any padded size from 64 on, any
// bits), lane l holding entries l, l + 64, ... of each (E = P / 64 registers a row),
// with the float steps of encode_vec (append.hip) in its order.  The
// left-to-right sum of
// squares is a chain of P dependent adds: the squares go to LDS and lane r
// walks row r's, so the R rows share one chain's time (rows start 4 banks
// apart: the 16-byte reads of up to 16 lanes do not conflict).  The
// butterflies of span 1..32 run between lanes (shfl_xor), the wider ones
// inside the lane; codes are gathered in LDS and the lanes pack the rows' words.
//
// Bound: the launch's latency for few rows (R = 1: the chain is about 1 us at
// P 256), VALU issue and LDS for many (R E = 32 registers of row data; 64 and
// 16 of them measured 1,037 and 1,072 us where 32 take 934, for 4,096 tokens of
// 256 heads at d256 K4/V2: 2.3 TB/s of input).  The kernel this replaced kept a
// lane's whole vector in scratch memory, 4 KB a lane, a launch a side: one
// token of those heads 608 + 740 us (here 4 us for both sides), 4,096 tokens
// 11.0 + 9.2 ms.
//
// t0: the first of the R rows, tokens t0 .. t0 + R - 1 (those below n_tok).
// s_sq: R * (P + 4) floats of LDS, this wave's own; the codes take the squares'
// place once the sums are done.
template <int P, int R>
__device__ __forceinline__ void encode_wide_rows(const HeadDesc *d, const RingState st, int n_tok,
                                                 int t0, const float *__restrict__ src, int dim,
                                                 int side, int B, int lane, float inv_sqrt_p,
                                                 float sqrt_p, const Q4Cell *s_q4,
                                                 float *s_sq) {
  constexpr int E = P / 64;
  constexpr int RS = P + 4;  // row stride of the squares
  const int cap = d->cap;
  const int mirror = mirror_count(st, n_tok, cap, d->hyb);
  const int nr = min(R, n_tok - t0);  // rows of this wave, at least 1
  if (t0 >= mirror && (cap <= 0 || t0 + nr <= n_tok - cap)) return;  // nothing is kept
  float v[R][E];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int e = 0; e < E; ++e)
      v[r][e] = r < nr && lane + 64 * e < dim ? src[(size_t)r * dim + lane + 64 * e] : 0.0f;
  if (t0 < mirror) {
    float *m = (side == 0 ? d->raw_k : d->raw_v) + (size_t)(st.raw_count + t0) * dim;
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (t0 + r < mirror)
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (lane + 64 * e < dim) m[(size_t)r * dim + lane + 64 * e] = v[r][e];
  }
  if (cap <= 0) return;
  uint8_t *codes = side == 0 ? d->k_codes : d->v_codes;
  float *scales = side == 0 ? d->k_scale : d->v_scale;
  const int slot0 = (int)(((long long)st.head + t0) % cap);
  // row r survives the call unless cap later tokens follow it
  auto kept = [&](int r) { return r < nr && t0 + r >= n_tok - cap; };
  auto slot_of = [&](int r) { return (int)(((long long)slot0 + r) % cap); };
  if (B == 16) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (kept(r)) {
        float *row = reinterpret_cast<float *>(codes) + (size_t)slot_of(r) * P;
#pragma unroll
        for (int e = 0; e < E; ++e) row[lane + 64 * e] = v[r][e];
        if (lane == 0) scales[slot_of(r)] = 1.0f;
      }
    return;
  }
  // lane r < R: the left-to-right sum of row r's squares (other lanes row 0's)
  auto seq_sumsq = [&]() {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int e = 0; e < E; ++e) s_sq[r * RS + lane + 64 * e] = __fmul_rn(v[r][e], v[r][e]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float4 *q4 = reinterpret_cast<const float4 *>(s_sq + (lane < R ? lane : 0) * RS);
    float acc = 0.0f;
#pragma unroll 4
    for (int b = 0; b < P / 16; ++b) {
      float4 x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = q4[4 * b + k];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        acc = __fadd_rn(acc, x[k].x);
        acc = __fadd_rn(acc, x[k].y);
        acc = __fadd_rn(acc, x[k].z);
        acc = __fadd_rn(acc, x[k].w);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // s_sq is read by every lane before it is rewritten
    return acc;
  };
  const float s = seq_sumsq();
  const float norm = sqrtf(__fadd_rn(s, 1e-12f));
  const float inv = 1.0f / norm;
  uint32_t flip[E];
#pragma unroll
  for (int e = 0; e < E; ++e) flip[e] = (~d->signs[2 * e + (lane >> 5)] >> (lane & 31)) << 31;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float iv = R == 1 ? inv : __shfl(inv, r, 64);
#pragma unroll
    for (int e = 0; e < E; ++e)
      v[r][e] = __uint_as_float(__float_as_uint(__fmul_rn(v[r][e], iv)) ^ flip[e]);
#pragma unroll
    for (int len = 1; len < 64; len <<= 1) {
      const bool upper = (lane & len) != 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float o = __shfl_xor(v[r][e], len, 64);
        v[r][e] = upper ? __fsub_rn(o, v[r][e]) : __fadd_rn(v[r][e], o);
      }
    }
#pragma unroll
    for (int len = 1; len < E; len <<= 1)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((e & len) == 0) {
          const float lo = v[r][e], hi = v[r][e | len];
          v[r][e] = __fadd_rn(lo, hi);
          v[r][e | len] = __fsub_rn(lo, hi);
        }
#pragma unroll
    for (int e = 0; e < E; ++e) v[r][e] = __fmul_rn(__fmul_rn(v[r][e], inv_sqrt_p), sqrt_p);
  }
  // bit r: row r is NaN (a NaN anywhere in the input reaches every entry
  // through the FWHT)
  uint32_t nan_rows = 0u;
#pragma unroll
  for (int r = 0; r < R; ++r) nan_rows |= (__any(v[r][0] != v[r][0]) ? 1u : 0u) << r;
  // The clamp (see encode_vec, whose bound holds up to padded 1024: the sums'
  // roundings are below 1,100 u = 7e-5): inert where every row has s >= 1e-10.
  if (!__all(lane >= nr || s >= 1e-10f)) {
    const float s2 = seq_sumsq();
    const float sigma = sqrtf(__fadd_rn(s2 / (float)P, 1e-12f));
    const float clip = __fmul_rn(3.0f, sigma);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float cr = R == 1 ? clip : __shfl(clip, r, 64);
#pragma unroll
      for (int e = 0; e < E; ++e) v[r][e] = __builtin_amdgcn_fmed3f(v[r][e], -cr, cr);
    }
  }
  if (lane < R && kept(lane)) scales[slot_of(lane)] = norm;
  uint8_t *s_code = reinterpret_cast<uint8_t *>(s_sq);
  const int age = t0 - (n_tok - cap);
  auto xm = [&](int bits) { return side == 0 ? (uint32_t)kperm_mask(P, bits) : 0u; };
  if (B == 4) store_wide_rows<P, R, 4>(v, nan_rows, codes, slot0, cap, nr, age, lane, xm(4), s_q4, s_code);
  else if (B == 3) store_wide_rows<P, R, 3>(v, nan_rows, codes, slot0, cap, nr, age, lane, xm(3), s_q4, s_code);
  else store_wide_rows<P, R, 2>(v, nan_rows, codes, slot0, cap, nr, age, lane, xm(2), s_q4, s_code);
}

}  // namespace aq
