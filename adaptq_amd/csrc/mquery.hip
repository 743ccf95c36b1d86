// mquery.hip -- decode of many queries per head (gfx950).
//
// With nq queries per head, the dense decode (attention.cpp:373-474 with
// v_mass <= 0) is two products per head over the ring:
//   logits   S[q][t] = sum_i qr[q][i] * CB_K[c_ti]        (qr = H (D . q))
//   output   O[q][d] = sum_t p[q][t] * vscale_t / sqrt(p) * CB_V[c_td]
// so each K/V tile can be read once for all the queries of its head instead
// of once per query (decode.hip's LUT kernel, one query per item).
//
// Logits are the reference's own floats.  On peaked softmaxes (outlier
// channels: logits of +-300, where one fp32 unit is 3e-5) the reference's
// rounding of the dot moves outputs by about 1e-4, so a more accurate dot
// (a double-precision matrix product was tried) lands as far from it on the
// other side.  Each logit is computed as attention.cpp:93-136 and :83-88
// compute it: eight fused multiply-add chains (chain L takes dims L, L + 8,
// ... in order), combined ((s0+s4)+(s1+s5)) + ((s2+s6)+(s3+s7)), times
// 1/(sqrt(dim) p), times the key's scale; the query rotation repeats the
// reference's float steps (attention.cpp:528-550, fwht.cpp:33-66).
//
// Both products run on the matrix cores.  v_mfma_f32_16x16x4 adds its four
// products to an entry one after another, in order, each a fused multiply-add
// rounded as fmaf (tests/test_gpu_mfma_chain.py: bit for bit, over normal,
// denormal and large operands), so a chain of it is a chain of the
// reference's: eight accumulators, chain L of a 16-token by 16-query tile fed
// dims L + 8 j, j ascending, four an instruction.  Operand layouts
// (established on the device): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16], register r of lane l is D[4 (l / 16) + r][l % 16].  Keys
// are A and queries B, so a lane holds all eight chain sums of its tokens and
// query, and combines them without leaving its registers.  The V sum takes
// queries as M and, at step r, tokens 4 k + r as K: A is the weight that the
// lane already has from the logits.  The softmax weight and
// the V scale are folded into A (fp32 accumulation, as the reference's).  The
// online softmax is the LUT kernel's with the reference's -1e30 seed, in
// natural units (exp2 of (logit - max) * log2 e, so the weights of the tokens
// near the maximum carry no rounding of the logit's magnitude); splits over
// tokens end in decode.hip's finalize kernel.
//
// Block: four waves, QG (1, 2 or 4) groups of 16 queries of one head, one
// token split.  The block takes TS = 4 / QG tiles of 16 tokens a step: its
// threads turn the tiles' codes into floats in LDS, a unit of 8 dims each
// (16-entry tables, distinct banks), one step ahead of their use; wave (slice
// ts, group) multiplies tile ts with its group's queries.  Lane (g, c) =
// (l / 16, l % 16) holds, for query c, the rotated entries of the 8-dim groups
// 4 i + g in registers; reads the same groups of token c's key (16-byte LDS
// reads, a step of four chains each) and, for tokens 4 g + r, the value's dims
// 4 c .. 4 c + 3 and 64 + 4 c .. (likewise).  Rows are padded so that 16
// lanes' reads cover the 64 banks.  Slices of the same queries merge in LDS at
// the end.
//
// Bound: the matrix cores' fp32 rate, and the vector ALU's work beside it
// (about 180 instructions a tile and wave, which the fp32 matrix rate does not
// hide: taking either product out shortens the launch by exactly its own 26
// us).  64 queries of 8 heads over 32,768 tokens at padded 128, K4/V4 (8.6
// GFLOP, 55 us at 157 TFLOP/s): 102 us under the profiler.  The kernel before
// it ran the logits' chains on the vector ALU, a token a lane, and passed them
// to the V product through LDS: 156 us.  With a wave dequantising its own
// tiles (codes read by the four lanes of a token, tables to registers) the
// matrix form took 175 us: sixteen code loads and 128 table reads a tile and
// wave, and 20 registers spilled.
#include <algorithm>

#include "launch.hpp"
#include "mquery_rule.hpp"

namespace aq {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMqThreads = 64 * kMqWaves;
constexpr float kLog2e = 1.44269504088896340736f;

// The codes of dims 8 j .. 8 j + 7 of a packed row (MSB-first,
// quantizer.cpp:156-209), as loaded: 4 bits a word, 2 bits a half word, 3 bits
// the two words that hold the 24-bit big-endian group (the second clamped to
// the row).  K rows of 2/4-bit codes are stored XOR-permuted (device.hpp
// kperm_mask; x = slot & mask, 0 for V): the unit's bytes sit at unit j ^ (x /
// unit bytes), permuted among themselves by x % unit bytes.
template <int B>
struct MqUnit {
  uint32_t w[B == 3 ? 2 : 1];
};

template <int P, int B>
__device__ __forceinline__ MqUnit<B> mq_load_unit(const uint8_t *codes, uint32_t slot, int j,
                                                  uint32_t x) {
  const uint8_t *row = codes + (size_t)slot * (P * B / 8);
  MqUnit<B> u;
  if constexpr (B == 4) {
    u.w[0] = reinterpret_cast<const uint32_t *>(row)[(uint32_t)j ^ (x >> 2)];
  } else if constexpr (B == 2) {
    u.w[0] = reinterpret_cast<const uint16_t *>(row)[(uint32_t)j ^ (x >> 1)];
  } else {
    const uint32_t *r32 = reinterpret_cast<const uint32_t *>(row);
    const int w0 = 3 * j / 4;
    u.w[0] = r32[w0];
    u.w[1] = r32[min(w0 + 1, P * 3 / 32 - 1)];
  }
  return u;
}

// The unit's eight values.
template <int B>
__device__ __forceinline__ void mq_unit_values(const MqUnit<B> &u, int j, uint32_t x,
                                               const float *s_cb, float (&v)[8]) {
  if constexpr (B == 4) {
    const uint32_t w = __builtin_amdgcn_perm(0u, u.w[0], 0x03020100u ^ ((x & 3u) * 0x01010101u));
#pragma unroll
    for (int d = 0; d < 8; ++d) v[d] = s_cb[(w >> (8 * (d >> 1) + ((d & 1) ? 0 : 4))) & 15u];
  } else if constexpr (B == 2) {
    const uint32_t w = __builtin_amdgcn_perm(0u, u.w[0], 0x0C0C0100u ^ ((x & 1u) * 0x0101u));
#pragma unroll
    for (int d = 0; d < 8; ++d) v[d] = s_cb[(w >> (8 * (d >> 2) + 6 - 2 * (d & 3))) & 3u];
  } else {
    // bytes 3 j .. 3 j + 2, from byte (3 j) % 4 of the word pair, big-endian
    const uint32_t a = __builtin_amdgcn_alignbyte(u.w[1], u.w[0], (uint32_t)(3 * j) & 3u);
    const uint32_t w = __builtin_amdgcn_perm(0u, a, 0x0C000102u);
#pragma unroll
    for (int d = 0; d < 8; ++d) v[d] = s_cb[(w >> (21 - 3 * d)) & 7u];
  }
}

// max(v) over the four lanes that share lane % 16.
__device__ __forceinline__ float quad_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Read-only global memory seen through the constant address space: loads at
// wave-uniform addresses become scalar loads.
typedef const __attribute__((address_space(4))) float cfloat;
// The descriptor read this way is uniform to the compiler too: loops over a
// ring's tokens stay scalar branches, barriers inside them included.
typedef const __attribute__((address_space(4))) HeadDesc cdesc;
__device__ __forceinline__ cdesc *desc_of(HeadDesc *const *item_desc, int i) {
  return (cdesc *)((const __attribute__((address_space(4))) uint64_t *)item_desc)[i];
}

// Rotated queries of query group qg of head h: rows of P floats at
// qrot[((h * qgroups + qg) * 16 + jj) * P], zero rows past nq.  One wave per
// query, lane l holding entries l and l + 64, with the reference's float steps
// (attention.cpp:528-550, fwht.cpp:33-66): qn = sqrt(sum q^2 + 1e-12) left to
// right, q / qn, signs, butterflies of span 1, 2, ..., P/2 (lo + hi, lo - hi),
// * RN(1/RN(sqrt p)), * RN(sqrt p * qn).
template <int P>
__global__ __launch_bounds__(256) void mq_rotate_kernel(HeadDesc *const *item_desc, int n_heads,
                                                        int nq, int qgroups,
                                                        const float *__restrict__ queries,
                                                        float *__restrict__ qrot) {
  constexpr int E = P / 64;  // entries per lane
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= qgroups * kMqQueries) return;
  const int j = row;  // query index: group row / 16, row % 16 within it
  const HeadDesc *d = item_desc[h];
  const int dim = d->dim;
  float *out = qrot + ((size_t)h * qgroups * kMqQueries + row) * P;
  if (j >= nq) {
#pragma unroll
    for (int i = 0; i < E; ++i) out[lane + 64 * i] = 0.0f;
    return;
  }
  const float *q = queries + (size_t)(j * n_heads + h) * dim;
  const cfloat *qs = (const cfloat *)q;
  // left to right: the row's 16-entry blocks come in as scalar loads ahead of
  // their squares
  float sq = 0.0f;
  const int nb = dim / 16;
  for (int b = 0; b < nb; ++b) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = qs[16 * b + k];
#pragma unroll
    for (int k = 0; k < 16; ++k) sq = __fadd_rn(sq, __fmul_rn(v[k], v[k]));
  }
  for (int e = 16 * nb; e < dim; ++e) sq = __fadd_rn(sq, __fmul_rn(qs[e], qs[e]));
  const float qn = sqrtf(__fadd_rn(sq, 1e-12f));
  const float inv = 1.0f / qn;
  float x[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane + 64 * i;
    float v = __fmul_rn(e < dim ? q[e] : 0.0f, inv);
    if (!((d->signs[e >> 5] >> (e & 31)) & 1u)) v = -v;
    x[i] = v;
  }
#pragma unroll
  for (int len = 1; len < 64; len <<= 1) {
    const bool upper = (lane & len) != 0;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const float other = __shfl_xor(x[i], len, 64);
      x[i] = upper ? __fsub_rn(other, x[i]) : __fadd_rn(x[i], other);
    }
  }
  if constexpr (E == 2) {
    const float lo = x[0], hi = x[1];
    x[0] = __fadd_rn(lo, hi);
    x[1] = __fsub_rn(lo, hi);
  }
  const float sqrt_p = sqrtf((float)P);
  const float inv_sqrt_p = 1.0f / sqrt_p;
  const float post = __fmul_rn(sqrt_p, qn);
#pragma unroll
  for (int i = 0; i < E; ++i) out[lane + 64 * i] = __fmul_rn(__fmul_rn(x[i], inv_sqrt_p), post);
}


// Block (split, head h, groups qg0 .. qg0 + QG - 1), 1-D grid with the split
// fastest.
template <int P, int KB, int VB, int QG>
__global__ __launch_bounds__(kMqThreads, QG == 4 ? 3 : 2) void decode_mq_kernel(
    HeadDesc *const *item_desc, int n_heads, int nq, int qgroups, int chunk, int n_splits,
    const float *__restrict__ qrot, float *__restrict__ partials) {
  constexpr int TS = kMqWaves / QG;         // tiles a step
  constexpr int NBUF = TS == 4 ? 1 : 2;     // LDS copies of a step's tiles
  constexpr int NT = P / 16;                // 16-column output tiles
  constexpr int NE = P / 4;                 // entries of a row a lane holds
  constexpr int KST = NE + 4;               // K: [token][g][group 4 i + g], stride of a (token, g)
  constexpr int VST = P + 4;                // V: [token][dim], stride of a token
  constexpr int TILE = kMqTile * (4 * KST + VST) + 2 * kMqTile;  // K, V, both scales
  constexpr int MST = P + 4;  // row stride of a wave's merge record: m, l, pad, pad, acc
  constexpr int UNITS = TS * kMqTile * P / 8;  // units of K (and of V) a step
  constexpr int UPT = (UNITS + kMqThreads - 1) / kMqThreads;
  static_assert(UNITS % kMqThreads == 0 || UNITS < kMqThreads, "units spread evenly");
  constexpr int SMEM = NBUF * TS * TILE;
  static_assert(TS == 1 || SMEM >= kMqWaves * kMqQueries * MST, "the merge records fit");
  __shared__ __align__(16) float s_buf[SMEM];
  __shared__ float s_cbk[16];
  __shared__ float s_cbv[16];

  const int bid = blockIdx.x;
  const int split = bid % n_splits, rest = bid / n_splits;
  const int h = rest % n_heads, qg0 = (rest / n_heads) * QG;
  cdesc *d = desc_of(item_desc, h);
  const int dim = d->dim, n = d->st.size;
  const int t_begin = split * chunk, t_end = min(n, t_begin + chunk);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int ts = wave / QG, qg = qg0 + wave % QG;
  const int j0 = qg * kMqQueries;  // first query of the wave
  auto part_of = [&](int j) {
    return partials + ((size_t)(j * n_heads + h) * n_splits + split) * (P + 4);
  };

  if (t_begin >= t_end) {
    // empty split: (m, l, acc) = (-inf, 0, 0) for the block's queries
    for (int i = threadIdx.x; i < QG * kMqQueries * (P + 4); i += kMqThreads) {
      const int jj = i / (P + 4), e = i - jj * (P + 4), j = qg0 * kMqQueries + jj;
      if (j < nq) part_of(j)[e] = e == 0 ? -INFINITY : 0.0f;
    }
    return;
  }

  const float attn_s = 1.0f / (sqrtf((float)dim) * (float)P);
  const float isp = 1.0f / sqrtf((float)P);
  const uint8_t *kbase = d->k_codes, *vbase = d->v_codes;
  const float *k_scale = d->k_scale, *v_scale = d->v_scale;

  // ---- a step's codes: units u = thread, thread + kMqThreads, ... of its TS
  // tiles, unit (token u / (P / 8), dims 8 (u % (P / 8)) ..); tokens past the
  // split's end are its last one (their weights are 0) ----
  MqUnit<KB> ku[UPT];
  MqUnit<VB> vu[UPT];
  float sc = 0.0f;
  const bool has_units = UNITS >= kMqThreads || (int)threadIdx.x < UNITS;
  auto slot_of = [&](int t) { return (uint32_t)min(t, t_end - 1); };
  auto load_step = [&](int tb) {
    if (has_units) {
#pragma unroll
      for (int i = 0; i < UPT; ++i) {
        const int u = (int)threadIdx.x + i * kMqThreads, tk = u / (P / 8), j = u % (P / 8);
        const uint32_t slot = slot_of(tb + tk);
        ku[i] = mq_load_unit<P, KB>(kbase, slot, j, slot & (uint32_t)kperm_mask(P, KB));
        vu[i] = mq_load_unit<P, VB>(vbase, slot, j, 0u);
      }
    }
    if (threadIdx.x < 2 * TS * kMqTile) {
      const int tk = threadIdx.x % (TS * kMqTile);
      sc = ((int)threadIdx.x < TS * kMqTile ? k_scale : v_scale)[slot_of(tb + tk)];
    }
  };
  auto store_step = [&](int tb, float *buf) {
    if (has_units) {
#pragma unroll
      for (int i = 0; i < UPT; ++i) {
        const int u = (int)threadIdx.x + i * kMqThreads, tk = u / (P / 8), j = u % (P / 8);
        float *tile = buf + (tk / kMqTile) * TILE;
        const int t16 = tk % kMqTile;
        const uint32_t x = slot_of(tb + tk) & (uint32_t)kperm_mask(P, KB);
        float kv[8], vv[8];
        mq_unit_values<KB>(ku[i], j, x, s_cbk, kv);
        float4 *kr = reinterpret_cast<float4 *>(tile + (t16 * 4 + (j & 3)) * KST + 8 * (j >> 2));
        kr[0] = make_float4(kv[0], kv[1], kv[2], kv[3]);
        kr[1] = make_float4(kv[4], kv[5], kv[6], kv[7]);
        mq_unit_values<VB>(vu[i], j, 0u, s_cbv, vv);
        float4 *vr = reinterpret_cast<float4 *>(tile + kMqTile * 4 * KST + t16 * VST + 8 * j);
        vr[0] = make_float4(vv[0], vv[1], vv[2], vv[3]);
        vr[1] = make_float4(vv[4], vv[5], vv[6], vv[7]);
      }
    }
    if (threadIdx.x < 2 * TS * kMqTile) {
      const int tk = threadIdx.x % (TS * kMqTile), side = (int)threadIdx.x / (TS * kMqTile);
      buf[(tk / kMqTile) * TILE + kMqTile * (4 * KST + VST) + side * kMqTile + tk % kMqTile] = sc;
    }
  };

  constexpr int kStep = kMqTile * TS;
  load_step(t_begin);
  if (threadIdx.x < (1 << KB)) s_cbk[threadIdx.x] = cb<KB>(threadIdx.x);
  if (threadIdx.x < (1 << VB)) s_cbv[threadIdx.x] = cb<VB>(threadIdx.x);
  // query c16's 8-dim groups 4 i + g (query groups past the last: unused)
  const bool live = qg < qgroups;
  float qe[NE];
  if (live) {
    const float *qr = qrot + ((size_t)(h * qgroups + qg) * kMqQueries + c16) * P + 8 * g;
#pragma unroll
    for (int j = 0; j < NE; ++j) qe[j] = qr[32 * (j / 8) + j % 8];
  }
  __syncthreads();
  store_step(t_begin, s_buf);
  __syncthreads();
  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY;  // query c16; the first tile seeds it with the reference's -1e30
  float l_part = 0.0f;      // this lane's tokens' share of query c16's sum

  int cur = 0;
  for (int tb = t_begin; tb < t_end; tb += kStep) {
    const bool more = tb + kStep < t_end;
    if (more) load_step(tb + kStep);
    const float *tile = s_buf + (cur * TS + ts) * TILE;
    const int tile_tb = tb + ts * kMqTile;
    if (live && tile_tb < t_end) {
      // ---- logits (attention.cpp:93-136, :83-88): eight chains ----
      f32x4 s8[8];
#pragma unroll
      for (int L = 0; L < 8; ++L) s8[L] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      const float4 *kr = reinterpret_cast<const float4 *>(tile + (c16 * 4 + g) * KST);
#pragma unroll
      for (int j = 0; j < NE / 4; ++j) {
        const float4 k4 = kr[j];
        const int L = 4 * (j & 1);
        s8[L] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.x, qe[4 * j], s8[L], 0, 0, 0);
        s8[L + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.y, qe[4 * j + 1], s8[L + 1], 0, 0, 0);
        s8[L + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.z, qe[4 * j + 2], s8[L + 2], 0, 0, 0);
        s8[L + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.w, qe[4 * j + 3], s8[L + 3], 0, 0, 0);
      }
      const float *sc_row = tile + kMqTile * (4 * KST + VST) + 4 * g;
      const float4 ks4 = *reinterpret_cast<const float4 *>(sc_row);
      const float4 vs4 = *reinterpret_cast<const float4 *>(sc_row + kMqTile);
      const float ks[4] = {ks4.x, ks4.y, ks4.z, ks4.w}, vs[4] = {vs4.x, vs4.y, vs4.z, vs4.w};
      // logits of query c16 and tokens 4 g + r of the tile
      float lg[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float dot = __fadd_rn(
            __fadd_rn(__fadd_rn(s8[0][r], s8[4][r]), __fadd_rn(s8[1][r], s8[5][r])),
            __fadd_rn(__fadd_rn(s8[2][r], s8[6][r]), __fadd_rn(s8[3][r], s8[7][r])));
        lg[r] = __fmul_rn(__fmul_rn(dot, attn_s), ks[r]);
      }
      if (tile_tb + kMqTile > t_end) {  // tokens past the split's end
#pragma unroll
        for (int r = 0; r < 4; ++r) lg[r] = tile_tb + 4 * g + r < t_end ? lg[r] : -INFINITY;
      }

      // ---- online softmax: the maximum moves, and the sums with it, only in
      // a tile that holds a larger logit (or seeds it) ----
      const float tmax = fmaxf(fmaxf(lg[0], lg[1]), fmaxf(lg[2], lg[3]));
      if (__any(tmax > m_run) || tb == t_begin) {
        const float m_new = fmaxf(m_run, fmaxf(quad_max(tmax), -1e30f));
        const float alpha = __builtin_amdgcn_exp2f(__fmul_rn(m_run - m_new, kLog2e));
        m_run = m_new;
        l_part *= alpha;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // O rows (query 4 g + r of the result layout) by their query's alpha
          const float a = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[nt][r] *= a;
        }
      }

      // ---- weighted V: O[q][dim] += sum_t w[q][t] V[t][dim], tile nt's column
      // c16 being dim 64 (nt / 4) + 4 c16 + nt % 4 ----
      const float *vr = tile + kMqTile * 4 * KST + 4 * g * VST + 4 * c16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(__fmul_rn(lg[r] - m_run, kLog2e));
        l_part += e;
        const float w = e * vs[r] * isp;
#pragma unroll
        for (int b = 0; b < NT / 4; ++b) {
          const float4 v4 = *reinterpret_cast<const float4 *>(vr + r * VST + 64 * b);
          acc[4 * b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, v4.x, acc[4 * b], 0, 0, 0);
          acc[4 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, v4.y, acc[4 * b + 1], 0, 0, 0);
          acc[4 * b + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, v4.z, acc[4 * b + 2], 0, 0, 0);
          acc[4 * b + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, v4.w, acc[4 * b + 3], 0, 0, 0);
        }
      }
    }
    if constexpr (NBUF == 1) __syncthreads();  // the tiles are read out
    else cur ^= 1;
    if (more) store_step(tb + kStep, s_buf + cur * TS * TILE);
    // the next step's tiles are written; this step's copy is read out.  (At the
    // loop's end: a barrier at its head, after the store's divergent branches,
    // was reached by the lanes of a wave one branch at a time.)
    __syncthreads();
  }

  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  auto dim_of = [&](int nt) { return 64 * (nt / 4) + 4 * c16 + (nt & 3); };
  if constexpr (TS == 1) {
    // the wave's records (m, l) of query c16 and acc rows 4 g + r
    if (!live) return;
    if (g == 0 && j0 + c16 < nq) {
      part_of(j0 + c16)[0] = m_run;
      part_of(j0 + c16)[1] = l_tot;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (j0 + 4 * g + r < nq) {
        float *po = part_of(j0 + 4 * g + r) + 4 + 4 * c16;
#pragma unroll
        for (int b = 0; b < NT / 4; ++b)
          *reinterpret_cast<float4 *>(po + 64 * b) = make_float4(
              acc[4 * b][r], acc[4 * b + 1][r], acc[4 * b + 2][r], acc[4 * b + 3][r]);
      }
    return;
  }
  // ---- merge the slices of each group (the tiles are read out) ----
  float *rec = s_buf + wave * (kMqQueries * MST);
  if (g == 0) {
    rec[c16 * MST] = m_run;
    rec[c16 * MST + 1] = l_tot;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) rec[(4 * g + r) * MST + 4 + dim_of(nt)] = acc[nt][r];
  __syncthreads();
  for (int i = threadIdx.x; i < QG * kMqQueries * (P + 4); i += kMqThreads) {
    const int jj = i / (P + 4), e = i - jj * (P + 4), j = qg0 * kMqQueries + jj;
    if (j >= nq || e == 2 || e == 3) continue;
    // slice w's record of this query: wave w QG + jj / 16
    auto rec_of = [&](int w) {
      return s_buf + ((w * QG + jj / kMqQueries) * kMqQueries + jj % kMqQueries) * MST;
    };
    float mw[TS], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < TS; ++w) {
      mw[w] = rec_of(w)[0];
      M = fmaxf(M, mw[w]);
    }
    float out;
    if (e == 0) {
      out = M;
    } else {
      out = 0.0f;
#pragma unroll
      for (int w = 0; w < TS; ++w) {
        // a slice without tokens has m = -inf and contributes 0
        const float f = __builtin_amdgcn_exp2f(__fmul_rn(mw[w] - M, kLog2e));
        out += rec_of(w)[e] * f;
      }
    }
    part_of(j)[e] = out;
  }
}

bool mq_eligible(int n_items, int n_heads, const DecodeShape &sh) {
  if (n_heads <= 0 || n_items % n_heads != 0) return false;
  const int nq = n_items / n_heads;
  const bool kq = sh.k_bits >= 2 && sh.k_bits <= 4, vq = sh.v_bits >= 2 && sh.v_bits <= 4;
  return !sh.raw && kq && vq && (sh.padded == 64 || sh.padded == 128) &&
         mq_pays(n_heads, nq, sh.max_n, sh.padded) && n_heads <= 65535 && (int64_t)n_heads * ((nq + kMqQueries - 1) / kMqQueries) *
                                      ((sh.max_n + 127) / 128) <
                                  (int64_t)1 << 31;
}

template <int P>
hipError_t dispatch_mq(const DecodeShape &sh, dim3 grid, HeadDesc *const *descs, int n_heads,
                       int nq, const MqPlan &mp, const float *q, float *qrot, float *part,
                       hipStream_t s) {
  mq_rotate_kernel<P><<<dim3((mp.qgroups * kMqQueries + 3) / 4, n_heads), 256, 0, s>>>(
      descs, n_heads, nq, mp.qgroups, q, qrot);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
#define AQ_MQ_QG(KB_, VB_, QG_)                                                             \
  decode_mq_kernel<P, KB_, VB_, QG_><<<grid, kMqThreads, 0, s>>>(                           \
      descs, n_heads, nq, mp.qgroups, mp.chunk, mp.splits, qrot, part)
#define AQ_MQ(KB_, VB_)                                                                     \
  if (sh.k_bits == KB_ && sh.v_bits == VB_) {                                               \
    if (mp.qg == 4) AQ_MQ_QG(KB_, VB_, 4);                                                  \
    else if (mp.qg == 2) AQ_MQ_QG(KB_, VB_, 2);                                             \
    else AQ_MQ_QG(KB_, VB_, 1);                                                             \
    return hipGetLastError();                                                               \
  }
  AQ_MQ(4, 2) AQ_MQ(4, 3) AQ_MQ(4, 4)
  AQ_MQ(3, 2) AQ_MQ(3, 3) AQ_MQ(3, 4)
  AQ_MQ(2, 2) AQ_MQ(2, 3) AQ_MQ(2, 4)
#undef AQ_MQ
#undef AQ_MQ_QG
  return hipErrorInvalidValue;
}

// Workspace of the multi-query path: the rotated queries (n_heads * qgroups
// * 16 rows of P floats), then the split partials (item, split) of P + 4.
size_t mq_qrot_floats(int n_heads, const MqPlan &mp, int padded) {
  return (size_t)n_heads * mp.qgroups * kMqQueries * padded;
}

}  // namespace

size_t decode_multi_workspace_floats(int n_items, int n_heads, const DecodeShape &sh) {
  if (!mq_eligible(n_items, n_heads, sh)) return decode_workspace_floats(n_items, sh);
  const MqPlan mp = mq_plan(n_heads, n_items / n_heads, sh.max_n);
  return mq_qrot_floats(n_heads, mp, sh.padded) + (size_t)n_items * mp.splits * (sh.padded + 4);
}

hipError_t launch_decode_multi(HeadDesc *const *descs, int n_items, int n_heads,
                               const DecodeShape &sh, const float *d_q, float *d_out,
                               float *d_ws, hipStream_t s) {
  if (n_items <= 0) return hipSuccess;
  if (!mq_eligible(n_items, n_heads, sh))
    return launch_decode(descs, n_items, sh, d_q, d_out, d_ws, s);
  const int nq = n_items / n_heads;
  const MqPlan mp = mq_plan(n_heads, nq, sh.max_n);
  const dim3 grid((unsigned)mp.splits * n_heads * mp.qblocks);
  float *qrot = d_ws, *part = d_ws + mq_qrot_floats(n_heads, mp, sh.padded);
  const hipError_t e =
      sh.padded == 64 ? dispatch_mq<64>(sh, grid, descs, n_heads, nq, mp, d_q, qrot, part, s)
                      : dispatch_mq<128>(sh, grid, descs, n_heads, nq, mp, d_q, qrot, part, s);
  if (e != hipSuccess) return e;
  return launch_finalize(descs, n_items, sh.padded, mp.splits, part, d_out, true, s);
}

}  // namespace aq
