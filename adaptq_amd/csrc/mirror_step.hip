// mirror_step.hip -- one decode step on the hybrid branch in one launch (gfx950).
//
// Restates attention.cpp:338-366 (append) and :491-523 (exact fp32 attention
// over the raw mirror) for one token and one query per head: a cache's first
// tokens, up to the hybrid threshold, are decoded this way.
//
// Block: one head, kTokWaves waves for the attention and two that encode the
// token's key and value into the ring and copy them to the mirror
// (encode_rows.hpp) beside them.  A thread takes one token: the reference's
// sequential, unfused dot product (attention.cpp:497-502) with the row in
// registers and the query read broadcast from LDS.  The new token's row comes
// from LDS, never from the mirror that the other waves are writing.  The
// weights go to LDS; then lane l of wave w adds dimensions l, l + 64, ... of
// tokens w, w + kTokWaves, ..., a coalesced row a load, and the waves' sums meet
// in LDS.
//
// Bound: latency, the dependent loads (descriptor, rows) and the dot's chain of
// dim adds.  A step of 14 heads d64, 0-32, 64-96 and 470-502 tokens: 8.0, 8.1
// and 12.4 us, where an append launch, the LUT kernel over the mirror and its
// finalize launch took 11.8, 14.8 and 14.5; 8 heads d128 9.3 (64-96 tokens) and
// 17.5 us (470-502), before 11.6 and 21.3; 16 heads d80, whose mirror decode
// took the generic kernel, 10.0 and 91 (200-232 tokens); 256 heads d64 24.9 and
// 30.8 (470-502).  So every step it can take goes to it.
#include "encode_rows.hpp"
#include "io.hpp"
#include "launch.hpp"

namespace aq {

namespace {

constexpr int kTokWaves = 8;
constexpr int kMaxTokens = 64 * kTokWaves;  // one token a thread
constexpr int kStepThreads = kMaxTokens + 128;

template <int P>
__global__ __launch_bounds__(kStepThreads) void mirror_step_kernel(
    HeadDesc *const *item_desc, const void *__restrict__ kin, const void *__restrict__ vin,
    const void *__restrict__ qin, void *__restrict__ out, IoType io, int dim, int kb, int vb,
    float inv_sqrt_p, float sqrt_p) {
  constexpr int E = P / 64;
  static constexpr Q4Table kTab = q4_table();
  __shared__ Q4Cell s_q4[kQ4Cells];
  __shared__ __align__(16) float s_q[P], s_k[P], s_v[P];
  __shared__ __align__(16) float s_sq[2][P + 4];
  __shared__ float s_w[kMaxTokens];
  __shared__ float s_red[2][kTokWaves];
  __shared__ float s_part[kTokWaves][P];
  const int item = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  HeadDesc *d = item_desc[item];
  const RingState st = d->st;
  const int n0 = __builtin_amdgcn_readfirstlane(st.raw_count);  // mirror rows before the step
  // (the host plans at most kMaxTokens; a captured step's ring goes on growing with
  // the replays, which attend over the oldest kMaxTokens from then on)
  const int n = min(n0 + 1, kMaxTokens);
  const float *raw_k = d->raw_k, *raw_v = d->raw_v;
  // the step's rows and query as fp32 in LDS, zeros past dim
  const size_t row0 = (size_t)item * dim;
  for (int j = tid; j < 3 * P; j += kStepThreads) {
    const int which = j / P, i = j % P;
    const void *src = which == 0 ? qin : which == 1 ? kin : vin;
    (which == 0 ? s_q : which == 1 ? s_k : s_v)[i] = i < dim ? io_load(src, row0 + i, io) : 0.0f;
  }
  if (tid < kQ4Cells) s_q4[tid] = kTab.c[tid];
  __syncthreads();  // also: every thread holds the old ring state

  float e = 0.0f;
  if (wave < kTokWaves) {
    if (wave * 64 < n) {
      // the sequential dot of this thread's token (clamped past the end)
      const bool mine = tid == n0;
      const float *kr = raw_k + (size_t)min(tid, n0 > 0 ? n0 - 1 : 0) * dim;
      float acc = 0.0f;
      if (n0 == 0) {  // no mirror row to read
        for (int i = 0; i < dim; ++i) acc = __fadd_rn(acc, __fmul_rn(s_q[i], s_k[i]));
      } else if (dim % 4 == 0) {
#pragma unroll 4
        for (int i = 0; i < dim; i += 16) {
          float4 r[4];
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (i + 4 * k < dim) r[k] = *reinterpret_cast<const float4 *>(kr + i + 4 * k);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (i + 4 * k < dim) {
              const float4 nk = *reinterpret_cast<const float4 *>(s_k + i + 4 * k);
              const float4 q4 = *reinterpret_cast<const float4 *>(s_q + i + 4 * k);
              acc = __fadd_rn(acc, __fmul_rn(q4.x, mine ? nk.x : r[k].x));
              acc = __fadd_rn(acc, __fmul_rn(q4.y, mine ? nk.y : r[k].y));
              acc = __fadd_rn(acc, __fmul_rn(q4.z, mine ? nk.z : r[k].z));
              acc = __fadd_rn(acc, __fmul_rn(q4.w, mine ? nk.w : r[k].w));
            }
        }
      } else {
        for (int i = 0; i < dim; ++i)
          acc = __fadd_rn(acc, __fmul_rn(s_q[i], mine ? s_k[i] : kr[i]));
      }
      const float logit = tid < n ? __fmul_rn(acc, 1.0f / sqrtf((float)dim)) : -INFINITY;
      e = logit;
      float m = logit;
#pragma unroll
      for (int k = 32; k >= 1; k >>= 1) m = fmaxf(m, __shfl_xor(m, k, 64));
      if (lane == 0) s_red[0][wave] = m;
    } else if (lane == 0) {
      s_red[0][wave] = -INFINITY;
    }
  } else {
    const int side = wave - kTokWaves;
    encode_wide_rows<P, 1>(d, st, 1, 0, side == 0 ? s_k : s_v, dim, side, side == 0 ? kb : vb, lane,
                           inv_sqrt_p, sqrt_p, s_q4, s_sq[side]);
  }
  __syncthreads();
  // the reference seeds the maximum at -1e30 (attention.cpp:496)
  float M = -1e30f;
#pragma unroll
  for (int w = 0; w < kTokWaves; ++w) M = fmaxf(M, s_red[0][w]);
  if (wave < kTokWaves) {
    e = tid < n ? expf(e - M) : 0.0f;
    s_w[tid] = e;
    float l = e;
#pragma unroll
    for (int k = 32; k >= 1; k >>= 1) l += __shfl_xor(l, k, 64);
    if (lane == 0) s_red[1][wave] = l;
  }
  __syncthreads();
  if (wave < kTokWaves) {
    float acc[E];
#pragma unroll
    for (int x = 0; x < E; ++x) acc[x] = 0.0f;
    constexpr int U = 8;  // rows in flight a wave
    for (int t = wave; t < n; t += U * kTokWaves) {
      float r[U][E];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int tt = t + u * kTokWaves;
#pragma unroll
        for (int x = 0; x < E; ++x) {
          const int i = lane + 64 * x;
          r[u][x] = tt < n0 && i < dim ? raw_v[(size_t)tt * dim + i] : 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int tt = t + u * kTokWaves;
        if (tt < n) {
          const float w = s_w[tt];
#pragma unroll
          for (int x = 0; x < E; ++x)
            acc[x] = fmaf(tt == n0 ? s_v[lane + 64 * x] : r[u][x], w, acc[x]);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < E; ++x) s_part[wave][lane + 64 * x] = acc[x];
  }
  if (tid == 0) d->st = ring_after(st, 1, d->cap, d->hyb);
  __syncthreads();
  float L = 0.0f;
#pragma unroll
  for (int w = 0; w < kTokWaves; ++w) L += s_red[1][w];
  // a zero or non-finite sum normalises by 1/n (attention.cpp:513)
  const float inv = L > 0.0f && isfinite(L) ? 1.0f / L : 1.0f / (float)n;
  if (tid < dim) {
    float a = 0.0f;
#pragma unroll
    for (int w = 0; w < kTokWaves; ++w) a += s_part[w][tid];
    io_store(out, row0 + tid, io, a * inv);
  }
}

__global__ __launch_bounds__(256) void to_f32_kernel(float *d0, float *d1, float *d2,
                                                     const void *s0, const void *s1,
                                                     const void *s2, size_t n, IoType io) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float *dst = blockIdx.y == 0 ? d0 : blockIdx.y == 1 ? d1 : d2;
  const void *src = blockIdx.y == 0 ? s0 : blockIdx.y == 1 ? s1 : s2;
  dst[i] = io_load(src, i, io);
}

__global__ __launch_bounds__(256) void from_f32_kernel(void *dst, const float *src, size_t n,
                                                       IoType io) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) io_store(dst, i, io, src[i]);
}

}  // namespace

bool mirror_step_supported(int n_items, int padded, int n) {
  return n_items > 0 && n > 0 && n <= kMaxTokens &&
         (padded == 64 || padded == 128 || padded == 256);
}

hipError_t launch_mirror_step(HeadDesc *const *descs, int n_items, int padded, int k_bits,
                              int v_bits, int dim, const void *k, const void *v, const void *q,
                              void *out, IoType io, hipStream_t s) {
  const float sp = sqrtf((float)padded), isp = 1.0f / sp;
#define AQ_MIRROR(P_)                                                                            \
  if (padded == P_) {                                                                            \
    mirror_step_kernel<P_><<<n_items, kStepThreads, 0, s>>>(descs, k, v, q, out, io, dim, k_bits, \
                                                            v_bits, isp, sp);                    \
    return hipGetLastError();                                                                    \
  }
  AQ_MIRROR(64) AQ_MIRROR(128) AQ_MIRROR(256)
#undef AQ_MIRROR
  return hipErrorInvalidValue;
}

hipError_t launch_to_f32(float *const dst[3], const void *const src[3], int n_arrays, size_t n,
                         IoType io, hipStream_t s) {
  if (n == 0) return hipSuccess;
  to_f32_kernel<<<dim3((unsigned)((n + 255) / 256), (unsigned)n_arrays), 256, 0, s>>>(
      dst[0], dst[1], dst[2], src[0], src[1], src[2], n, io);
  return hipGetLastError();
}

hipError_t launch_from_f32(void *dst, const float *src, size_t n, IoType io, hipStream_t s) {
  if (n == 0) return hipSuccess;
  from_f32_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(dst, src, n, io);
  return hipGetLastError();
}

}  // namespace aq
