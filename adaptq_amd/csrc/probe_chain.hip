// probe_chain.hip -- the arithmetic that the many-query decode rests on
// (mquery.hip): a chain of v_mfma_f32_16x16x4 against the chain of fmaf that it
// stands for (in the same library as probe_rows.hip; never part of
// libadaptq.so).
//
// One wave per problem: D = C + A B with A [16][K], B [K][16], C and D [16][16],
// K a multiple of 4, k ascending.  Operand layouts as in mquery.hip: lane l
// supplies A[l % 16][k + l / 16] and B[k + l / 16][l % 16], register r of lane l
// is D[4 (l / 16) + r][l % 16].
#include <hip/hip_runtime.h>

namespace aq {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(64) void probe_chain_kernel(const float *a, const float *b,
                                                         const float *c, float *d_mfma,
                                                         float *d_fmaf, int K) {
  const int l = threadIdx.x, col = l & 15, g = l >> 4;
  const size_t i = blockIdx.x;
  a += i * 16 * K;
  b += i * 16 * K;
  f32x4 acc, ref;
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = ref[r] = c[i * 256 + (4 * g + r) * 16 + col];
  for (int k = 0; k < K; k += 4)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[col * K + k + g], b[(k + g) * 16 + col], acc, 0,
                                               0, 0);
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) ref[r] = fmaf(a[(4 * g + r) * K + k], b[k * 16 + col], ref[r]);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    d_mfma[i * 256 + (4 * g + r) * 16 + col] = acc[r];
    d_fmaf[i * 256 + (4 * g + r) * 16 + col] = ref[r];
  }
}

}  // namespace
}  // namespace aq

// n problems of K: a and b hold n * 16 * K floats, c, d_mfma and d_fmaf n * 256
// (device memory).  Returns 0, or -1 for arguments outside these (nothing
// launched), or the HIP error.
extern "C" int adaptq_probe_chain(const float *a, const float *b, const float *c, float *d_mfma,
                                  float *d_fmaf, int n, int K, void *stream) {
  if (n <= 0 || n > 1 << 20 || K <= 0 || K > 4096 || K % 4 != 0 || !a || !b || !c || !d_mfma ||
      !d_fmaf)
    return -1;
  aq::probe_chain_kernel<<<n, 64, 0, (hipStream_t)stream>>>(a, b, c, d_mfma, d_fmaf, K);
  return (int)hipGetLastError();
}
