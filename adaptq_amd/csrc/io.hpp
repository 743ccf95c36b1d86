// io.hpp -- rows of fp32, fp16 or bf16 values, read as fp32 and written rounded
// to nearest even.
#pragma once

#include "launch.hpp"

namespace aq {

__device__ __forceinline__ float io_load(const void *p, size_t i, IoType io) {
  if (io == IoType::F32) return static_cast<const float *>(p)[i];
  if (io == IoType::F16) return (float)static_cast<const _Float16 *>(p)[i];
  return __uint_as_float((uint32_t)static_cast<const uint16_t *>(p)[i] << 16);
}

__device__ __forceinline__ void io_store(void *p, size_t i, IoType io, float v) {
  if (io == IoType::F32) {
    static_cast<float *>(p)[i] = v;
  } else if (io == IoType::F16) {
    static_cast<_Float16 *>(p)[i] = (_Float16)v;
  } else {
    const uint32_t b = __float_as_uint(v);
    static_cast<uint16_t *>(p)[i] =
        v != v ? 0x7FC0u : (uint16_t)((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
  }
}

}  // namespace aq
