// Common device helpers for the MI355X (gfx950 / CDNA4) kernels.
//
// Design notes:
//  * wavefront = 64 lanes; all block sizes are multiples of 64
//  * bf16 global loads are vectorized as ushort4/ushort8 (8-16 B per lane)
//  * fp32 accumulation everywhere; bf16 storage
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#define XLLM_WAVE 64
#define XLLM_DEV __device__ __forceinline__

namespace xllm {

using bf16 = __hip_bfloat16;

// ---- vector types for wide loads -------------------------------------------------
struct alignas(8) ushort4_t { unsigned short x[4]; };
struct alignas(16) ushort8_t { unsigned short x[8]; };
struct alignas(16) float4_t { float x[4]; };

XLLM_DEV float bf16_to_f32(unsigned short u) {
  union { float f; unsigned int i; } c;
  c.i = ((unsigned int)u) << 16;
  return c.f;
}

XLLM_DEV unsigned short f32_to_bf16(float f) {
  union { float f; unsigned int i; } c;
  c.f = f;
  // round-to-nearest-even
  unsigned int lsb = (c.i >> 16) & 1;
  c.i += 0x7fff + lsb;
  return (unsigned short)(c.i >> 16);
}

// ---- wave reductions -------------------------------------------------------------
XLLM_DEV float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

XLLM_DEV float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Reduce within a contiguous group of `W` lanes (W a power of two <= 64).
template <int W>
XLLM_DEV float group_reduce_sum(float v) {
#pragma unroll
  for (int off = W / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ---- block reduction through LDS (for 256-thread blocks = 4 waves) ---------------
// `tmp` must have >= blockDim.x / 64 floats.
XLLM_DEV float block_reduce_sum(float v, float* tmp) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  v = wave_reduce_sum(v);
  if (lane == 0) tmp[wid] = v;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  v = (threadIdx.x < nw) ? tmp[threadIdx.x] : 0.0f;
  if (wid == 0) {
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  }
  if (threadIdx.x == 0) tmp[0] = v;
  __syncthreads();
  return tmp[0];
}

// tanh below 1/2: the odd Taylor series up to x^15 (the next term is under 2^-26 of
// the value)
XLLM_DEV float tanh_near(float v) {
  const float w = v * v;
  float y = fmaf(w, -929569.0f / 638512875.0f, 21844.0f / 6081075.0f);
  y = fmaf(y, w, -1382.0f / 155925.0f);
  y = fmaf(y, w, 62.0f / 2835.0f);
  y = fmaf(y, w, -17.0f / 315.0f);
  y = fmaf(y, w, 2.0f / 15.0f);
  y = fmaf(y, w, -1.0f / 3.0f);
  return fmaf(y * w, v, v);
}
// 1 - 2 / (e^2x + 1): from 1/2 on; a NaN stays one
XLLM_DEV float tanh_far(float v) {
  const float e = __expf(2.0f * (v > 15.0f ? 15.0f : v));
  return 1.0f - 2.0f / (e + 1.0f);
}

}  // namespace xllm
