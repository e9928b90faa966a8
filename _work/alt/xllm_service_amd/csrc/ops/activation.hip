// Fused activation kernels (SwiGLU / GEGLU) for MI355X (gfx950).
//
// out[t, i] = act(x[t, i]) * x[t, I + i] — one fused pass, 16 B per lane. The
// lanes are dealt through the rows without gaps, whatever I is: a row of
// workgroups per token leaves lanes idle where I is not a multiple of 2048. The
// division by the row length is a product with a fixed reciprocal.
// Us, 64-bit divisions in a fixed grid | a row of workgroups per token | here:
// 300 x 1408 2.10 | 2.23 | 2.02, 1024 x 2816 4.20 | 4.69 | 3.94, 8192 x 512 5.25 |
// 6.00 | 4.92, 8192 x 2816 21.8 | 24.0 | 20.5, 8192 x 14336 137 | 122 | 123 (5.7
// TB/s); 300 x 14336 5.49 | 5.10 | 5.21.
#include "common.h"

namespace xllm {

struct ActRows {           // v / per_row for v < 2^31
  unsigned per_row, mul;
  int shift;
};

template <bool GELU>
__global__ __launch_bounds__(256) void act_and_mul_kernel(
    unsigned short* __restrict__ out,      // [T, I]
    const unsigned short* __restrict__ x,  // [T, 2*I]
    const int I, const unsigned total, const ActRows rows) {
  const unsigned v = blockIdx.x * 256u + threadIdx.x;
  if (v < total) {
    const unsigned q = (unsigned)(((unsigned long long)v * rows.mul) >>
                                  rows.shift);
    const long row = q;
    const int col = (int)(v - q * rows.per_row) * 8;
    ushort8_t g = *reinterpret_cast<const ushort8_t*>(x + row * 2 * I + col);
    ushort8_t u = *reinterpret_cast<const ushort8_t*>(x + row * 2 * I + I + col);
    ushort8_t r;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float gf = bf16_to_f32(g.x[j]);
      float uf = bf16_to_f32(u.x[j]);
      float a;
      if constexpr (GELU) {
        float t = tanhf(0.7978845608028654f * (gf + 0.044715f * gf * gf * gf));
        a = 0.5f * gf * (1.0f + t);
      } else {
        a = gf / (1.0f + __expf(-gf));
      }
      r.x[j] = f32_to_bf16(a * uf);
    }
    *reinterpret_cast<ushort8_t*>(out + row * I + col) = r;
  }
}

template <bool GELU>
static void act_launch(unsigned short* out, const unsigned short* x, int T,
                       int I, hipStream_t stream) {
  if (T <= 0 || I < 8) return;
  const unsigned per_row = I / 8;
  // 2^(31 + l) / per_row rounded up, l bits hold per_row - 1: exact below 2^31
  int l = 0;
  while ((1L << l) < per_row) l++;
  const ActRows rows = {per_row,
                        (unsigned)((1ULL << (31 + l)) / per_row + 1), 31 + l};
  const int most = (int)((1L << 30) / per_row);      // rows of one launch
  for (long t = 0; t < T; t += most) {
    const unsigned total = (unsigned)(T - t < most ? T - t : most) * per_row;
    hipLaunchKernelGGL((act_and_mul_kernel<GELU>), dim3((total + 255) / 256),
                       dim3(256), 0, stream, out + t * I,
                       x + t * 2 * I, I, total, rows);
  }
}

void launch_silu_and_mul(unsigned short* out, const unsigned short* x, int T,
                         int I, hipStream_t stream) {
  act_launch<false>(out, x, T, I, stream);
}

void launch_gelu_and_mul(unsigned short* out, const unsigned short* x, int T,
                         int I, hipStream_t stream) {
  act_launch<true>(out, x, T, I, stream);
}

}  // namespace xllm
