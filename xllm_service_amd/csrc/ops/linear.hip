// y = x W^T (+ bias) in bf16 for the row counts of serving steps: decode batches
// and short prompts. Longer ones stay with the library (rule and measurements
// at linear_takes).
//
// W [N, K] and x [M, K] both have their contraction index innermost, so tiles of
// both are rows x 128 entries, loaded straight to LDS (global_load_lds, 16 B per
// lane, 256 B of a row at a time) with the 16 B chunks of a row permuted by the
// row: whole-row reads then meet no bank twice. W rows are the A operand, x rows
// the B operand of 32x32x16 products (layouts: mfma_rows.h); sums are fp32.
//
// The LDS reads are asm with their wait: in front of a builtin the compiler
// waits for every load to LDS in flight.
#include "mfma_rows.h"

namespace xllm {

#define LN_K 128           // entries of a row per step

// bytes into a [rows][128] image of chunk 2 ks + h of a lane's row
XLLM_DEV void ln_addresses(unsigned base, int row, int h, unsigned (&at)[8]) {
#pragma unroll
  for (int ks = 0; ks < 8; ks++)
    at[ks] = base + 2 * (row * LN_K + (((2 * ks + h) ^ (row & 15)) << 3));
}
// four steps of 32 rows
XLLM_DEV void ln_read(const unsigned* at, bf16x8* v) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
      "ds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
      : "memory");
}
XLLM_DEV void ln_read2(const unsigned* a, const unsigned* b, bf16x8* v,
                       bf16x8* u) {
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %4, %12\n\t"
      "ds_read_b128 %1, %9\n\tds_read_b128 %5, %13\n\t"
      "ds_read_b128 %2, %10\n\tds_read_b128 %6, %14\n\t"
      "ds_read_b128 %3, %11\n\tds_read_b128 %7, %15\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(u[0]),
        "=&v"(u[1]), "=&v"(u[2]), "=&v"(u[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]),
        "v"(b[2]), "v"(b[3])
      : "memory");
}

// Rows r0 .. of a matrix into an image: instruction i moves four rows
template <int ROWS>
struct LnTile {
  static constexpr int NI = ROWS / 4;
  unsigned off[NI];        // bytes from the matrix' start, but for the step
  // rows past the last one repeat it: their results go nowhere
  XLLM_DEV void init(long first, long rows, long stride, int lane) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int r = i * 4 + (lane >> 4);
      const long row = min(first + r, rows - 1) - first;
      off[i] = (unsigned)(row * stride * 2 +
                          (((lane & 15) ^ (r & 15)) << 4));
    }
  }
  XLLM_DEV void load(const unsigned short* p, unsigned short* dst) const {
#pragma unroll
    for (int i = 0; i < NI; i++)
      __builtin_amdgcn_global_load_lds(
          (glb_void*)(reinterpret_cast<const char*>(p) + off[i]),
          (lds_void*)(dst + i * 512), 16, 0, 0);
  }
};

// ---- decode batches: a stream over W -------------------------------------------
// A workgroup owns 16 rows of W and up to 16 MT rows of x (16x16x32 products);
// its NW waves take the steps of K in turn, each through tiles of its own and
// without a barrier. The sums of the waves meet in LDS. Sixteen rows and not
// more, because the projections of a layer have few thousand of them: N = 4096
// fills the 256 CUs once, and what a CU moves besides W, the rows of x, comes
// from L2.
template <int MT, int NW>
__global__ __launch_bounds__(NW * 64) void linear_stream_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias, const int M, const int N,
    const int K, const long x_stride) {
  constexpr int T = 16 * LN_K, TILE = T * (1 + MT);
  constexpr int ROW = 20;                        // fp32 of a part's row, padded
  constexpr int PART = NW * 16 * MT * ROW * 2;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[NW * TILE > PART ? NW * TILE : PART];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const long n0 = blockIdx.x * 16L;
  unsigned short* wt = lds + wid * TILE;
  unsigned short* xt = wt + T;
  LnTile<16> lw;
  LnTile<16 * MT> lx;
  lw.init(n0, N, K, lane);
  lx.init(0, M, x_stride, lane);
  const unsigned short* wp = w + n0 * K;
  unsigned at[4];                                // chunk 4 ks + g of row c16
#pragma unroll
  for (int ks = 0; ks < 4; ks++)
    at[ks] = (unsigned)(unsigned long long)(const lds_u16*)wt +
             2 * (c16 * LN_K + (((4 * ks + g) ^ c16) << 3));
  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = K / LN_K;
  if (wid < steps) {
    lw.load(wp + wid * LN_K, wt);
    lx.load(x + wid * LN_K, xt);
  }
  for (int t = wid; t < steps; t += NW) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bf16x8 a[4], b[MT][4];
    unsigned xat[MT][4];
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int ks = 0; ks < 4; ks++) xat[j][ks] = at[ks] + (1 + j) * (2 * T);
    ln_read2(at, xat[0], a, b[0]);
    if (t + NW < steps) lw.load(wp + (t + NW) * LN_K, wt);
#pragma unroll
    for (int j = 1; j < MT; j++) ln_read(xat[j], b[j]);
    if (t + NW < steps) lx.load(x + (t + NW) * LN_K, xt);
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
      for (int j = 0; j < MT; j++)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks], b[j][ks],
                                                         acc[j], 0, 0, 0);
  }
  // acc[j][r] = y[m = 16 j + c16][n = 4 g + r]
  __syncthreads();
  float* part = reinterpret_cast<float*>(lds);   // [NW][16 MT][ROW]
#pragma unroll
  for (int j = 0; j < MT; j++)
    *reinterpret_cast<float4*>(part + ((wid * MT + j) * 16 + c16) * ROW +
                               4 * g) =
        make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
  __syncthreads();
  for (int i = tid; i < 16 * MT * 4; i += NW * 64) {
    const int m = i >> 2, col = (i & 3) * 4;
    const long n = n0 + col;
    if (m >= M || n >= N) continue;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < NW; k++) {
      const float4 z = *reinterpret_cast<const float4*>(
          part + (k * 16 * MT + m) * ROW + col);
      s[0] += z.x; s[1] += z.y; s[2] += z.z; s[3] += z.w;
    }
    if (bias != nullptr) {
#pragma unroll
      for (int k = 0; k < 4; k++) s[k] += bf16_to_f32(bias[n + k]);
    }
    uint2 o;
    o.x = pack_bf16(s[0], s[1]);
    o.y = pack_bf16(s[2], s[3]);
    *reinterpret_cast<uint2*>(y + (long)m * N + n) = o;
  }
}

// ---- short prompts: 64 x 64 tiles -----------------------------------------------
// Four waves, a quarter of the tile each; one barrier per step. S buffers: four
// where a workgroup has a CU to itself (three steps are on the way while one
// is multiplied: 300 x 2048 x 2048 10.8 us, with two 11.8), two where two share
// it (300 x 4096 x 2048 16.6 us, with four 21.6). Bound by the chain of a step:
// LDS reads, their wait, four products on one accumulator.
template <int S>
__global__ __launch_bounds__(256, S == 4 ? 1 : 2) void linear_tile_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, const int M, const int N,
    const int K, const long x_stride, const int n_tiles_n) {
  constexpr int HALF = 64 * LN_K, TILE = 2 * HALF;
  __shared__ __attribute__((aligned(1024))) unsigned short lds[S * TILE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;
  const long n0 = (blockIdx.x % n_tiles_n) * 64L;
  const long m0 = (blockIdx.x / n_tiles_n) * 64L;
  const int wn = wid & 1, wm = wid >> 1;
  // a wave loads 16 rows of both
  LnTile<16> lw, lx;
  const long nr = min(n0 + wid * 16, (long)N - 1);
  const long mr = min(m0 + wid * 16, (long)M - 1);
  lw.init(nr, N, K, lane);
  lx.init(mr, M, x_stride, lane);
  const unsigned short* wp = w + nr * K;
  const unsigned short* xp = x + mr * x_stride;
  unsigned short* mine = lds + wid * 16 * LN_K;
  unsigned wat[8], xat[8];
  const unsigned base = (unsigned)(unsigned long long)(const lds_u16*)lds;
  ln_addresses(base, wn * 32 + c32, h, wat);
  ln_addresses(base + 2 * HALF, wm * 32 + c32, h, xat);
  f32x16 acc = mr_zero();
  const int steps = K / LN_K;
  auto stage = [&](int t) {                      // eight loads
    unsigned short* dst = mine + (t & (S - 1)) * TILE;
    lw.load(wp + t * LN_K, dst);
    lx.load(xp + t * LN_K, dst + HALF);
  };
  for (int t = 0; t < min(S - 1, steps); t++) stage(t);
  for (int t = 0; t < steps; t++) {
    const int buf = t & (S - 1);
    // this step has arrived; what was issued later may be on the way
    if (S == 4 && t + 2 < steps)
      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else if (S == 4 && t + 1 < steps)
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t + S - 1 < steps) stage(t + S - 1);
#pragma unroll
    for (int k = 0; k < 8; k += 4) {
      unsigned a_at[4], b_at[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        a_at[i] = wat[k + i] + buf * (2 * TILE);
        b_at[i] = xat[k + i] + buf * (2 * TILE);
      }
      bf16x8 a[4], b[4];
      ln_read2(a_at, b_at, a, b);
#pragma unroll
      for (int i = 0; i < 4; i++) acc = mr_mma(a[i], b[i], acc);
    }
  }
  // through LDS to whole rows
  __syncthreads();
  constexpr int ROW = 64 + 8;                    // bf16 of a row, padded
#pragma unroll
  for (int r = 0; r < 16; r += 4) {
    uint2 o;
    o.x = pack_bf16(acc[r], acc[r + 1]);
    o.y = pack_bf16(acc[r + 2], acc[r + 3]);
    *reinterpret_cast<uint2*>(lds + (wm * 32 + c32) * ROW + wn * 32 + 2 * r +
                              4 * h) = o;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int idx = tid + i * 256, row = idx >> 3, col = (idx & 7) * 8;
    if (m0 + row < M && n0 + col < N)
      *reinterpret_cast<uint4*>(y + (m0 + row) * N + n0 + col) =
          *reinterpret_cast<const uint4*>(lds + row * ROW + col);
  }
}

// 0: the library's; 1: stream; 2: tiles. Besides its time on the GPU a library
// call costs 28 us of host time (its choice of a kernel), these cost 6.
// Measured, us on the GPU, here | library, weights from memory (N x K):
//   M 1-8    2048 x 2048 4.2 | 8.3, 4096 x 4096 8.5 | 14.5, 8192 x 4096 15.1 |
//            17, 4096 x 14336 24 | 26, 28672 x 4096 42 | 61, 32000 x 4096 46 | 58
//   M 24-32  2048 x 2048 5.0 | 8.6, 4096 x 4096 10.5 | 12.7, 6144 x 4096 16.5 |
//            16, 8192 x 4096 19 | 17.5: x rows weigh as much as W from here on
//   M 64     4096 x 2048 9.9 | 12.4, 4096 x 4096 14.2 | 14.6, 6144 x 4096 22 | 18
//   M 96-192 4096 x 2048 12 | 14-21, 4096 x 4096 20 | 21-31, 4096 x 14336 60-68
//            | 50-104 (tuned 50)
//   M 300    2048 x 2048 10.8 | 10.5, 4096 x 2048 16.6 | 15.7, 4096 x 4096 29 | 25
//   M 512    3072 x 2048 16.5 | 15.3, 4096 x 2048 17.6 | 17.1; M 1024 30 | 24
//   M 96-256, few tiles   512 x 4096 17.7 | 8.8-12, 1024 x 2048 10.5 | 8.4, 1536 x 3072
//            16 | 10.7, 2048 x 4096 18.8-20.4 | 12.8-15.9, 2560 x 4096 19 | 13; 1024 x
//            1024 and 3072 x 4096 are still faster here
//   M 16     32000 x 4096 as above, 128256 x 4096 193 | 189 (tuned 178); 8 177 | 188
// With a bias the library chooses among other kernels, which are faster from 65 rows
// on, here | library: 96 x 2048 x 2048 11.8 | 6.9, 128 x 2048 x 1536 9.9 | 6.3, 300 x
// 4096 x 2048 16.1 | 13.6, 96 x 4608 x 3584 18.2 | 16.5, 512 x 3072 x 2048 16.5 | 13.6.
// A tuned choice of the library is preferred above 48 rows (linear in bindings.cpp):
//   4096 x 4096, here | tuned | not   M 48 12.6 | 13.7 | 13.7, 64 14.5 | 13.6 | 15.1,
//            96 19.6 | 17.2 | 22.0, 128 21.4 | 16.9 | 24.5
int linear_takes(long M, long N, long K, bool bias) {
  if (M <= 0 || K < LN_K || K % LN_K != 0 || N % 8 != 0) return 0;
  if (N * K >= (1L << 31) || M * K >= (1L << 30)) return 0;
  if (M <= 16) return M <= 8 || N * K <= 1L << 28 ? 1 : 0;
  if (M <= 64) return N * K <= 4096L * 4096 ? 1 : 0;
  if (bias) return 0;
  const long tiles = ((M + 63) / 64) * ((N + 63) / 64);
  // few tiles with long rows leave most of the chip waiting for their chain
  if (tiles <= 128 && ((K > 2048 && N < 3072) || (K > 1024 && N < 2048))) return 0;
  return K <= 4096 && (tiles <= 256 || (tiles <= 512 && K <= 2048)) ? 2 : 0;
}

void launch_linear(unsigned short* y, const unsigned short* x,
                   const unsigned short* w, const unsigned short* bias, int M,
                   int N, int K, long x_stride, int kind, hipStream_t stream) {
  if (kind == 1) {
    const dim3 grid((N + 15) / 16);
    const bool few = grid.x <= 256;              // a CU each
#define LN_STREAM(MT, NW)                                                      \
  hipLaunchKernelGGL((linear_stream_kernel<MT, NW>), grid, dim3(NW * 64), 0,   \
                     stream, y, x, w, bias, M, N, K, x_stride)
    if (M <= 16) LN_STREAM(1, 8);
    else if (M <= 32) { if (few) LN_STREAM(2, 8); else LN_STREAM(2, 4); }
    else if (M <= 48) { if (few) LN_STREAM(3, 8); else LN_STREAM(3, 4); }
    else LN_STREAM(4, 4);
#undef LN_STREAM
    return;
  }
  const int tn = (N + 63) / 64, tm = (M + 63) / 64;
  if (tn * tm <= 256)
    hipLaunchKernelGGL((linear_tile_kernel<4>), dim3(tn * tm), dim3(256), 0,
                       stream, y, x, w, M, N, K, x_stride, tn);
  else
    hipLaunchKernelGGL((linear_tile_kernel<2>), dim3(tn * tm), dim3(256), 0,
                       stream, y, x, w, M, N, K, x_stride, tn);
}

}  // namespace xllm
