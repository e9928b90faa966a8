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
// A workgroup owns 16 NT rows of W and XR rows of x (16x16x32 products); its NW
// waves take the steps of K in turn, each through a ring of D tiles of its own and
// without a barrier. The sums of the waves meet in LDS.
//   What bounds it: W from memory (a kernel that only reads takes 7.0 us for 32 MB,
// 12.4 for 64, 47 for 256), and beside it the rows of x, which every workgroup
// fetches from L2: 24 of them weigh as much as 24 rows of W. So no more rows of x
// are loaded than there are (in steps of eight), and two row tiles of W share them
// where that leaves a workgroup for most CUs. Workgroups start at different
// steps, so that not all ask for the same columns of x at a time. Us, N x K, before
// (16 rows of W, 16 or 32 of x, one tile a wave) -> here:
//   M 8   4096 x 4096 8.7 -> 7.7, 6144 x 4096 12.7 -> 10.7, 8192 x 4096 14.9 -> 12.8
//   M 24  4096 x 4096 10.1 -> 9.1, 6144 x 4096 15.2 -> 12.4, 8192 x 4096 16.9 -> 14.3,
//         32000 x 4096 57 -> 48, 4096 x 14336 27.5 -> 25.3
//   M 64  4096 x 4096 14.4 -> 13.2, 6144 x 4096 22.0 -> 17.2, 8192 x 4096 23.5 -> 18.5
template <int NT, int XR, int NW, int D>
__global__ __launch_bounds__(NW * 64) void linear_stream_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias, const int M, const int N,
    const int K, const long x_stride) {
  constexpr int WR = 16 * NT;                    // rows of W
  constexpr int MT = (XR + 15) / 16;             // row tiles of x
  constexpr int T = WR * LN_K, TILE = T + XR * LN_K;
  constexpr int ROW = WR + 4;                    // fp32 of a part's row, padded
  constexpr int PART = NW * 16 * MT * ROW * 2;
  constexpr int RING = NW * D * TILE;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[RING > PART ? RING : PART];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const long n0 = blockIdx.x * (long)WR;
  unsigned short* wt = lds + wid * (D * TILE);
  LnTile<WR> lw;
  LnTile<XR> lx;
  lw.init(n0, N, K, lane);
  lx.init(0, M, x_stride, lane);
  const unsigned short* wp = w + n0 * K;
  // bytes of chunk 4 ks + g of row c16; a last tile of eight rows is read twice
  const unsigned base = (unsigned)(unsigned long long)(const lds_u16*)wt;
  const int half = XR % 16 != 0 ? c16 & 7 : c16;
  unsigned at[4], last[4];
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    at[ks] = 2 * (c16 * LN_K + (((4 * ks + g) ^ c16) << 3));
    last[ks] = 2 * (half * LN_K + (((4 * ks + g) ^ half) << 3));
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = K / LN_K, turn = blockIdx.x % steps;
  const int mine = (steps - wid + NW - 1) / NW;  // of this wave
  auto load = [&](int i, int slot) {
    int t = wid + i * NW + turn;
    t = (t >= steps ? t - steps : t) * LN_K;
    lw.load(wp + t, wt + slot * TILE);
    lx.load(x + t, wt + slot * TILE + T);
  };
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < mine) load(d, d);
  for (int i = 0, slot = 0; i < mine; i++, slot = slot + 1 == D ? 0 : slot + 1) {
    if (D == 2 && i + 1 < mine)                  // the next tile may be on the way
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((WR + XR) / 4) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    constexpr int TILES = NT + MT;               // row tiles of W, then of x
    bf16x8 v[TILES][4];
    auto rows = [&](int r, unsigned (&to)[4]) {
#pragma unroll
      for (int ks = 0; ks < 4; ks++)
        to[ks] = base + slot * (2 * TILE) + r * (2 * 16 * LN_K) +
                 (r == TILES - 1 ? last[ks] : at[ks]);
    };
    unsigned r0[4], r1[4];
#pragma unroll
    for (int r = 0; r + 1 < TILES; r += 2) {
      rows(r, r0);
      rows(r + 1, r1);
      ln_read2(r0, r1, v[r], v[r + 1]);
    }
    if constexpr (TILES % 2 != 0) {
      rows(TILES - 1, r0);
      ln_read(r0, v[TILES - 1]);
    }
    if (i + D < mine) load(i + D, slot);
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < MT; j++)
          acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              v[n][ks], v[NT + j][ks], acc[n][j], 0, 0, 0);
  }
  // acc[n][j][r] = y[m = 16 j + c16][16 n + 4 g + r]
  __syncthreads();
  float* part = reinterpret_cast<float*>(lds);   // [NW][16 MT][ROW]
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int j = 0; j < MT; j++)
      *reinterpret_cast<float4*>(part + ((wid * MT + j) * 16 + c16) * ROW +
                                 16 * n + 4 * g) =
          make_float4(acc[n][j][0], acc[n][j][1], acc[n][j][2], acc[n][j][3]);
  __syncthreads();
  constexpr int C4 = WR / 4;                     // columns in fours
  for (int i = tid; i < 16 * MT * C4; i += NW * 64) {
    const int m = i / C4, col = (i % C4) * 4;
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
//   M 8      2048 x 2048 4.1 | 8.9, 4096 x 4096 7.7 | 15.3, 4096 x 14336 21 | 25, 28672 x
//            4096 39 | 60, 32000 x 4096 44 | 57
//   M 16     32000 x 4096 48 | 57; 128256 x 4096, another kernel, 193 | 189
//   M 24-32  512 x 14336 20.4 | 18.1, 23.1 | 24.5; 4096 x 4096 9.1-10 | 13.2, 8192 x 4096
//            14.4-15 | 16, 14336 x 4096 24.5-26.1 | 25.6, 32000 x 4096 48.4-50.6 | 62;
//            12288 x 8192 45-46.5 | 41
//   M 48     4096 x 4096 11.8 | 13.6, 8192 x 4096 16.9 | 17.9, 14336 x 4096 28.4 | 26.2,
//            28672 x 4096 53 | 60, 14336 x 2048 16.4 | 16.8; 512 x 8192 12.7 | 9.7, 2048 x
//            8192 17.9 | 15.1, 6144 x 14336 47 | 52
//   M 64     4096 x 4096 13.2 | 14.9, 8192 x 4096 18.5 | 18.9, 12288 x 4096 31.4 | 24.7, 12288
//            x 2048 18.8 | 16.1; 1024 x 8192 20 | 13.6, 4096 x 8192 22.7 | 23.9, 6144 x
//            8192 30 | 29.3, 4096 x 14336 38.8 | 38.8
//   M 96-192 4096 x 2048 12 | 14-21, 4096 x 4096 20 | 21-31, 4096 x 14336 60-68
//            | 50-104 (tuned 50)
//   M 300    2048 x 2048 10.8 | 10.5, 4096 x 2048 16.6 | 15.7, 4096 x 4096 29 | 25
//   M 512    3072 x 2048 16.5 | 15.3, 4096 x 2048 17.6 | 17.1; M 1024 30 | 24
//   M 96-256, few tiles   512 x 4096 17.7 | 8.8-12, 1024 x 2048 10.5 | 8.4, 1536 x 3072
//            16 | 10.7, 2048 x 4096 18.8-20.4 | 12.8-15.9, 2560 x 4096 19 | 13; 1024 x
//            1024 and 3072 x 4096 are still faster here
// With a bias the library chooses among other kernels, which are faster from 65 rows
// on, here | library: 96 x 2048 x 2048 11.8 | 6.9, 128 x 2048 x 1536 9.9 | 6.3, 300 x
// 4096 x 2048 16.1 | 13.6, 96 x 4608 x 3584 18.2 | 16.5, 512 x 3072 x 2048 16.5 | 13.6.
// A tuned choice of the library is preferred above 48 rows, above 32 where N > 8192
// (linear in bindings.cpp): M 32, 28672 x 4096 48.9 | 48.2, M 48 53.5 | 49.3 | 60.5 not,
//   4096 x 4096, here | tuned | not   M 48 11.8 | 13.7 | 13.7, 64 13.2 | 13.6 | 15.1,
//            96 19.6 | 17.2 | 22.0, 128 21.4 | 16.9 | 24.5
int linear_takes(long M, long N, long K, bool bias) {
  if (M <= 0 || K < LN_K || K % LN_K != 0 || N % 8 != 0) return 0;
  if (N * K >= (1L << 31) || M * K >= (1L << 30)) return 0;
  if (M <= 16) return M <= 8 || N * K <= 1L << 28 ? 1 : 0;
  // few workgroups with long rows
  if (M <= 32)
    return (N > 1024 || K <= 8192) &&
           (N <= 8192 || (K <= 4096 && N * K <= 1L << 28)) ? 1 : 0;
  if (M <= 48)
    return N <= 8192 ? (N > 2048 || K < 8192 ? 1 : 0)
                     : N * K <= 1L << 28 &&
                       (K <= 2048 || (K <= 4096 && N >= 18432)) ? 1 : 0;
  if (M <= 64)
    return N <= 8192 && (K <= 4096 || (N >= 2048 && N <= 4096 && K <= 8192)) ? 1 : 0;
  if (bias) return 0;
  const long tiles = ((M + 63) / 64) * ((N + 63) / 64);
  // few tiles with long rows leave most of the chip waiting for their chain
  if (tiles <= 128 && ((K > 2048 && N < 3072) || (K > 1024 && N < 2048))) return 0;
  return K <= 4096 && (tiles <= 256 || (tiles <= 512 && K <= 2048)) ? 2 : 0;
}

// Row tiles of W: one up to 4096 rows of it, one workgroup a CU then; two above.
// Up to 16 rows of x weigh little, and where W has many columns and its row
// tiles leave few CUs without one in the last turn, one tile is the better again:
// M 8, 8192 x 4096 12.8 one | 13.5 two, 12288 x 4096 17.9 | 19.9, 8192 x 8192 26.2 |
// 29.8; but 4608 x 4096 10.5 | 9.4 (a ninth of the CUs have two), 14336 x 4096
// 22.2 | 21.1, 8192 x 2048 9.1 | 8.0; M 24, 8192 x 4096 15.6 | 14.4.
static bool linear_one_tile(int M, int N, int K) {
  const int wgs = (N + 15) / 16;
  return wgs <= 256 ||
         (M <= 16 && K >= 4096 && 10 * wgs >= 9 * ((wgs + 255) / 256 * 256));
}
// A workgroup that has a CU to itself takes all of its LDS: two tiles a wave, or
// more waves. Where there are more than CUs, two of them share one: M 24, 32000 x
// 4096 48.4, with two tiles 49.2; 18944 x 4096 33.4 | 34.5.
static void launch_stream(unsigned short* y, const unsigned short* x,
                          const unsigned short* w, const unsigned short* bias,
                          int M, int N, int K, long x_stride,
                          hipStream_t stream) {
  const bool one = linear_one_tile(M, N, K);
  const dim3 grid((N + (one ? 15 : 31)) / (one ? 16 : 32));
  const bool few = grid.x <= 256;
#define LN_STREAM(NT, XR, NW, D)                                               \
  hipLaunchKernelGGL((linear_stream_kernel<NT, XR, NW, D>), grid,              \
                     dim3(NW * 64), 0, stream, y, x, w, bias, M, N, K, x_stride)
  if (one) {
    if (M <= 8) LN_STREAM(1, 8, 4, 2);
    else if (M <= 16) LN_STREAM(1, 16, 4, 2);
    else if (M <= 24) LN_STREAM(1, 24, 4, 2);
    else if (M <= 32) LN_STREAM(1, 32, 4, 2);
    else if (M <= 48) LN_STREAM(1, 48, 4, 2);
    else LN_STREAM(1, 64, 4, 2);
  } else {
    if (M <= 8) LN_STREAM(2, 8, 4, 2);
    else if (M <= 16) { if (few) LN_STREAM(2, 16, 4, 2); else LN_STREAM(2, 16, 2, 2); }
    else if (M <= 24) { if (few) LN_STREAM(2, 24, 4, 2); else LN_STREAM(2, 24, 4, 1); }
    else if (M <= 32) { if (few) LN_STREAM(2, 32, 4, 2); else LN_STREAM(2, 32, 4, 1); }
    else if (M <= 48) { if (few) LN_STREAM(2, 48, 7, 1); else LN_STREAM(2, 48, 4, 1); }
    else LN_STREAM(2, 64, 6, 1);
  }
#undef LN_STREAM
}

void launch_linear(unsigned short* y, const unsigned short* x,
                   const unsigned short* w, const unsigned short* bias, int M,
                   int N, int K, long x_stride, int kind, hipStream_t stream) {
  if (kind == 1) {
    launch_stream(y, x, w, bias, M, N, K, x_stride, stream);
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
