// y = x W^T (+ bias) in bf16 for the row counts of serving steps: decode batches
// and short prompts. Longer ones stay with the library (rule and measurements
// at linear_takes).
//
// W [N, K] and x [M, K] both have their contraction index innermost, so tiles of
// both are rows x 128 entries, loaded straight to LDS (global_load_lds, 16 B per
// lane, 256 B of a row at a time) with the 16 B chunks of a row permuted by the
// row: whole-row reads then meet no bank twice. W rows are the A operand, x rows
// the B operand of 16x16x32 products; sums are fp32.
#include <stdexcept>

#include "linear.h"
#include "mfma_rows.h"

namespace xllm {

#define LN_K 128           // entries of a row per step

// Four chunks of a lane's row, with their wait in the same asm: after loads to LDS through
// global addresses the compiler waits for more than it has to.
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

// Gated products: W = [gates | ups] by rows, half of each, and a tile of ROWS rows has
// as many of both. Row of the matrix that row r of the tile from gate `first` on is;
// rows past the last one repeat it
template <int ROWS>
XLLM_DEV long ln_gate_row(long first, long half, int r) {
  return r < ROWS / 2 ? min(first + r, half - 1)
                      : half + min(first + r - ROWS / 2, half - 1);
}
// Rotated products: a tile of ROWS rows has ROWS / 2 of the first half of a head and
// their partners of the other one. Its first row, and row r of it from there
template <int ROWS> XLLM_DEV int ln_rope_first(int tile) {
  constexpr int TILES = LN_HEAD / ROWS;          // of a head
  return tile / TILES * LN_HEAD + tile % TILES * (ROWS / 2);
}
template <int ROWS> XLLM_DEV int ln_rope_row(int r) {
  return r < ROWS / 2 ? r : LN_HEAD / 2 + r - ROWS / 2;
}
// what becomes of row m of the columns from `first` on: the columns' place, null for
// none, in a query, a key or a value
struct LnRope {
  long pos, slot;
  XLLM_DEV void init(const LinearEnds& e, long m, bool ok) {
    pos = ok ? e.positions[m] : 0;
    slot = ok ? e.slots[m] : -1;
  }
  XLLM_DEV unsigned short* place(const LinearEnds& e, unsigned short* y, long m,
                                 int first) const {
    const int h = first / LN_HEAD, at = first % LN_HEAD;
    if (h < e.n_q) return y + (m * e.n_q + h) * LN_HEAD + at;
    if (slot < 0) return nullptr;
    const long blk = slot >> 31 == 0 ? (unsigned)slot / (unsigned)e.block
                                     : slot / e.block;
    const bool val = h >= e.n_q + e.n_kv;
    return (val ? e.v_cache : e.k_cache) +
           ((blk * e.n_kv + h - e.n_q - (val ? e.n_kv : 0)) * e.block +
            (slot - blk * e.block)) * LN_HEAD + at;
  }
  // cos and sin of four columns' pairs
  XLLM_DEV void angles(const LinearEnds& e, int first, float4& c, float4& s) const {
    const float* p = e.cos_sin + pos * LN_HEAD + first % LN_HEAD;
    c = make_float4(1.f, 1.f, 1.f, 1.f);
    s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (first / LN_HEAD >= e.n_q + e.n_kv) return;   // values stay
    c = *reinterpret_cast<const float4*>(p);
    s = *reinterpret_cast<const float4*>(p + LN_HEAD / 2);
  }
};
// four pairs
XLLM_DEV void ln_turn(float* a, float* b, const float4& c, const float4& s) {
  const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float x = a[e], y = b[e];
    a[e] = x * cc[e] - y * ss[e];
    b[e] = y * cc[e] + x * ss[e];
  }
}
// silu(gate) up of two sums
XLLM_DEV float ln_gated(float gate, float up) {
  return gate / (1.0f + __expf(-gate)) * up;
}

// two neighbours: joined with the residual's, their squares added to sq
XLLM_DEV unsigned ln_join(float a, float b, unsigned& r, unsigned w, float& sq) {
  a += __uint_as_float(r << 16);
  b += __uint_as_float(r & 0xffff0000u);
  sq += a * a + b * b;
  r = pack_bf16(a, b);
  return pack_bf16(a * __uint_as_float(w << 16),
                   b * __uint_as_float(w & 0xffff0000u));
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
  // the first half of the rows from `first` on, the other half as many rows further
  // on as there are in a half of the matrix
  XLLM_DEV void init_gate(long first, long half, long stride, int lane) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int r = i * 4 + (lane >> 4);
      const long row = ln_gate_row<ROWS>(first, half, r) - first;
      off[i] = (unsigned)(row * stride * 2 +
                          (((lane & 15) ^ (r & 15)) << 4));
    }
  }
  XLLM_DEV void init_rope(long stride, int lane) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int r = i * 4 + (lane >> 4);
      off[i] = (unsigned)(ln_rope_row<ROWS>(r) * stride * 2 +
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
template <int NT, int XR, int NW, int D, int MODE>
__global__ __launch_bounds__(NW * 64) void linear_stream_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias, const int M, const int N,
    const int K, const long x_stride, const unsigned turns,
    const LinearEnds ends) {
  constexpr bool GATE = MODE & LN_GATE, SCALE = MODE & LN_SCALE,
                 ADD = MODE & LN_ADD, ROPE = MODE & LN_ROPE;
  constexpr bool PAIR = GATE || ROPE;            // two rows of W to a column
  constexpr int WR = 16 * NT;                    // rows of W
  constexpr int MT = (XR + 15) / 16;             // row tiles of x
  constexpr int T = WR * LN_K, TILE = T + XR * LN_K;
  constexpr int ROW = WR + 4;                    // fp32 of a part's row, padded
  constexpr int PART = NW * 16 * MT * ROW * 2;
  constexpr int RING = NW * D * TILE;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[RING > PART + 32 * MT ? RING : PART + 32 * MT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  constexpr int OUT = PAIR ? WR / 2 : WR;        // columns of the result
  const int n_out = GATE ? N / 2 : N;
  const long n0 = ROPE ? (long)ln_rope_first<WR>(blockIdx.x) : blockIdx.x * (long)OUT;
  unsigned short* wt = lds + wid * (D * TILE);
  LnTile<WR> lw;
  LnTile<XR> lx;
  if (ROPE) lw.init_rope(K, lane);
  else if (GATE) lw.init_gate(n0, n_out, K, lane);
  else lw.init(n0, N, K, lane);
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
  // squares of this wave's rows, wid + NW i: fetched here, summed at the end
  constexpr int SR = SCALE ? (XR + NW - 1) / NW : 1;
  uint4 sq[SR];
  if constexpr (SCALE) {
#pragma unroll
    for (int i = 0; i < SR; i++) {
      const int m = wid + NW * i;
      sq[i] = mr_load(mr_buffer(ends.squares + (long)m * ends.n_squares,
                                m < M ? ends.n_squares * 4 : 0), lane * 16);
    }
  }
  // what is added at the end: this lane's columns of up to OWN rows
  constexpr int C4 = OUT / 4;                    // columns in fours
  constexpr int OWN = (16 * MT * C4 + NW * 64 - 1) / (NW * 64);
  uint2 res[ADD ? OWN : 1], norm[ADD ? OWN : 1];
  if constexpr (ADD) {
#pragma unroll
    for (int k = 0; k < OWN; k++) {
      const int i = tid + k * NW * 64, m = i / C4;
      const long n = n0 + (i % C4) * 4;
      res[k] = norm[k] = make_uint2(0u, 0u);
      if (m >= M || n >= n_out) continue;
      res[k] = *reinterpret_cast<const uint2*>(ends.residual +
                                               (long)m * n_out + n);
      norm[k] = *reinterpret_cast<const uint2*>(ends.norm + n);
    }
  }
  LnRope rope[ROPE ? OWN : 1];
  float4 cosv[ROPE ? OWN : 1], sinv[ROPE ? OWN : 1];
  if constexpr (ROPE) {
#pragma unroll
    for (int k = 0; k < OWN; k++) {
      const int i = tid + k * NW * 64, m = i / C4;
      rope[k].init(ends, m, m < M);
      rope[k].angles(ends, (int)n0 + (i % C4) * 4, cosv[k], sinv[k]);
    }
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = K / LN_K;
  const int turn = (int)__umulhi(blockIdx.x * turns, (unsigned)steps);
  const int mine = (steps - wid + NW - 1) / NW;  // of this wave
  auto column = [&](int i) {
    const int t = wid + i * NW + turn;
    return (t >= steps ? t - steps : t) * LN_K;
  };
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < mine) {
      lw.load(wp + column(d), wt + d * TILE);
      lx.load(x + column(d), wt + d * TILE + T);
    }
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
      // W is read, its next tile may come: 64 rows, 2560 x 2560 9.4 -> 9.1 us
      if (r < NT && r + 2 >= NT && i + D < mine)
        lw.load(wp + column(i + D), wt + slot * TILE);
    }
    if constexpr (TILES % 2 != 0) {
      rows(TILES - 1, r0);
      ln_read(r0, v[TILES - 1]);
    }
    if (i + D < mine) lx.load(x + column(i + D), wt + slot * TILE + T);
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
  float* factor = reinterpret_cast<float*>(lds + PART);
  if constexpr (SCALE) {
    // all rows in step: one after the other they took 2 us
    float v[SR];
#pragma unroll
    for (int i = 0; i < SR; i++)
      v[i] = __uint_as_float(sq[i].x) + __uint_as_float(sq[i].y) +
             __uint_as_float(sq[i].z) + __uint_as_float(sq[i].w);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      float u[SR];
#pragma unroll
      for (int i = 0; i < SR; i++) u[i] = __shfl_xor(v[i], off, 64);
#pragma unroll
      for (int i = 0; i < SR; i++) v[i] += u[i];
    }
    float mine = v[0];
#pragma unroll
    for (int i = 1; i < SR; i++) mine = lane == i ? v[i] : mine;
    const int m = wid + NW * lane;
    if (lane < SR && m < 16 * MT)
      factor[m] = rsqrtf(mine / (float)K + ends.eps);
  }
  __syncthreads();
  auto sum = [&](int m, int col, float (&s)[4]) {
#pragma unroll
    for (int k = 0; k < NW; k++) {
      const float4 z = *reinterpret_cast<const float4*>(
          part + (k * 16 * MT + m) * ROW + col);
      if (k == 0) { s[0] = z.x; s[1] = z.y; s[2] = z.z; s[3] = z.w; }
      else { s[0] += z.x; s[1] += z.y; s[2] += z.z; s[3] += z.w; }
    }
  };
#pragma unroll
  for (int k = 0; k < OWN; k++) {
    const int i = tid + k * NW * 64;
    if (i >= 16 * MT * C4) break;
    const int m = i / C4, col = (i % C4) * 4;
    const long n = n0 + col;
    const bool ok = m < M && n < n_out;
    if (!ADD && !ok) continue;
    float s[4];
    sum(m, col, s);
    const float f = SCALE ? factor[m] : 1.0f;
    if constexpr (GATE) {
      float u[4];
      sum(m, OUT + col, u);
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] = ln_gated(s[e] * f, u[e] * f);
    } else if constexpr (ROPE) {
      float u[4];
      sum(m, OUT + col, u);
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] *= f, u[e] *= f;
      ln_turn(s, u, cosv[k], sinv[k]);
      unsigned short* to = rope[k].place(ends, y, m, (int)n);
      if (to == nullptr) continue;
      *reinterpret_cast<uint2*>(to) =
          make_uint2(pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]));
      *reinterpret_cast<uint2*>(to + LN_HEAD / 2) =
          make_uint2(pack_bf16(u[0], u[1]), pack_bf16(u[2], u[3]));
      continue;
    } else if constexpr (SCALE) {
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] *= f;
    }
    if (!ROPE && MODE % 4 != LN_GATE && !ADD && bias != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] += bf16_to_f32(bias[n + e]);
    }
    uint2 o;
    o.x = pack_bf16(s[0], s[1]);
    o.y = pack_bf16(s[2], s[3]);
    const long at = (long)m * n_out + n;
    if constexpr (ADD) {
      float q = 0.0f;
      if (ok) {
        o.x = ln_join(s[0], s[1], res[k].x, norm[k].x, q);
        o.y = ln_join(s[2], s[3], res[k].y, norm[k].y, q);
        *reinterpret_cast<uint2*>(ends.residual + at) = res[k];
      }
#pragma unroll
      for (int off = C4 / 2; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
      if (col == 0 && m < M)
        ends.sums[(long)m * gridDim.x + blockIdx.x] = q;
      if (!ok) continue;
    }
    *reinterpret_cast<uint2*>(y + at) = o;
  }
}

// ---- short prompts ---------------------------------------------------------------
// A workgroup owns 16 NW rows of W and 16 MT of x. Tiles of LK columns go through a
// ring of S buffers; a wave multiplies 32 rows of W by all of x over one half of a
// tile's columns, with the operands of the next tile read from LDS meanwhile and one
// barrier per tile. At the end the waves of the two halves swap a row tile of W.
//   What bounds it: what a CU pulls from L2, (16 NW + 16 MT) K entries at 70 KB/us with
// W from memory (98 where it is cached; a loop of loads alone 107-115): without
// products 300 x 3072 x 2048 takes 10.2 us of 11.6, without the epilogue 10.5. Longer
// rings and other orders of the columns changed nothing, and rows of 64 B instead of
// 256, as the products want their operands straight from memory, come at a third of
// the rate. So the shape that a CU pulls least for is taken (linear_shape), all
// products run beside the loads, and loads go through buffers: after global ones the
// compiler lets no LDS read pass another. Us, 64 x 64 tiles of four waves, a quarter
// of the products each -> here: 300 x 2048 x 2048 11.2 -> 9.4, 4096 x 2048 16.3 -> 13.2,
// 4096 x 4096 29.5 -> 22.5, 3072 x 2048 11.7 -> 11.6; 96 x 3072 x 2048 10.9 -> 9.6;
// 192 x 6144 x 4096 30.1 -> 25.7; 256 x 3072 x 2048, as many
// tiles of 64 x 64 either way, 12.0 -> 11.9 (a ring of five there 12.2).
template <int NW, int MT, int LK, int S, int MODE>
__global__ __launch_bounds__(NW * 64) void linear_tile_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, const int M, const int N,
    const int K, const long x_stride, const int n_tiles_n,
    const LinearEnds ends) {
  constexpr bool GATE = MODE & LN_GATE, SCALE = MODE & LN_SCALE,
                 ADD = MODE & LN_ADD, ROPE = MODE & LN_ROPE;
  constexpr bool PAIR = GATE || ROPE;            // two rows of W to a column
  constexpr int WR = 16 * NW;                    // rows of W
  constexpr int WT = WR * LK, TILE = WT + 16 * MT * LK;
  constexpr int KS = LK / 64;                    // products a wave makes of a step
  constexpr int CPR = LK / 8, RPI = 64 / CPR;    // chunks of a row, rows a load
  constexpr int WI = 16 / RPI, XI = 16 * MT / (RPI * NW);   // loads of a wave
  static_assert(XI * RPI * NW == 16 * MT, "");
  __shared__ __attribute__((aligned(1024))) unsigned short lds[S * TILE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  constexpr int OUT = PAIR ? WR / 2 : WR;        // columns of the result
  const int n_out = GATE ? N / 2 : N;
  const int tile_n = blockIdx.x % n_tiles_n;
  const long n0 = ROPE ? (long)ln_rope_first<WR>(tile_n) : tile_n * (long)OUT;
  const long m0 = (blockIdx.x / n_tiles_n) * (16L * MT);
  const int n_cols = (int)min((long)OUT, n_out - n0);
  const int m_rows = (int)min(16L * MT, M - m0);
  const unsigned short* wp = w + n0 * K;
  const unsigned short* xp = x + m0 * x_stride;
  const unsigned w_bytes =
      (unsigned)(n_cols + (GATE ? n_out : ROPE ? LN_HEAD / 2 : 0)) * K * 2;
  const unsigned x_bytes = (unsigned)((m_rows - 1) * x_stride + K) * 2;
  // a wave loads 16 rows of W and its share of x, RPI at a time; rows past the last
  // one repeat it: their results go nowhere
  unsigned w_off[WI], x_off[XI];
  auto offset = [&](int r, long row, long stride) {
    const int swz = LK == 128 ? r & 15 : (r >> 1) & 7;
    return (unsigned)(row * stride * 2) + (((lane % CPR) ^ swz) << 4);
  };
#pragma unroll
  for (int i = 0; i < WI; i++) {
    const int r = (wid * WI + i) * RPI + lane / CPR;
    w_off[i] = offset(r, ROPE   ? ln_rope_row<WR>(r)
                         : GATE ? ln_gate_row<WR>(n0, n_out, r) - n0
                                : min(r, n_cols - 1), K);
  }
#pragma unroll
  for (int i = 0; i < XI; i++) {
    const int r = (wid * XI + i) * RPI + lane / CPR;
    x_off[i] = offset(r, min(r, m_rows - 1), x_stride);
  }
  // squares of the rows, SL lanes to each: fetched here, summed at the end
  constexpr int SL = NW * 64 / (16 * MT) >= 8 ? 8 : NW * 64 / (16 * MT) >= 4 ? 4 : 2;
  constexpr int SQ = SCALE ? 64 / (4 * SL) : 1;
  uint4 sq[SQ];
  if constexpr (SCALE) {
    const auto src = mr_buffer(ends.squares + m0 * ends.n_squares,
                               (unsigned)m_rows * ends.n_squares * 4);
#pragma unroll
    for (int i = 0; i < SQ; i++) {
      const int p = (i * SL + tid % SL) * 4;
      sq[i] = mr_load(src, p < ends.n_squares
                               ? (tid / SL * ends.n_squares + p) * 4 : ~15u);
    }
  }
  constexpr int C8 = OUT / 8;                    // columns in eights
  constexpr int OWN = (16 * MT * C8 + NW * 64 - 1) / (NW * 64);
  LnRope rope[ROPE ? OWN : 1];
  if constexpr (ROPE) {
#pragma unroll
    for (int k = 0; k < OWN; k++) {
      const int row = (tid + k * NW * 64) / C8;
      rope[k].init(ends, m0 + row, row < m_rows);
    }
  }
  const int steps = K / LK;
  auto stage = [&](int t, int slot) {
    // past the end: zeros, by an empty buffer; an offset in front of its bounds check
    // would be taken from a size of 0
    const bool on = t < steps;
    const unsigned col = on ? t * (LK * 2) : 0u;
    const auto ws = mr_buffer(wp, on ? w_bytes : 0u);
    const auto xs = mr_buffer(xp, on ? x_bytes : 0u);
    unsigned short* dst = lds + slot * TILE;
#pragma unroll
    for (int i = 0; i < WI; i++)
      mr_to_lds(ws, w_off[i], dst + (wid * WI + i) * 512, col);
#pragma unroll
    for (int i = 0; i < XI; i++)
      mr_to_lds(xs, x_off[i], dst + WT + (wid * XI + i) * 512, col);
  };
  // a wave multiplies 32 rows of W by all of x over half of the step's columns
  const int hw = wid % (NW / 2), hk = wid / (NW / 2);
  int at[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
    at[ks] = c16 * LK + (((4 * (KS * hk + ks) + g) ^
                          (LK == 128 ? c16 : c16 >> 1)) << 3);
  struct Frags { bf16x8 w[KS][2], x[KS][MT]; };
  auto fetch = [&](Frags& f, int slot) {
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const lds_u16* p = (const lds_u16*)lds + slot * TILE + at[ks];
#pragma unroll
      for (int i = 0; i < 2; i++)
        f.w[ks][i] =
            *reinterpret_cast<const lds_bf16x8*>(p + (hw * 2 + i) * 16 * LK);
#pragma unroll
      for (int j = 0; j < MT; j++)
        f.x[ks][j] = *reinterpret_cast<const lds_bf16x8*>(p + WT + j * 16 * LK);
    }
  };
  f32x4 acc[2][MT];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < S - 1; t++) stage(t, t);
  // the next step's tile has arrived, those after it may be on the way
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * (WI + XI)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * (WI + XI)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f[2];
  fetch(f[0], 0);
  int slot = 0;
  auto step = [&](int t, const Frags& now, Frags& next) {
    meet();
    stage(t + S - 1, slot == 0 ? S - 1 : slot - 1);
    slot = slot == S - 1 ? 0 : slot + 1;
    fetch(next, slot);
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < MT; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              now.w[ks][i], now.x[ks][j], acc[i][j], 0, 0, 0);
  };
  for (int t = 0;;) {
    step(t, f[0], f[1]);
    if (++t == steps) break;
    step(t, f[1], f[0]);
    if (++t == steps) break;
  }
  float4 cosv[ROPE ? OWN : 1][2], sinv[ROPE ? OWN : 1][2];
  if constexpr (ROPE) {
#pragma unroll
    for (int k = 0; k < OWN; k++)
#pragma unroll
      for (int e = 0; e < 2; e++)
        rope[k].angles(ends, (int)n0 + (tid + k * NW * 64) % C8 * 8 + 4 * e,
                       cosv[k][e], sinv[k][e]);
  }
  // acc[i][j][r] = a half of y[m = 16 j + c16][n = 32 hw + 16 i + 4 g + r]. The
  // waves of the two halves swap a row tile of W, then whole rows go out.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  f32x4* swap = reinterpret_cast<f32x4*>(lds);   // [NW][MT][64]
#pragma unroll
  for (int j = 0; j < MT; j++) swap[(wid * MT + j) * 64 + lane] = hk ? acc[0][j] : acc[1][j];
  __syncthreads();
  // rows on their way out: bf16, or what something is still done to, padded
  constexpr bool WIDE = PAIR || ADD;
  constexpr int ROW = WIDE ? 2 * (WR + 4) : WR + 8;
  unsigned short* out = lds + NW * MT * 64 * 8;
  const int col0 = 32 * hw + 16 * hk + 4 * g;
  float* factor = reinterpret_cast<float*>(out + 16 * MT * ROW);
  if constexpr (SCALE) {
    float v = 0.0f;
#pragma unroll
    for (int i = 0; i < SQ; i++)
      v += __uint_as_float(sq[i].x) + __uint_as_float(sq[i].y) +
           __uint_as_float(sq[i].z) + __uint_as_float(sq[i].w);
#pragma unroll
    for (int off = SL / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (tid % SL == 0 && tid / SL < 16 * MT)
      factor[tid / SL] = rsqrtf(v / (float)K + ends.eps);
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < MT; j++) {
    f32x4 z = (hk ? acc[1][j] : acc[0][j]) +
              swap[((wid ^ (NW / 2)) * MT + j) * 64 + lane];
    if (SCALE) z *= factor[16 * j + c16];
    if constexpr (WIDE) {
      *reinterpret_cast<f32x4*>(out + (16 * j + c16) * ROW + 2 * col0) = z;
    } else {
      uint2 o;
      o.x = pack_bf16(z[0], z[1]);
      o.y = pack_bf16(z[2], z[3]);
      *reinterpret_cast<uint2*>(out + (16 * j + c16) * ROW + col0) = o;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < OWN; k++) {
    const int idx = tid + k * NW * 64;
    const int row = idx / C8, col = idx % C8 * 8;
    const bool ok = row < m_rows && col < n_cols;
    if (!ADD && !ok) continue;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    float f[8];
    if constexpr (WIDE) {
      auto eight = [&](int at, float (&to)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *reinterpret_cast<f32x4*>(to + e) = *reinterpret_cast<const f32x4*>(
              out + row * ROW + 2 * (at + e));
      };
      if (ok) eight(col, f);
      if constexpr (ROPE) {
        float u[8];
        eight(OUT + col, u);
        ln_turn(f, u, cosv[k][0], sinv[k][0]);
        ln_turn(f + 4, u + 4, cosv[k][1], sinv[k][1]);
        unsigned short* to = rope[k].place(ends, y, m0 + row, (int)n0 + col);
        if (to == nullptr) continue;
        *reinterpret_cast<uint4*>(to) =
            make_uint4(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]),
                       pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
        *reinterpret_cast<uint4*>(to + LN_HEAD / 2) =
            make_uint4(pack_bf16(u[0], u[1]), pack_bf16(u[2], u[3]),
                       pack_bf16(u[4], u[5]), pack_bf16(u[6], u[7]));
        continue;
      }
      if constexpr (GATE) {
        float u[8];
        eight(OUT + col, u);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = ln_gated(f[e], u[e]);
        v = make_uint4(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]),
                       pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
      }
    } else {
      v = *reinterpret_cast<const uint4*>(out + row * ROW + col);
    }
    const long at = (m0 + row) * n_out + n0 + col;
    if constexpr (ADD) {
      float q = 0.0f;
      if (ok) {
        uint4 r = *reinterpret_cast<const uint4*>(ends.residual + at);
        const uint4 n = *reinterpret_cast<const uint4*>(ends.norm + n0 + col);
        v = make_uint4(ln_join(f[0], f[1], r.x, n.x, q),
                       ln_join(f[2], f[3], r.y, n.y, q),
                       ln_join(f[4], f[5], r.z, n.z, q),
                       ln_join(f[6], f[7], r.w, n.w, q));
        *reinterpret_cast<uint4*>(ends.residual + at) = r;
      }
#pragma unroll
      for (int off = C8 / 2; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
      if (idx % C8 == 0 && row < m_rows)
        ends.sums[(m0 + row) * n_tiles_n + blockIdx.x % n_tiles_n] = q;
      if (!ok) continue;
    }
    *reinterpret_cast<uint4*>(y + at) = v;
  }
}

// More tiles of 64 x 64 than CUs, rows of W up to 2048: two workgroups share a CU, four
// waves, a quarter of the tile each; two buffers, one barrier per step of 128 columns.
// Bound by what comes before and after its few steps, which two workgroups cover for
// each other. Us, linear_tile_kernel | here: 256 x 6912 x 640 9.9 | 8.0, 300 x 4864 x 1024
// 11.2 | 9.9, 500 x 4096 x 1536 14.5 | 13.8, 256 x 6912 x 128 5.1 | 4.1.
__global__ __launch_bounds__(256, 2) void linear_square_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, const int M, const int N,
    const int K, const long x_stride, const int n_tiles_n) {
  constexpr int HALF = 64 * LN_K, TILE = 2 * HALF;
  __shared__ __attribute__((aligned(1024))) unsigned short lds[2 * TILE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;
  const long n0 = (blockIdx.x % n_tiles_n) * 64L;
  const long m0 = (blockIdx.x / n_tiles_n) * 64L;
  const int wn = wid & 1, wm = wid >> 1;
  // a wave loads 16 rows of both; rows past the last one repeat it
  LnTile<16> lw, lx;
  const long nr = min(n0 + wid * 16, (long)N - 1);
  const long mr = min(m0 + wid * 16, (long)M - 1);
  lw.init(nr, N, K, lane);
  lx.init(mr, M, x_stride, lane);
  const unsigned short* wp = w + nr * K;
  const unsigned short* xp = x + mr * x_stride;
  unsigned short* mine = lds + wid * 16 * LN_K;
  // bytes of chunk 2 k + h of a lane's row in either half
  const unsigned base = (unsigned)(unsigned long long)(const lds_u16*)lds;
  unsigned wat[8], xat[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int rw = wn * 32 + c32, rx = wm * 32 + c32;
    wat[k] = base + 2 * (rw * LN_K + (((2 * k + h) ^ (rw & 15)) << 3));
    xat[k] = base + 2 * (HALF + rx * LN_K + (((2 * k + h) ^ (rx & 15)) << 3));
  }
  f32x16 acc = mr_zero();
  const int steps = K / LN_K;
  auto stage = [&](int t) {
    unsigned short* dst = mine + (t & 1) * TILE;
    lw.load(wp + t * LN_K, dst);
    lx.load(xp + t * LN_K, dst + HALF);
  };
  stage(0);
  for (int t = 0; t < steps; t++) {
    const unsigned buf = (t & 1) * (2 * TILE);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t + 1 < steps) stage(t + 1);
#pragma unroll
    for (int k = 0; k < 8; k += 4) {
      unsigned a_at[4], b_at[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        a_at[i] = wat[k + i] + buf;
        b_at[i] = xat[k + i] + buf;
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

// 0: the library's; 1: stream; 2: tiles; 3: square ones, without LinearEnds' options.
// Besides its time on the GPU a library call costs 28 us of host time (its choice of a
// kernel), these cost 6.
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
//   M 96-192 2048 x 2048 9.2 | 11.2-12, 4096 x 2048 10-11 | 13.3-21.5, 4096 x 4096
//            16.6-18.7 | 22-33, 6144 x 4096 20.6-25.7 | 23-34, 8192 x 4096 23.5-28.5 | 24.3-35,
//            4096 x 8192 30-34 | 36-59, 3584 x 18944 55-67 | 98-124
//   M 300    2048 x 2048 9.3 | 12.9, 4096 x 2048 13.1 | 15.5, 4096 x 4096 22.4 | 25.8, 6144 x
//            4096 30.3 | 30, 4096 x 14336 71 | 75; not in one turn of the CUs: 8192 x 4096
//            46 | 37, 14336 x 2048 49 | 30
//   M 512-1024   3072 x 2048 16.7 | 15.2, 4096 x 4096 30.7 | 30.2, 2048 x 2048 12-17.3 |
//            12.8-17.1, 1024 x 4096 15.5-20.7 | 15.8-21.1; M 2048, 512 x 2048 13 | 10.8, M 3072 18 |
//            12.9; but M 8192, 64 x 2048 8.7 | 10
//   long rows, few tiles   M 96, 1024 x 4096 15.2 | 11.8, 2560 x 4096 15.9 | 13.2; M 128,
//            1536 x 3072 12.7 | 10.5, 2048 x 4096 15.4 | 12.6, M 192 15.3 | 15.8; M 192, 1024 x
//            4096 15 | 12.3, M 300 13.9 | 15.4; at K 2048 1024 x 2048 6.6 | 8.3
// With a bias the library chooses among other kernels, which were faster from 65 rows
// on: 96 x 2048 x 2048 6.9, 128 x 2048 x 1536 6.3, 96 x 4608 x 3584 16.5.
// A tuned choice of the library is preferred above 48 rows, above 32 where N > 8192
// (linear in bindings.cpp): M 32, 28672 x 4096 48.9 | 48.2, M 48 53.5 | 49.3 | 60.5 not,
//   4096 x 4096, here | tuned | not   M 48 11.8 | 13.7 | 13.7, 64 13.2 | 13.6 | 15.1,
//            96 16.6 | 17.2 | 22.0, 128 16.6 | 16.9 | 24.5

// Of the shapes that linear_tile_kernel has, the one that a CU pulls least for: turns
// of the CUs times the rows of a tile. x rows of 64 rows of W, or 0: 64 of 128.
// Three row tiles of 48 without a smaller fourth one, which would fetch W ahead of
// the others, cost long rows more than two of 64 and a rest: M 144, 4096 x 14336 59.7 |
// 52.7, 4096 x 8192 34.4 | 31.2, 3584 x 18944 74.6 | 66.1; M 152 48.3 | 54.8.
static int linear_shape(long M, long N, long K, long* turns) {
  int best = 0;
  long least = 0;
  for (int mt = 0; mt <= 6; mt++) {
    if (mt == 1 || (mt == 3 && K > 4096 && M > 128 && M <= 144)) continue;
    const long wr = mt == 0 ? 128 : 64, xr = mt == 0 ? 64 : 16 * mt;
    const long t = ((N + wr - 1) / wr * ((M + xr - 1) / xr) + 255) / 256;
    const long cost = t * (wr + xr);
    if (least != 0 && cost >= least) continue;
    least = cost;
    best = mt;
    *turns = t;
  }
  return best;
}

// The choice (0 to 3, see above). ends: LinearEnds' options are wanted, which save a launch
// of 2.5 to 5 us. Then products are taken too that the library is faster at by less than
// that, and the answer is never 3.
int linear_takes(long M, long N, long K, bool bias, bool ends) {
  if (M <= 0 || K < LN_K || K % LN_K != 0 || N % 8 != 0) return 0;
  if (N * K >= (1L << 31) || M * K >= (1L << 30)) return 0;
  if (M <= 16) return M <= 8 || N * K <= 1L << 28 ? 1 : 0;
  // The library splits long rows of whole 1024s over workgroups: few workgroups here
  // wait longer for theirs. Here | library, 512 x 8192 | 512 x 8448: M 24 8.2 | 8.1, 8.6 |
  // 17.7, M 40 10.9 | 7.9, 11.4 | 17.5, M 64 13.5 | 8.4, 14 | 17.8; M 32, 512 x 16384 18.4 | 19.2
  const bool split = K >= 6144 && K % 1024 == 0;
  if (M <= 32) {
    if (N <= 8192)
      return N > 1024 || K <= 8192 || !split || M > 24 || N <= 256 ? 1 : 0;
    if (ends) return K <= 4096 && N * K <= 1L << 28 ? 1 : 0;
    // More than 8192 columns: x rows weigh more and more, and the last turn of the CUs
    // counts. Here | library, M 20, M 28-32: 50272 x 768 20.7 | 20, 21.6 | 20.4; 9216 x 4096
    // 22.6 | 20.5, 24.1 | 21.4; 12288 x 4096 24.2 | 23.4, 25.6 | 24; 14336 x 4096 25.2 | 25.8,
    // 27.2 | 26.3; 16384 x 4096 27.1 | 32.5, 28.5 | 32.6; 24576 x 3072 31.5 | 31.3, 33.2 | 31.5;
    // 37888 x 3584 53.6 | 54.9, 57 | 55.7
    if (K <= 2048) return N <= 32768 ? 1 : 0;
    return K <= 4096 && (M <= 24 ? N >= 14336 && N * K <= 1L << 28
                                 : N >= 16384 && K > 3072 && N * K <= 1L << 27) ? 1 : 0;
  }
  // M 40: 14336 x 2048 16.9 | 17.4, 32000 x 1024 18.6 | 25.9; 24576 x 2048 25.4 | 25, 28672 x
  // 4096 53.1 | 48.3 (M 48 55.4 | 58.5), 50272 x 768 23.7 | 21.7, 18944 x 3584 36.7 | 33.9
  if (M <= 48) {
    if (N <= 8192) return N > 2048 || !split || (N >= 1536 && K < 8192) ? 1 : 0;
    if (ends)
      return N * K <= 1L << 28 && (K <= 2048 || (K <= 4096 && N >= 18432)) ? 1 : 0;
    return (K <= 2048 && N <= 16384) || (K <= 1024 && N <= 32768) ? 1 : 0;
  }
  if (M <= 64) {
    if (N > 8192) return N * K <= 1L << 23 ? 1 : 0;   // M 57, 9600 x 384 6.7 | 8.2
    if (K <= 4096 || (N >= 2048 && N <= 4096 && K <= 8192)) return 1;
    return split ? (N >= 1280 && N <= 2048 && K < 8192 ? 1 : 0)
                 : (N * K <= 1L << 24 ? 1 : 0);
  }
  if (bias) return 0;
  long turns;
  const int shape = linear_shape(M, N, K, &turns);
  const long squares = (M + 63) / 64 * ((N + 63) / 64);
  // Up to two turns of square tiles where none of the others takes one, or has tiles
  // of 128 rows: library | square, 126 x 8448 x 640 11.1 | 7.9, 160 x 9856 x 1536 19.8 | 17.3,
  // 300 x 4864 x 1024 13.9 | 9.9, 256 x 6912 x 1536 20.8 | 14.9, 689 x 2688 x 1920 20.5 | 17,
  // 160 x 8448 x 2048 24.2 | 19.8, 512 x 3072 x 2048 15.3 | 16.4
  if (!ends && squares > 256 && squares <= 512 &&
      K <= (shape == 0 || turns > 1 ? 2048 : 512))
    return 3;
  if (turns > 1 || (M > 2048 && N > 128 && K > 1024)) return 0;
  if (N > 8192 && (N > 16384 || K > 2048 || shape == 0)) return 0;
  // 128 rows of W a tile, the library has as large ones from 257 rows on: M 512, 3584 x
  // 3584 27.6 | 25.8, M 300, 4608 x 3584 26.9 | 23.8; but M 256, 6144 x
  // 4096 31.1 | 40.3, and short rows, M 512, 4096 x 1024 10.9 | 13.1
  if (!ends && shape == 0 && M > 256 && K > 1536) return 0;
  // M 80: 4096 x 14336 48.8 | 43.1, 4096 x 11008 40.9 | 35, 3584 x 8192 27.9 | 25.4 and at
  // M 76 47.3 | 49.2, 39.6 | 40.7, 27 | 28.1; 3584 x 18944 61 | 130
  if (K > 4096)
    return N >= 3072 && N <= 4608 && M <= 192 &&
           !(M > 76 && M <= 80 && N > 3072 && K <= 16384) ? 2 : 0;
  // Fewer than 1024 columns in up to 32 tiles of 128 by 64, where the library steps to its
  // next time: 512 x 3072, M 320 8.4 | 8.6; 768 x 3072, M 300 8.6 | 8.7, M 350 11.6 | 8.8;
  // 768 x 4096, M 300 12.1 | 13.8, M 400 14.2 | 14.3, M 768 19.4 | 16.6; but 768 x 2560, M 300
  // 9.6 | 8.3
  if (!ends && K > 2560 && N < 1024 && (N + 127) / 128 * ((M + 63) / 64) <= 32)
    return 0;
  // few tiles with long rows leave most of the chip waiting for their chain, many of
  // them wait for each other: 256 x 4096, M 300 10 | 8.9, M 2048 16.2 | 13.8; M 1536, 640 x
  // 2560 14.7 | 12.4, M 2048, 512 x 2048 13 | 10.8, 1024 x 4096 32.6 | 28.5. Where the tiles of
  // W are no multiple of four, those that share one lie on several XCDs: 576 x 4096, M 300,
  // 12.2 | 10.2, 832 x 3072, M 260, 11.1 | 8.7
  if (K > 2048)
    return N >= 512 && (N >= 1024 || N % 256 == 0) && M <= 1024 &&
           !((N < 3072 && M <= 128) || (N < 2048 && M <= 256)) ? 2 : 0;
  return M <= 1536 || K <= 1536 || N <= 128 ? 2 : 0;
}

// Row tiles of W: one up to 4096 rows of it, one workgroup a CU then; two above.
// Up to 16 rows of x weigh little, and where W has long rows and many columns, one
// tile is the better again if the last turn of the CUs leaves fewer of them idle with
// it, or as few and no more than a tenth. M 8, one | two: 8192 x 4096 13.7 | 14.2, 9216 x
// 4096 17.3 | 19.7, 12288 x 4096 19.5 | 21.6, 18944 x 3584 26.8 | 27.9, 28672 x 4096 40.4 |
// 42.7; but 4608 x 3584 10.4 | 9.5 (a ninth of the CUs have two), 14336 x 4096 23.7 | 22.4,
// 22016 x 4096 33.6 | 33, 24576 x 2048 22.9 | 19.8; M 24, 8192 x 4096 16.6 | 15.3.
// Short rows have little to share: M 8, 8192 x 640 4.4 | 4.7, 7424 x 1536 6.5 | 6.7, 10240 x
// 1536 8.3 | 9.3, but 4352 x 1536 5.8 | 5.6.
static bool linear_one_tile(int M, int N, int K) {
  const int wgs = (N + 15) / 16, turns = (wgs + 255) / 256;
  const int of_two = ((N + 31) / 32 + 255) / 256;
  if (wgs <= 256) return true;
  if (M > 16) return false;
  if (K >= 2048)
    return K >= 2560 && (turns < 2 * of_two || 10 * wgs >= 9 * 256 * turns);
  if (N <= 8192) return K <= 640 || (K <= 1536 && N > 6656);
  return turns < 2 * of_two && K >= (M <= 8 ? 1024 : 1536);
}
// A workgroup that has a CU to itself takes all of its LDS: two tiles a wave, or
// more waves. Where there are more than CUs, two of them share one: M 24, 32000 x
// 4096 48.4, with two tiles 49.2; 18944 x 4096 33.4 | 34.5. Of short rows eight waves with one
// tile are faster: M 10, 8192 x 640 4.5 -> 4.4, M 32, 2560 x 2560 7.3 -> 6.9, but 4096 x 4096
// 10.4 | 10.5.
template <int MODE>
static void launch_stream(unsigned short* y, const unsigned short* x,
                          const unsigned short* w, const unsigned short* bias,
                          int M, int N, int K, long x_stride,
                          const LinearEnds& ends, hipStream_t stream) {
  constexpr int PAIR = MODE & (LN_GATE | LN_ROPE) ? 2 : 1;
  const bool one = linear_one_tile(M, N, K);
  const int out = (one ? 16 : 32) / PAIR, n_out = N / PAIR;
  const dim3 grid((n_out + out - 1) / out);
  const bool few = grid.x <= 256;
  // Workgroup b starts at step b mod steps, which its product with 2^32 / steps holds in
  // the upper bits: 10 rows, 768 x 768 2.9 us, with a division 3.0; 4096 x 4096 8.2, all
  // at the first step 9.1.
  const int steps = K / LN_K;
  const unsigned turns = (unsigned)(((1L << 32) + steps - 1) / steps);
#define LN_STREAM(NT, XR, NW, D)                                               \
  hipLaunchKernelGGL((linear_stream_kernel<NT, XR, NW, D, MODE>), grid,        \
                     dim3(NW * 64), 0, stream, y, x, w, bias, M, N, K,         \
                     x_stride, turns, ends)
  if (one) {
    const bool eight = !few && K <= 1536;        // many workgroups of short rows
    if (M <= 8) { if (eight) LN_STREAM(1, 8, 8, 1); else LN_STREAM(1, 8, 4, 2); }
    else if (M <= 16) { if (eight) LN_STREAM(1, 16, 8, 1); else LN_STREAM(1, 16, 4, 2); }
    else if (M <= 24) LN_STREAM(1, 24, 4, 2);
    else if (M <= 32) { if (K <= 2560) LN_STREAM(1, 32, 8, 1); else LN_STREAM(1, 32, 4, 2); }
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

template <int MODE>
static void launch_tile(unsigned short* y, const unsigned short* x,
                        const unsigned short* w, int M, int N, int K,
                        long x_stride, const LinearEnds& ends,
                        hipStream_t stream) {
  constexpr int PAIR = MODE & (LN_GATE | LN_ROPE) ? 2 : 1;
  const int n_out = N / PAIR;
#define LN_TILE(NW, MT, LK, S)                                                 \
  do {                                                                         \
    constexpr int OUT = 16 * NW / PAIR;                                         \
    const int tn = (n_out + OUT - 1) / OUT, tm = (M + 16 * MT - 1) / (16 * MT); \
    hipLaunchKernelGGL((linear_tile_kernel<NW, MT, LK, S, MODE>),              \
                       dim3((unsigned)(tn * tm)), dim3(NW * 64), 0, stream, y, \
                       x, w, M, N, K, x_stride, tn, ends);                     \
  } while (0)
  // a ring longer than a row costs what its empty steps do: 300 x 1344 x 128 3.5 -> 3.1,
  // 500 x 2048 x 256 4.3 -> 3.8
  const bool short_row = K <= 384;
  long turns;
  switch (linear_shape(M, N, K, &turns)) {
    case 0: LN_TILE(8, 4, 64, 6); break;
    case 2: if (short_row) LN_TILE(4, 2, 64, 4); else LN_TILE(4, 2, 128, 6); break;
    case 3: if (short_row) LN_TILE(4, 3, 128, 3); else LN_TILE(4, 3, 128, 5); break;
    case 4: if (short_row) LN_TILE(4, 4, 64, 4); else LN_TILE(4, 4, 128, 4); break;
    case 5: LN_TILE(4, 5, 128, 4); break;
    default: LN_TILE(4, 6, 128, 4);
  }
#undef LN_TILE
}

// Tiles of N that such a product has: parts of LN_ADD's sums
int linear_tiles(int M, int N, int K, int kind) {
  if (kind == 1) return linear_one_tile(M, N, K) ? (N + 15) / 16 : (N + 31) / 32;
  long turns;
  return linear_shape(M, N, K, &turns) == 0 ? (N + 127) / 128 : (N + 63) / 64;
}

// mode: LN_GATE: W = [gates | ups], y [M, N / 2] = silu(x gates^T) (x ups^T);
// LN_SCALE with or without it, LN_ADD alone, LN_SCALE | LN_ROPE: see there
void launch_linear(unsigned short* y, const unsigned short* x,
                   const unsigned short* w, const unsigned short* bias, int M,
                   int N, int K, long x_stride, int kind, int mode,
                   const LinearEnds& ends, hipStream_t stream) {
  if (kind == 3 && mode == 0 && bias == nullptr) {
    const int tn = (N + 63) / 64, tm = (M + 63) / 64;
    hipLaunchKernelGGL(linear_square_kernel, dim3((unsigned)(tn * tm)), dim3(256),
                       0, stream, y, x, w, M, N, K, x_stride, tn);
    return;
  }
  if (kind != 1 && kind != 2) throw std::invalid_argument("linear: kernels");
#define LN_MODE(MODE)                                                          \
  case MODE:                                                                   \
    if (kind == 1)                                                             \
      launch_stream<MODE>(y, x, w, bias, M, N, K, x_stride, ends, stream);     \
    else                                                                       \
      launch_tile<MODE>(y, x, w, M, N, K, x_stride, ends, stream);             \
    break
  switch (mode) {
    LN_MODE(0);
    LN_MODE(LN_GATE);
    LN_MODE(LN_SCALE);
    LN_MODE(LN_SCALE | LN_GATE);
    LN_MODE(LN_ADD);
    LN_MODE(LN_SCALE | LN_ROPE);
    default: throw std::invalid_argument("linear: mode");
  }
#undef LN_MODE
}

}  // namespace xllm
