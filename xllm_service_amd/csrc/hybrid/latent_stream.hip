// Latent attention of decoded rows (bf16) for gfx950: rank 512 with a rotated
// tail of 0 or 64 entries, 16-token pages, at most 32 heads. Prompt rows:
// latent_rows.hip, other sizes: latent_attn_mfma.hip.
//
// One new token per sequence; its heads attend to the SAME cached rows of W =
// 512 + tail entries, values are the first 512 of a row. The step is a stream
// over the cache: a workgroup (4 waves, two of them share a CU) walks tiles of
// 32 rows for 16 heads of one sequence. Tiles go from memory straight to LDS
// (global_load_lds, 16 B per lane: a page is one contiguous piece), two buffers,
// one barrier per tile, so that a tile is on the way while the other is
// computed. Before, tiles went through registers between two barriers.
//
//   S^T[key][head] = K Q^T       16x16x32 products, a wave multiplies a quarter of
//                                the columns (A = K rows from LDS, B = Q in
//                                registers); shares are added through LDS
//   online softmax               a lane holds 8 keys of ONE head
//   O^T[col][head] += V^T P^T    wave w owns columns 128 w .. 128 w + 127;
//                                A = V^T by transpose reads of the same image,
//                                P split exactly into three bf16 terms
//
// K row (m>>2)*8 + half*4 + (m&3) is fed as A row m of half 0 / 1, so that the
// C registers of a lane are the keys g*8 .. g*8+7 its B operand wants.
//
// LDS image: row-major [32][W], 16 B chunk c of row k at c ^ swz(k). Rows of 512
// start on the same bank and need four bits of it, rows of 576 alternate
// between the halves of the banks and need three; either way the 16 rows (or 8
// pieces of 32 B) that share an LDS cycle fall on different banks.
//
// Measured, 32 sequences of 1.5-2.5 k keys, 16 heads, rows of 576: 67 + 5 us before,
// 23.5 us with the merge now (25.6 when every wave made all scores, and read all of a
// tile for them); the rows alone take 15 us at the rate of a large copy. Bound by a tile's
// chain of LDS reads, products and weights, 1.7 us for 36 KB: more tiles on their way
// (four buffers) did not help, nor did two teams of waves with tiles of their own in a
// workgroup, which beside 144 KB of LDS gained nothing over more parts.
//
// The LDS reads are asm with their wait: in front of a builtin the compiler
// waits for every load to LDS in flight.
//
// Fragments of 16x16x32 (lane l, g = l >> 4): A[l&15][g*8 + j], B[g*8 +
// j][l&15], C[g*4 + r][l&15].
#include "../ops/paged_merge.h"
#include "hybrid_common.h"

namespace xllm {
namespace hyb {

constexpr int LS_KT = 32;       // keys per tile (two pages)
constexpr int LS_R = 512;       // value columns

template <int W> XLLM_DEV int ls_swz(int k) {
  const int lo = (((k >> 3) & 1) << 1) | ((k >> 4) & 1);
  return W == 512 ? ((k & 3) << 2) | lo : (((k >> 1) & 1) << 2) | lo;
}

// K fragments of four steps, both halves
template <int W>
XLLM_DEV void ls_keys(const unsigned* at, bf16x8 (&k)[2][4]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
      "ds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
      "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\t"
      "ds_read_b128 %6, %10 offset:%12\n\tds_read_b128 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]),
        "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2]), "=&v"(k[1][3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(8 * W)
      : "memory");
}
// of one step
template <int W>
XLLM_DEV void ls_key(unsigned at, bf16x8 (&k)[2]) {
  asm volatile(
      "ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0]), "=&v"(k[1])
      : "v"(at), "n"(8 * W)
      : "memory");
}
// The waves' shares of the scores, [wave][half][lane]: `mine` goes out, their sum
// comes back, added in the same order by all
XLLM_DEV void ls_share(unsigned to, unsigned from, f32x4 (&sc)[2]) {
  // the compiler does not see what an asm block reads of a product under way: it
  // ends within 16 states
  asm volatile(
      "s_nop 15\n\ts_nop 7\n\tds_write_b128 %0, %1\n\tds_write_b128 %0, %2 offset:1024\n\t"
      "s_waitcnt lgkmcnt(0)" ::"v"(to), "v"(sc[0]), "v"(sc[1])
      : "memory");
  __builtin_amdgcn_s_barrier();
  f32x4 x[8];
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:1024\n\t"
      "ds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %8 offset:3072\n\t"
      "ds_read_b128 %4, %8 offset:4096\n\tds_read_b128 %5, %8 offset:5120\n\t"
      "ds_read_b128 %6, %8 offset:6144\n\tds_read_b128 %7, %8 offset:7168\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]),
        "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7])
      : "v"(from)
      : "memory");
#pragma unroll
  for (int i = 0; i < 2; i++) sc[i] = (x[i] + x[2 + i]) + (x[4 + i] + x[6 + i]);
}
// Four V^T fragments (16 columns, 32 keys each)
template <int W>
XLLM_DEV void ls_values(unsigned a0, unsigned a1, unsigned a2, unsigned a3,
                        bf16x8 (&v)[4]) {
  typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
  u32x2 t[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(t[4]),
        "=&v"(t[5]), "=&v"(t[6]), "=&v"(t[7])
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "n"(8 * W)
      : "memory");
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const unsigned x[4] = {t[2 * i][0], t[2 * i][1], t[2 * i + 1][0],
                           t[2 * i + 1][1]};
    __builtin_memcpy(&v[i], x, 16);
  }
}
XLLM_DEV f32x4 ls_mma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Parts of a sequence of n tiles: one for every `per` of them, or of up to `few` one for
// every two
XLLM_DEV int ls_own(int n, int n_part, int per, int few) {
  return max(paged_parts(n, n_part, per), paged_parts(n, min(n_part, few), 2));
}

template <int W>
__global__ void __launch_bounds__(256, 2) latent_stream_kernel(
    float* __restrict__ out,               // [S, H, 512] (n_part == 1)
    float* __restrict__ ws_o,              // [S*H][n_part][512]
    float* __restrict__ ws_ml,             // [S*H][n_part][2]
    const unsigned short* __restrict__ q,  // [S, H, W]
    const unsigned short* __restrict__ cache,   // [blocks, 16, W]
    const int* __restrict__ block_tables, const int* __restrict__ seq_lens,
    int heads, int table_width, float scale, int n_part, int per, int few,
    int window) {
  constexpr int CPR = W / 8;                     // 16 B chunks of a row
  constexpr int IPP = 16 * CPR / 64;             // load instructions per page
  constexpr int NI = 2 * IPP / 4;                // ... of a wave per tile
  constexpr int KS = W / 32;                     // steps of a score product
  constexpr int TILE = LS_KT * W;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[2 * TILE + 4 * 2 * 64 * 8];            // and the shares of the scores

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, n = lane & 15;
  const int n_seqs = gridDim.x / n_part;
  const int part = blockIdx.x / n_seqs, s = blockIdx.x % n_seqs;  // idle last
  const int h0 = blockIdx.y * 16;                // first head
  const int seq_len = seq_lens[s];
  const int n_tiles = (seq_len + LS_KT - 1) / LS_KT;
  const int lo = window > 0 ? max(0, seq_len - window) : 0;
  const int t_first = lo / LS_KT;
  const int parts = ls_own(n_tiles - t_first, n_part, per, few);
  if (part >= parts) return;
  const int tpp = (n_tiles - t_first + parts - 1) / parts;
  const int t_begin = t_first + part * tpp;
  const int t_end = min(n_tiles, t_begin + tpp);

  const bool on = h0 + n < heads;
  const long row = (long)s * heads + (on ? h0 + n : h0);
  const short flip = scale < 0.0f ? (short)0x8000 : (short)0;
  const float c = paged_factor(scale);
  // this wave's steps of the score product
  const int k0 = W == 512 ? 4 * w : 4 * w + min(w, 2);
  const bool five = W == 576 && w < 2;
  bf16x8 qf[5];
#pragma unroll
  for (int i = 0; i < 5; i++)
    qf[i] = *reinterpret_cast<const bf16x8*>(
                q + row * W + min(k0 + i, KS - 1) * 32 + g * 8) ^
            flip;

  // ---- loads: instruction i of wave w is the (4 i + w)-th of the tile --------
  const int last_blk = (seq_len - 1) / 16, last_row = (seq_len - 1) % 16;
  const int* table = block_tables + (long)s * table_width;
  unsigned off[NI];                              // bytes into the page
  int rowin[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int j = 4 * i + w, p = j >= IPP;
    const int chunk = (j - p * IPP) * 64 + lane;
    const int r = chunk / CPR, pos = chunk - r * CPR;
    rowin[i] = r;
    off[i] = (unsigned)(r * (2 * W) + ((pos ^ ls_swz<W>(p * 16 + r)) << 4));
  }
  // ids of the pages of 32 tiles from the tb-th on, two lanes a tile
  int tb = t_begin;
  auto pages_from = [&](int t) {
    return table[min(2 * t + lane, table_width - 1)];
  };
  auto stage = [&](int t, int pages, int buf) {
    const int p0 = __builtin_amdgcn_readlane(pages, 2 * (t - tb));
    const int p1 = 2 * t + 1 > last_blk
        ? p0 : __builtin_amdgcn_readlane(pages, 2 * (t - tb) + 1);
    const char* src0 =
        reinterpret_cast<const char*>(cache) + (long)p0 * (32 * W);
    const char* src1 =
        reinterpret_cast<const char*>(cache) + (long)p1 * (32 * W);
    unsigned short* dst = lds + buf * TILE;
    if (2 * t + 1 < last_blk) {
#pragma unroll
      for (int i = 0; i < NI; i++)
        __builtin_amdgcn_global_load_lds(
            (glb_void*)((4 * i + w >= IPP ? src1 : src0) + off[i]),
            (lds_void*)(dst + (4 * i + w) * 512), 16, 0, 0);
      return;
    }
    // rows past the last key repeat it: masked below, and finite
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int p = 4 * i + w >= IPP, pg = 2 * t + p, r = rowin[i];
      const int rr = pg < last_blk ? r : pg > last_blk ? last_row
                                       : min(r, last_row);
      __builtin_amdgcn_global_load_lds(
          (glb_void*)((p ? src1 : src0) + off[i] + (rr - r) * (2 * W)),
          (lds_void*)(dst + (4 * i + w) * 512), 16, 0, 0);
    }
  };

  // ---- LDS addresses (bytes, first buffer) -------------------------------------
  const unsigned base = (unsigned)(unsigned long long)(const lds_u16*)lds;
  const int km = (n >> 2) * 8 + (n & 3);         // key of A row n, half 0
  unsigned kat[5];
#pragma unroll
  for (int i = 0; i < 5; i++)
    kat[i] = base + 2 * (km * W + (((min(k0 + i, KS - 1) * 4 + g) ^
                                    ls_swz<W>(km)) << 3));
  const unsigned from = base + 2 * (2 * TILE) + lane * 16, to = from + w * 2048;
  const int vk = g * 8 + (n >> 2);               // key of a value piece
  unsigned vat[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int ch = (w * 8 + i) * 2 + ((n & 3) >> 1);
    vat[i] = base + 2 * (vk * W + ((ch ^ ls_swz<W>(vk)) << 3) + (n & 1) * 4);
  }

  f32x4 acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.0f;

  int pages = 0;
  if (t_begin < t_end) {
    pages = pages_from(t_begin);
    stage(t_begin, pages, 0);
  }
  for (int t = t_begin; t < t_end; t++) {
    const int buf = (t - t_begin) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + 1 < t_end) {
      if (t + 1 - tb == 32) {
        tb += 32;
        pages = pages_from(tb);
      }
      stage(t + 1, pages, buf ^ 1);
    }
    const unsigned shift = buf * (2 * TILE);
    unsigned ka[5];
#pragma unroll
    for (int i = 0; i < 5; i++) ka[i] = kat[i] + shift;
    // ---- scores ----------------------------------------------------------------
    f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    {
      bf16x8 k[2][4];
      ls_keys<W>(ka, k);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sc[0] = ls_mma(k[0][i], qf[i], sc[0]);
        sc[1] = ls_mma(k[1][i], qf[i], sc[1]);
      }
      if (five) {
        bf16x8 e[2];
        ls_key<W>(ka[4], e);
        sc[0] = ls_mma(e[0], qf[4], sc[0]);
        sc[1] = ls_mma(e[1], qf[4], sc[1]);
      }
    }
    ls_share(to, from, sc);
    // sc[h2][r]: key t*32 + g*8 + h2*4 + r, head n
    if (t == n_tiles - 1 || t * LS_KT < lo) {    // uniform
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int key = t * LS_KT + g * 8 + i;
        if (key >= seq_len || key < lo) sc[i >> 2][i & 3] = -INFINITY;
      }
    }
    // ---- online softmax: weights are 2^(c (s - m)) --------------------------------
    float mt = sc[0][0];
#pragma unroll
    for (int i = 1; i < 8; i++) mt = fmaxf(mt, sc[i >> 2][i & 3]);
    mt = pair_max(mt);
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    if (__any(mt > m)) {
      const float m_new = fmaxf(m, mt);
      const float alpha =
          __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < 8; i++) acc[i] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    bf16x8 p[3];
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      float a = __builtin_amdgcn_exp2f(fmaf(sc[i >> 2][i & 3], c, -mc));
      float b = __builtin_amdgcn_exp2f(fmaf(sc[i >> 2][(i & 3) + 1], c, -mc));
      l += a + b;
#pragma unroll
      for (int e = 0; e < 3; e++) {
        const unsigned u = pack_bf16(a, b);
        reinterpret_cast<unsigned*>(&p[e])[i >> 1] = u;
        drop_bf16(a, b, u);
      }
    }
    // ---- O^T += V^T P^T -------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < 8; i += 4) {
      bf16x8 v[4];
      ls_values<W>(vat[i] + shift, vat[i + 1] + shift, vat[i + 2] + shift,
                   vat[i + 3] + shift, v);
#pragma unroll
      for (int e = 0; e < 3; e++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i + j] = ls_mma(v[j], p[e], acc[i + j]);
    }
  }
  // acc[i][r] = O[head n][column w*128 + i*16 + g*4 + r]
  l = pair_sum(l);
  l += __shfl_xor(l, 16, 64);
  if (!on) return;
  const int col = w * 128 + g * 4;
  if (parts == 1) {
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;
    float* o = out + row * LS_R + col;
#pragma unroll
    for (int i = 0; i < 8; i++)
      *reinterpret_cast<float4*>(o + i * 16) = make_float4(
          acc[i][0] * inv, acc[i][1] * inv, acc[i][2] * inv, acc[i][3] * inv);
    return;
  }
  const long slot = row * n_part + part;
  if (w == 0 && g == 0) {
    ws_ml[slot * 2] = m * c;
    ws_ml[slot * 2 + 1] = t_begin < t_end ? l : PAGED_ABSENT;
  }
  if (t_begin >= t_end) return;
  float* o = ws_o + slot * LS_R + col;
#pragma unroll
  for (int i = 0; i < 8; i++)
    *reinterpret_cast<float4*>(o + i * 16) =
        make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
}

// out[row] = sum_p o[row][p] 2^(m_p - M) / sum_p l_p 2^(m_p - M): half a
// workgroup per row, four columns per lane
__global__ void __launch_bounds__(256) latent_stream_merge_kernel(
    float* __restrict__ out, const float* __restrict__ ws_o,
    const float* __restrict__ ws_ml, int n_part, int per, int few, long rows,
    int heads, const int* __restrict__ seq_lens, int window) {
  const long row = blockIdx.x * 2L + (threadIdx.x >> 7);
  const int col = (threadIdx.x & 127) * 4;
  if (row >= rows) return;
  const int len = seq_lens[row / heads];
  const int parts = ls_own(
      (len + LS_KT - 1) / LS_KT -
          (window > 0 ? max(0, len - window) / LS_KT : 0), n_part, per, few);
  if (parts == 1) return;                        // written where it belongs
  float M = -INFINITY, L = 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const float2* ml = reinterpret_cast<const float2*>(ws_ml) + row * n_part;
  const float* o = ws_o + row * n_part * LS_R + col;
  paged_add_parts<8>(
      [&](int p) { return ml[p]; },
      [&](int p) { return *reinterpret_cast<const float4*>(o + (long)p * LS_R); },
      parts, M, L, a);
  const float inv = L != 0.0f ? 1.0f / L : 0.0f;
  *reinterpret_cast<float4*>(out + row * LS_R + col) =
      make_float4(a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv);
}

bool latent_stream_takes(int W, int r, int heads, int block_size) {
  return r == LS_R && (W == 512 || W == 576) && heads <= 32 && block_size == 16;
}

// Room for parts from what the host knows; how many there are follows a sequence's own
// length in the kernel (ls_own). Few workgroups: one per CU, parts of at least two
// tiles. Measured (us, by parts): 1 x 700 keys, 16 heads 16 (4), 12 (8); 8 x 4000 35
// (8), 23 (16), 20 (32); 16 x 2000 18.5 (16), 20.3 (32). More, where a part is a long
// chain: parts of four tiles up to one turn of two workgroups per CU, 24 x 2000 22.8
// (10), 22.3 (21), 24 x 0.1-6 k 34.8 (10), 29.1 (21), 32 x 2000 24.8 (8), 23.8 (16), 32 x
// 0.1-6 k 40.9 (8), 33.0 (16), 43 x 1500 28 (5), 25 (10), 43 x 0.1-6 k 62 (5), 42 (10), 64
// x 1000 25 (4), 24 (8), 64 x 0.1-6 k 78 (4), 55 (8); and what one per CU leaves room for of
// two: 24 x 500 15.8 (8), 17.7 (4), 32 x 1000 18.6 (8), 19.3 (16). Still more in tables of
// 512 to 1024 keys the same: 90 x 600 33 (parts of 16 tiles), 23 (of 4), 128 x 0.1-0.9 k
// 35, 27, but 256 x 300 26.5, 32. Else parts of 16 tiles, so that a long sequence among
// short ones is no chain that outlasts the rest: 90 x 0.1-6 k 74 (6), 84 (5, of 4 tiles),
// 300 x 0.1-4 k 188 (2), 210 (1).
struct LsParts { long room, per, few; };
static LsParts ls_parts(long wgs, long table_width, int window) {
  long tiles = (table_width + 1) / 2;
  if (window > 0) tiles = std::min<long>(tiles, window / LS_KT + 2);
  LsParts x;
  if (wgs < 24) x = {256 / wgs, 2, 0};
  else if (wgs < 86) x = {512 / wgs, 4, 256 / wgs};
  else if (wgs <= 256 && tiles > 16 && tiles <= 32) x = {512 / wgs, 4, 0};
  else x = {(512 + wgs - 1) / wgs, 16, 0};
  const long most = std::max((tiles + x.per - 1) / x.per,
                             std::min(x.few, (tiles + 1) / 2));
  x.room = std::min<long>({x.room, most, 32});
  return x;
}
static long ls_wgs(int n_seqs, int heads) {
  return std::max<long>(1, (long)n_seqs * ((heads + 15) / 16));
}
int latent_stream_parts(int n_seqs, int heads, long table_width, int window) {
  return (int)ls_parts(ls_wgs(n_seqs, heads), table_width, window).room;
}

// q, cache and out 16 B aligned
void launch_latent_stream(float* out, float* ws_o, float* ws_ml,
                          const unsigned short* q, const unsigned short* cache,
                          const int* block_tables, const int* seq_lens,
                          int n_seqs, int heads, int W, int table_width,
                          float scale, int n_part, int window, hipStream_t st) {
  if (n_seqs == 0) return;
  const dim3 grid(n_seqs * n_part, (heads + 15) / 16);
  const LsParts p = ls_parts(ls_wgs(n_seqs, heads), table_width, window);
  auto k = W == 512 ? latent_stream_kernel<512> : latent_stream_kernel<576>;
  hipLaunchKernelGGL(k, grid, dim3(256), 0, st, out, ws_o, ws_ml, q, cache,
                     block_tables, seq_lens, heads, table_width, scale, n_part,
                     (int)p.per, (int)p.few, window);
  if (n_part > 1) {
    const long rows = (long)n_seqs * heads;
    hipLaunchKernelGGL(latent_stream_merge_kernel,
                       dim3((unsigned)((rows + 1) / 2)), dim3(256), 0, st, out,
                       ws_o, ws_ml, n_part, (int)p.per, (int)p.few, rows, heads,
                       seq_lens, window);
  }
}

}  // namespace hyb
}  // namespace xllm
