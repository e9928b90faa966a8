// Latent attention of decoded rows (bf16) for gfx950: rank 512 with a rotated
// tail of 0 or 64 entries, 16-token pages, at most 32 heads. Other sizes and
// prompt rows: latent_attn_mfma.hip.
//
// One new token per sequence; its heads attend to the SAME cached rows of W =
// 512 + tail entries, values are the first 512 of a row. The step is a stream
// over the cache: a workgroup (4 waves, two of them share a CU) walks tiles of
// 32 rows for 16 heads of one sequence. Tiles go from memory straight to LDS
// (global_load_lds, 16 B per lane: a page is one contiguous piece), two buffers,
// one barrier per tile, so that a tile is on the way while the other is
// computed. Before, tiles went through registers between two barriers.
//
//   S^T[key][head] = K Q^T       16x16x32 products, every wave makes all of it
//                                (A = K rows from LDS, B = Q in registers)
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
// Measured, 32 sequences of 1.5-2.4 k keys, 16 heads, rows of 576: 67 + 5 us before,
// 24 us with the merge now; the rows alone take 15 us at the rate of a large copy.
//
// The LDS reads are asm with their wait: in front of a builtin the compiler
// waits for every load to LDS in flight.
//
// Fragments of 16x16x32 (lane l, g = l >> 4): A[l&15][g*8 + j], B[g*8 +
// j][l&15], C[g*4 + r][l&15].
#include "../ops/paged_merge.h"
#include "hybrid_common.h"
#include <cstdlib>

namespace xllm {
namespace hyb {

constexpr int LS_KT = 32;       // keys per tile (two pages)
constexpr int LS_R = 512;       // value columns

template <int W> XLLM_DEV int ls_swz(int k) {
  const int lo = (((k >> 3) & 1) << 1) | ((k >> 4) & 1);
  return W == 512 ? ((k & 3) << 2) | lo : (((k >> 1) & 1) << 2) | lo;
}

// Eight K fragments: four steps of both halves. W == 512: one address per step;
// W == 576: two, and two offsets.
template <int W, int OFF>
XLLM_DEV void ls_keys(const unsigned (&at)[4], bf16x8 (&k)[2][4]) {
  constexpr int H = 8 * W;                       // bytes of four rows
  constexpr int O1 = W == 512 ? OFF : OFF + 128;
  asm volatile(
      "ds_read_b128 %0, %8 offset:%12\n\tds_read_b128 %1, %9 offset:%12\n\t"
      "ds_read_b128 %2, %10 offset:%13\n\tds_read_b128 %3, %11 offset:%13\n\t"
      "ds_read_b128 %4, %8 offset:%14\n\tds_read_b128 %5, %9 offset:%14\n\t"
      "ds_read_b128 %6, %10 offset:%15\n\tds_read_b128 %7, %11 offset:%15\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]),
        "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2]), "=&v"(k[1][3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(OFF), "n"(O1),
        "n"(OFF + H), "n"(O1 + H)
      : "memory");
}
// the last two steps of 576
template <int OFF>
XLLM_DEV void ls_keys_end(const unsigned (&at)[4], bf16x8 (&k)[2][2]) {
  asm volatile(
      "ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\t"
      "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %5 offset:%7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[1][0]), "=&v"(k[1][1])
      : "v"(at[0]), "v"(at[1]), "n"(OFF), "n"(OFF + 8 * 576)
      : "memory");
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

template <int W, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS, 2) latent_stream_kernel(
    float* __restrict__ out,               // [S, H, 512] (n_part == 1)
    float* __restrict__ ws_o,              // [S*H][n_part][512]
    float* __restrict__ ws_ml,             // [S*H][n_part][2]
    const unsigned short* __restrict__ q,  // [S, H, W]
    const unsigned short* __restrict__ cache,   // [blocks, 16, W]
    const int* __restrict__ block_tables, const int* __restrict__ seq_lens,
    int heads, int table_width, float scale, int n_part, int per, int window) {
  constexpr int CPR = W / 8;                     // 16 B chunks of a row
  constexpr int IPP = 16 * CPR / 64;             // load instructions per page
  constexpr int NI = 2 * IPP / 4;                // ... of a wave per tile
  constexpr int KS = W / 32;                     // steps of a score product
  constexpr int TILE = LS_KT * W;
  __shared__ __attribute__((aligned(1024))) unsigned short lds[TEAMS * 2 * TILE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
  const int team = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int g = lane >> 4, n = lane & 15;
  const int n_seqs = gridDim.x / n_part;
  const int part = blockIdx.x / n_seqs, s = blockIdx.x % n_seqs;  // idle last
  const int h0 = blockIdx.y * 16;                // first head
  const int seq_len = seq_lens[s];
  const int n_tiles = (seq_len + LS_KT - 1) / LS_KT;
  const int lo = window > 0 ? max(0, seq_len - window) : 0;
  const int t_first = lo / LS_KT;
  const int parts = paged_parts(n_tiles - t_first, n_part, per);
  if (part >= parts) return;
  const int tpp = (n_tiles - t_first + parts - 1) / parts;
  const int t_begin = t_first + part * tpp;
  const int t_end = min(n_tiles, t_begin + tpp);

  const bool on = h0 + n < heads;
  const long row = (long)s * heads + (on ? h0 + n : h0);
  const short flip = scale < 0.0f ? (short)0x8000 : (short)0;
  const float c = paged_factor(scale);
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
    qf[ks] = *reinterpret_cast<const bf16x8*>(q + row * W + ks * 32 + g * 8) ^
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
    unsigned short* dst = lds + (team * 2 + buf) * TILE;
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
  const unsigned base =
      (unsigned)(unsigned long long)(const lds_u16*)(lds + team * 2 * TILE);
  const int km = (n >> 2) * 8 + (n & 3);         // key of A row n, half 0
  unsigned kat[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int ch = W == 512 ? i * 4 + g : (i & 1) * 4 + g;
    kat[i] = base + 2 * (km * W + ((ch ^ ls_swz<W>(km)) << 3));
  }
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
    if (t_begin + team < t_end) stage(t_begin + team, pages, 0);
  }
  for (int i = 0; t_begin + i * TEAMS < t_end; i++) {   // as often for all teams
    const int t = t_begin + i * TEAMS + team, buf = i & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + TEAMS < t_end) {
      if (t + TEAMS - tb >= 32) {
        tb += 32;
        pages = pages_from(tb);
      }
      stage(t + TEAMS, pages, buf ^ 1);
    }
    if (t >= t_end) break;                       // the last turn
    const unsigned shift = buf * (2 * TILE);
    unsigned ka[4];
#pragma unroll
    for (int i = 0; i < 4; i++) ka[i] = kat[i] + shift;
    // ---- scores ----------------------------------------------------------------
    f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    auto four = [&](const bf16x8 (&k)[2][4], int ks) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sc[0] = ls_mma(k[0][i], qf[ks + i], sc[0]);
        sc[1] = ls_mma(k[1][i], qf[ks + i], sc[1]);
      }
    };
    {
      bf16x8 k[2][4];
      ls_keys<W, 0>(ka, k); four(k, 0);
      ls_keys<W, 256>(ka, k); four(k, 4);
      ls_keys<W, 512>(ka, k); four(k, 8);
      ls_keys<W, 768>(ka, k); four(k, 12);
      if constexpr (W == 576) {
        bf16x8 e[2][2];
        ls_keys_end<1024>(ka, e);
#pragma unroll
        for (int i = 0; i < 2; i++) {
          sc[0] = ls_mma(e[0][i], qf[16 + i], sc[0]);
          sc[1] = ls_mma(e[1][i], qf[16 + i], sc[1]);
        }
      }
    }
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
  if constexpr (TEAMS > 1) {
    __syncthreads();                             // the tiles have been read
    f32x4* const o = reinterpret_cast<f32x4*>(lds);   // [8][256]
    float2* const ml = reinterpret_cast<float2*>(lds + 8 * 256 * 8);
    if (team == 1) {
#pragma unroll
      for (int i = 0; i < 8; i++) o[i * 256 + (tid & 255)] = acc[i];
      ml[tid & 255] = make_float2(m, l);
    }
    __syncthreads();
    if (team == 1) return;
    const float2 other = ml[tid];
    const float top = fmaxf(m, other.x), from = top == -INFINITY ? 0.f : top;
    const float mine = __builtin_amdgcn_exp2f((m - from) * c);
    const float its = __builtin_amdgcn_exp2f((other.x - from) * c);
    m = top;
    l = l * mine + other.y * its;
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = acc[i] * mine + o[i * 256 + tid] * its;
  }
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
    const float* __restrict__ ws_ml, int n_part, int per, long rows, int heads,
    const int* __restrict__ seq_lens, int window) {
  const long row = blockIdx.x * 2L + (threadIdx.x >> 7);
  const int col = (threadIdx.x & 127) * 4;
  if (row >= rows) return;
  const int len = seq_lens[row / heads];
  const int parts = paged_parts(
      (len + LS_KT - 1) / LS_KT -
          (window > 0 ? max(0, len - window) / LS_KT : 0), n_part, per);
  if (parts == 1) return;                        // written where it belongs
  float M = -INFINITY, L = 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  paged_add_parts<8>(reinterpret_cast<const float2*>(ws_ml) + row * n_part,
                     ws_o + row * n_part * LS_R + col, parts, LS_R, M, L, a);
  const float inv = L != 0.0f ? 1.0f / L : 0.0f;
  *reinterpret_cast<float4*>(out + row * LS_R + col) =
      make_float4(a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv);
}

bool latent_stream_takes(int W, int r, int heads, int block_size) {
  return r == LS_R && (W == 512 || W == 576) && heads <= 32 && block_size == 16;
}

// Room for parts from what the host knows, one part for every `per` tiles of a
// sequence's own in the kernel. Few workgroups: one per CU, parts of at least two
// tiles. Measured (us, by parts): 32 x 2000 keys, 16 heads 92 (1), 32 (4), 24
// (8), 27 (16); 8 x 4000 173 (1), 32 (8), 23 (16), 21 (32); 64 x 1000 51 (1), 24
// (4), 26 (8); 1 x 700 36 (1), 13 (12). More: parts of 16 tiles, so that a long
// sequence among short ones is no chain that outlasts the rest; 128 x 600 35
// (1), 28 (2), 30 (4).
static int ls_per(long wgs) { if (getenv("LSE")) return atoi(getenv("LSE")); return wgs < 86 ? 2 : 16; }
int latent_stream_parts(int n_seqs, int heads, long table_width, int window) {
  const long wgs = std::max<long>(1, (long)n_seqs * ((heads + 15) / 16));
  long tiles = (table_width + 1) / 2;
  if (window > 0) tiles = std::min<long>(tiles, window / LS_KT + 2);
  const long per = ls_per(wgs);
  if (getenv("LSP")) return atoi(getenv("LSP"));
  const long p = wgs < 86 ? 256 / wgs : (512 + wgs - 1) / wgs;
  return (int)std::min<long>({p, (tiles + per - 1) / per, 32});
}

// q, cache and out 16 B aligned
void launch_latent_stream(float* out, float* ws_o, float* ws_ml,
                          const unsigned short* q, const unsigned short* cache,
                          const int* block_tables, const int* seq_lens,
                          int n_seqs, int heads, int W, int table_width,
                          float scale, int n_part, int window, hipStream_t st) {
  if (n_seqs == 0) return;
  const dim3 grid(n_seqs * n_part, (heads + 15) / 16);
  const int per = ls_per((long)n_seqs * grid.y);
  const bool deep = getenv("LSD") ? atoi(getenv("LSD")) : grid.x * grid.y <= 256;
  auto k = W == 512 ? (deep ? latent_stream_kernel<512, 2>
                            : latent_stream_kernel<512, 1>)
                    : (deep ? latent_stream_kernel<576, 2>
                            : latent_stream_kernel<576, 1>);
  hipLaunchKernelGGL(k, grid, dim3(deep ? 512 : 256), 0, st, out, ws_o, ws_ml, q, cache,
                     block_tables, seq_lens, heads, table_width, scale, n_part,
                     per, window);
  if (n_part > 1) {
    const long rows = (long)n_seqs * heads;
    hipLaunchKernelGGL(latent_stream_merge_kernel,
                       dim3((unsigned)((rows + 1) / 2)), dim3(256), 0, st, out,
                       ws_o, ws_ml, n_part, per, rows, heads, seq_lens, window);
  }
}

}  // namespace hyb
}  // namespace xllm
