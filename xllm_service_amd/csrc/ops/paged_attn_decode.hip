// Paged-attention DECODE kernel for MI355X (gfx950 / CDNA4) — MFMA-based.
//
// One new token per sequence: for one (sequence, kv_head) the G query heads
// (G <= 32) are the columns of S^T = K Q^T and of O^T += V^T P^T, as in
// paged_attn_prefill.hip (layouts: mfma_rows.h); most columns are padding and
// the matrix pipe does not notice, the kernel is a stream over the cache.
//
//   * every WAVE streams tiles of 32 keys (2 pages) of its own, through 16 KB
//     of LDS of its own, straight from memory (global_load_lds, 16 B per lane):
//     no registers hold data in flight, no barrier in the loop. While the
//     scores of a tile are made its values are on the way, while its values
//     are multiplied the next keys are: counted waits, each for the older half
//   * 8 waves a CU (LDS-bound) keep 64-128 KB in flight per CU, four times
//     what memory latency times bandwidth asks for
//   * waves of a workgroup merge through LDS at the end; when there are too
//     few (sequence, kv_head) pairs to fill the chip the keys are split over
//     P workgroups, whose fp32 results a second kernel merges
//
// Measured, 32 query / 8 key heads of 128: 128 sequences of 1-2 k keys 160 ->
// 143 us, 5.6 TB/s (a large copy: 4.9); 24 x 0.6-1.3 k 24 + 9 -> 18 us; one of
// 776: 16 -> 8 us. 28/4 heads, 6 x 9-20 k: 54 + 16 -> 28 + 4 us. Before: K in
// registers a tile ahead, V loaded in the tile that used it, one result per
// wave through memory.
//
// Parity: reference engine's paged-attention decode.
#include "mfma_rows.h"

namespace xllm {

#define PA_BS 16           // cache block size (tokens)
#define PA_KT 32           // keys per tile (2 cache blocks)
#define PA_NW 4            // waves per workgroup

// Columns [0, D) of 16 rows of a V image: the A operands of one step of
// O^T += V^T P^T. The wait is part of it: a builtin here would make the compiler
// wait for every load in flight to LDS, the next keys among them.
template <int D, int OFF>
XLLM_DEV void pa_cols(const unsigned (&at)[D / 32], bf16x8 (&v)[D / 32]) {
  typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
  u32x2 t[2 * (D / 32)];
  if constexpr (D == 128)
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8 offset:%12\n\t"
        "ds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
        "ds_read_b64_tr_b16 %2, %9 offset:%12\n\t"
        "ds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
        "ds_read_b64_tr_b16 %4, %10 offset:%12\n\t"
        "ds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
        "ds_read_b64_tr_b16 %6, %11 offset:%12\n\t"
        "ds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(t[4]),
          "=&v"(t[5]), "=&v"(t[6]), "=&v"(t[7])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(OFF),
          "n"(OFF + 8 * D)
        : "memory");
  else
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4 offset:%6\n\t"
        "ds_read_b64_tr_b16 %1, %4 offset:%7\n\t"
        "ds_read_b64_tr_b16 %2, %5 offset:%6\n\t"
        "ds_read_b64_tr_b16 %3, %5 offset:%7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3])
        : "v"(at[0]), "v"(at[1]), "n"(OFF), "n"(OFF + 8 * D)
        : "memory");
#pragma unroll
  for (int i = 0; i < D / 32; i++) {
    const unsigned x[4] = {t[2 * i][0], t[2 * i][1], t[2 * i + 1][0],
                           t[2 * i + 1][1]};
    __builtin_memcpy(&v[i], x, 16);
  }
}

// 32 rows of a K image: the A operands of S^T = K Q^T, with their wait (as above)
template <int D>
XLLM_DEV void pa_rows(const unsigned (&at)[D / 16], bf16x8 (&k)[D / 16]) {
  if constexpr (D == 128)
    asm volatile(
        "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
        "ds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %12\n\tds_read_b128 %5, %13\n\t"
        "ds_read_b128 %6, %14\n\tds_read_b128 %7, %15\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3]), "=&v"(k[4]),
          "=&v"(k[5]), "=&v"(k[6]), "=&v"(k[7])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "v"(at[4]),
          "v"(at[5]), "v"(at[6]), "v"(at[7])
        : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
        "ds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
        : "memory");
}

// TERMS: bf16 terms a softmax weight is split into (1: rounded; 3: all of its
// 32 bits).
template <int D, int TERMS>
__global__ __launch_bounds__(PA_NW * 64, 2) void paged_attn_decode_kernel(
    unsigned short* __restrict__ out,        // [S, n_qheads, D]
    float* __restrict__ ws_o,                // [S*n_qheads][P][D] (P > 1)
    float* __restrict__ ws_ml,               // [S*n_qheads][P][2]
    const unsigned short* __restrict__ q,    // [num_seqs, n_qheads, D] bf16
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, BS, D]
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ seq_lens,        // [num_seqs]
    const float scale, const int G, const int n_kv, const int max_blocks,
    const long q_stride, const long out_stride, const int P) {
  constexpr int NW = PA_NW, KS = D / 16, DT = D / 32;
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = PA_KT / RPI;            // ... instructions per tile
  constexpr int TILE = PA_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short kv_lds[NW * 2 * TILE];
  __shared__ float ml_lds[NW][32][2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;
  const int part = blockIdx.x % P, unit = blockIdx.x / P;
  const int seq = unit / n_kv, kvh = unit % n_kv;
  const int seq_len = seq_lens[seq];
  const int n_tiles = (seq_len + PA_KT - 1) / PA_KT;
  const int step = P * NW;                   // tiles from one to a wave's next
  const int t0 = part * NW + wid;

  const bool row_ok = c32 < G;
  const int head = kvh * G + c32;
  // weights are 2^(c (s - m)); a negative scale turns the queries' signs
  const short flip = scale < 0.0f ? (short)0x8000 : (short)0;
  const float c = fmaxf(fabsf(scale) * 1.4426950408889634f, 1e-30f);
  // padding columns hold the first head's query: their results go nowhere
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
    qf[ks] = *reinterpret_cast<const bf16x8*>(
                 q + (long)seq * q_stride +
                 (long)(row_ok ? head : kvh * G) * D + ks * 16 + h * 8) ^
             flip;
  f32x16 o_acc[DT];
#pragma unroll
  for (int i = 0; i < DT; i++) o_acc[i] = mr_zero();
  float m = -INFINITY, l = 0.0f;

  // ---- loads: pages 2t and 2t + 1 of the sequence --------------------------
  const int* btab = block_tables + (long)seq * max_blocks;
  const int last_blk = (seq_len - 1) / PA_BS;
  const int last_row = (seq_len - 1) % PA_BS;
  const int srow = lane / CPR, spos = lane % CPR;
  unsigned short* kt = kv_lds + wid * 2 * TILE;
  unsigned short* vt = kt + TILE;
  auto off_of = [&](int r, bool val) {       // bytes into a page
    const int x = val ? mr_swz_cols<D>(r) : mr_swz_rows<D>(r);
    return (unsigned)(r * (2 * D) + ((spos ^ x) << 4));
  };
  unsigned koff[NI / 2], voff[NI / 2];
#pragma unroll
  for (int i = 0; i < NI / 2; i++) {
    koff[i] = off_of(i * RPI + srow, false);
    voff[i] = off_of(i * RPI + srow, true);
  }
  // ids of 32 of the wave's tiles from the tb-th on, two lanes a tile
  int tb = 0;
  // (read without waiting for the length: what lies past the last page is not
  // used)
  auto pages_from = [&](int n) {
    return btab[min(2 * (t0 + (n + (lane >> 1)) * step) + (lane & 1),
                    max_blocks - 1)];
  };
  auto load = [&](int t, int n, int pages, bool val) {
    const char* cache = reinterpret_cast<const char*>(val ? v_cache : k_cache);
    unsigned short* dst = val ? vt : kt;
    const int page0 = __builtin_amdgcn_readlane(pages, 2 * (n - tb));
    const int page1 = 2 * t + 1 > last_blk
        ? page0 : __builtin_amdgcn_readlane(pages, 2 * (n - tb) + 1);
    const char* src0 = cache + ((long)page0 * n_kv + kvh) * (PA_BS * D * 2);
    const char* src1 = cache + ((long)page1 * n_kv + kvh) * (PA_BS * D * 2);
    auto move = [&](int i, unsigned off) {
      __builtin_amdgcn_global_load_lds(
          (glb_void*)((i < NI / 2 ? src0 : src1) + off),
          (lds_void*)(dst + i * RPI * D), 16, 0, 0);
    };
    if (2 * t + 1 < last_blk) {
#pragma unroll
      for (int i = 0; i < NI; i++)
        move(i, val ? voff[i % (NI / 2)] : koff[i % (NI / 2)]);
      return;
    }
    // rows past the last key repeat it: masked below, and finite
    unsigned off[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int ii = i % (NI / 2), r = ii * RPI + srow;
      const int pg = 2 * t + i / (NI / 2);
      const int rr = pg < last_blk ? r : pg > last_blk ? last_row
                                       : min(r, last_row);
      off[i] = (val ? voff[ii] : koff[ii]) + (rr - r) * (2 * D);
    }
#pragma unroll
    for (int i = 0; i < NI; i++) move(i, off[i]);
  };
  // everything but the NI loads issued last has arrived
  auto wait_older = [&] {
    if constexpr (NI == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  };
  auto wait_all = [&] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

  const int kbase = mr_row_base<D>(lane), vbase = mr_col_base<D>(lane);
  unsigned kat[KS], vat[DT];                   // LDS bytes
#pragma unroll
  for (int i = 0; i < KS; i++)
    kat[i] = (unsigned)(unsigned long long)((const lds_u16*)kt +
                                            (kbase ^ (i << 4)));
#pragma unroll
  for (int i = 0; i < DT; i++)
    vat[i] = (unsigned)(unsigned long long)((const lds_u16*)vt +
                                            (vbase ^ (i << 5)));
  int pages = pages_from(0);
  if (t0 < n_tiles) {
    load(t0, 0, pages, false);
    load(t0, 0, pages, true);
  }
  for (int t = t0, n = 0; t < n_tiles; t += step, n++) {
    const bool more = t + step < n_tiles;
    wait_older();                              // K of this tile is there
    bf16x8 k[KS];
    pa_rows<D>(kat, k);
    f32x16 s = mr_zero();
#pragma unroll
    for (int ks = 0; ks < KS; ks++) s = mr_mma(k[ks], qf[ks], s);
    int ids = pages;
    if (more) {
      if (n + 1 - tb == 32) {
        ids = pages_from(n + 1);
        asm volatile("" : "+v"(ids));          // the wait for them stays here
        tb += 32;
      }
      load(t + step, n + 1, ids, false);
    }
    if (t == n_tiles - 1) {
#pragma unroll
      for (int r = 0; r < 16; r++)
        if (t * PA_KT + mr_key_of(r, h) >= seq_len) s[r] = -INFINITY;
    }
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mt = fmaxf(mt, s[r]);
    mt = pair_max(mt);
    if (__any(mt > m)) {
      const float m_new = fmaxf(m, mt);
      const float alpha =
          __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o_acc[i][r] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    bf16x8 p[TERMS][2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      float a = __builtin_amdgcn_exp2f(fmaf(s[r], c, -mc));
      float b = __builtin_amdgcn_exp2f(fmaf(s[r + 1], c, -mc));
      l += a + b;
#pragma unroll
      for (int x = 0; x < TERMS; x++) {
        const unsigned u = pack_bf16(a, b);
        reinterpret_cast<unsigned*>(&p[x][r >> 3])[(r & 7) >> 1] = u;
        drop_bf16(a, b, u);
      }
    }
    if (more) wait_older();                    // V of this tile is there
    else wait_all();
    bf16x8 v[DT];
    pa_cols<D, 0>(vat, v);
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
      for (int x = 0; x < TERMS; x++)
        o_acc[i] = mr_mma(v[i], p[x][0], o_acc[i]);
    pa_cols<D, 32 * D>(vat, v);
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
      for (int x = 0; x < TERMS; x++)
        o_acc[i] = mr_mma(v[i], p[x][1], o_acc[i]);
    if (more) load(t + step, n + 1, ids, true);
    pages = ids;
  }
  l = pair_sum(l);

  // ---- the waves' results meet in LDS ----------------------------------------
  __syncthreads();
  float* mo = reinterpret_cast<float*>(kv_lds);          // [NW][G][D]
  if (row_ok) {
    if (h == 0) {
      ml_lds[wid][c32][0] = m == -INFINITY ? m : m * c;
      ml_lds[wid][c32][1] = l;
    }
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4*>(mo + (wid * G + c32) * D + i * 32 + 2 * r +
                                   4 * h) =
            make_float4(o_acc[i][r], o_acc[i][r + 1], o_acc[i][r + 2],
                        o_acc[i][r + 3]);
  }
  __syncthreads();
  for (int idx = tid; idx < G * (D / 4); idx += NW * 64) {
    const int row = idx / (D / 4), col = idx % (D / 4) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; w++) M = fmaxf(M, ml_lds[w][row][0]);
    const float Mu = M == -INFINITY ? 0.0f : M;
    float L = 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = __builtin_amdgcn_exp2f(ml_lds[w][row][0] - Mu);
      L += ml_lds[w][row][1] * f;
      const float4 x =
          *reinterpret_cast<const float4*>(mo + (w * G + row) * D + col);
      a[0] += x.x * f; a[1] += x.y * f; a[2] += x.z * f; a[3] += x.w * f;
    }
    if (P == 1) {
      const float inv = L > 0.0f ? 1.0f / L : 0.0f;
      uint2 y;
      y.x = pack_bf16(a[0] * inv, a[1] * inv);
      y.y = pack_bf16(a[2] * inv, a[3] * inv);
      *reinterpret_cast<uint2*>(out + (long)seq * out_stride +
                                (long)(kvh * G + row) * D + col) = y;
    } else {
      const long slot = ((long)seq * n_kv * G + kvh * G + row) * P + part;
      if (col == 0) {
        ws_ml[slot * 2] = M;
        ws_ml[slot * 2 + 1] = L;
      }
      *reinterpret_cast<float4*>(ws_o + slot * D + col) =
          make_float4(a[0], a[1], a[2], a[3]);
    }
  }
}

// out[row] = sum_p o[row][p] 2^(m_p - M) / sum_p l_p 2^(m_p - M): D/4 lanes per
// row, four columns each
template <int D>
__global__ __launch_bounds__(256) void paged_attn_merge_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ ws_o,
    const float* __restrict__ ws_ml, const int n_qheads, const int n_part,
    const long out_stride, const long rows) {
  constexpr int LPR = D / 4;
  const long row = (blockIdx.x * 256L + threadIdx.x) / LPR;
  const int col = (threadIdx.x % LPR) * 4;
  if (row >= rows) return;
  const float2* ml = reinterpret_cast<const float2*>(ws_ml) + row * n_part;
  const float* o = ws_o + row * n_part * D + col;
  float M = -INFINITY;
  for (int p = 0; p < n_part; p++) M = fmaxf(M, ml[p].x);
  if (M == -INFINITY) M = 0.0f;
  float L = 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int p = 0; p < n_part; p++) {
    const float2 z = ml[p];
    const bool on = z.y > 0.0f;              // else nothing was written
    const float w = on ? __builtin_amdgcn_exp2f(z.x - M) : 0.0f;
    const float4 x = *reinterpret_cast<const float4*>(o + (long)p * D);
    L += on ? z.y * w : 0.0f;
    a[0] += on ? x.x * w : 0.0f; a[1] += on ? x.y * w : 0.0f;
    a[2] += on ? x.z * w : 0.0f; a[3] += on ? x.w * w : 0.0f;
  }
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  uint2 y;
  y.x = pack_bf16(a[0] * inv, a[1] * inv);
  y.y = pack_bf16(a[2] * inv, a[3] * inv);
  const long tok = row / n_qheads;
  *reinterpret_cast<uint2*>(out + tok * out_stride +
                            (row - tok * n_qheads) * D + col) = y;
}

void launch_paged_attn_merge(unsigned short* out, const float* ws_o,
                             const float* ws_ml, int n_qheads, int D,
                             int n_part, long out_stride, long rows,
                             hipStream_t stream) {
  const dim3 grid((unsigned)((rows * (D / 4) + 255) / 256));
  if (D == 128)
    hipLaunchKernelGGL((paged_attn_merge_kernel<128>), grid, dim3(256), 0,
                       stream, out, ws_o, ws_ml, n_qheads, n_part, out_stride,
                       rows);
  else
    hipLaunchKernelGGL((paged_attn_merge_kernel<64>), grid, dim3(256), 0,
                       stream, out, ws_o, ws_ml, n_qheads, n_part, out_stride,
                       rows);
}

// ---------------- other head widths: shuffle-reduce design -------------------
template <int G>
__global__ __launch_bounds__(256) void paged_attn_decode_small_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ q,
    const unsigned short* __restrict__ k_cache,
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ seq_lens,
    const float scale, const int n_kv_heads, const int D,
    const int max_blocks_per_seq, const long q_stride, const long out_stride) {
  const int seq = blockIdx.x / n_kv_heads;
  const int kvh = blockIdx.x % n_kv_heads;
  const int n_qheads = n_kv_heads * G;
  const int seq_len = seq_lens[seq];
  const int n_blocks = (seq_len + PA_BS - 1) / PA_BS;
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int tg = lane >> 4;
  const int d8 = lane & 15;
  const int dvalid = (8 * d8) < D;

  float qf[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const long qoff = (long)seq * q_stride + (long)(kvh * G + g) * D + 8 * d8;
    if (dvalid) {
      ushort8_t v = *reinterpret_cast<const ushort8_t*>(q + qoff);
#pragma unroll
      for (int j = 0; j < 8; j++) qf[g][j] = bf16_to_f32(v.x[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) qf[g][j] = 0.0f;
    }
  }
  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    m[g] = -INFINITY; l[g] = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) acc[g][j] = 0.0f;
  }
  const int* btab = block_tables + (long)seq * max_blocks_per_seq;
  const long head_stride = (long)PA_BS * D;
  for (int bi = wid; bi < n_blocks; bi += 4) {
    const long base = ((long)btab[bi] * n_kv_heads + kvh) * head_stride;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int t = j * 4 + tg;
      const int tok = bi * PA_BS + t;
      if (tok >= seq_len) continue;
      const long roff = base + (long)t * D + 8 * d8;
      float kf[8], vf[8];
      if (dvalid) {
        ushort8_t k8 = *reinterpret_cast<const ushort8_t*>(k_cache + roff);
        ushort8_t v8 = *reinterpret_cast<const ushort8_t*>(v_cache + roff);
#pragma unroll
        for (int u = 0; u < 8; u++) { kf[u] = bf16_to_f32(k8.x[u]); vf[u] = bf16_to_f32(v8.x[u]); }
      } else {
#pragma unroll
        for (int u = 0; u < 8; u++) { kf[u] = 0.0f; vf[u] = 0.0f; }
      }
#pragma unroll
      for (int g = 0; g < G; g++) {
        float s = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) s += qf[g][u] * kf[u];
        s = group_reduce_sum<16>(s) * scale;
        const float m_new = fmaxf(m[g], s);
        const float a = __expf(m[g] - m_new);
        const float p = __expf(s - m_new);
        m[g] = m_new;
        l[g] = l[g] * a + p;
#pragma unroll
        for (int u = 0; u < 8; u++) acc[g][u] = acc[g][u] * a + p * vf[u];
      }
    }
  }
  __shared__ float ml[16][G][2];
  __shared__ float accs[16][G][16][8];
  const int part = wid * 4 + tg;
  if (d8 == 0) {
#pragma unroll
    for (int g = 0; g < G; g++) { ml[part][g][0] = m[g]; ml[part][g][1] = l[g]; }
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
#pragma unroll
    for (int u = 0; u < 8; u++) accs[part][g][d8][u] = acc[g][u];
  }
  __syncthreads();
  for (int g = wid; g < G; g += 4) {
    float m_star = -INFINITY;
#pragma unroll
    for (int p = 0; p < 16; p++) m_star = fmaxf(m_star, ml[p][g][0]);
    float l_tot = 0.0f, o0 = 0.0f, o1 = 0.0f;
    const int pd8 = lane >> 2;
    const int pu = (2 * lane) & 7;
#pragma unroll
    for (int p = 0; p < 16; p++) {
      const float mw = ml[p][g][0];
      const float w = (mw == -INFINITY) ? 0.0f : __expf(mw - m_star);
      l_tot += w * ml[p][g][1];
      o0 += w * accs[p][g][pd8][pu];
      o1 += w * accs[p][g][pd8][pu + 1];
    }
    const float inv = (l_tot > 0.0f) ? 1.0f / l_tot : 0.0f;
    if (2 * lane < D) {
      const long ooff = (long)seq * out_stride + (long)(kvh * G + g) * D + 2 * lane;
      out[ooff] = f32_to_bf16(o0 * inv);
      out[ooff + 1] = f32_to_bf16(o1 * inv);
    }
  }
}

// Workgroups the keys of a (sequence, kv_head) pair are split over, from what
// the host knows: the pairs and the widest table. One workgroup per CU is
// enough to split for (more of them only add results to merge), a part of less
// than eight tiles (two a wave) is not worth its share of the merge, and
// neither is a split in two. Measured (us, 32/8 heads of 128), whole | split:
// 1 x 776 keys 10.2 | 7.8, 1 x 2000 18.8 | 8.9, 1 x 20000 143 | 20 (16 parts),
// 8 x 2000 19.9 | 15.8, 8 x 14000 144 | 82; 1 x 200 5.4 | 6.6, 8 x 500 8.6 |
// 9.7, 16 x 1000 13.6 | 15.7, 32 x 1500 36.7 | 40.2. Eight waves in a workgroup
// instead of four: within 5 % where that many keys are split at all, slower
// for many pairs (128 x 300 keys: 41 against 33).
int paged_attn_decode_parts(int num_seqs, int n_kv_heads, int max_blocks) {
  const long units = (long)num_seqs * n_kv_heads;
  const long tiles = ((long)max_blocks * PA_BS + PA_KT - 1) / PA_KT;
  long p = units > 0 ? 256 / units : 1;
  if (p > tiles / 8) p = tiles / 8;
  return (int)(p < 3 ? 1 : p > 16 ? 16 : p);
}

void launch_paged_attn_decode(unsigned short* out, const unsigned short* q,
                              const unsigned short* k_cache,
                              const unsigned short* v_cache,
                              const int* block_tables, const int* seq_lens,
                              float* ws_ml, float* ws_o, float scale,
                              int num_seqs, int n_qheads, int n_kv_heads, int D,
                              int max_blocks_per_seq, long q_stride,
                              long out_stride, int parts,
                              hipStream_t stream) {
  const int G = n_qheads / n_kv_heads;
  if (num_seqs == 0) return;
  if (D != 128 && D != 64) {
    const dim3 grid(num_seqs * n_kv_heads), block(256);
#define PA_SMALL(GV)                                                           \
  hipLaunchKernelGGL((paged_attn_decode_small_kernel<GV>), grid, block, 0,     \
                     stream, out, q, k_cache, v_cache, block_tables, seq_lens, \
                     scale, n_kv_heads, D, max_blocks_per_seq, q_stride,       \
                     out_stride)
    switch (G) {
      case 1: PA_SMALL(1); break;
      case 2: PA_SMALL(2); break;
      case 3: PA_SMALL(3); break;
      case 4: PA_SMALL(4); break;
      case 5: PA_SMALL(5); break;
      case 6: PA_SMALL(6); break;
      case 7: PA_SMALL(7); break;
      case 8: PA_SMALL(8); break;
      default: break;  // validated host-side
    }
#undef PA_SMALL
    return;
  }
  const dim3 grid((unsigned)(num_seqs * n_kv_heads * parts));
#define PA_LAUNCH(DV, TERMS)                                                   \
  hipLaunchKernelGGL((paged_attn_decode_kernel<DV, TERMS>), grid,              \
                     dim3(PA_NW * 64), 0, stream, out, ws_o, ws_ml, q,         \
                     k_cache, v_cache, block_tables, seq_lens, scale, G,       \
                     n_kv_heads, max_blocks_per_seq, q_stride, out_stride,     \
                     parts)
  // 64-wide heads have 32-bit weights, as every other width but 128
  if (D == 128) PA_LAUNCH(128, 1);
  else PA_LAUNCH(64, 3);
#undef PA_LAUNCH
  if (parts > 1)
    launch_paged_attn_merge(out, ws_o, ws_ml, n_qheads, D, parts, out_stride,
                            (long)num_seqs * n_qheads, stream);
}

}  // namespace xllm
