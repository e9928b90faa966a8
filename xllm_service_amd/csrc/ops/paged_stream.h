// Paged attention of decoded rows on MI355X (gfx950 / CDNA4).
//
// One new token per sequence: for one (sequence, kv_head) the G query heads
// (G <= 32) are the columns of S^T = K Q^T and of O^T += V^T P^T, as in
// paged_rows.h (layouts: mfma_rows.h); most columns are padding and
// the matrix pipe does not notice, the kernel is a stream over the cache.
//
//   * every WAVE streams tiles of 32 keys (2 pages) of its own, through 16 KB
//     of LDS of its own, straight from memory (global_load_lds, 16 B per lane):
//     no registers hold data in flight, no barrier in the loop. While the
//     scores of a tile are made its values are on the way, while its values
//     are multiplied the next keys are: counted waits, each for the older half
//   * 8 waves a CU (LDS-bound) keep 64-128 KB in flight per CU, four times
//     what memory latency times bandwidth asks for
//   * waves of a workgroup merge through LDS at the end; where there are too
//     few (sequence, kv_head) pairs to fill the chip, or tables long enough for
//     one sequence to outlast the others, the keys are split over up to P
//     workgroups, as many as a sequence's own length asks for, of whose fp32
//     results the last one to finish makes the sequence's (paged_meet)
//
// Measured, 32 query / 8 key heads of 128: 128 sequences of 1-2 k keys 160 ->
// 143 us, 5.6 TB/s (a large copy: 4.9); 24 x 0.6-1.3 k 24 + 9 -> 18 us; one of
// 776: 16 -> 8 us. 28/4 heads, 6 x 9-20 k: 54 + 16 -> 28 + 4 us. Before: K in
// registers a tile ahead, V loaded in the tile that used it, one result per
// wave through memory. What a second kernel for the merge cost, and parts that
// were larger for it, us with its launch -> here: one of 776 10.6 -> 7.5, 6 x 9-20 k
// 38.4 -> 37.0, 16 x 0.5-4 k 31.3 -> 25.5. What is left of it is a chain of three
// trips to memory: results out, the count, all results in.
#pragma once
#include <algorithm>

#include "paged_merge.h"

namespace xllm {

#define PA_BS 16           // cache block size (tokens)
#define PA_KT 32           // keys per tile (2 cache blocks)

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

// TERMS: bf16 terms a softmax weight is split into (2: its upper 16 bits of
// mantissa; 3: all of them). MORE: the options of PagedMore.
//   Two terms cost no product of their own: columns 16 and up are padding where
// at most 8 heads share a key head. They hold the queries of columns 0 to 15
// again, and their lanes, which make the same weights, keep the second terms.
// With one rounded term the results' error depended on how many weights were the
// largest of their wave, and so exact: 24 x 0.6-1.4 k keys 0.00192 of the result,
// by 32 waves a row 0.00186; with two 0.00166, which is the rounding to bf16. Us,
// one term | two by a product of their own | here: 1 x 776 keys 9.0 | 9.6 | 9.5,
// 24 x 0.6-1.4 k 18.9 | 19.6 | 19.1, 128 x 1-2 k 142.5 | 142.8 | 142.0.
//   NW: waves of a workgroup, four but where the host asks for two. SPLIT: there is room
// for parts (without the code for them 5.05 -> 4.93 us for a few keys).
template <int D, int TERMS, bool MORE, int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64, NW == 2 && D == 64 ? 8 : 2) void
paged_attn_stream_kernel(
    void* __restrict__ out,                  // [S, n_qheads, D]
    float* __restrict__ ws_o,                // [S*n_qheads][P][D] (P > 1)
    float* __restrict__ ws_ml,               // [S*n_qheads][P][2]
    const unsigned short* __restrict__ q,    // [num_seqs, n_qheads, D] bf16
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, BS, D]
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ seq_lens,        // [num_seqs]
    const float scale, const int G, const int n_kv, const int max_blocks,
    const long q_stride, const long out_stride, const PagedSplit split,
    const PagedMeet meet, const PagedMore x) {
  constexpr int KS = D / 16, DT = D / 32;
  constexpr bool FOLD = TERMS == 2;          // G <= 8
  constexpr int NP = FOLD ? 1 : TERMS;       // products per weight
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = PA_KT / RPI;            // ... instructions per tile
  constexpr int TILE = PA_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short kv_lds[NW * 2 * TILE];
  __shared__ float ml_lds[NW][32][2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;
  // first the first parts of all: idle ones are then the last and not all of one
  // XCD (16 x 1000 keys of 8 heads with room for 8: 55 us the other way, 22 so)
  const int P = SPLIT ? split.parts : 1, units = gridDim.x / P;
  const int part = blockIdx.x / units, unit = blockIdx.x % units;
  const int seq = unit / n_kv, kvh = unit % n_kv;
  const int seq_len = seq_lens[seq];
  const int n_tiles = (seq_len + PA_KT - 1) / PA_KT;
  // a wave's tiles are every step-th of the list, from the i0-th on
  const PagedTiles list =
      paged_tiles<MORE>(x, seq_len, seq_len, n_tiles, PA_KT);
  const int parts = SPLIT ? split.of(list.n) : 1;
  if (SPLIT && part >= parts) return;
  u64 seen = 0;
  if (SPLIT && parts > 1 && tid == 0) seen = paged_seen(meet.count + unit);
  const int step = parts * NW, i0 = part * NW + wid;
  const int lo = paged_first<MORE>(x, seq_len);   // first key in the window

  const int col = FOLD ? c32 & 15 : c32;
  const bool second = FOLD && c32 >= 16;     // second terms of column col
  const unsigned first = second ? 0xffff0000u : 0u;   // what the others keep
  const bool row_ok = col < G;
  const int head = kvh * G + col;
  const PagedScore sc = paged_score<MORE>(x, scale, row_ok ? head : kvh * G);
  // padding columns hold the first head's query: their results go nowhere
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
    qf[ks] = *reinterpret_cast<const bf16x8*>(
                 q + (long)seq * q_stride +
                 (long)(row_ok ? head : kvh * G) * D + ks * 16 + h * 8) ^
             sc.flip;
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
  // used; a table without columns has no entry to read)
  auto pages_from = [&](int n) {
    return max_blocks <= 0
        ? 0
        : btab[min(2 * list.at(i0 + (n + (lane >> 1)) * step) + (lane & 1),
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
  if (SPLIT && parts > 1 && tid == 0) paged_open(meet.count + unit, seen, meet.tag);
  if (i0 < list.n) {
    load(list.at(i0), 0, pages, false);
    load(list.at(i0), 0, pages, true);
  }
  for (int i = i0, n = 0; i < list.n; i += step, n++) {
    const int t = list.at(i);
    const bool more = i + step < list.n;
    wait_older();                              // K of this tile is there
    bf16x8 k[KS];
    pa_rows<D>(kat, k);
    f32x16 s[1] = {mr_zero()};
#pragma unroll
    for (int ks = 0; ks < KS; ks++) s[0] = mr_mma(k[ks], qf[ks], s[0]);
    int ids = pages;
    if (more) {
      if (n + 1 - tb == 32) {
        ids = pages_from(n + 1);
        asm volatile("" : "+v"(ids));          // the wait for them stays here
        tb += 32;
      }
      load(list.at(i + step), n + 1, ids, false);
    }
    if (MORE && x.cap > 0.0f) paged_cap<1>(s, sc.pre, x.cap);
    if (t == n_tiles - 1 || (MORE && t * PA_KT < lo)) {      // uniform
      paged_mask<MORE>(x, s, seq_len, lo, [&](int, int r) {
        return t * PA_KT + mr_key_of(r, h);
      });
    }
    const float c = sc.c;                      // weights are 2^(c (s - m))
    float mt = s[0][0];
#pragma unroll
    for (int r = 1; r < 16; r++) mt = fmaxf(mt, s[0][r]);
    mt = pair_max(mt);
    if (__any(mt > m)) {
      const float m_new = fmaxf(m, mt);
      const float alpha =
          __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int j = 0; j < DT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o_acc[j][r] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    bf16x8 p[NP][2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      float a = __builtin_amdgcn_exp2f(fmaf(s[0][r], c, -mc));
      float b = __builtin_amdgcn_exp2f(fmaf(s[0][r + 1], c, -mc));
      l += a + b;
#pragma unroll
      for (int e = 0; e < NP; e++) {
        unsigned u;
        if constexpr (FOLD) {
          a -= __uint_as_float(__float_as_uint(a) & first);
          b -= __uint_as_float(__float_as_uint(b) & first);
          u = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a),
                                    0x07060302u);
        } else {
          u = pack_bf16(a, b);
          drop_bf16(a, b, u);
        }
        reinterpret_cast<unsigned*>(&p[e][r >> 3])[(r & 7) >> 1] = u;
      }
    }
    if (more) wait_older();                    // V of this tile is there
    else wait_all();
    bf16x8 v[DT];
    pa_cols<D, 0>(vat, v);
#pragma unroll
    for (int j = 0; j < DT; j++)
#pragma unroll
      for (int e = 0; e < NP; e++)
        o_acc[j] = mr_mma(v[j], p[e][0], o_acc[j]);
    pa_cols<D, 32 * D>(vat, v);
#pragma unroll
    for (int j = 0; j < DT; j++)
#pragma unroll
      for (int e = 0; e < NP; e++)
        o_acc[j] = mr_mma(v[j], p[e][1], o_acc[j]);
    if (more) load(list.at(i + step), n + 1, ids, true);
    pages = ids;
  }
  l = pair_sum(l);

  // ---- the waves' results meet in LDS ----------------------------------------
  __syncthreads();
  const int R = FOLD ? 2 * G : G;                        // second terms apart
  constexpr int DP = FOLD ? D + 4 : D;                   // rows on other banks
  float* mo = reinterpret_cast<float*>(kv_lds);          // [NW][R][DP]
  if (row_ok) {
    if (h == 0 && !second) {
      ml_lds[wid][col][0] = m == -INFINITY ? m : m * sc.c;
      ml_lds[wid][col][1] = l;
    }
    float* mine = mo + (wid * R + (second ? G : 0) + col) * DP + 4 * h;
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4*>(mine + i * 32 + 2 * r) =
            make_float4(o_acc[i][r], o_acc[i][r + 1], o_acc[i][r + 2],
                        o_acc[i][r + 3]);
  }
  __syncthreads();
  // parts of this unit's rows
  const long rows_at = ((long)seq * n_kv + kvh) * G * P;
  const auto unit_o = mr_buffer(ws_o + rows_at * D, parts == 1 ? 0 : G * P * D * 4);
  const auto unit_ml = mr_buffer(ws_ml + rows_at * 2, parts == 1 ? 0 : G * P * 8);
  for (int idx = tid; idx < G * (D / 4); idx += NW * 64) {
    const int row = idx / (D / 4), at = idx % (D / 4) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; w++) M = fmaxf(M, ml_lds[w][row][0]);
    const float Mu = M == -INFINITY ? 0.0f : M;
    float L = 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = __builtin_amdgcn_exp2f(ml_lds[w][row][0] - Mu);
      L += ml_lds[w][row][1] * f;
      const float* from = mo + (w * R + row) * DP + at;
      float4 y = *reinterpret_cast<const float4*>(from);
      if (FOLD) {
        const float4 z = *reinterpret_cast<const float4*>(from + G * DP);
        y.x += z.x; y.y += z.y; y.z += z.z; y.w += z.w;
      }
      a[0] += y.x * f; a[1] += y.y * f; a[2] += y.z * f; a[3] += y.w * f;
    }
    if (!SPLIT || parts == 1) {
      if (MORE && x.sink != nullptr) L += paged_sink(x, kvh * G + row, M);
      const float inv = L != 0.0f ? 1.0f / L : 0.0f;
      paged_put<MORE>(x, out, (long)seq * out_stride +
                      (long)(kvh * G + row) * D + at,
                      a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv);
    } else {
      const int slot = row * P + part;
      if (at == 0) mr_store_far2(unit_ml, slot * 8, make_float2(M, L));
      mr_store_far(unit_o, (slot * D + at) * 4,
                   make_float4(a[0], a[1], a[2], a[3]));
    }
  }
  int* flag = reinterpret_cast<int*>(kv_lds);
  if (!SPLIT || parts == 1 || !paged_last(meet.count + unit, parts, flag)) return;
  // ---- all parts are there ----------------------------------------------------
  for (int idx = tid; idx < G * (D / 4); idx += NW * 64) {
    const int row = idx / (D / 4), at = idx % (D / 4) * 4;
    const bool sink = MORE && x.sink != nullptr;
    float M = sink ? x.sink[kvh * G + row] * 1.4426950408889634f : -INFINITY;
    float L = sink ? 1.0f : 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int slot = row * P;
    paged_add_parts<8>(
        [&](int p) { return mr_load_far2(unit_ml, (slot + p) * 8); },
        [&](int p) { return mr_load_far(unit_o, ((slot + p) * D + at) * 4); },
        parts, M, L, a);
    const float inv = L != 0.0f ? 1.0f / L : 0.0f;
    paged_put<MORE>(x, out, (long)seq * out_stride +
                    (long)(kvh * G + row) * D + at,
                    a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv);
  }
}

// Parts the keys of a (sequence, kv_head) pair are split into: room for P of them
// from what the host knows (the pairs and the widest table), as many as a sequence's
// own tiles ask for in the kernel (PagedSplit::of).
//   Few pairs: one workgroup per CU is enough to split for. Up to eight parts one tile
// for each wave is best, beyond them two, and what is done in three turns of a wave not
// worth the merge. Us, 8 key heads, by parts: 1 x 776 keys 12.2 whole, 8.9 (4), 8.1 (8);
// 1 x 2000 21, 9.4 (8), 10.0 (16); 1 x 20000 182, 22.8 (16); 1 x 300 7.7, 7.6 (3), 1 x 400
// 8.7, 8.4 (2), 7.5 (4); 8 x 500 9.5, 9.1 (4), 8 x 2000 26, 17.7 (4); 64-wide, 4 x 400 7.9,
// 7.5 (4), but 7 x 400, with room for three, 7.9, 8.4.
//   With options (a window, a cap, a sink) weights have 32 bits and a tile is longer: four
// tiles a part however many, from nine on (4 key heads, 1 x 300 keys, capped 10.5 whole,
// 8.3 in three, 1 x 1000 19.7, 8.5 in eight; a window of 512 12.0, 8.2 in five).
//   Up to 128 pairs in tables of up to 4096 keys, two parts, whose 256 workgroups fill one
// turn, of sequences over 24 tiles (40 from 118 pairs on, which lose by it when they are
// equal); us, whole | two: 13 x 1.9-2.6 k 31.8 | 26.8, 11 x 0.5-4 k 31.0 | 21.6, 4 key heads, 29 x
// 0.9-2.5 k 29.7 | 24.8, 24 x 0.4-1.25 k 14.9 | 13.0, 31 x 1.1-1.4 k 16.1 | 18.2. Three or four fill
// it and a bit: 11 x 2000 23.8, 21.6 in two. Longer tables by 32 tiles, as those of more pairs,
// so that none of a batch outlasts the rest: by 16 | at most two | by 32, 11 x 0.9-8 k 51.6 |
// 52.3 | 44.5, 4 key heads, 26 x 0.3-4.9 k in tables of 8192 42.0 | 37.9 | 35.3.
//   More pairs fill the chip, and equal ones lose by a split what the merge costs (24 x
// 0.6-1.4 k 22.8 | 26.4; 32 x 1-2 k 38.2 | 41.3), but a long sequence among short ones is a
// chain of tiles that outlasts the rest. By parts of 32 tiles, at most 8: 8 key heads, 16 x
// 2-16 k 173 | 142, 48 x 0.3-8 k 184 | 159, 32 x 0.3-6 k 83.3 | 82.4. The host sees no
// lengths, and in a captured step the widest table there can be: whole up to 4096 keys.
// From 768 pairs on they are whole in any table: idle parts and the merge cost short
// sequences up to twice their time (tables of 8192, 8 key heads, 128 x 16 keys 12.3 whole
// | 18.1, x 64 15.4 | 19.2; 32 key heads, 256 x 16 65 | 113), and neither even nor uneven
// lengths gain by parts there. 512 to 767 pairs do: 8 key heads, 66 x 3.6-7.3 k 232 | 212, 32
// key heads, 22 x 0.2-8.7 k 277 | 241, against 64 x 16 keys 7.9 | 10.9, x 200 15.5 | 16.7.
//   Capped scores take twice as long: with many pairs below 512, from 1500 keys on at most
// four parts of 20 tiles (1024 pairs of 16 keys in tables of 4096 8.6 in one | 16.5). 4 key
// heads: 32 x 0.7-3 k 47 | 30, 32 x 0-4 k 61 | 37, 64 x 0.3-3 k 54 | 51, 24 x 0.1-1 k in tables
// of 4096 20 | 19 (parts of 16: 31, 37, 50, 17; of 32: 31, 36, 54, 22).
//   Eight waves in a workgroup instead of four: within 5 % where keys are split and where
// they are not, slower for many pairs (128 x 300 keys: 41 against 33).
inline PagedSplit paged_stream_split(long num_seqs, int n_kv_heads,
                                     long max_blocks, bool options = false,
                                     bool capped = false) {
  const long units = num_seqs * n_kv_heads;
  // a table without columns, of sequences without keys, is one part like any other
  const long table = std::max<long>(1, (max_blocks * PA_BS + PA_KT - 1) / PA_KT);
  PagedSplit x;
  if (units == 0) return x;
  if (units < 86) {
    x.parts = (int)std::min<long>(256 / units, 16);
    x.per = options ? 4 : 8;
    x.near = 4;
    x.least = options ? 9 : x.parts < 4 ? 17 : 13;
    x.parts = x.of((int)std::min<long>(table, 1 << 20));
    return x;
  }
  if (units <= 128 && !options && table <= 128) {
    x.per = units < 118 ? 24 : 40;
    x.parts = table > x.per ? 2 : 1;
    return x;
  }
  const long f = capped ? 2 : 1, tiles = f * table;
  x.per = capped ? 20 : 32;
  if (tiles < 96 || (units > 128 && !capped && tiles <= 128) ||
      (capped && units >= 512) || (!options && units >= 768))
    return x;
  x.parts = (int)std::min<long>(8 / f, (tiles + 31) / 32);
  return x;
}

// Decoded rows (at most 32 query heads per key head, 8 with two terms) and the
// merge of their parts
template <int D, int TERMS, bool MORE>
inline void paged_stream(void* out, float* ws_o, float* ws_ml,
                         const unsigned short* q, const unsigned short* k_cache,
                         const unsigned short* v_cache, const int* block_tables,
                         const int* seq_lens, int num_seqs, float scale,
                         int n_qheads, int n_kv, int max_blocks, long q_stride,
                         long out_stride, PagedSplit split, const PagedMore& x,
                         hipStream_t stream) {
  if (num_seqs == 0) return;
  const dim3 grid((unsigned)(num_seqs * n_kv * split.parts));
  PagedMeet meet;
  if (split.parts > 1)
    meet = paged_meet(ws_ml, (long)num_seqs * n_qheads, split.parts);
#define PS_GO(NW, SPLIT)                                                       \
  hipLaunchKernelGGL((paged_attn_stream_kernel<D, TERMS, MORE, NW, SPLIT>),    \
                     grid, dim3(NW * 64), 0, stream, out, ws_o, ws_ml, q,      \
                     k_cache, v_cache, block_tables, seq_lens, scale,          \
                     n_qheads / n_kv, n_kv, max_blocks, q_stride, out_stride,  \
                     split, meet, x)
  if (split.parts > 1) PS_GO(4, true);
  else if (!MORE && split.waves == 2) PS_GO((MORE ? 4 : 2), false);
  else PS_GO(4, false);
#undef PS_GO
}

}  // namespace xllm
