// Paged attention of prompt rows on MI355X (gfx950 / CDNA4), MFMA-based.
//
// Flash-style online-softmax attention where K/V come from the paged KV
// cache (chunked prefill and prefix-cache hits share this one code path:
// new tokens' K/V are scattered into the cache first, then this runs).
//
// The G query heads of a key/value head attend to the same keys, so the
// (query, head) pairs of a sequence are rows of one matrix, row = query * G +
// head in group. A workgroup (4 waves) owns 128 rows of one key/value head, a
// wave 32; two workgroups share a CU. Short chunks fill their tiles better
// that way (93 queries x 7 heads: 6 tiles, not 7 x 1) and a workgroup's rows
// span few positions, so little of a tile on the diagonal is masked.
//
// Per tile of 64 keys:
//   S^T[key][row] = K Q^T        32x32x16 products, A = K rows from LDS, B = Q
//                                in registers for the whole kernel
//   online softmax               a lane holds 32 of the tile's scores of ONE
//                                row and its partner lane (l ^ 32) the others:
//                                a row maximum is a chain of v_max and one lane
//                                swap, the sums meet once, at the very end
//   O^T[d][row] += V^T P^T       A = V^T by hardware transpose reads, B = the
//                                lane's own weights, rounded to bf16: no trip
//                                through LDS
// K and V tiles go from memory straight to LDS (no registers, no ds_write),
// double-buffered with one barrier per tile. The loads place 16 B per lane in
// lane order, so rows cannot be padded; the 16 B chunks of a row are permuted
// by its key instead (on the side of the memory address), which makes both
// the row reads of K and the transpose reads of V free of bank conflicts.
//
// Few row tiles over a long context leave most of the chip idle: then the
// keys are split over n_part workgroups and a second kernel merges the fp32
// partial results.
//
// Bound by the matrix pipe and the vector unit in turn: a tile costs a wave
// 32 products (about 1000 cycles) and about as many cycles of exponentials,
// maxima and conversions, which the second wave of the SIMD overlaps; LDS
// reads feed 32 rows each and stay just below the pipe's rate. Measured, 4
// prompts of 1.6-2.3 k tokens over up to 3.1 k cached ones, 32 heads: 371 us,
// 873 TFLOP/s (a large bf16 matrix product: 1466); one head and 16 rows per
// wave on 16x16x32 products, P through LDS: 1209 us. 3 chunks of 93-261 tokens
// over 0.5-1.8 k, 28 heads, with the key split: 31 us, without a list of tiles
// made on the host; before: 110 us and 48 us of copies and waiting. 8 prompts
// of 109-438 tokens, 12 heads of 64: 13.6 us, an eager loop before: 14 ms.
//
// Fragment layouts, the order of the keys and of the LDS images: mfma_rows.h.
#pragma once
#include "paged_merge.h"

namespace xllm {

#define PF_ROWS 128        // rows per workgroup
#define PF_KT 64           // keys per tile
#define PF_BS 16           // cache block size

// Row tile `b` of the batch -> sequence and tile within it; later tiles of a
// sequence (more keys) come first. False: past the last one. One wave looks
// 64 sequences over at a time.
XLLM_DEV bool pf_locate(int b, const int* cu_q, int n_seqs, int G, int lane,
                        int* s, int* lt) {
  int acc = 0;
  for (int base = 0; base < n_seqs; base += 64) {
    const int i = base + lane;
    int nt = 0;
    if (i < n_seqs)
      nt = ((cu_q[i + 1] - cu_q[i]) * G + PF_ROWS - 1) / PF_ROWS;
    int sum = nt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(sum, off, 64);
      if (lane >= off) sum += up;
    }
    const unsigned long long hit = __ballot(b < acc + sum);
    if (hit != 0) {
      const int first = __ffsll(hit) - 1;
      *s = __builtin_amdgcn_readfirstlane(base + first);
      *lt = __builtin_amdgcn_readfirstlane(acc + __shfl(sum, first, 64) - 1 -
                                           b);
      return true;
    }
    acc += __shfl(sum, 63, 64);
  }
  return false;
}

// TERMS: bf16 terms a softmax weight is split into. One rounds it to bf16;
// three (8 + 8 + 8 mantissa bits) hold all of its 32-bit value, each with a
// product of its own into the same fp32 sums. MORE: the options of PagedMore.
template <int D, int TERMS, bool MORE>
__global__ __launch_bounds__(256, 2) void paged_attn_rows_kernel(
    void* __restrict__ out,                  // [total_q, n_qheads, D]
    float* __restrict__ ws_o,                // [total_q*n_qheads][n_part][D]
    float* __restrict__ ws_ml,               // [total_q*n_qheads][n_part][2]
    const unsigned short* __restrict__ q,    // [total_q, n_qheads, D] bf16
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, 16, D]
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ cu_q,            // [num_seqs+1] query offsets
    const int* __restrict__ seq_lens,        // [num_seqs] total key len
    const int n_seqs, const float scale, const int G, const int n_kv,
    const int max_blocks, const long q_stride, const long out_stride,
    const int n_part, const PagedMore x) {
  constexpr int KS = D / 16;                 // k steps of a score product
  constexpr int DT = D / 32;                 // 32-wide tiles of the head
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = 16 / RPI;               // ... instructions per page
  constexpr int TILE = PF_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short kv_lds[4 * TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;

  const int kvh = blockIdx.x % n_kv;
  const int part = (blockIdx.x / n_kv) % n_part;
  int seq, lt;
  if (!pf_locate(blockIdx.x / (n_kv * n_part), cu_q, n_seqs, G, lane, &seq,
                 &lt))
    return;
  const int q_start = cu_q[seq];
  const int q_len = cu_q[seq + 1] - q_start;
  const int seq_len = seq_lens[seq];
  const int ctx = seq_len - q_len;
  const int rows = q_len * G;
  const int n_qheads = n_kv * G;

  const int row0 = lt * PF_ROWS;
  const int kmax = ctx + (min(row0 + PF_ROWS, rows) - 1) / G + 1;
  const int n_tiles = (kmax + PF_KT - 1) / PF_KT;
  const PagedTiles list = paged_tiles<MORE>(x, ctx + row0 / G + 1, kmax,
                                            n_tiles, PF_KT);
  // parts of at least four tiles; the rest of them stay empty
  const int parts = min(n_part, (list.n + 3) / 4);
  const int tpp = parts > 0 ? (list.n + parts - 1) / parts : 0;
  const int i_begin = part * tpp;
  const int i_end = min(list.n, i_begin + tpp);

  // ---- this lane's row -----------------------------------------------------
  const int wrow0 = row0 + wid * 32;
  const bool wave_on = wrow0 < rows;
  const int rho = wrow0 + c32;
  const bool row_ok = rho < rows;
  const int qi = rho / G;
  const int head = kvh * G + rho - qi * G;
  const int limit = row_ok ? ctx + qi + 1 : 0;   // keys this row sees
  const int wmin = ctx + wrow0 / G + 1;          // fewest of a row in the wave
  const int wmax = ctx + (min(wrow0 + 32, rows) - 1) / G + 1;

  // keys below lo are out of sight but for the kept ones
  const int lo = paged_first<MORE>(x, row_ok ? limit : 1);
  const int wlo = paged_first<MORE>(x, wmin), whi = paged_first<MORE>(x, wmax);
  const PagedScore sc = paged_score<MORE>(x, scale, row_ok ? head : kvh * G);
  // rows past the last one hold its query: their results go nowhere
  const int qr = min(rho, rows - 1), qq = qr / G;
  const unsigned short* qp = q + (long)(q_start + qq) * q_stride +
                             (long)(kvh * G + qr - qq * G) * D + h * 8;
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
    qf[ks] = *reinterpret_cast<const bf16x8*>(qp + ks * 16) ^ sc.flip;
  f32x16 o_acc[DT];
#pragma unroll
  for (int i = 0; i < DT; i++) o_acc[i] = mr_zero();
  float m = -INFINITY, l = 0.0f;

  // ---- staging: a wave moves the tile's page `wid` ---------------------------
  const int* btab = block_tables + (long)seq * max_blocks;
  const int last_blk = (seq_len - 1) / PF_BS;
  const int srow = lane / CPR, spos = lane % CPR;
  // byte offset in a page of what this lane moves: row r of the page, its
  // chunk permuted by the row's key
  unsigned koff[NI], voff[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int r = i * RPI + srow;
    koff[i] = (unsigned)(r * (2 * D) + ((spos ^ mr_swz_rows<D>(r)) << 4));
    voff[i] = (unsigned)(r * (2 * D) + ((spos ^ mr_swz_cols<D>(r)) << 4));
  }
  // Where this wave's pages of 64 tiles from the tb-th on are and how much of each
  // is keys, one tile per lane: a tile's addresses are a few v_readlane then, and no
  // scalar load, which would make every wait for LDS a wait for it too. Rows past
  // the last key are out of the bounds: zeros, masked below.
  int tb = i_begin;
  unsigned at_lo = 0, at_hi = 0, bytes = 0;
  auto look_up = [&]() {
    const int pg = list.at(min(tb + lane, i_end - 1)) * (PF_KT / PF_BS) + wid;
    const long at =
        ((long)btab[min(pg, last_blk)] * n_kv + kvh) * (PF_BS * D * 2);
    at_lo = (unsigned)at;
    at_hi = (unsigned)(at >> 32);
    bytes = min(max(seq_len - pg * PF_BS, 0), PF_BS) * (D * 2);
    asm volatile("" : "+v"(at_lo), "+v"(at_hi), "+v"(bytes));   // waited for here
  };
  auto stage = [&](int it, int buf) {
    const int i = it - tb;
    const long at =
        (long)((unsigned long long)__builtin_amdgcn_readlane(at_hi, i) << 32 |
               (unsigned)__builtin_amdgcn_readlane(at_lo, i));
    const unsigned n = __builtin_amdgcn_readlane(bytes, i);
    const auto kp = mr_buffer((const char*)k_cache + at, n);
    const auto vp = mr_buffer((const char*)v_cache + at, n);
    unsigned short* dst = kv_lds + buf * 2 * TILE + wid * 16 * D;
#pragma unroll
    for (int k = 0; k < NI; k++) {
      mr_to_lds(kp, koff[k], dst + k * RPI * D);
      mr_to_lds(vp, voff[k], dst + TILE + k * RPI * D);
    }
  };

  const int kbase = mr_row_base<D>(lane), vbase = mr_col_base<D>(lane);

  if (i_begin < i_end) {
    look_up();
    stage(i_begin, 0);
  }
  for (int it = i_begin; it < i_end; it++) {
    const int buf = (it - i_begin) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (it + 1 < i_end) {
      if (it + 1 - tb == 64) {
        tb += 64;
        look_up();
      }
      stage(it + 1, buf ^ 1);
    }
    const int k0 = list.at(it) * PF_KT;
    if (!wave_on || k0 >= wmax) continue;
    if (MORE && k0 + PF_KT <= wlo && k0 >= x.keep_first) continue;
    const lds_u16* kt = (const lds_u16*)kv_lds + buf * 2 * TILE;
    const lds_u16* vt = kt + TILE;

    // ---- scores: keys [32 i, 32 i + 32) of the tile ------------------------
    // (two independent chains of products, four K rows in flight)
    f32x16 s[2] = {mr_zero(), mr_zero()};
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
#pragma unroll
      for (int i = 0; i < 2; i++)
        s[i] = mr_mma(*reinterpret_cast<const lds_bf16x8*>(
                          kt + (kbase ^ (ks << 4)) + i * 32 * D),
                      qf[ks], s[i]);
    }
    // three steps of K are on the way while one is multiplied
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
    for (int ks = 0; ks < KS - 3; ks++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
    if (MORE && x.cap > 0.0f) paged_cap<2>(s, sc.pre, x.cap);
    // uniform: a tile on the diagonal or on the edge of a window
    if (k0 + PF_KT > wmin || (MORE && k0 < whi)) {
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int key = k0 + i * 32 + mr_key_of(r, h);
          if (key >= limit || (MORE && key < lo && key >= x.keep_first))
            s[i][r] = -INFINITY;
        }
    }
    // ---- online softmax: weights are 2^(c (s - m)) ---------------------------
    const float c = sc.c;
    float mt = s[0][0];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[i][r]);
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
    bf16x8 p[TERMS][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        float a = __builtin_amdgcn_exp2f(fmaf(s[i][r], c, -mc));
        float b = __builtin_amdgcn_exp2f(fmaf(s[i][r + 1], c, -mc));
        if (TERMS > 1) l += a + b;
#pragma unroll
        for (int e = 0; e < TERMS; e++) {
          const unsigned u = pack_bf16(a, b);
          reinterpret_cast<unsigned*>(
              &p[e][i * 2 + (r >> 3)])[(r & 7) >> 1] = u;
          if (TERMS == 1) l = sum_bf16(u, l);
          drop_bf16(a, b, u);
        }
      }
    // ---- O^T += V^T P^T ------------------------------------------------------
#pragma unroll
    for (int st = 0; st < 4; st++)
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const bf16x8 a = mr_cols_own<D>(vt + (vbase ^ (dt << 5)) + st * 16 * D);
#pragma unroll
        for (int e = 0; e < TERMS; e++)
          o_acc[dt] = mr_mma(a, p[e][st], o_acc[dt]);
      }
  }

  // ---- epilogue: o_acc[dt][r] = O[row][dt*32 + 8*(r>>2) + 4h + (r&3)] --------
  l = pair_sum(l);
  if (!row_ok) return;
  const long grow = (long)(q_start + qi) * n_qheads + head;
  if (n_part == 1) {
    if (MORE && x.sink != nullptr)
      l += __builtin_amdgcn_exp2f(x.sink[head] * 1.4426950408889634f -
                                  m * sc.c);
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;
    const long at = (long)(q_start + qi) * out_stride + (long)head * D + 4 * h;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        paged_put<MORE>(x, out, at + dt * 32 + 2 * r, o_acc[dt][r] * inv,
                        o_acc[dt][r + 1] * inv, o_acc[dt][r + 2] * inv,
                        o_acc[dt][r + 3] * inv);
    return;
  }
  const long slot = grow * n_part + part;
  if (h == 0) {
    ws_ml[slot * 2] = m * sc.c;
    ws_ml[slot * 2 + 1] = i_begin < i_end ? l : PAGED_ABSENT;
  }
  if (i_begin >= i_end) return;
  float* o = ws_o + slot * D + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<float4*>(o + dt * 32 + 2 * r) =
          make_float4(o_acc[dt][r], o_acc[dt][r + 1], o_acc[dt][r + 2],
                      o_acc[dt][r + 3]);
}

// Row tiles a batch has at most, and the parts its keys are split into: about
// two workgroups per CU are wanted, and parts of at least eight tiles of keys
// (four with 32-bit weights, whose tiles take twice as long): the merge costs
// more than smaller ones save. Measured (us, by parts 1 | 2 | 4 | 8), 32-bit
// weights: 2 x 64 rows of 32 heads over 4000 keys 191 | 104 | 60 | 40; 300 of 16
// over 600 37 | 26 | 24 | 28; 1024 of 32 over 8000 (264 row tiles) 374 | 298 |
// 302 | 325; 4096 of 16 in a window (520 row tiles) 69 | 87 | 111 | 182.
inline long paged_rows_tiles(long tokens, int n_seqs, int G) {
  return tokens * G / PF_ROWS + n_seqs;
}
inline int paged_rows_parts(long tokens, int n_seqs, int G, int n_kv,
                            long max_blocks, int terms) {
  const long wgs = paged_rows_tiles(tokens, n_seqs, G) * n_kv;
  const long most = max_blocks * PF_BS / ((terms > 1 ? 4 : 8) * PF_KT);
  long p = wgs > 0 ? (512 + wgs / 2) / wgs : 1;
  if (p > most) p = most;
  return (int)(p < 1 ? 1 : p > 16 ? 16 : p);
}

// Prompt rows and the merge of their parts
template <int D, int TERMS, bool MORE>
inline void paged_rows(void* out, float* ws_o, float* ws_ml,
                       const unsigned short* q, const unsigned short* k_cache,
                       const unsigned short* v_cache, const int* block_tables,
                       const int* cu_q, const int* seq_lens, long tokens,
                       int n_seqs, float scale, int n_qheads, int n_kv,
                       int max_blocks, long q_stride, long out_stride,
                       int n_part, const PagedMore& x, hipStream_t stream) {
  const int G = n_qheads / n_kv;
  if (tokens == 0 || n_seqs <= 0) return;
  const dim3 grid(
      (unsigned)(paged_rows_tiles(tokens, n_seqs, G) * n_kv * n_part));
  hipLaunchKernelGGL((paged_attn_rows_kernel<D, TERMS, MORE>), grid, dim3(256),
                     0, stream, out, ws_o, ws_ml, q, k_cache, v_cache,
                     block_tables, cu_q, seq_lens, n_seqs, scale, G, n_kv,
                     max_blocks, q_stride, out_stride, n_part, x);
  if (n_part > 1)
    paged_merge<D, MORE>(out, ws_o, ws_ml, n_qheads, n_part, out_stride,
                         tokens * n_qheads, x, stream, nullptr, 1, 1, cu_q,
                         n_seqs);
}

}  // namespace xllm
