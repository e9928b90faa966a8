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
// keys of a tile are split over workgroups, by the length of its own sequence
// (pf_parts). Of up to eight parts the last one to finish merges the fp32 partial results
// of all (PagedMeet), of more a second kernel does, which all CUs share.
//
// Bound by the matrix pipe and the vector unit in turn: a tile costs a wave
// 32 products (about 1000 cycles) and about as many cycles of exponentials,
// maxima and conversions, which the second wave of the SIMD overlaps; LDS
// reads feed 32 rows each and stay just below the pipe's rate. Loads to LDS go
// through buffers: after those through global addresses, which are flat
// instructions to the compiler, every use of an LDS read waited for all reads in
// flight, and the first transpose read for the next tile too. With that and
// three steps of K on the way ahead of their products, before -> after: 4 prompts
// of 1.6-2.3 k tokens over up to 3.1 k cached ones, 32 heads 366 -> 353 us,
// 3 chunks of 93-261 tokens over 0.5-1.8 k, 28 heads, keys split 30.9 -> 30.1, 2
// of 1.8-2.3 k in a window of 1024, three terms 63.3 -> 61.3, 8 prompts of 109-438,
// 12 heads of 64 13.6. (One head and 16 rows per wave on 16x16x32 products, P
// through LDS: 1209 us for the first; an eager loop 14 ms for the last.)
//
// Fragment layouts, the order of the keys and of the LDS images: mfma_rows.h.
#pragma once
#include <algorithm>
#include <climits>

#include "paged_merge.h"

namespace xllm {

#define PF_ROWS 128        // rows per workgroup
#define PF_KT 64           // keys per tile
#define PF_BS 16           // cache block size

// x / d for 0 <= x < 2^31 by a multiplication with pf_inverse(d) and a shift by pf_shift(d):
// the compiler's division by what it does not know takes 25 instructions, of which a wave
// alone on its SIMD issues one in six cycles. Exact: with s the shift, 2^s >= d, and
// e = d pf_inverse(d) - 2^(31+s) < d, the product is too large by x e / (2^(31+s) d),
// less than the 1/d that x / d is at least below the next whole number. Eight of them, and
// the pages' ids asked for before them: 12.6 to 12.3 us for a sequence of 192 to 512 tokens at
// 4 heads over 1, 12.0 to 11.55 for six of 60 to 400 at 64-wide heads, 18.2 to 18.1 for 700.
XLLM_DEV int pf_div(int x, unsigned inverse, int shift) {
  return (int)(__umulhi(2u * (unsigned)x, inverse) >> shift);
}
__host__ __device__ __forceinline__ int pf_shift(int d) {
  return 31 - __builtin_clz(2u * (unsigned)d - 1);
}
inline unsigned pf_inverse(int d) {
  return (unsigned)(((1ull << (31 + pf_shift(d))) + d - 1) / d);
}

// Where a workgroup's rows are: tile lt of sequence seq
struct PfPlace { int seq, lt, q_start, q_len, seq_len; };

// Which of `total` units, the longest first, workgroup b takes where a CU holds two and
// `turn` come one to a CU: what is left over joins the shortest of those, the very shortest
// the longest of them, so that the longest have a CU to themselves. (Joined to the longest
// of all, 500 and 695 tokens of 28/4 heads, 268 workgroups, took 24.1 us, 22.7 so.) (More
// than two turns with the second reversed: 1318 drawn batches, no faster.)
XLLM_DEV int pf_fold(int b, int total, int turn) {
  const int over = total - turn;
  if (over <= 0 || over > turn) return b;
  return b >= turn ? turn + total - 1 - b : b < over ? turn - over + b : b - over;
}

// What there is to know of a single sequence, fetched together
struct PfOnly {
  int start, len, keys;
  XLLM_DEV PfOnly(const int* cu_q, const int* seq_lens) {
    const int end = cu_q[1];
    start = cu_q[0];
    keys = seq_lens[0];
    asm volatile("" ::"s"(start), "s"(end), "s"(keys));
    len = end - start;
  }
};
// Row tile `b` of a single sequence, without scans: 0.4 us of a small call
template <int ROWS>
XLLM_DEV bool pf_only(int b, int turn, const int* cu_q, const int* seq_lens, int G,
                      PfPlace* place) {
  const PfOnly s(cu_q, seq_lens);
  const int all = (s.len * G + ROWS - 1) / ROWS;
  if (b >= all) return false;
  b = pf_fold(b, all, turn);
  *place = {0, all - 1 - b, s.start, s.len, s.keys};
  return true;
}

// Row tile `b` of the batch; later tiles of a sequence (more keys) come first. False:
// past the last one. One wave looks 64 sequences over at a time, and what it
// found of the one it wants is taken from its lane: fetched again by a scalar load it
// was one more latency in a chain of four before the first product: 8 short prompts, 12
// heads of 64, 13.55 -> 13.3 us, 3 chunks over 0.5-1.8 k 30.2 -> 29.75.
template <int ROWS>
XLLM_DEV bool pf_locate(int b, const int* cu_q, const int* seq_lens, int n_seqs,
                        int G, int lane, PfPlace* at) {
  int acc = 0;
  for (int base = 0; base < n_seqs; base += 64) {
    const int i = base + lane;
    int start = 0, len = 0, keys = 0;
    if (i < n_seqs) {
      start = cu_q[i];
      len = cu_q[i + 1] - start;
      keys = seq_lens[i];
    }
    const int nt = i < n_seqs ? (len * G + ROWS - 1) / ROWS : 0;
    int sum = nt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(sum, off, 64);
      if (lane >= off) sum += up;
    }
    const unsigned long long hit = __ballot(b < acc + sum);
    if (hit != 0) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll(hit) - 1);
      *at = {base + l, acc + __builtin_amdgcn_readlane(sum, l) - 1 - b,
             __builtin_amdgcn_readlane(start, l),
             __builtin_amdgcn_readlane(len, l),
             __builtin_amdgcn_readlane(keys, l)};
      return true;
    }
    acc += __builtin_amdgcn_readlane(sum, 63);
  }
  return false;
}

// Sums (maxima) of the lanes up to and with this one, on the vector unit alone
template <bool SUM>
XLLM_DEV int pf_scan(int v) {
#define PF_STEP(CTRL, ROWS)                                                    \
  {                                                                            \
    const int u = __builtin_amdgcn_update_dpp(SUM ? 0 : INT_MIN, v, CTRL, ROWS, \
                                              0xf, false);                     \
    v = SUM ? v + u : max(v, u);                                               \
  }
  PF_STEP(0x111, 0xf) PF_STEP(0x112, 0xf) PF_STEP(0x114, 0xf)   // row_shr
  PF_STEP(0x118, 0xf)
  PF_STEP(0x142, 0xa) PF_STEP(0x143, 0xc)                       // row_bcast
#undef PF_STEP
  return v;
}

// Row tile `b` of the batch, the longest chains of keys first whatever their
// sequences: a tile of a sequence has ROWS rows (of query and head) fewer before it
// than the next one, so all tiles sort into levels of WIDTH of those with at most
// WIDTH tiles of a sequence to a level, which share its keys and stay together. The level
// of tile b is found by halves, a lane counting its sequence's tiles above one. Up to 64
// sequences; of more, one sequence after the other (pf_locate).
//   Two turns of workgroups come folded (pf_fold). By sequences, the tiles of two equal
// prompts met their likes: 2 x 1.8-2.3 k in a window of 1024 59.5 -> 54.8 us, 4 x 512 of
// 32/8 heads 28.3 -> 22.8, 3 x 500 capped 51.5 -> 40.2. WIDTH 1, 2 and 4: 40 x 60 behind
// 500, whose two tiles read the same keys, 48.6, 46.0, 46.5 (46.7 by sequences), 1500
// and 300 of 64-wide heads 26.6, 26.6, 27.6.
template <int ROWS, int WIDTH>
XLLM_DEV bool pf_longest(int b, int turn, const int* cu_q, const int* seq_lens,
                         int n_seqs, int G, int lane, PfPlace* place) {
  if (n_seqs > 64)
    return pf_locate<ROWS>(b, cu_q, seq_lens, n_seqs, G, lane, place);
  if (n_seqs == 1) return pf_only<ROWS>(b, turn, cu_q, seq_lens, G, place);
  int start = 0, len = 0, keys = 0;              // of sequence `lane`
  if (lane < n_seqs) {
    start = cu_q[lane];
    len = cu_q[lane + 1] - start;
    keys = seq_lens[lane];
  }
  const int nt = (len * G + ROWS - 1) / ROWS, top = keys * G;
  const int most = __builtin_amdgcn_readlane(
      pf_scan<false>(nt > 0 ? top : INT_MIN), 63);
  const int total = __builtin_amdgcn_readlane(pf_scan<true>(nt), 63);
  if (b >= total) return false;
  b = pf_fold(b, total, turn);
  // its tiles from the top: [first, first + nt)
  const int first = nt > 0 ? (most - top) / ROWS : 0;
  const int depth = __builtin_amdgcn_readlane(pf_scan<false>(first + nt), 63);
  const int deepest = (depth - 1) / WIDTH;       // level, in tiles; tiles over it
  int level = 0, above = 0;
  for (int step = deepest > 0 ? 1 << (31 - __builtin_clz(deepest)) : 0; step > 0;
       step >>= 1) {
    const int mine = level + step * WIDTH;
    const int c = __builtin_amdgcn_readlane(
        pf_scan<true>(min(max(mine - first, 0), nt)), 63);
    if (c <= b) level = mine, above = c;         // uniform
  }
  // sequence `lane`'s tiles over the level, and with those in it
  const int over = min(max(level - first, 0), nt);
  const int with = min(max(level + WIDTH - first, 0), nt);
  const int upto = pf_scan<true>(with - over);
  const int r = b - above;
  const int i = __builtin_amdgcn_readfirstlane(__ffsll(__ballot(r < upto)) - 1);
  const int k = r - __builtin_amdgcn_readlane(upto - with, i);
  *place = {i, __builtin_amdgcn_readlane(nt, i) - 1 - k,
            __builtin_amdgcn_readlane(start, i),
            __builtin_amdgcn_readlane(len, i),
            __builtin_amdgcn_readlane(keys, i)};
  return true;
}

#define PF_UNITS 448       // groups of waves that a batch's keys are split over,
#define PF_TURN 512        // and that the CUs hold at once
// parts that the last one merges, at most, by groups of waves
#define PF_MEET(KG) ((KG) > 1 ? 8 : 4)

// Unit `b` of a batch whose keys are split: a row tile and one of its parts, b - part the
// tile's first. One sequence: up to `most` equal parts, of at least four tiles of keys.
// Several: parts of `per` tiles, so that all of the batch walk about as many, whatever its
// sequences' lengths; if the last part merges, four of them and more only of twelve tiles.
// Never more parts than ceil(n / per), or than `most`: the grid and the scratch hold that
// many units (PagedRows), and a row whose unit was not in the grid would leave the merge
// without its place. PF_UNITS: just under two groups of waves to a CU.
//   The same number of parts for all, as many as the longest's table asks for, left one
// sequence's chain to be waited for: 50, 60, 300 and 20 tokens behind 9000, 100, 0 and 700
// of 32/8 heads 59.4 -> 34.4 us, of 28/4 51.4 -> 29, 31, 322 and 416 behind 4052, 20 and
// 27 of 32/32 56 -> 30.5, 2 x 200 behind 3000 52.3 -> 41.1; equal ones (8 x 100 behind 500,
// 20.1) gain nothing.
template <int ROWS, bool MORE>
XLLM_DEV bool pf_parts(int b, int least, int most, int groups, int turn,
                       const PagedMore& x,
                       const int* cu_q, const int* seq_lens, int n_seqs, int G,
                       int n_kv, int lane, PfPlace* at, int* part, int* parts,
                       int* first) {
  if (n_seqs == 1) {
    const PfOnly s(cu_q, seq_lens);
    const int p = paged_equal<MORE>(x, s.keys, PF_KT, most);
    const int nt = (s.len * G + ROWS - 1) / ROWS, all = nt * p;
    if (b >= all) return false;
    b = pf_fold(b, all, turn);
    const int t = b / p;                         // a division takes 0.05 us
    *part = b - t * p;
    *parts = p;
    *first = t * p;
    *at = {0, nt - 1 - t, s.start, s.len, s.keys};
    return true;
  }
  int start = 0, len = 0, keys = 0, nt = 0, n = 0;
  auto look = [&](int i) {                       // sequence i, one to a lane
    start = len = keys = 0;
    if (i < n_seqs) {
      start = cu_q[i];
      len = cu_q[i + 1] - start;
      keys = seq_lens[i];
    }
    nt = (len * G + ROWS - 1) / ROWS;
    n = paged_walk<MORE>(x, keys, PF_KT);
  };
  int work = 0;
  for (int base = 0; base < n_seqs; base += 64) {
    look(base + lane);
    work += __builtin_amdgcn_readlane(pf_scan<true>(nt * n), 63);
  }
  const int some = PF_UNITS / groups;
  int per = max(least, (work * n_kv + some - 1) / some);
  const bool few = most <= 8;
  auto parts_of = [&](int q) {
    const int p = max(min((n + q - 1) / q, most), 1);
    return few ? min(p, max(4, (n + 11) / 12)) : p;
  };
  if (n_seqs <= 64) {
    auto fits = [&](int p) {
      return __builtin_amdgcn_readlane(pf_scan<true>(nt * p), 63) * n_kv <=
             PF_TURN / groups;
    };
    auto chain = [&](int p) {
      return __builtin_amdgcn_readlane(
          pf_scan<false>(nt > 0 ? (n + p - 1) / p : 0), 63);
    };
    // Units left for another turn are waited for: parts are lengthened until there are
    // none, unless that takes longer than the turn. 2 x 600 behind 500 of 28/4 in a window
    // 53.9 us in two parts of 6 tiles, 39.1 in one of 11, 2 x 420 behind 3600-6900 of 32/8,
    // capped, 232 and 194; but 1000 and 1100 of 16/4, capped, 50.4 in two of up to 9, 65.9 in
    // one. Two groups of waves, 6 x 337 behind 230 of 8/1 in a window 34.9 and 24.8.
    if (!fits(parts_of(per))) {
      // of a causal prompt the row tiles are half as long on average as the last of them
      auto turns = [&]() {
        const int now = chain(parts_of(per));
        if (groups > 1) return 2 * now;
        const int seen = min(n, (max(keys - len / 2, 0) + PF_KT - 1) / PF_KT);
        const int mean = __builtin_amdgcn_readlane(pf_scan<true>(nt * seen), 63);
        return now + (int)((float)now * mean / max(work, 1)) + (MORE ? 2 : 4);
      };
      const int step = max(per / 8, 1);
      for (int q = per + step; q <= 2 * per; q += step)
        if (fits(parts_of(q))) {
          // two groups of waves: a quarter more is no turn
          if ((groups > 1 && q <= per + per / 4) || chain(parts_of(q)) <= turns())
            per = q;
          break;
        }
    }
  }
  int acc = 0;
  for (int base = 0; base < n_seqs; base += 64) {
    if (n_seqs > 64) look(base + lane);
    const int p = parts_of(per);
    const int upto = acc + pf_scan<true>(nt * p);
    const unsigned long long hit = __ballot(b < upto);
    if (hit != 0) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll(hit) - 1);
      const int pl = __builtin_amdgcn_readlane(p, l);
      const int r = b - __builtin_amdgcn_readlane(upto - nt * p, l);
      const int t = r / pl;
      *part = r - t * pl;
      *parts = pl;
      *first = b - *part;
      *at = {base + l, __builtin_amdgcn_readlane(nt, l) - 1 - t,
             __builtin_amdgcn_readlane(start, l),
             __builtin_amdgcn_readlane(len, l),
             __builtin_amdgcn_readlane(keys, l)};
      return true;
    }
    acc = __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// TERMS: bf16 terms a softmax weight is split into. One rounds it to bf16;
// three (8 + 8 + 8 mantissa bits) hold all of its 32-bit value, each with a
// product of its own into the same fp32 sums. MORE: the options of PagedMore.
// KG: groups of four waves, each with the same rows and its share of the tiles: what
// splitting keys over workgroups does, without partial results in memory.
// SORT: the longest chains first, where keys are not split.
template <int D, int TERMS, bool MORE, int KG, bool SPLIT, bool SORT = true>
__global__ __launch_bounds__(KG * 256, 2) void paged_attn_rows_kernel(
    // (what the first loads need comes first: these are in registers)
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ cu_q,            // [num_seqs+1] query offsets
    const int* __restrict__ seq_lens,        // [num_seqs] total key len
    const int n_seqs, const int G, const int n_kv, const int max_blocks,
    const unsigned by_kv, const unsigned by_G,   // pf_inverse of n_kv and G
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, 16, D]
    const unsigned short* __restrict__ q,    // [total_q, n_qheads, D] bf16
    const unsigned short* __restrict__ v_cache,
    void* __restrict__ out,                  // [total_q, n_qheads, D]
    float* __restrict__ ws_o,                // [blocks][PF_ROWS * D], a block for a part
    float* __restrict__ ws_ml,               // [blocks][PF_ROWS][2]
    int2* __restrict__ ws_at,                // [total_q*n_qheads]: first slot, parts;
                                             // of several prompts, for the merge
    const PagedMeet meet,                    // [blocks]: its first part's counts
    const float scale, const long q_stride, const long out_stride,
    const int least, const int most, const int turn, const PagedMore x,
    const PagedAhead ahead) {
  constexpr int KS = D / 16;                 // k steps of a score product
  constexpr int DT = D / 32;                 // 32-wide tiles of the head
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = 16 / RPI;               // ... instructions per page
  constexpr int TILE = PF_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short
      kv_lds[KG * 4 * TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wid = wave & 3, kg = KG > 1 ? wave >> 2 : 0;
  const int h = lane >> 5, c32 = lane & 31;

  if (!MORE && (int)blockIdx.x >= ahead.from) {
    paged_fetch(ahead, blockIdx.x - ahead.from, kv_lds);
    return;
  }
  const int sG = pf_shift(G);
  const int unit = pf_div(blockIdx.x, by_kv, pf_shift(n_kv));
  const int kvh = blockIdx.x - unit * n_kv;
  int part = 0, parts = 1, first = 0;
  PfPlace at;
  if constexpr (SPLIT) {
    if (!pf_parts<PF_ROWS, MORE>(unit, least, most, KG, turn, x, cu_q,
                                 seq_lens, n_seqs, G, n_kv, lane, &at, &part,
                                 &parts, &first))
      return;
  } else if constexpr (SORT) {
    if (!pf_longest<PF_ROWS, 2>(unit,
                                KG > 1 ? INT_MAX / 2 : 256 / n_kv, cu_q, seq_lens,
                                n_seqs, G, lane, &at))
      return;
  } else {
    if (!pf_locate<PF_ROWS>(unit, cu_q, seq_lens, n_seqs, G, lane, &at))
      return;
  }
  const int seq = at.seq, lt = at.lt, q_start = at.q_start, q_len = at.q_len,
            seq_len = at.seq_len;
  const int ctx = seq_len - q_len;
  const int rows = q_len * G;
  const int n_qheads = n_kv * G;

  const int row0 = lt * PF_ROWS;
  const int kmax = ctx + pf_div(min(row0 + PF_ROWS, rows) - 1, by_G, sG) + 1;
  const int n_tiles = (kmax + PF_KT - 1) / PF_KT;
  const PagedTiles list = paged_tiles<MORE>(x, ctx + pf_div(row0, by_G, sG) + 1, kmax,
                                            n_tiles, PF_KT);
  const int tpp = (max(list.n, 0) + parts - 1) / parts;
  // its parts' place: their blocks lie together
  const long block = SPLIT ? (long)first * n_kv + kvh * parts : 0;
  u64 seen = 0;
  const bool meets = SPLIT && parts > 1 && meet.count != nullptr;
  if (meets && threadIdx.x == 0) seen = paged_seen(meet.count + block);
  const int p_begin = part * tpp;
  const int i_end = min(list.n, p_begin + tpp);
  const int i_begin = p_begin + kg;              // every KG-th of a group's

  // ids of this wave's pages of 64 of its tiles, one per lane: a scalar load per tile would
  // make every wait for LDS a wait for it too. The first are asked for here: what comes
  // before the tile is 0.8 us.
  const int* btab = block_tables + (long)seq * max_blocks;
  const int last_blk = (seq_len - 1) / PF_BS;
  const int last_row = (seq_len - 1) % PF_BS;
  int tb = 0;                                    // from this one on
  auto pages_from = [&](int n) {
    return btab[min(list.at(i_begin + (n + lane) * KG) * (PF_KT / PF_BS) + wid,
                    last_blk)];
  };
  int pages = 0;
  if (i_begin < i_end) pages = pages_from(0);

  // ---- this lane's row -----------------------------------------------------
  const int wrow0 = row0 + wid * 32;
  const bool wave_on = wrow0 < rows;
  const int rho = wrow0 + c32;
  const bool row_ok = rho < rows;
  const int qi = pf_div(rho, by_G, sG);
  const int head = kvh * G + rho - qi * G;
  const int limit = row_ok ? ctx + qi + 1 : 0;   // keys this row sees
  const int wmin = ctx + pf_div(wrow0, by_G, sG) + 1;   // fewest of a row in the wave
  const int wmax = ctx + pf_div(min(wrow0 + 32, rows) - 1, by_G, sG) + 1;

  // keys below lo are out of sight but for the kept ones
  const int lo = paged_first<MORE>(x, row_ok ? limit : 1);
  const int wlo = paged_first<MORE>(x, wmin), whi = paged_first<MORE>(x, wmax);
  const PagedScore sc = paged_score<MORE>(x, scale, row_ok ? head : kvh * G);
  // rows past the last one hold its query: their results go nowhere
  const int qr = min(rho, rows - 1), qq = pf_div(qr, by_G, sG);
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
  const int srow = lane / CPR, spos = lane % CPR;
  // byte offset in a page of what this lane moves: row r of the page, its
  // chunk permuted by the row's key
  auto off_of = [&](int r, int key, bool val) {
    const int x = val ? mr_swz_cols<D>(key) : mr_swz_rows<D>(key);
    return (unsigned)(r * (2 * D) + ((spos ^ x) << 4));
  };
  unsigned koff[NI], voff[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int r = i * RPI + srow;
    koff[i] = off_of(r, r, false);
    voff[i] = off_of(r, r, true);
  }
  auto put = [&](__amdgpu_buffer_rsrc_t kp, __amdgpu_buffer_rsrc_t vp,
                 unsigned ko, unsigned vo, unsigned short* dst) {
    mr_to_lds(kp, ko, dst);
    mr_to_lds(vp, vo, dst + TILE);
  };
  auto stage = [&](int t, int page, int buf) {
    const int pg = t * (PF_KT / PF_BS) + wid;
    const long base = ((long)page * n_kv + kvh) * (PF_BS * D);
    const auto kp = mr_buffer(k_cache + base, PF_BS * D * 2);
    const auto vp = mr_buffer(v_cache + base, PF_BS * D * 2);
    unsigned short* dst = kv_lds + (kg * 2 + buf) * 2 * TILE + wid * 16 * D;
    if (pg < last_blk) {
#pragma unroll
      for (int i = 0; i < NI; i++)
        put(kp, vp, koff[i], voff[i], dst + i * RPI * D);
      return;
    }
    // rows past the last key repeat it: masked below, and finite
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int r = i * RPI + srow;
      const int rr = pg > last_blk ? last_row : min(r, last_row);
      put(kp, vp, off_of(rr, r, false), off_of(rr, r, true), dst + i * RPI * D);
    }
  };

  const int kbase = mr_row_base<D>(lane), vbase = mr_col_base<D>(lane);

  if (i_begin < i_end) {
    stage(list.at(i_begin), __builtin_amdgcn_readlane(pages, 0), 0);
  }
  // a step: a tile of every group, the last of which may have none left
  for (int at = p_begin, n = 0; at < i_end; at += KG, n++) {
    const int buf = n & 1, it = at + kg;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (it + KG < i_end) {
      if (n + 1 - tb == 64) {
        tb += 64;
        pages = pages_from(tb);
      }
      stage(list.at(it + KG), __builtin_amdgcn_readlane(pages, n + 1 - tb),
            buf ^ 1);
    }
    if (KG > 1 && it >= i_end) continue;
    const int k0 = list.at(it) * PF_KT;
    if (!wave_on || k0 >= wmax) continue;
    if (MORE && k0 + PF_KT <= wlo && k0 >= x.keep_first) continue;
    const lds_u16* kt = (const lds_u16*)kv_lds + (kg * 2 + buf) * 2 * TILE;
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
      paged_mask<MORE>(x, s, limit, lo, [&](int i, int r) {
        return k0 + i * 32 + mr_key_of(r, h);
      });
    }
    // ---- online softmax: weights are 2^(c (s - m)) ---------------------------
    const float c = sc.c;
    float mt = s[0][0];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[i][r]);
    mt = pair_max(mt);
    // Some row of 32 has a new maximum in most tiles. Weights of 32 bits and sums round the
    // same whatever they are scaled by, so there sums are scaled only where one has grown
    // by more than 2^8: 2 of 1.5-2.6 k in a window of 1024 53.4 -> 51.4 us, 911 and 1317
    // capped 64.5 -> 61.8, errors 1-2% smaller. (One rounded to bf16 is exact where it is 1.)
    if (TERMS > 1 ? __any((mt - m) * c > 8.0f) : __any(mt > m)) {
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
        l += a + b;
#pragma unroll
        for (int e = 0; e < TERMS; e++) {
          const unsigned u = pack_bf16(a, b);
          reinterpret_cast<unsigned*>(
              &p[e][i * 2 + (r >> 3)])[(r & 7) >> 1] = u;
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
  m = m == -INFINITY ? m : m * sc.c;
  if (meets && threadIdx.x == 0) paged_open(meet.count + block, seen, meet.tag);
  constexpr int OWN = DT / KG;                   // column tiles a group finishes
  const int dt0 = kg * OWN;
  constexpr unsigned GONE = 0x7ffffff0;          // out of the bounds: no store, zeros
  const int row = wid * 32 + c32;
  const unsigned size_o = SPLIT && parts > 1 ? parts * (PF_ROWS * D * 4) : 0;
  const auto unit_o = mr_buffer(SPLIT ? ws_o + block * (PF_ROWS * D) : nullptr, size_o);
  const auto unit_ml =
      mr_buffer(SPLIT ? ws_ml + block * (PF_ROWS * 2) : nullptr, size_o / D * 2);
  auto piece = [&](int b, int j, int r) {        // of part b: 1 KB of a wave's
    return (unsigned)(((((b * 4 + wid) * DT + dt0 + j) * 4 + r) * 64 + lane) * 16);
  };
  if constexpr (KG > 1) {
    // the groups swap halves of their sums
    __syncthreads();
    f32x4* swap = reinterpret_cast<f32x4*>(kv_lds);   // [8 waves][OWN][4][64]
    float2* ml = reinterpret_cast<float2*>(swap + 8 * OWN * 4 * 64);   // [8][32]
    if (h == 0) ml[wave * 32 + c32] = make_float2(m, l);
#pragma unroll
    for (int j = 0; j < OWN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const f32x16 o = kg ? o_acc[j] : o_acc[OWN + j];
        swap[((wave * OWN + j) * 4 + r) * 64 + lane] =
            f32x4{o[4 * r], o[4 * r + 1], o[4 * r + 2], o[4 * r + 3]};
      }
    __syncthreads();
    const float2 z = ml[(wave ^ 4) * 32 + c32];
    // a group without tiles has no part in the row
    const bool mine = i_begin < i_end, other = p_begin + (kg ^ 1) < i_end;
    float top = fmaxf(m, z.x);                   // which skips a NaN
    if (m != m || z.x != z.x) top = NAN;
    const float to = top == -INFINITY ? 0.0f : top;
    const float f = mine ? __builtin_amdgcn_exp2f(m - to) : 0.0f;
    const float g = other ? __builtin_amdgcn_exp2f(z.x - to) : 0.0f;
    l = (mine ? l * f : 0.0f) + (other ? z.y * g : 0.0f);
    m = top;
#pragma unroll
    for (int j = 0; j < OWN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const f32x4 y = swap[(((wave ^ 4) * OWN + j) * 4 + r) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float x = kg ? o_acc[OWN + j][4 * r + e] : o_acc[j][4 * r + e];
          o_acc[j][4 * r + e] =
              (mine ? x * f : 0.0f) + (other ? y[e] * g : 0.0f);
        }
      }
  }
  if (meets) {
    // ---- the last of a few parts merges them -------------------------------
    // A wave writes and reads its sums as its lanes hold them, 1 KB at a time: 3-4 us
    // less than the kernel of merges takes, with its start, its rows' places, and one part
    // more to read. More parts by fours, and those again, took longer than that kernel
    // (7 to 25% of calls of 20 to 50 us).
    constexpr int MEET = PF_MEET(KG);
    mr_store_far2(unit_ml, h == 0 && kg == 0 ? (part * PF_ROWS + row) * 8 : GONE,
                  make_float2(m, l));
#pragma unroll
    for (int j = 0; j < OWN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        mr_store_far(unit_o, piece(part, j, r),
                     make_float4(o_acc[j][4 * r], o_acc[j][4 * r + 1],
                                 o_acc[j][4 * r + 2], o_acc[j][4 * r + 3]));
    if (!paged_last(meet.count + block, parts, reinterpret_cast<int*>(kv_lds)))
      return;
    float2 z[MEET];
    bool on[MEET];                            // without keys: no part in the row
#pragma unroll
    for (int k = 0; k < MEET; k++) {
      on[k] = k < parts && k * tpp < list.n;
      if (k < 4 || parts > 4)
        z[k] = mr_load_far2(unit_ml, on[k] ? (k * PF_ROWS + row) * 8 : GONE);
    }
    float top = -INFINITY;
#pragma unroll
    for (int k = 0; k < MEET; k++) {
      if (k == part) z[k] = make_float2(m, l);
      if (on[k]) top = fmaxf(top, z[k].x);
    }
    m = top;
    if (top == -INFINITY) top = 0.0f;
    l = 0.0f;
    float w[MEET];
#pragma unroll
    for (int k = 0; k < MEET; k++) {
      w[k] = on[k] ? __builtin_amdgcn_exp2f(z[k].x - top) : 0.0f;
      l += on[k] ? z[k].y * w[k] : 0.0f;
    }
    // in the order of the parts, whichever is the last
    constexpr int JB = OWN < 2 ? OWN : 2, KB = 4;
#pragma unroll
    for (int j0 = 0; j0 < OWN; j0 += JB) {
      float4 sum[JB][4];
#pragma unroll
      for (int k0 = 0; k0 < MEET; k0 += KB) {
        if (k0 >= parts) break;                  // uniform
        float4 y[KB][JB][4];
#pragma unroll
        for (int k = 0; k < KB; k++)
#pragma unroll
          for (int j = 0; j < JB; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              y[k][j][r] = mr_load_far(
                  unit_o, on[k0 + k] && k0 + k != part ? piece(k0 + k, j0 + j, r)
                                                       : GONE);
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float4 mine =
                make_float4(o_acc[j0 + j][4 * r], o_acc[j0 + j][4 * r + 1],
                            o_acc[j0 + j][4 * r + 2], o_acc[j0 + j][4 * r + 3]);
            float4 a = k0 > 0 ? sum[j][r] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int k = k0; k < k0 + KB; k++) {
              const float4 v = k == part ? mine : y[k - k0][j][r];
              a.x += on[k] ? v.x * w[k] : 0.0f;
              a.y += on[k] ? v.y * w[k] : 0.0f;
              a.z += on[k] ? v.z * w[k] : 0.0f;
              a.w += on[k] ? v.w * w[k] : 0.0f;
            }
            sum[j][r] = a;
          }
      }
#pragma unroll
      for (int j = 0; j < JB; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          o_acc[j0 + j][4 * r] = sum[j][r].x;
          o_acc[j0 + j][4 * r + 1] = sum[j][r].y;
          o_acc[j0 + j][4 * r + 2] = sum[j][r].z;
          o_acc[j0 + j][4 * r + 3] = sum[j][r].w;
        }
    }
  }
  if (!row_ok) return;
  const long grow = (long)(q_start + qi) * n_qheads + head;
  // for the merge, the parts of a row lie together (strided, it took up to 9 us more)
  const long slot = block * PF_ROWS + row * parts + part;
  if (SPLIT && ws_at != nullptr && part == 0 && h == 0 && kg == 0)
    ws_at[grow] = make_int2((int)slot, parts);
  if (!SPLIT || meets || parts == 1) {
    if (MORE && x.sink != nullptr) l += paged_sink(x, head, m);
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;
    const long to = (long)(q_start + qi) * out_stride + (long)head * D + 4 * h;
#pragma unroll
    for (int j = 0; j < OWN; j++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        paged_put<MORE>(x, out, to + (dt0 + j) * 32 + 2 * r, o_acc[j][r] * inv,
                        o_acc[j][r + 1] * inv, o_acc[j][r + 2] * inv,
                        o_acc[j][r + 3] * inv);
    return;
  }
  if (h == 0 && kg == 0) {
    ws_ml[slot * 2] = m;
    ws_ml[slot * 2 + 1] = p_begin < i_end ? l : PAGED_ABSENT;
  }
  if (p_begin >= i_end) return;
  float* o = ws_o + slot * D + 4 * h;
#pragma unroll
  for (int j = 0; j < OWN; j++)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<float4*>(o + (dt0 + j) * 32 + 2 * r) =
          make_float4(o_acc[j][r], o_acc[j][r + 1], o_acc[j][r + 2],
                      o_acc[j][r + 3]);
}

// Row tiles a batch has at most
template <int ROWS>
inline long paged_rows_tiles(long tokens, int n_seqs, int G) {
  return (tokens * G + n_seqs * (ROWS - 1L)) / ROWS;
}
// Groups of waves, and parts of the keys (pf_parts): about two groups of waves per CU are
// wanted, and parts of at least eight tiles of keys (four with 32-bit weights, whose
// tiles take twice as long): the merge costs more than smaller ones save. Measured (us,
// by parts 1 | 2 | 4 | 8), 32-bit weights: 2 x 64 rows of 32 heads over 4000 keys 191 |
// 104 | 60 | 40; 300 of 16 over 600 37 | 26 | 24 | 28; 1024 of 32 over 8000 (264 row tiles)
// 374 | 298 | 302 | 325; 4096 of 16 in a window (520 row tiles) 69 | 87 | 111 | 182.
//   Two groups of waves and one part where these fill one turn of the CUs: 128-wide
// heads, up to 24 tiles, or for a single sequence that fills most of the CUs; us, as
// before (parts) | two groups: 1024 tokens of 32/8 heads 34.5 (2) | 25.5, 28/4 32.5 (2)
// | 24.8, 3 x 300 behind 1000 44 (2) | 33, 1000 behind 1000 49.5 (2) | 42.2, 700 20.9
// (1) | 20.0, but 300 13.2 (1) | 14.1; 300 behind 1000, 28/4 (66 workgroups) 27.3 |
// 28.5, 16/4 1000 behind 1000 (125) 34.9 (4) | 37.5; and one prompt in up to 448
// workgroups, whose chains differ: 1200 of 32/32 (19 tiles) 44 | 30, 1400 of 32/8 39 |
// 32.8, 2048 of 28/4 (448) 54.2 | 50, 32/8 (512) 55.5 | 56.4, 850 of 64/8 (14 tiles) 29
// | 31.4. 32-bit weights, 2 x 400 behind 500 of 32/8 in a window 46.3 (2) | 33, in one
// of 512 41 (2) | 29.5, capped 51.8 | 40, but 300 behind 1000 (75) 37 (4) | 42, 2000 of
// 16/4 capped 71 (2) | 73.7. 64-wide, two workgroups to a CU: 8 prompts of 64-448 13.3
// (1) | 12.4, 1700 (168) 27.8 (3) | 32.7; but two turns of short chains start and end
// together: several in 300 workgroups and more, up to 7 tiles 0.94 to 0.98 of the time before | 1.02 to
// 1.21, from 350 on up to 11 tiles 0.92 to 0.98 | 1.04, 12 and more 0.82 to 0.94 | 0.80 to 0.88,
// capped 0.91 | 0.76.
// groups: KG; least: tiles of a part, 0 without parts; most: parts of a tile; units: tiles
// and parts a grid holds; scratch: floats
struct PagedRows {
  int groups = 1, least = 0, most = 1;
  bool meet = false;
  long units = 0, scratch = 0;
};
// Parts of a single sequence: of two groups of waves, which leave half the partial
// results in memory, where at least three of them make 200 to 256 units; us, one | two
// groups: 300 behind 2000 of 32/8 37.2 | 31.5, 300 behind 12000 of 16/4 64.8 | 48.7, of
// 28/4 (204 units) 91 | 78, capped 1900 and 32/8 47.1 | 44; two parts (256 units) of 1000
// behind 500 of 16/4 capped 38.6 | 42.8. The last part merges (meet) or a kernel of its
// own; us, kernel | last: 1700 of 64-wide heads 28.8 | 23.3, 300 behind 2000 of 32/8 31.3 |
// 26.4, 700 in a window 32.2 | 26.4; four parts of few tiles, whose merge is short, 60
// behind 2000 (64 units) 20.6 | 22.4, of 32 heads (128) 21.3 | 23.5; up to eight 60 behind
// 4000 23.4 | 28.2.
inline void paged_rows_one(PagedRows& x, long wgs, long tiles, int D, int terms) {
  const int least = terms == 1 ? 8 : 4;
  if (x.groups > 1 || wgs > 340 || tiles < 2 * least) return;
  const long twos = std::min<long>({256 / wgs, tiles / (terms == 1 ? 8 : 5), 16});
  if (D == 128 && twos > 2 && wgs * twos >= 200) x.groups = 2;
  x.most = x.groups == 2
               ? (int)twos
               : (int)std::min<long>({(512 + wgs / 2) / wgs, tiles / least, 16});
  x.least = x.groups == 2 ? 12 : least;
  x.meet = x.most <= 2 || (x.most <= 4 && wgs * x.most >= 160);
}
// Parts of several sequences, whose lengths only the kernel knows. Where their row tiles
// are many, parts are few: the last one merges. Where they are few a long sequence has
// many, which a kernel of its own merges sooner, and which are shorter. thin: so few rows
// that what the last part reads would be mostly padding.
//   712 drawn batches of 2 to 70 sequences, time over that of as many parts for all and a
// kernel for the merge, by workgroups before keys are split; one group of waves and a
// kernel | two and a kernel | one and the last | two and the last part. bf16 weights: up
// to 19 0.90 | 0.96 | 1.17 | 1.12, 39 0.85 | 0.87 | 0.98 | 0.93, 63 0.92 | 0.88 | 0.99 |
// 0.91, 95 0.93 | 0.88 | 0.90 | 0.82, 144 0.88 | 0.88 | 0.87 | 0.82, 199 0.92 | 0.99 | 0.85 |
// 0.88, 259 0.90 | 0.94 | 0.83 | 0.87, 340 0.97 | 1.01 | 0.89 | 0.95; thin ones from 64 on
// 0.90 | 0.99 | 0.95 | 0.97. 128-wide, 32-bit weights: 39 0.94 | 0.92 | 1.20 | 1.09, 63
// 0.96 | 0.96 | 0.94 | 0.93, 144 0.97 | 0.92 | 0.91 | 0.84, 256 0.96 | 0.99 | 0.87 | 0.92, 340
// 0.95 | 0.91 | 0.87 | 0.85. 64-wide from 64 on 0.97 | - | 0.82 | 0.85.
//   By two groups in 13 to 24 tiles too, below 145 workgroups (one part of two groups | by
// parts): 16 x 17-27 behind up to 1500 of 28/4 31.0 | 20.8, 3 x 19-127 of 32/32 27.1 | 20.2, 2
// x 168-385 behind 400-1100 of 16/4 29.3 | 21.5.
inline void paged_rows_several(PagedRows& x, long wgs, long tiles, int D, int terms,
                               bool thin) {
  if (wgs > 340) return;
  if (terms == 1) {
    if (x.groups > 1 ? wgs >= 145 || tiles < 13 : tiles < 16) return;
    x.meet = !thin && wgs >= 64 && (wgs >= 145 || tiles <= 128);
    if (x.meet) {
      x.groups = wgs < 145 ? 2 : 1;
      x.least = x.groups == 1 || tiles < 17 ? 12 : 8;
    } else {
      x.groups = thin || wgs < 20 || (wgs < 40 && tiles > 64) ? 1 : 2;
      x.least = wgs < 20 ? 4 : 6;
    }
  } else if (D == 128) {
    if (x.groups > 1 || tiles < 8) return;
    x.meet = !thin && wgs >= 40 && (wgs >= 64 || tiles <= 16) &&
             (wgs >= 96 || tiles <= 64);
    if (x.meet) {
      x.groups = wgs >= 64 && wgs < 145 ? 2 : 1;
      x.least = wgs < 64 ? 4 : wgs < 257 ? 6 : 8;
    } else {
      x.groups = tiles > 16 && !thin ? 2 : 1;
      x.least = 4;
    }
  } else {
    if (x.groups > 1 || tiles < 8) return;
    x.meet = !thin && wgs >= 64;
    x.least = x.meet ? 6 : 4;
  }
  x.most = x.meet ? PF_MEET(x.groups) : 16;
}
inline PagedRows paged_rows_plan(long tokens, int n_seqs, int G, int n_kv, int D,
                                 long max_blocks, int terms, bool options) {
  PagedRows x;
  const long row_tiles = paged_rows_tiles<PF_ROWS>(tokens, n_seqs, G);
  const long wgs = row_tiles * n_kv;
  const long keys = max_blocks * PF_BS, tiles = keys / PF_KT;
  const bool alone = n_seqs == 1 && 2 * keys < 3 * tokens;
  if (wgs == 0) return x;
  if (D == 64) {
    const bool brief = !options && n_seqs > 1 && wgs >= 300 &&
                       tiles <= (wgs < 350 ? 7 : 11);
    x.groups = keys >= 384 && wgs >= 200 && wgs <= 448 && !brief ? 2 : 1;
  } else if (terms > 1) {
    x.groups = keys >= 512 && tiles <= 20 && wgs >= 200 && wgs <= 256 ? 2 : 1;
  } else if (keys >= 640 && wgs >= 72) {
    x.groups = wgs <= 256 ? (tiles <= 24 || (n_seqs == 1 && wgs >= 200) ? 2 : 1)
                          : (wgs <= 448 && alone && tiles >= 18 ? 2 : 1);
  }
  if (n_seqs == 1) paged_rows_one(x, wgs, tiles, D, terms);
  else paged_rows_several(x, wgs, tiles, D, terms, tokens * G <= 64L * n_seqs);
  if (x.least == 0) return x;
  x.units = n_seqs > 1 ? row_tiles + PF_UNITS / x.groups / n_kv + 1
                       : row_tiles * x.most;
  x.scratch = x.units * n_kv * (PF_ROWS * (D + 2) + (x.meet ? 2 : 0)) +
              (x.meet || n_seqs == 1 ? 0 : tokens * G * n_kv * 2);
  return x;
}

inline long paged_rows_wgs(const PagedRows& p, long tokens, int n_seqs, int G,
                           int n_kv) {
  return (p.least > 0 ? p.units : paged_rows_tiles<PF_ROWS>(tokens, n_seqs, G)) *
         n_kv;
}

// Prompt rows and the merge of their parts
template <int D, int TERMS, bool MORE>
inline void paged_rows(void* out, float* ws_o, const unsigned short* q,
                       const unsigned short* k_cache,
                       const unsigned short* v_cache, const int* block_tables,
                       const int* cu_q, const int* seq_lens, long tokens,
                       int n_seqs, float scale, int n_qheads, int n_kv,
                       int max_blocks, long q_stride, long out_stride,
                       const PagedRows& plan, const PagedMore& x,
                       const PagedAhead& ahead, hipStream_t stream) {
  const int G = n_qheads / n_kv;
  if (tokens == 0 || n_seqs <= 0) return;
  const long wgs = paged_rows_wgs(plan, tokens, n_seqs, G, n_kv);
  PagedMeet meet;
  float* ws_ml = ws_o + wgs * PF_ROWS * D;
  if (plan.meet) meet = paged_meet(ws_ml, wgs * PF_ROWS, 1);
  int2* ws_at = plan.least > 0 && !plan.meet && n_seqs > 1
                    ? reinterpret_cast<int2*>(ws_ml + wgs * PF_ROWS * 2) : nullptr;
  const int turn = 256 / n_kv;
  // Batches that the CUs hold one to each come as they are, without a search: 8 x 38-140 of
  // 28/4 9.62 -> 9.46 us, 325 drawn ones 0.941 -> 0.934 of the time before there was one.
  const bool as_is = n_seqs > 1 && wgs <= 256;
#define PF_GO(KG, SPLIT, SORT)                                                 \
  hipLaunchKernelGGL((paged_attn_rows_kernel<D, TERMS, MORE, KG, SPLIT, SORT>),\
                     dim3((unsigned)(wgs + ahead.wgs)), dim3(KG * 256), 0,     \
                     stream, block_tables, cu_q, seq_lens, n_seqs, G, n_kv,    \
                     max_blocks, pf_inverse(n_kv), pf_inverse(G), k_cache, q,  \
                     v_cache, out, ws_o, ws_ml, ws_at,                         \
                     meet, scale, q_stride, out_stride, plan.least, plan.most, \
                     turn, x, ahead)
  if (plan.groups == 2 && plan.least > 0) PF_GO(2, true, true);
  else if (plan.groups == 2) PF_GO(2, false, true);
  else if (plan.least > 0) PF_GO(1, true, true);
  else if (as_is) PF_GO(1, false, false);
  else PF_GO(1, false, true);
#undef PF_GO
  if (plan.least > 0 && !plan.meet)
    paged_merge<D, MORE, PF_ROWS, PF_KT>(out, ws_o, ws_ml, ws_at, n_qheads, out_stride,
                                         tokens * n_qheads, x, stream, cu_q, seq_lens,
                                         n_seqs, n_kv, plan.most);
}

}  // namespace xllm
