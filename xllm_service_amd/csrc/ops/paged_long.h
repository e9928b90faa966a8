// Paged attention of long prompts, 128-wide heads, bf16 in and out, causal: waves that
// multiply and weigh in turn.
//
// Rows, tiles, products and LDS images are those of paged_rows.h. There each wave
// does a tile's products and then its weights, and what the two waves of a SIMD overlap
// is left to chance: 2610 cycles a tile and wave, a whole call's by counters, of which
// the matrix pipe works 1024 and the vector unit 1130. Here a workgroup has eight waves
// and 256 rows, two waves to a SIMD, which take turns: while waves 0-3 multiply (weights
// of the last tile by its values, keys of this one by the queries, 32 products without a
// pause), waves 4-7 make weights of their scores, then the other way round, a barrier
// between two half steps. Operands of the next four products are read from LDS during
// each four, the first ones before the barrier. Four tiles of K and V in LDS: loads have
// two steps to arrive. A wave's share of a step is one page, whose address three
// v_readlane fetch from a table of 64 tiles made at once: by scalar arithmetic on the way
// a step's loads cost 700 cycles.
//
// Bound by the card's power: 640 k cycles at 1.8 GHz while calls follow each other, 623 k at
// 2.35 with zeros for data (350 | 265 us). So what takes fewer cycles and as much energy gains
// nothing (all operands in registers before their products: 1660 -> 1380 cycles for a tile's
// 32, 328 -> 333 us), and what is left out counts: without exponentials 328 -> 313, without
// three quarters of the operands' reads 308, without the scaling of sums 321. Scaling them
// only in the lanes whose maximum has grown: 353.5 -> 348.0 (runs of one side differ by 0.7%;
// cards differ by 8%). 4 prompts of 1.6-2.3 k tokens over up to 3.1 k cached ones, 32 heads
// of 128. What it costs is one workgroup per CU: nothing covers its start and its end, so it
// is taken for whole turns of workgroups with long chains only (paged_long_takes).
#pragma once
#include "paged_rows.h"

namespace xllm {

#define PL_ROWS 256        // rows per workgroup
#define PL_BUFS 4          // tiles of K and V in LDS

__global__ __launch_bounds__(512) void paged_attn_long_kernel(
    unsigned short* __restrict__ out,        // [total_q, n_qheads, D]
    const unsigned short* __restrict__ q,    // [total_q, n_qheads, D] bf16
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, 16, D]
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ cu_q,            // [num_seqs+1] query offsets
    const int* __restrict__ seq_lens,        // [num_seqs] total key len
    const int n_seqs, const float scale, const int G, const int n_kv,
    const int max_blocks, const long q_stride, const long out_stride) {
  constexpr int D = 128;
  constexpr int KS = D / 16;                 // k steps of a score product
  constexpr int DT = D / 32;                 // 32-wide tiles of the head
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = 16 / RPI;               // ... instructions per page
  constexpr int TILE = PF_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short
      kv_lds[2 * PL_BUFS * TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;

  const int kvh = blockIdx.x % n_kv;
  PfPlace place;
  if (!pf_longest<PL_ROWS, 1>(blockIdx.x / n_kv, INT_MAX / 2, cu_q, seq_lens,
                              n_seqs, G, lane, &place))
    return;
  const int seq = place.seq, lt = place.lt, q_start = place.q_start,
            q_len = place.q_len, seq_len = place.seq_len;
  const int ctx = seq_len - q_len;
  const int rows = q_len * G;

  const int row0 = lt * PL_ROWS;
  const int kmax = ctx + (min(row0 + PL_ROWS, rows) - 1) / G + 1;
  const int n = (max(kmax, 0) + PF_KT - 1) / PF_KT;   // tiles; rows without keys: 0

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

  const PagedScore sc = paged_score<false>(PagedMore{}, scale, 0);
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

  // ---- staging: waves 0-3 move a page of K each, waves 4-7 one of V ----------
  const int half = wid >> 2, page4 = wid & 3;
  const int* btab = block_tables + (long)seq * max_blocks;
  const int last_blk = (seq_len - 1) / PF_BS;
  const int srow = lane / CPR, spos = lane % CPR;
  const unsigned short* cache = half ? v_cache : k_cache;
  // byte offset in a page of what this lane moves: row r of the page, its
  // chunk permuted by the row's key
  unsigned off[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int r = i * RPI + srow;
    off[i] = (unsigned)(r * (2 * D) +
                        ((spos ^ (half ? mr_swz_cols<D>(r) : mr_swz_rows<D>(r)))
                         << 4));
  }
  // Where this wave's pages of 64 tiles from the tb-th on are and how much of each
  // is keys, one tile per lane: what is left to do per tile is three v_readlane. A
  // row past the last key, and a tile past the last one, is out of the bounds.
  int tb = 0;
  unsigned from_lo = 0, from_hi = 0, bytes = 0;
  auto look_up = [&]() {
    const int t = tb + lane,
              pg = max(min(t, n - 1), 0) * (PF_KT / PF_BS) + page4;
    const long id = btab[min(pg, last_blk)];
    const unsigned long long at = (unsigned long long)(
        cache + (id * n_kv + kvh) * (PF_BS * D));
    from_lo = (unsigned)at;
    from_hi = (unsigned)(at >> 32);
    bytes = t < n ? min(max(seq_len - pg * PF_BS, 0), PF_BS) * (D * 2) : 0;
    asm volatile("" : "+v"(from_lo), "+v"(from_hi), "+v"(bytes));  // now
  };
  // Bundle j: keys of the j-th tile and values of the one before, which are read
  // together. This wave's share of it:
  auto stage = [&](unsigned j) {
    const int i = (int)j - half - tb;
    const unsigned lo = __builtin_amdgcn_readlane(from_lo, i);
    const unsigned hi = __builtin_amdgcn_readlane(from_hi, i);
    const auto src = mr_buffer((const void*)((unsigned long long)hi << 32 | lo),
                               __builtin_amdgcn_readlane(bytes, i));
    unsigned short* dst =
        kv_lds + (j % PL_BUFS * 2 + half) * TILE + page4 * 16 * D;
#pragma unroll
    for (int k = 0; k < NI; k++) mr_to_lds(src, off[k], dst + k * RPI * D);
  };
  // before bundle j is staged
  auto ready = [&](unsigned j) {
    if ((int)j - half - tb < 64) return;
    tb += 64;
    look_up();
  };
  // A half step ends. `later` bundles of this wave may be on the way
  auto meet = [&](int later) {
    __builtin_amdgcn_sched_barrier(0);
    if (later == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  const int kbase = mr_row_base<D>(lane), vbase = mr_col_base<D>(lane);
  const float c = sc.c;
  f32x16 s[2];
  bf16x8 p[4];
  float mc = 0.0f;
  // weights of keys [16 st, 16 st + 16) of a tile
  auto weigh = [&](int st) {
    const int i = st >> 1;
#pragma unroll
    for (int r = 8 * (st & 1); r < 8 * (st & 1) + 8; r += 2) {
      const float a = __builtin_amdgcn_exp2f(fmaf(s[i][r], c, -mc));
      const float b = __builtin_amdgcn_exp2f(fmaf(s[i][r + 1], c, -mc));
      l += a + b;
      reinterpret_cast<unsigned*>(&p[st])[(r & 7) >> 1] = pack_bf16(a, b);
    }
  };
  // operands of four products: 16 values' rows, or two steps of the keys'
  auto fetch_v = [&](bf16x8 (&f)[DT], const lds_u16* vt, int st) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
      f[dt] = mr_cols_own<D>(vt + (vbase ^ (dt << 5)) + st * 16 * D);
  };
  auto fetch_k = [&](bf16x8 (&f)[4], const lds_u16* kt, int ks) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      f[i] = *reinterpret_cast<const lds_bf16x8*>(
          kt + (kbase ^ ((ks + (i >> 1)) << 4)) + (i & 1) * 32 * D);
  };
  auto values = [&](const bf16x8 (&f)[DT], int st) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
      o_acc[dt] = mr_mma(f[dt], p[st], o_acc[dt]);
  };
  auto scores = [&](const bf16x8 (&f)[4], int ks) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      s[i & 1] = mr_mma(f[i], qf[ks + (i >> 1)], s[i & 1]);
  };
  // all of a tile's, the next operands on the way during each four products
  auto all_scores = [&](bf16x8 (&f)[4], const lds_u16* kt) {
    s[0] = s[1] = mr_zero();
    bf16x8 g[4];
#pragma unroll
    for (int ks = 0; ks < KS; ks += 4) {
      fetch_k(g, kt, ks + 2);
      scores(f, ks);
      __builtin_amdgcn_sched_barrier(0);
      if (ks + 4 < KS) fetch_k(f, kt, ks + 4);
      scores(g, ks + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // scores of tile j to weights
  auto settle = [&](int j) {
    const int k0 = j * PF_KT;
    if (k0 + PF_KT > wmin) {                     // uniform: a tile on the diagonal
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if (k0 + i * 32 + mr_key_of(r, h) >= limit) s[i][r] = -INFINITY;
        }
    }
    // online softmax: weights are 2^(c (s - m))
    float mt = s[0][0];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[i][r]);
    mt = pair_max(mt);
    if (mt > m) {                                // lanes without a new one rest
      const float alpha = __builtin_amdgcn_exp2f((m - mt) * c);
      m = mt;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o_acc[i][r] *= alpha;
    }
    mc = m == -INFINITY ? 0.0f : m * c;
    // made here: the compiler would move them behind the barrier, to their use
#pragma unroll
    for (int st = 0; st < 4; st++) {
      weigh(st);
      asm volatile("" : "+v"(p[st]));
    }
  };

  // tiles with keys that this wave's rows see
  const unsigned mine =
      wave_on ? (unsigned)(max(wmax, 0) + PF_KT - 1) / PF_KT : 0;
  look_up();
#pragma unroll
  for (int i = 0; i < PL_BUFS - 1; i++)
    if (i > 0 || !half) stage(i);
  if (half) meet(2);
  unsigned j = 0;
  const lds_u16 *kt, *vt;                      // of bundle j; values of the next
  auto open = [&]() {
    ready(j + PL_BUFS - 1);
    meet(1);
    __builtin_amdgcn_s_setprio(1);
    kt = (const lds_u16*)kv_lds + (j % PL_BUFS) * (2 * TILE);
    vt = (const lds_u16*)kv_lds + ((j + 1) % PL_BUFS) * (2 * TILE) + TILE;
  };
  if (mine > 0) {
    bf16x8 f[DT], g[DT], fk[4];
    open();
    fetch_k(fk, kt, 0);
    stage(j + PL_BUFS - 1);
    all_scores(fk, kt);
    __builtin_amdgcn_s_setprio(0);
    for (;;) {
      meet(2);
      settle(j);
      fetch_v(f, vt, 0);
      const lds_u16* v = vt;
      j++;
      open();
      if (j == mine) break;
      fetch_v(g, v, 1);
      values(f, 0);
      __builtin_amdgcn_sched_barrier(0);
      fetch_v(f, v, 2);
      values(g, 1);
      __builtin_amdgcn_sched_barrier(0);
      fetch_v(g, v, 3);
      values(f, 2);
      stage(j + PL_BUFS - 1);
      __builtin_amdgcn_sched_barrier(0);
      fetch_k(fk, kt, 0);
      values(g, 3);
      __builtin_amdgcn_sched_barrier(0);
      all_scores(fk, kt);
      __builtin_amdgcn_s_setprio(0);
    }
    stage(j + PL_BUFS - 1);
    values(f, 0);
#pragma unroll
    for (int st = 1; st < 4; st++) {
      fetch_v(f, kt + TILE, st);
      values(f, st);
    }
    __builtin_amdgcn_s_setprio(0);
    if ((int)j < n) meet(2);
    j++;
  }
  for (; (int)j <= n; j++) {
    open();
    stage(j + PL_BUFS - 1);
    __builtin_amdgcn_s_setprio(0);
    if ((int)j < n) meet(2);
  }
  if (!half) meet(2);
  // loads past the ends are still on their way to LDS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- epilogue: o_acc[dt][r] = O[row][dt*32 + 8*(r>>2) + 4h + (r&3)] --------
  l = pair_sum(l);
  if (!row_ok) return;
  const float inv = l != 0.0f ? 1.0f / l : 0.0f;
  const long at = (long)(q_start + qi) * out_stride + (long)head * D + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      paged_put<false>(PagedMore{}, out, at + dt * 32 + 2 * r,
                       o_acc[dt][r] * inv, o_acc[dt][r + 1] * inv,
                       o_acc[dt][r + 2] * inv, o_acc[dt][r + 3] * inv);
}

// Workgroups that fill their turns, one to a CU: the host knows the width of the tables,
// not the lengths, and counts as if sequences were equal. Us, paged_rows.h | here, by
// query/key heads, workgroups in parentheses:
//   nearly two turns   32/8: 4096 153 | 139 (512), 3760 133 | 120 (470), 3 x 1253 behind
//            3132 246 | 225 (480); 64/8: 1880 behind 4700 348 | 321 (470); but fewer, 2500
//            71.5 | 74 (320), 1024 behind 1024 50 | 56 (136)
//   up to two and a half, a third turn for a few   32/8: 4128 behind 4128 453 | 467
//            (516), 2 x 2064 behind 1444 184 | 202 (528), 3 x 1376 behind 3440 307 | 335
//            (528); 64/8: 3 x 688 behind 1720 164 | 182 (528), 2064 85.7 | 87.9 (520);
//            but 4200 and 100 behind 3000 205 | 161 (544), for the order of its chains
//   more     32/8: 3 x 1866 behind 4665 512 | 481 (720), 5600 behind 14000 1484 | 1369
//            (704); 64/8: 3 x 933 behind 2332 268 | 259 (720), but in tables of 2243 keys
//            2 x 1320 behind 923 152 | 156 (672). One sequence with little before it has
//            short chains for the last turn in both kernels: 64/8: 2800 141 | 149 (704),
//            32/32: 5600 270 | 278 (704); but of 7200, 32/8, 414 | 398 (904)
// Not many short prompts beside a long one, 2200 and 20 x 100 65 | 68.5 (688), 40 x 100
// behind 2000 207 | 217 (816), nor, of more than four turns, short ones at all: with
// eight query heads to each 7 x 500 and 2100 143 | 160 (1464), but 4096 294 | 284 (1032).
inline bool paged_long_takes(long tokens, int n_seqs, int G, int n_kv,
                             long max_blocks) {
  const long keys = max_blocks * PF_BS, rows = tokens * G;
  const long wgs = (rows + n_seqs * (long)PL_ROWS - 1) / (n_seqs * (long)PL_ROWS) *
                   n_seqs * n_kv;
  if (wgs < 440 || keys < 2048 || tokens < 256L * n_seqs) return false;
  if (wgs <= 512) return true;
  if (wgs <= 640 || keys < 3072) return false;
  if (wgs > 1100 && tokens < 1024L * n_seqs) return false;
  return n_seqs > 1 || 2 * keys >= 3 * tokens || keys >= 6144;
}

inline void paged_long(unsigned short* out, const unsigned short* q,
                       const unsigned short* k_cache,
                       const unsigned short* v_cache, const int* block_tables,
                       const int* cu_q, const int* seq_lens, long tokens,
                       int n_seqs, float scale, int n_qheads, int n_kv,
                       int max_blocks, long q_stride, long out_stride,
                       hipStream_t stream) {
  const int G = n_qheads / n_kv;
  if (tokens == 0 || n_seqs <= 0) return;
  hipLaunchKernelGGL(
      paged_attn_long_kernel,
      dim3((unsigned)(paged_rows_tiles<PL_ROWS>(tokens, n_seqs, G) * n_kv)),
      dim3(512), 0, stream, out, q, k_cache, v_cache, block_tables, cu_q,
      seq_lens, n_seqs, scale, G, n_kv, max_blocks, q_stride, out_stride);
}

}  // namespace xllm
