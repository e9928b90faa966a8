// Latent attention of prompt rows (bf16) for gfx950: rank 512 with a rotated tail
// of 0 or 64 entries, 16-token pages. Other sizes: latent_attn_mfma.hip, decoded rows
// latent_stream.hip.
//
// All heads of a token attend to the SAME cached rows [latent | rotated key], so
// (query, head) pairs are rows of one matrix, row = query * heads + head. A workgroup
// (8 waves, a CU to itself) owns 128 of them, two waves 32, or half as many where that
// leaves fewer CUs idle, four waves 32 (lr_plan). Per tile of 32 keys, by two:
//   S^T[key][row] = K Q^T        32x32x16 products, A = K rows from LDS, B = Q in
//                                registers. Each of the two waves takes half of the
//                                columns; they add each other's sums through LDS
//   online softmax               by both: a lane holds 16 keys of ONE row
//   O^T[col][row] += V^T P^T     each wave owns 256 columns; A = V^T by transpose
//                                reads of the same image, P split exactly into three
//                                bf16 terms, a product each
// So a wave keeps its queries (64 registers; two steps of 18 are in LDS) and sums (128)
// where they are, and a CU reads 320 KB of LDS per tile, 2560 cycles beside the 4224 of its
// products (66 of 32 cycles a wave, two waves a SIMD). (16 rows a wave, 16x16x32 products
// and a tile at a time read as long as they multiplied, and waited for each tile.)
//
// The two waves of a SIMD belong to different rows, and one's exponentials meet the
// other's products: half of the waves pass the barrier of the next tile between the
// scores of this one and its weights, the others after both. Hence three tiles in LDS:
// the one being weighed late, this one, and the one on its way, which the early waves ask
// for while the sums of scores are on theirs. The two waves of the same rows wait for
// each other's sums by flags in LDS, not at a barrier of all: both come to every tile that
// one comes to, and neither waits for anything else between its own sums and its flag.
//
// Measured, us, before | here: 16 heads, rows of 576, 1800 and 2200 tokens 1002 | 229 (1090
// TFLOP/s executed), 1000 tokens 247 | 75, 434 and 45 behind 5000 1244 | 128 (parts), by
// four waves 256 tokens 68 | 24, 16 25 | 9.2 (two waves 33 and 13.6); 32 heads, rows of 512 in
// a window of 1024, 3077 and 63 560 | 161. A tile takes about 7000 cycles of a CU (2.9 us),
// its products 4224; the clock is 1.9 GHz meanwhile (2.39 with zeros for data, in as many
// cycles). Of a wave's, steps of K asked for as they were needed took 900 more, and
// loads at the start of a tile 1000: their instructions queue. Error against 64 bits,
// the first three: 3.6e-7 | 3.0e-7, 3.3 | 2.1, 7.0 | 2.5.
//
// LDS image: rows 1152 B apart (those of 512 entries too), 16 B chunk c of row k at
// c ^ lr_swz(k). Rows alternate between the halves of the banks; with that the 16 rows of
// a row read, and the four 64 B pieces of a transpose read, fall on different ones.
#include <cmath>

#include "../ops/paged_rows.h"
#include "hybrid_common.h"

namespace xllm {
namespace hyb {

constexpr int LR_ROWS = 128;    // rows per workgroup, or half of them
constexpr int LR_KT = 32;       // keys per tile
constexpr int LR_SPLIT = 64;    // keys that parts are counted in
constexpr int LR_R = 512;       // value columns
constexpr int LR_W = 576;       // entries from row to row in LDS
constexpr int LR_TILE = LR_KT * LR_W;

XLLM_DEV int lr_swz(int k) { return (((k >> 1) & 1) << 2) | ((k >> 2) & 3); }

// V^T of what the caller has waited for: through a pointer without alias information the
// compiler waits for all loads to LDS first.
XLLM_DEV bf16x8 lr_cols(const lds_u16* __restrict__ p, int first, int second) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + first));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + second));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// SH: waves that share 32 rows
template <int W, int SH>
__global__ __launch_bounds__(512) void latent_rows_kernel(
    float* __restrict__ out,                     // [T, heads, 512]
    float* __restrict__ ws_o,                    // [units * LR_ROWS][512]
    float* __restrict__ ws_ml,                   // [units * LR_ROWS][2]
    int2* __restrict__ ws_at,                    // [T * heads]: first slot, parts
    const unsigned short* __restrict__ q,        // [T, heads, W]
    const unsigned short* __restrict__ cache,    // [blocks, 16, W]
    const int* __restrict__ block_tables, const int* __restrict__ cu_q,
    const int* __restrict__ seq_lens, const int n_seqs, const int heads,
    const int table_width, const float scale, const int least, const int most,
    const PagedMore x) {
  constexpr int ROWS = 8 / SH * 32;
  constexpr int NS = W / 16 / SH;                // steps of a wave's share of a score
  constexpr int COLS = LR_R / SH, CT = COLS / 32;   // its columns of the values
  constexpr int IPP = 16 * W / 512;              // load instructions per page
  constexpr int NI = 2 * IPP / 4;                // ... of a wave of four per tile
  constexpr int CPR = W / 8;                     // 16 B chunks of a row
  // steps with Q in registers, not LDS
  constexpr int QR = SH > 2 ? NS : W == LR_W ? 16 : 14;
  // One object: with several the compiler tells their accesses apart, but lets reads of
  // one wait for all loads to it. Three tiles, sums that waves swap, queries of
  // the last steps, 8 flags, keys that the rows see.
  constexpr int SWAP = 3 * LR_TILE, LAST = SWAP + 8 * 4 * 64 * 8,
                FLAG = LAST + 8 * (NS - QR) * 64 * 8, LIMIT = FLAG + 16;
  __shared__ __attribute__((aligned(1024))) unsigned short lds[LIMIT + 2 * ROWS];
  typedef volatile __attribute__((address_space(3))) int lds_flag;
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
  typedef __attribute__((address_space(3))) float lds_f32;
  lds_flag* flag = (lds_flag*)((lds_u16*)lds + FLAG);
  lds_f32x4* swap = (lds_f32x4*)((lds_u16*)lds + SWAP);

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int share = w % SH, rg = w / SH;         // columns, rows of the wave
  const bool late = w >= 4;
  const int h = lane >> 5, c32 = lane & 31;
  if (tid < 8) flag[tid] = 0;                    // seen after the first barrier

  int part = 0, parts = 1, first = 0;
  PfPlace at;
  if (least > 0) {
    if (!pf_parts<ROWS, true>(blockIdx.x, least, most, 2, INT_MAX / 2, x, cu_q,
                                 seq_lens, n_seqs, heads, 1, lane, &at, &part,
                                 &parts, &first))
      return;
  } else {
    if (!pf_longest<ROWS, 1>(blockIdx.x, INT_MAX / 2, cu_q, seq_lens, n_seqs,
                                heads, lane, &at))
      return;
  }
  at = {__builtin_amdgcn_readfirstlane(at.seq), __builtin_amdgcn_readfirstlane(at.lt),
        __builtin_amdgcn_readfirstlane(at.q_start),
        __builtin_amdgcn_readfirstlane(at.q_len),
        __builtin_amdgcn_readfirstlane(at.seq_len)};
  part = __builtin_amdgcn_readfirstlane(part);
  parts = __builtin_amdgcn_readfirstlane(parts);
  first = __builtin_amdgcn_readfirstlane(first);
  const int ctx = at.seq_len - at.q_len, rows = at.q_len * heads;
  const int row0 = at.lt * ROWS;
  const int kmax = ctx + (min(row0 + ROWS, rows) - 1) / heads + 1;
  const PagedTiles list =
      paged_tiles<true>(x, ctx + row0 / heads + 1, kmax,
                        (kmax + LR_SPLIT - 1) / LR_SPLIT, LR_SPLIT);
  const int tpp = (max(list.n, 0) + parts - 1) / parts;
  const int p_begin = part * tpp, p_end = min(list.n, p_begin + tpp);
  const int t_begin = list.at(p_begin) * (LR_SPLIT / LR_KT);
  const int t_end = min((p_end + list.gap) * (LR_SPLIT / LR_KT),
                        (kmax + LR_KT - 1) / LR_KT);

  // first key of a row that sees those below `limit`
  auto first_of = [&](int limit) { return x.window > 0 ? max(0, limit - x.window) : 0; };

  // ---- this lane's row: those past the last one repeat it, and go nowhere ------
  const int wrow0 = row0 + rg * 32;
  const bool wave_on = wrow0 < rows;
  const bool row_ok = wrow0 + c32 < rows;
  const int rho = min(wrow0 + c32, rows - 1);
  typedef __attribute__((address_space(3))) int lds_int;
  lds_int* limits = (lds_int*)((lds_u16*)lds + LIMIT) + rg * 32 + c32;
  *limits = ctx + rho / heads + 1;               // read by lanes that wrote the same
  const int wmin = ctx + min(wrow0, rows - 1) / heads + 1;   // ... of the wave
  const int wmax = ctx + (min(wrow0 + 32, rows) - 1) / heads + 1;
  // ... and of its half of the workgroup
  const int seen = late ? kmax : ctx + (min(row0 + ROWS / 2, rows) - 1) / heads + 1;
  const int wlo = first_of(wmin), whi = first_of(wmax);
  const long row = (long)at.q_start * heads + rho;
  const short flip = scale < 0.0f ? (short)0x8000 : (short)0;
  const float c = __uint_as_float(                // in a scalar register
      __builtin_amdgcn_readfirstlane(__float_as_uint(paged_factor(scale))));
  // step i: two of every 2 SH, an odd last one of those that are left (W 576, SH 4)
  constexpr int PAIRS = NS / 2 * 2;
  auto step_of = [&](int i) {
    return i < PAIRS ? 2 * SH * (i >> 1) + (i & 1) + 2 * share : PAIRS * SH + share;
  };
  bf16x8 qf[QR];
  lds_bf16x8* qlast =
      (lds_bf16x8*)((lds_u16*)lds + LAST) + w * (NS - QR) * 64 + lane;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const bf16x8 z =
        *reinterpret_cast<const bf16x8*>(
            q + row * W + step_of(i) * 16 + h * 8) ^ flip;
    if (i < QR) qf[i] = z;
    else qlast[(i - QR) * 64] = z;               // read by this lane alone
  }

  // ---- loads: instruction i of wave w, 0 to 3, is the (4 i + w)-th of the tile -------
  const int* table = block_tables + (long)at.seq * table_width;
  const int last_blk = (at.seq_len - 1) / 16;
  int tb = t_begin;                              // ids of the pages of 32 tiles from here
  auto pages_from = [&](int t) { return table[min(2 * t + lane, last_blk)]; };
  int pages = 0;
  auto stage = [&](int t, int buf) {
    const auto page = [&](int p) {               // keys that no row sees: zeros
      const int id = __builtin_amdgcn_readlane(pages, 2 * (t - tb) + p);
      // (a clamp of both ends is a vector instruction)
      const int n = __builtin_amdgcn_readfirstlane(
          min(max(kmax - (2 * t + p) * 16, 0), 16));
      return mr_buffer(cache + (long)id * (16 * W), n * (2 * W));
    };
    const auto p0 = page(0), p1 = page(1);
    unsigned short* dst = lds + buf * LR_TILE;
    // places in the page are computed for each tile: kept, they would be five registers
    // of the 256, and others would go to memory
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int j = 4 * i + w;
      const unsigned chunk = (j - (j >= IPP ? IPP : 0)) * 64 + ln;
      const unsigned r = chunk / CPR, pos = chunk - r * CPR;
      mr_to_lds(j >= IPP ? p1 : p0, r * (2 * W) + ((pos ^ lr_swz(r)) << 4),
                dst + (W == LR_W ? j * 512 : j * LR_W));
    }
  };

  // ---- LDS addresses (entries, first buffer) -------------------------------------
  // step i of K: ^ 16 (i % 2) + 32 SH (i / 2)
  const int kat = c32 * LR_W + (((4 * share + h) ^ lr_swz(c32)) << 3);
  const int klast = c32 * LR_W + 16 * PAIRS * SH + (((2 * share + h) ^ lr_swz(c32)) << 3);
  // V^T of keys r .. r + 3 (and 4 further on in the upper lanes), column tile ct: ^ 32
  // (ct % 2) + 64 (ct / 2). Keys from `most` on, whose weights are zero, give way to the
  // one before: their values may be infinite or NaN.
  auto place = [&](int r, int most) {
    int i = lane & 15;
    asm volatile("" : "+v"(i));                  // not kept in registers meanwhile
    r = min(r + 4 * h + (i >> 2), most - 1);
    const int chunk = ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
    return r * LR_W + share * COLS + ((chunk ^ lr_swz(r)) << 3) + (i & 1) * 4;
  };
  const int vat = place(0, LR_KT);               // 8 keys on: ^ 16 + 8 rows

  f32x16 acc[CT], s;
#pragma unroll
  for (int i = 0; i < CT; i++) acc[i] = mr_zero();
  float m = -INFINITY, l = 0.0f;

  // n: of the tile, from 1 on; between: while the other wave's sums are on their way
  auto score = [&](int n, int buf, const auto& between) {
    __builtin_amdgcn_s_setprio(1);
    const int k = kat + buf * LR_TILE;
    auto key = [&](int i) {
      return *reinterpret_cast<const lds_bf16x8*>(
          (const lds_u16*)lds +
          (i < PAIRS ? (k ^ (i & 1) * 16) + (i >> 1) * (32 * SH)
                     : klast + buf * LR_TILE));
    };
    // rows of KA steps on their way ahead of the products
    constexpr int KA = 4;
    bf16x8 f[KA + 1], ql[NS > QR ? NS - QR : 1];
#pragma unroll
    for (int i = 0; i < KA; i++) f[i] = key(i);
    __builtin_amdgcn_sched_group_barrier(0x100, KA, 0);
    s = mr_zero();
#pragma unroll
    for (int i = 0; i < NS; i++) {
      if (i + KA < NS) f[(i + KA) % (KA + 1)] = key(i + KA);
      if (i + 2 >= QR && i + 2 < NS) ql[i + 2 - QR] = qlast[(i + 2 - QR) * 64];
      s = mr_mma(f[i % (KA + 1)], i < QR ? qf[i < QR ? i : 0] : ql[i < QR ? 0 : i - QR],
                 s);
      if (i + KA < NS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (i + 2 >= QR && i + 2 < NS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
      swap[(w * 4 + r) * 64 + lane] =
          f32x4{s[4 * r], s[4 * r + 1], s[4 * r + 2], s[4 * r + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    flag[w] = n;
    __builtin_amdgcn_s_setprio(0);
    between();
    // the waves of these rows add up in the same order: all come to the same weights
    if constexpr (SH == 2) {
      while (__builtin_amdgcn_readfirstlane(flag[w ^ 1]) < n) {}
      asm volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const f32x4 y = swap[((w ^ 1) * 4 + r) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; e++) s[4 * r + e] += y[e];
      }
    } else {
#pragma unroll
      for (int i = 1; i < SH; i++)
        while (__builtin_amdgcn_readfirstlane(flag[w ^ i]) < n) {}
      asm volatile("" ::: "memory");
      const int w0 = w - share;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        f32x4 y[SH];
#pragma unroll
        for (int i = 0; i < SH; i++) y[i] = swap[((w0 + i) * 4 + r) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; e++)
          s[4 * r + e] = (y[0][e] + y[1][e]) + (y[2][e] + y[3][e]);
      }
    }
  };
  auto weigh = [&](int t, int buf) {
    const int k0 = t * LR_KT;
    if (k0 + LR_KT > wmin || k0 < whi) {         // uniform
      const int limit = *limits, lo = first_of(limit);
      const unsigned span = (unsigned)max(limit - lo, 0);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const unsigned key = (unsigned)(k0 + 8 * (r >> 2) + 4 * h + (r & 3) - lo);
        s[r] = key < span ? s[r] : -INFINITY;
      }
    }
    // weights are 2^(c (s - m))
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mt = fmaxf(mt, s[r]);
    mt = pair_max(mt);
    // Sums are scaled only where a maximum has grown by more than 2^8: scaled weights and
    // sums round the same, and some row of 32 has a new maximum in most tiles.
    if (__any((mt - m) * c > 8.0f)) {
      const float m_new = fmaxf(m, mt);
      const float alpha =
          __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < CT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    const int v = vat + buf * LR_TILE;
#pragma unroll
    for (int st = 0; st < 2; st++) {
      bf16x8 p[3];
#pragma unroll
      for (int r = 0; r < 8; r += 2) {
        float a = __builtin_amdgcn_exp2f(fmaf(s[8 * st + r], c, -mc));
        float b = __builtin_amdgcn_exp2f(fmaf(s[8 * st + r + 1], c, -mc));
        l += a + b;
#pragma unroll
        for (int e = 0; e < 3; e++) {
          const unsigned u = pack_bf16(a, b);
          reinterpret_cast<unsigned*>(&p[e])[r >> 1] = u;
          drop_bf16(a, b, u);
        }
      }
      int at0 = v + st * (16 * LR_W), at1 = (at0 ^ 16) + 8 * LR_W;
      if (k0 + LR_KT > seen) {                   // uniform
        at0 = place(st * 16, seen - k0) + buf * LR_TILE;
        at1 = place(st * 16 + 8, seen - k0) + buf * LR_TILE;
      }
      // values of the next tiles on the way during the products of one; even tiles first,
      // so that there are two addresses at a time
      constexpr int AHEAD = SH > 2 || W != LR_W ? 2 : 1, EVEN = CT / 2;
      auto value = [&](int i) {
        const int y = i < EVEN ? 0 : 32;
        return lr_cols((const lds_u16*)lds + i % EVEN * 64, at0 ^ y, at1 ^ y);
      };
      bf16x8 f[AHEAD + 1];
#pragma unroll
      for (int i = 0; i < AHEAD; i++) f[i] = value(i);
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);
#pragma unroll
      for (int i = 0; i < CT; i++) {
        const int ct = 2 * (i % EVEN) + i / EVEN;
        if (i + AHEAD < CT) f[(i + AHEAD) % (AHEAD + 1)] = value(i + AHEAD);
#pragma unroll
        for (int e = 0; e < 3; e++)
          acc[ct] = mr_mma(f[i % (AHEAD + 1)], p[e], acc[ct]);
        if (i + AHEAD < CT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
      }
    }
  };

  // tile t is there, and nobody reads the one before the last
  auto meet = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (t_begin < t_end) {
    pages = pages_from(t_begin);
    if (!late) stage(t_begin, 0);
    meet();
  }
  for (int t = t_begin, buf = 0; t < t_end; t++) {
    const int k0 = t * LR_KT, next = buf == 2 ? 0 : buf + 1;
    auto ahead = [&]() {
      if (late || t + 1 >= t_end) return;
      if (t + 1 - tb == 32) {
        tb += 32;
        pages = pages_from(tb);
      }
      stage(t + 1, next);
    };
    // uniform, and the same for the two waves of these rows
    const bool on = wave_on && k0 < wmax && k0 + LR_KT > wlo;
    if (on) score(t - t_begin + 1, buf, ahead);
    else ahead();
    if (late && t + 1 < t_end) meet();
    if (on) weigh(t, buf);
    if (!late && t + 1 < t_end) meet();
    buf = next;
  }

  // acc[ct][r] = O[row][COLS share + 32 ct + 8 (r / 4) + 4 h + r % 4]
  l = pair_sum(l);
  // parts of a row lie together
  const long slot0 = (long)first * ROWS + part;
  if (row_ok && share == 0 && h == 0) {
    const int in = rg * 32 + c32;
    if (ws_at != nullptr && part == 0)
      ws_at[row] = make_int2(first * ROWS + in * parts, parts);
    if (parts > 1) {
      const long slot = slot0 + in * parts;
      ws_ml[slot * 2] = m == -INFINITY ? m : m * c;
      ws_ml[slot * 2 + 1] = t_begin < t_end ? l : PAGED_ABSENT;
    }
  }
  if (parts > 1 && t_begin >= t_end) return;     // uniform
  // Through LDS, two column tiles at a time: a lane's four columns of a row alone are
  // 16 B to memory, 16 lanes' are 256.
  const float inv = parts > 1 ? 1.0f : l != 0.0f ? 1.0f / l : 0.0f;
  constexpr int OW = 64 + 4;                     // of a row, padded
  __syncthreads();
  lds_f32* o = (lds_f32*)((lds_u16*)lds) + w * (32 * OW);
  const int orow = lane >> 4, ocol = (lane & 15) * 4;
  float* to = parts > 1 ? ws_o + (slot0 + (long)rg * 32 * parts) * LR_R
                        : out + ((long)at.q_start * heads + wrow0) * LR_R;
  const int stride = (parts > 1 ? parts : 1) * LR_R;
  const int here = rows - wrow0;                 // rows of the wave
#pragma unroll
  for (int ct = 0; ct < CT; ct += 2) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *(lds_f32x4*)(o + c32 * OW + i * 32 + 2 * r + 4 * h) =
            f32x4{acc[ct + i][r] * inv, acc[ct + i][r + 1] * inv,
                  acc[ct + i][r + 2] * inv, acc[ct + i][r + 3] * inv};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int r = i * 4 + orow;
      const f32x4 y = *(const lds_f32x4*)(o + r * OW + ocol);
      if (r < here)
        *reinterpret_cast<f32x4*>(to + (long)r * stride + share * COLS + ct * 32 +
                                  ocol) = y;
    }
  }
}

bool latent_rows_takes(int W, int r, int block_size) {
  return r == LR_R && (W == 512 || W == LR_W) && block_size == 16;
}

// least: 64-key tiles of a part, 0 without parts; most: parts of a row tile; units: row
// tiles and parts that the grid holds
// A row tile is a chain of 3 us per 64 keys, so keys are split where row tiles leave CUs
// idle: a single sequence's evenly (paged_equal: parts of four tiles and more), several by
// their lengths (pf_parts). Us, not split | in parts: 16 tokens of 16 heads behind 7000 521
// | 42 (least 4 46, 8 60), 45 and 434 behind 5000 416 | 132, 34-309 behind 1000 93 | 54,
// 1000 alone 90 | 74. Between 128 and 200 row tiles short tables gain nothing: 44 and 1024
// of 32 heads 55 | 61, 389 and 1250 85 | 91; long ones do: 210-828 behind 150-4000 206 | 154.
// Parts take scratch: at most 67 MB for one sequence (256 units of 128 rows), 112 MB for
// several (425).
struct LrPlan { int rows = LR_ROWS, least = 0, most = 1; long units = 0, scratch = 0; };
static LrPlan lr_split(int rows, long wgs, int n_seqs, long tiles) {
  LrPlan x;
  x.rows = rows;
  x.units = wgs;
  if (wgs == 0 || tiles < 8) return x;
  if (n_seqs == 1) {
    x.most = (int)std::min<long>({256 / wgs, tiles / 2, 32});
    if (x.most > 1) x.least = 2;
  } else if (wgs <= 128 || (wgs <= 200 && tiles >= 32)) {
    x.most = 16;
    x.least = 2;
  }
  return x;
}
// Estimated time of a call, us. tokens, keys: of a sequence on average, of the longest
// there can be; walked: of them those that a row sees at most. A tile of 64 keys takes a
// workgroup 5.8 us, 4.1 with 64 rows (they read the same keys, swap as many sums and make
// as many weights), and where all CUs are busy 8 and 5.2. A part's sums go out and come
// back, 0.07 us for each 128 rows on top of 3.
static double lr_time(const LrPlan& p, int n_seqs, double tokens, double keys,
                      double walked) {
  const bool half = p.rows < LR_ROWS;
  const double units = p.units, tiles = std::max(1.0, walked / LR_SPLIT);
  const double fixed = half ? 7.0 : 10.0, tile = half ? 4.1 : 5.8;
  if (p.least > 0) {
    const double all = units * tiles * 0.6;      // of several: their lengths differ
    const double per = n_seqs == 1 ? std::ceil(tiles / p.most)
                                   : std::max(2.0, all / (PF_UNITS / 2));
    const double parts = n_seqs == 1 ? units * p.most : std::max(units, all / per);
    return fixed + tile * per + 3.0 + parts * (half ? 0.035 : 0.07);
  }
  // The first `climb` rows of a prompt see ever more keys, from `least` on. Workgroups
  // past a turn of the CUs, the shortest chains, follow others that are hardly longer.
  const double climb = std::max(0.0, walked - std::max(0.0, keys - tokens));
  const double rising = std::min(1.0, climb / std::max(1.0, tokens));
  const double least = tiles * (walked - climb) / std::max(1.0, walked);
  const double left = std::min(std::max(0.0, units - 256.0), 256.0) / units;
  const double next = left <= 0.0 ? 0.0 : left >= rising
      ? tiles : least + (tiles - least) * left / rising;
  const double all = units * (tiles - rising * (tiles - least) / 2) / 256.0;
  return fixed + std::max(tile * std::max(tiles, 2 * next), (half ? 5.2 : 8.0) * all);
}
// Row tiles of 64 rows, 32 of which four waves share, where they are estimated to be
// faster: for calls that leave CUs idle, or that few chains outlast. Us, 128 | 64 rows, row
// tiles of 128 in parentheses: 16 heads, one prompt of 16 tokens 13.6 | 9.2 (2), 64 17.2 |
// 11.8 (8), 256 33 | 24 (32), 512 46.8 | 38.3 (64), 1000 73 | 71.8 (125), 1300 115 | 93 (163),
// 4 of 128 24.9 | 18.5 (67), 8 of 64-200 30.9 | 24.9 (145), 351-1771 95 | 76 (199), 40 behind
// 3000 42.9 | 34.6 (5); but 300 behind 3000 81 | 91 (38), of 32 heads 133 | 208 (75), 533
// behind 3900 356 | 508 (133), 200-500 behind 100-2000 67 | 92 (75), 2031 in a window of
// 1024 109 | 154 (254), 5 of 221-475 behind 39-257 85 | 113 (451).
static LrPlan lr_plan(long tokens, int n_seqs, int heads, long table_width,
                      int window) {
  const long keys = table_width * 16;
  long tiles = (keys + LR_SPLIT - 1) / LR_SPLIT;
  if (window > 0) tiles = std::min<long>(tiles, window / LR_SPLIT + 3);
  LrPlan x = lr_split(LR_ROWS, paged_rows_tiles<LR_ROWS>(tokens, n_seqs, heads), n_seqs,
                      tiles);
  const LrPlan y =
      lr_split(LR_ROWS / 2, paged_rows_tiles<LR_ROWS / 2>(tokens, n_seqs, heads), n_seqs,
               tiles);
  const double each = (double)tokens / std::max(n_seqs, 1);
  const double walked = window > 0 ? std::min<double>(keys, window + LR_SPLIT) : keys;
  if (x.units > 0 && lr_time(y, n_seqs, each, keys, walked) <
                         0.93 * lr_time(x, n_seqs, each, keys, walked))
    x = y;                                       // (7%: what the estimate is off by)
  if (x.least == 0) return x;
  x.units = n_seqs > 1 ? x.units + PF_UNITS / 2 + 1 : x.units * x.most;
  x.scratch = x.units * x.rows * (LR_R + 2) + (n_seqs > 1 ? tokens * heads * 2 : 0);
  return x;
}
// floats
long latent_rows_scratch(long tokens, int n_seqs, int heads, long table_width,
                         int window) {
  return lr_plan(tokens, n_seqs, heads, table_width, window).scratch;
}

void latent_rows_way(long tokens, int n_seqs, int heads, long table_width, int window,
                     int* rows, int* least, int* most) {
  const LrPlan p = lr_plan(tokens, n_seqs, heads, table_width, window);
  *rows = p.rows;
  *least = p.least;
  *most = p.most;
}

// q, cache and out 16 B aligned
void launch_latent_rows(float* out, float* ws, const unsigned short* q,
                        const unsigned short* cache, const int* block_tables,
                        const int* cu_q, const int* seq_lens, long tokens,
                        int n_seqs, int heads, int W, int table_width, float scale,
                        int window, hipStream_t st) {
  if (tokens == 0 || n_seqs == 0) return;
  const LrPlan p = lr_plan(tokens, n_seqs, heads, table_width, window);
  PagedMore x;
  x.window = window;
  x.out_f32 = 1;
  float* ws_ml = ws + p.units * p.rows * LR_R;
  int2* ws_at = p.least > 0 && n_seqs > 1
                    ? reinterpret_cast<int2*>(ws_ml + p.units * p.rows * 2) : nullptr;
  const bool few = p.rows < LR_ROWS;
  auto k = W == LR_W ? (few ? latent_rows_kernel<LR_W, 4> : latent_rows_kernel<LR_W, 2>)
                     : (few ? latent_rows_kernel<512, 4> : latent_rows_kernel<512, 2>);
  hipLaunchKernelGGL(k, dim3((unsigned)p.units), dim3(512), 0, st, out, ws, ws_ml,
                     ws_at, q, cache, block_tables, cu_q, seq_lens, n_seqs, heads,
                     table_width, scale, p.least, p.most, x);
  if (p.least > 0) {
    auto merge = few ? paged_merge<LR_R, true, LR_ROWS / 2, LR_SPLIT>
                     : paged_merge<LR_R, true, LR_ROWS, LR_SPLIT>;
    merge(out, ws, ws_ml, ws_at, heads, (long)heads * LR_R, tokens * heads, x, st, cu_q,
          seq_lens, n_seqs, 1, p.most);
  }
}

}  // namespace hyb
}  // namespace xllm
