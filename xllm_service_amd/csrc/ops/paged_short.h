// Paged attention of few prompt rows, bf16 in and out, causal.
//
// Rows, tiles, products and LDS images are those of paged_rows.h, but where row
// tiles leave CUs idle, what counts is the chain: 300 tokens of 16/4 heads are 40
// workgroups of 128 rows there, which walk up to five tiles of keys each, a barrier and
// a wait for every one. Here a workgroup has 32 rows, and its four waves walk every
// fourth tile, each through LDS of its own and without a barrier; their results meet
// in LDS at the end. The keys of a wave's next tile are fetched while this one's
// weights and values are multiplied, its values during the next scores.
//
// Bound by that chain and the launch. Measured (us, paged_rows.h, with its merge where
// it splits | here): 300 tokens of 16/4 heads of 128 11.9 | 10.3, 512 of them
// 16.8 | 11.7, 1000 of 8/1 25.1 | 14.9, 100 of 32/8 behind 800 22.8 | 14.6, 1000 of 12/12
// heads of 64 19.8 | 14.6, 300 of 16/4 in a window 17.3 | 13.7, capped 22.2 | 16.1. What a CU
// pulls (61 KB/us: each wave has tiles of its own) bounds longer chains: 64 rows a wave,
// half as much to pull, were slower (300 tokens 17, 100 behind 4000 60 | 40 for 32 rows).
// A single sequence's chain begins with its pages and arguments at once (a kernel of its
// own: a branch costs the others what it saves here): 300 tokens of 16/4 heads 9.9 -> 9.0,
// 100 behind 800 of 32/8 13.8 -> 12.4, 60 behind 1000 of 28/4 15.4 -> 14.1.
// A SIMD has one wave, whose products' sums would lie in the half of its registers that
// only products read: with them in the other half (a flag of the build) 60 behind 500 of
// 32/8 heads 13.1 -> 12.4, 100 behind 1000 18.0 -> 17.3, 2 x 500 of 12/12 of 64 14 -> 13.3.
#pragma once
#include "paged_rows.h"

namespace xllm {

#define PS_ROWS 32         // rows per workgroup
#define PS_WAVES 4
#define PS_KEYS 2048       // that a row sees, at most

// ONE: there is a single sequence
template <int D, int TERMS, bool MORE, bool ONE>
__global__ __launch_bounds__(PS_WAVES * 64) void paged_attn_short_kernel(
    const int* __restrict__ block_tables,    // [num_seqs, max_blocks]
    const int* __restrict__ cu_q,            // [num_seqs+1] query offsets
    const int* __restrict__ seq_lens,        // [num_seqs] total key len
    const int n_seqs, const int G, const int n_kv, const int max_blocks,
    const unsigned short* __restrict__ k_cache,  // [blocks, n_kv, 16, D]
    const unsigned short* __restrict__ q,    // [total_q, n_qheads, D] bf16
    const unsigned short* __restrict__ v_cache,
    void* __restrict__ out,                  // [total_q, n_qheads, D]
    const float scale, const long q_stride, const long out_stride,
    const PagedMore x, const PagedAhead ahead) {
  constexpr int KS = D / 16;                 // k steps of a score product
  constexpr int DT = D / 32;                 // 32-wide tiles of the head
  constexpr int CPR = D / 8;                 // 16 B chunks of a row
  constexpr int RPI = 64 / CPR;              // rows one load instruction fills
  constexpr int NI = 16 / RPI;               // ... instructions per page
  constexpr int PAGES = PF_KT / PF_BS;       // of a tile
  constexpr int TILE = PF_KT * D;            // elements of a K or V tile
  __shared__ __attribute__((aligned(1024))) unsigned short
      kv_lds[PS_WAVES * 2 * TILE];
  __shared__ float2 ml[PS_WAVES][PS_ROWS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;

  // Of a single sequence the pages of the wave's 16 tiles are asked for before its length
  // is known: what lies past the last one is not used. The arguments come together, as the
  // compiler would not ask for them: each wait for some of them is 0.2 us. (Several
  // sequences' first pages, a sequence to a lane, delay the search: 3 x 40-120 behind
  // 100-500 of 16/4 heads 10.0 -> 10.2.)
  const int tile = wid + PS_WAVES * (lane / PAGES);   // of this lane's page
  const bool early = ONE && (!MORE || x.window <= 0);
  int id = 0;
  if (early) id = block_tables[min(tile * PAGES + lane % PAGES, max_blocks - 1)];
  if (!MORE && (int)blockIdx.x >= ahead.from) {
    paged_fetch(ahead, blockIdx.x - ahead.from, kv_lds);
    return;
  }
  if constexpr (ONE)
    asm volatile("" ::"s"(q), "s"(k_cache), "s"(v_cache), "s"(q_stride), "s"(scale));
  const int kvh = blockIdx.x % n_kv;
  PfPlace place;
  if (ONE ? !pf_only<PS_ROWS>(blockIdx.x / n_kv, INT_MAX / 2, cu_q, seq_lens, G, &place)
          : !pf_locate<PS_ROWS>(blockIdx.x / n_kv, cu_q, seq_lens, n_seqs, G, lane,
                                &place))
    return;
  const int q_start = place.q_start, q_len = place.q_len,
            seq_len = place.seq_len;
  const int ctx = seq_len - q_len;
  const int rows = q_len * G;
  const int row0 = place.lt * PS_ROWS;
  const int rho = row0 + c32;
  const bool row_ok = rho < rows;
  const int qi = rho / G;
  const int head = kvh * G + rho - qi * G;
  const int limit = row_ok ? ctx + qi + 1 : 0;   // keys this row sees
  const int wmin = ctx + row0 / G + 1;           // fewest of a row
  const int kmax = ctx + (min(row0 + PS_ROWS, rows) - 1) / G + 1;
  const PagedTiles list = paged_tiles<MORE>(x, wmin, kmax,
                                            (kmax + PF_KT - 1) / PF_KT, PF_KT);
  const int n = list.n;                          // this wave's tiles: wid + 4 i
  // keys below lo are out of sight but for the kept ones
  const int lo = paged_first<MORE>(x, row_ok ? limit : 1);
  const int whi = paged_first<MORE>(x, kmax);

  const PagedScore sc = paged_score<MORE>(x, scale, row_ok ? head : kvh * G);
  const float c = sc.c;
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

  // ---- staging -----------------------------------------------------------------
  const int* btab = block_tables + (long)place.seq * max_blocks;
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
  // Where the pages of this wave's tiles are, and how much of each is keys, one page
  // per lane: 16 tiles, where a row that sees PS_KEYS keys has up to 9 for a wave and one
  // past them is asked for. Rows past the last key, and tiles past the last one, are out
  // of the bounds: zeros.
  static_assert((PS_KEYS / PF_KT / PS_WAVES + 2) * PAGES <= 64, "pages per lane");
  unsigned at_lo = 0, at_hi = 0, bytes = 0;
  auto look_up = [&]() {
    const int pg = list.at(min(tile, n - 1)) * PAGES + lane % PAGES;
    if (!early) id = btab[min(pg, last_blk)];
    const long at = ((long)id * n_kv + kvh) * (PF_BS * D * 2);
    at_lo = (unsigned)at;
    at_hi = (unsigned)(at >> 32);
    bytes = tile < n ? min(max(seq_len - pg * PF_BS, 0), PF_BS) * (D * 2) : 0;
    asm volatile("" : "+v"(at_lo), "+v"(at_hi), "+v"(bytes));   // waited for here
  };
  unsigned short* kv = kv_lds + wid * (2 * TILE);
  // keys (values) of this wave's i-th tile
  auto stage = [&](int i, bool val) {
#pragma unroll
    for (int p = 0; p < PAGES; p++) {
      const int at = i * PAGES + p;
      const unsigned a = __builtin_amdgcn_readlane(at_lo, at);
      const unsigned b = __builtin_amdgcn_readlane(at_hi, at);
      const auto src = mr_buffer(
          (const char*)(val ? v_cache : k_cache) +
              (long)((unsigned long long)b << 32 | a),
          __builtin_amdgcn_readlane(bytes, at));
#pragma unroll
      for (int k = 0; k < NI; k++)
        mr_to_lds(src, val ? voff[k] : koff[k],
                  kv + (val ? TILE : 0) + (p * 16 + k * RPI) * D);
    }
  };
  // the last tile's worth of loads of this wave may be on the way
  auto arrived = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI * PAGES) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto read = [&]() {                            // what is loaded over has been read
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  const int kbase = mr_row_base<D>(lane), vbase = mr_col_base<D>(lane);
  const lds_u16* kt = (const lds_u16*)kv;
  const lds_u16* vt = kt + TILE;
  if (wid < n) {
    look_up();
    stage(0, false);
    stage(0, true);
  }
  for (int i = 0; wid + PS_WAVES * i < n; i++) {
    const int k0 = list.at(wid + PS_WAVES * i) * PF_KT;
    arrived();                                   // keys
    f32x16 s[2] = {mr_zero(), mr_zero()};
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        s[j] = mr_mma(*reinterpret_cast<const lds_bf16x8*>(
                          kt + (kbase ^ (ks << 4)) + j * 32 * D),
                      qf[ks], s[j]);
    read();
    stage(i + 1, false);
    if (MORE && x.cap > 0.0f) paged_cap<2>(s, sc.pre, x.cap);
    // uniform: a tile on the diagonal or on the edge of a window
    if (k0 + PF_KT > wmin || (MORE && k0 < whi))
      paged_mask<MORE>(x, s, limit, lo, [&](int j, int r) {
        return k0 + j * 32 + mr_key_of(r, h);
      });
    // online softmax: weights are 2^(c (s - m))
    float mt = s[0][0];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[j][r]);
    mt = pair_max(mt);
    const float m_new = fmaxf(m, mt);
    const float alpha =
        __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < DT; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) o_acc[j][r] *= alpha;
    const float mc = m == -INFINITY ? 0.0f : m * c;
    bf16x8 p[TERMS][4];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        float a = __builtin_amdgcn_exp2f(fmaf(s[j][r], c, -mc));
        float b = __builtin_amdgcn_exp2f(fmaf(s[j][r + 1], c, -mc));
        l += a + b;
#pragma unroll
        for (int e = 0; e < TERMS; e++) {
          const unsigned u = pack_bf16(a, b);
          reinterpret_cast<unsigned*>(
              &p[e][j * 2 + (r >> 3)])[(r & 7) >> 1] = u;
          drop_bf16(a, b, u);
        }
      }
    arrived();                                   // values
#pragma unroll
    for (int st = 0; st < 4; st++)
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const bf16x8 a = mr_cols_own<D>(vt + (vbase ^ (dt << 5)) + st * 16 * D);
#pragma unroll
        for (int e = 0; e < TERMS; e++)
          o_acc[dt] = mr_mma(a, p[e][st], o_acc[dt]);
      }
    read();
    stage(i + 1, true);
  }

  // ---- the waves' results ------------------------------------------------------
  // loads past the last tile are still on their way to LDS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  l = pair_sum(l);
  __syncthreads();
  f32x4* part = reinterpret_cast<f32x4*>(kv_lds);   // [waves][DT][4][64]
  if (h == 0) ml[wid][c32] = make_float2(m == -INFINITY ? m : m * c, l);
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 4; r++)
      part[((wid * DT + dt) * 4 + r) * 64 + lane] =
          f32x4{o_acc[dt][4 * r], o_acc[dt][4 * r + 1], o_acc[dt][4 * r + 2],
                o_acc[dt][4 * r + 3]};
  __syncthreads();
  if (!row_ok) return;
  float top = -INFINITY, sum = 0.0f, f[PS_WAVES];
  bool lost = false;                             // fmaxf skips a NaN
#pragma unroll
  for (int w = 0; w < PS_WAVES; w++) {
    const float2 z = ml[w][c32];
    top = fmaxf(top, z.x);
    lost |= z.x != z.x;
  }
  if (lost) top = NAN;
#pragma unroll
  for (int w = 0; w < PS_WAVES; w++) {
    const float2 z = ml[w][c32];
    // a wave without keys has no part in the row
    f[w] = w < n ? __builtin_amdgcn_exp2f(z.x - (top == -INFINITY ? 0.0f : top))
                 : 0.0f;
    if (w < n) sum += z.y * f[w];
  }
  if (MORE && x.sink != nullptr) sum += paged_sink(x, head, top);
  const float inv = sum != 0.0f ? 1.0f / sum : 0.0f;
  // a wave writes one (two) of every four pieces of its rows
  const long to = (long)(q_start + qi) * out_stride + (long)head * D + 4 * h;
#pragma unroll
  for (int i = 0; i < DT; i++) {
    const int piece = wid * DT + i, dt = piece >> 2, r = piece & 3;
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < PS_WAVES; w++)
      if (w < n) o += part[((w * DT + dt) * 4 + r) * 64 + lane] * f[w];
    paged_put<MORE>(x, out, to + dt * 32 + 8 * r, o[0] * inv, o[1] * inv,
                    o[2] * inv, o[3] * inv);
  }
}

// One turn of workgroups (at 128 wide LDS holds one per CU, at 64 two) over 128 to 2048
// keys, half of that for 64-wide heads, 768 with options, where a tile takes twice as
// long. More workgroups take a second turn for what fewer waves do over the same keys
// (us, paged_rows.h | here): 300 tokens of 32/8 heads (304 workgroups) 12.3 | 13.3, in a
// window 17.5 | 19.2, 8 prompts of 64-448 of 12/12 of 64 (764) 12.4 | 17.4, 594 behind up to
// 3000 keys (616) 50 | 68; but 2 x 600 behind 200 (456) 22.3 | 16.5; over up to 192
// keys 12 x 58-115 (504) 0.96 | 1.10 of the time of the kernel before, 20 x 17-49 behind 43-84
// (480) 0.97 | 1.17, but 8 x 27-231 0.99 | 0.85. In one or two tiles of keys
// there is nothing to share: 20 tokens 6.3 | 7.0, 64 of 64-wide heads 5.4 | 6.1. Longer
// tables go to more workgroups there: 32 tokens of 28/4 heads behind 1000 keys 18.5 | 15.9,
// 100 of 32/8 behind 1600 22.0 | 20.5, but 32 behind 3000 21.9 | 29.4; 16 of 64-wide heads
// behind 1000 11.9 | 12.0; 100 of 16/4 behind 1000, capped, 25.2 | 28.3, 30 of them in a window
// of 1024 20.1 | 21.9. From 1536 keys on, where there are three parts, only rows that fill
// a tile: 17 of 32/32 heads behind 1400 21.3 | 19.2, behind 1600 18.1 | 21.2, 60 of them
// 22.7 | 19.3, 19.8 | 21.3; 30 of 16/4 (120 rows) behind 1600 19.1 | 19.7, 45 behind 1930
// 21.8 | 21.7.
inline bool paged_short_takes(long tokens, int n_seqs, int G, int n_kv, int D,
                              long max_blocks, bool options) {
  const long keys = max_blocks * PF_BS;
  return paged_rows_tiles<PS_ROWS>(tokens, n_seqs, G) * n_kv <=
             (D == 64 ? keys >= 192 || options ? 512 : 400 : 256) &&
         keys >= 128 &&
         keys <= (options ? 768 : D == 64 ? PS_KEYS / 2 : PS_KEYS) &&
         (keys < 1536 || tokens * G >= (long)PF_ROWS * n_seqs);
}

template <int D, int TERMS, bool MORE>
inline void paged_short(void* out, const unsigned short* q,
                        const unsigned short* k_cache,
                        const unsigned short* v_cache, const int* block_tables,
                        const int* cu_q, const int* seq_lens, long tokens,
                        int n_seqs, float scale, int n_qheads, int n_kv,
                        int max_blocks, long q_stride, long out_stride,
                        const PagedMore& x, const PagedAhead& ahead,
                        hipStream_t stream) {
  const int G = n_qheads / n_kv;
  auto go = n_seqs == 1 ? paged_attn_short_kernel<D, TERMS, MORE, true>
                        : paged_attn_short_kernel<D, TERMS, MORE, false>;
  hipLaunchKernelGGL(
      go,
      dim3((unsigned)(paged_rows_tiles<PS_ROWS>(tokens, n_seqs, G) * n_kv +
                      ahead.wgs)),
      dim3(PS_WAVES * 64), 0, stream, block_tables, cu_q, seq_lens, n_seqs, G, n_kv,
      max_blocks, k_cache, q, v_cache, out, scale, q_stride, out_stride, x, ahead);
}

// How a batch of prompts is run: by this kernel, or by paged_rows.h. max_blocks: pages
// that a row sees
struct PagedPrompts : PagedRows {
  bool few = false;
};
inline PagedPrompts paged_prompts(long tokens, int n_seqs, int G, int n_kv, int D,
                                  long max_blocks, int terms, bool options) {
  PagedPrompts p;
  p.few = paged_short_takes(tokens, n_seqs, G, n_kv, D, max_blocks, options);
  if (!p.few)
    static_cast<PagedRows&>(p) =
        paged_rows_plan(tokens, n_seqs, G, n_kv, D, max_blocks, terms, options);
  return p;
}

}  // namespace xllm
