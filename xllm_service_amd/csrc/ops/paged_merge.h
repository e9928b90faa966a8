// What the paged attention kernels (paged_rows.h, paged_stream.h) share: their
// options, and the merge of keys that were split over workgroups.
#pragma once
#include <algorithm>
#include <atomic>
#include <climits>
#include <random>

#include "mfma_rows.h"

namespace xllm {

// Options of a call. A kernel instantiated without MORE ignores them: bf16
// results, every earlier key seen, scores scale * q.k.
struct PagedMore {
  int window = 0;         // > 0: a row sees the last `window` keys ...
  int keep_first = 0;     // ... and the first keep_first
  int chunked = 0;        // `window` is a chunk size: a row sees its own chunk
  int out_f32 = 0;        // results in fp32
  float cap = 0.0f;       // > 0: scores become cap * tanh(score / cap)
  const float* sink = nullptr;        // [heads]: e^sink joins the denominator
  const float* head_scale = nullptr;  // [heads]: one more score multiplier
};

// What later kernels read from memory, for the CUs that attention over a few rows leaves
// idle: workgroups past the last one's rows bring it into the cache in front of memory
// (256 MB), and the products that follow find their weights there: 300 x 4096 x 2048 12.9 ->
// 10.3 us, 3072 x 2048 11.3 -> 8.8, 4096 x 4096 21.6 -> 16.6. 8 layers, 300 rows of 2048
// 532 -> 490, 120 448 -> 392, 2 x 90 471 -> 427, 600 795 -> 745; of 4096, 300 1145 -> 1120,
// 90 774 -> 743, 150 826 -> 827. (Loads of the next weights among those of a product
// itself cost 30 us instead: they return in order, and each step waited for memory
// again. Decoded rows stream their weights at the rate of memory, and gained nothing.)
struct PagedAhead {
  static constexpr int N = 4;
  int from = INT_MAX;                 // the first that does so (a kernel that asks for the
  int wgs = 0;                        // size of its grid waits for it), how many do
  const unsigned short* at[N] = {};
  unsigned bytes[N] = {};
};
// by workgroup `mine` of them, through LDS that it does not look at: 1 KB a wave
XLLM_DEV void paged_fetch(const PagedAhead& a, int mine, unsigned short* lds) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned waves = blockDim.x >> 6, lane = threadIdx.x & 63;
  const unsigned step = a.wgs * waves * 1024u;
  for (int i = 0; i < PagedAhead::N; i++) {
    const auto src = mr_buffer(a.at[i], a.bytes[i]);
    for (unsigned at = (mine * waves + wave) * 1024u; at < a.bytes[i]; at += step)
      mr_to_lds(src, at + lane * 16, lds + wave * 512);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// What the CUs that `wgs` workgroups leave can fetch of N pieces while those run: a CU
// pulls 60 KB/us, memory 5 MB/us. Rows that see few keys are done sooner. Us a layer,
// nothing fetched | 300 | 450 KB a CU: 40 rows of 4096 71.8 | 69.8 | 70.2, 200 (keys) 107.8
// | 106.9 | 109.0, 300 137.2 | 134.9 | 134.7; of 2048 100 49.6 | 47.1 | 47.0, 300 61.5 | 58.9 |
// 56.8, 600 93.8 | 89.8 | 89.5. 60 and 120 KB gain nothing: the first product reads most of
// its weights from memory all the same.
//   streamed: what decoded rows of the same step read of their caches before the first
// weight is used, through the same cache in front of memory. Us a layer, nothing | 300 KB a
// CU beside rows of 600-1400 keys, MB of their pages: 100 rows of 2048 and 16 (46 MB) 64.4 |
// 59.4, 64 (180) 79.7 | 77.6, 96 (270) 95.3 | 97.6, 128 106.5 | 108.9; of 4096 16 (90) 110.9 |
// 106.5, 32 (180) 127.9 | 124.1, 48 (270) 143 | 144, 64 154.8 | 158.1; 300 rows, which fetch
// 48 MB, and 16 157.1 | 154.9, 32 174.2 | 176.6.
inline PagedAhead paged_ahead(long wgs, long keys, const void* const* at,
                              const long* bytes, long streamed) {
  PagedAhead a;
  if (at == nullptr || wgs > 256 - 32) return a;
  const long cus = 256 - wgs;
  const long most =
      std::min<long>(48 << 20, cus * ((keys <= 256 ? 300L : 450L) << 10));
  if (most + streamed > 224L << 20) return a;
  a.from = (int)wgs;
  a.wgs = (int)cus;
  long room = most;
  for (int i = 0; i < PagedAhead::N; i++) {
    const long n = std::min(bytes[i], room) / 1024 * 1024;
    if (n <= 0) continue;
    a.at[i] = static_cast<const unsigned short*>(at[i]);
    a.bytes[i] = (unsigned)n;
    room -= n;
  }
  return a;
}

// first key that a row which sees keys below `limit` has in its window
template <bool MORE>
XLLM_DEV int paged_first(const PagedMore& x, int limit) {
  if (!MORE || x.window <= 0) return 0;
  return x.chunked ? (limit - 1) / x.window * x.window
                   : max(0, limit - x.window);
}

// The tiles a workgroup walks: those that hold kept keys, then from the first
// one that its earliest row (which sees keys below `limit`) sees.
struct PagedTiles {
  int keep, gap, n;       // at(i): i below keep as it is, else + gap
  XLLM_DEV int at(int i) const { return i < keep ? i : i + gap; }
};
template <bool MORE>
XLLM_DEV PagedTiles paged_tiles(const PagedMore& x, int limit, int kmax,
                                int n_tiles, int kt) {
  if (!MORE || x.window <= 0) return {0, 0, n_tiles};
  const int first = paged_first<MORE>(x, limit) / kt;
  const int keep = min((min(x.keep_first, kmax) + kt - 1) / kt, first);
  return {keep, first - keep, n_tiles - (first - keep)};
}

// |scale| log2(e), above zero; a NaN stays one
XLLM_DEV float paged_factor(float scale) {
  const float c = fabsf(scale) * 1.4426950408889634f;
  return c < 1e-30f ? 1e-30f : c;
}

// How a row's scores become weights 2^(c (s - m)): a negative factor turns the
// signs of the query's entries, so that c is positive; with a cap, s is the
// capped score and pre goes in front of the tanh.
struct PagedScore { short flip; float c, pre; };
template <bool MORE>
XLLM_DEV PagedScore paged_score(const PagedMore& x, float scale, int head) {
  constexpr float log2e = 1.4426950408889634f;
  if (MORE && x.head_scale != nullptr) scale *= x.head_scale[head];
  if (MORE && x.cap > 0.0f) return {0, log2e, scale / x.cap};
  return {scale < 0.0f ? (short)0x8000 : (short)0,
          paged_factor(scale), 0.0f};
}

// s <- cap * tanh(pre * s). Tiles without large scores, nearly all of them, skip
// the exponentials and divisions.
template <int N>
XLLM_DEV void paged_cap(f32x16 (&s)[N], float pre, float cap) {
  float big = 0.0f;
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      s[i][r] *= pre;
      big = fmaxf(big, fabsf(s[i][r]));
    }
  const bool far = __any(!(big < 0.5f));
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float v = s[i][r];
      float y = tanh_near(v);
      if (far) {
        const float z = tanh_far(v);
        y = fabsf(v) < 0.5f ? y : z;
      }
      s[i][r] = cap * y;
    }
}

// Scores of keys that a row does not see are -inf: those from `limit` on and those below
// lo but for the first keep_first. key(r): of entry r. Without kept keys that is one
// comparison; written with || the compiler branched around each of the entries.
template <bool MORE, int N, class Key>
XLLM_DEV void paged_mask(const PagedMore& x, f32x16 (&s)[N], int limit, int lo,
                         const Key& key) {
  if (!MORE || x.keep_first <= 0) {
    const unsigned span = (unsigned)max(limit - (MORE ? lo : 0), 0);
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const unsigned at = (unsigned)(key(i, r) - (MORE ? lo : 0));
        s[i][r] = at < span ? s[i][r] : -INFINITY;
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int k = key(i, r);
      const bool on = (k < limit) & ((k >= lo) | (k < x.keep_first));
      s[i][r] = on ? s[i][r] : -INFINITY;
    }
}

// Decoded rows: parts that a list of n tiles is really split into, of the P that
// the host, which does not know the lengths, made room for: one for every `per` tiles,
// of up to eight one for every `near`
__host__ __device__ inline int paged_parts(int n, int P, int per) {
  const int p = (n + per - 1) / per;
  return p < 1 ? 1 : p > P ? P : p;
}
struct PagedSplit {
  int parts = 1, per = 1;
  int near = 1 << 20;        // tiles
  int least = 0;             // tiles of the shortest list that is split
  int waves = 4;             // of a workgroup
  __host__ __device__ int of(int n) const {
    const int far = paged_parts(n, parts, per);
    const int most = paged_parts(n, parts < 8 ? parts : 8, near);
    if (n < least) return 1;
    return far > most ? far : most;
  }
};

// What the sink of a head adds to the sum of a row whose maximum is `top` (with the
// factor of its scores). Rows without keys have no maximum, and a sink of -inf has no
// weight for them either.
XLLM_DEV float paged_sink(const PagedMore& x, int head, float top) {
  return __builtin_amdgcn_exp2f(x.sink[head] * 1.4426950408889634f -
                                (top == -INFINITY ? 0.0f : top));
}

// four neighbouring results
template <bool MORE>
XLLM_DEV void paged_put(const PagedMore& x, void* out, long at, float a,
                        float b, float c, float d) {
  if (MORE && x.out_f32) {
    *reinterpret_cast<float4*>((float*)out + at) = make_float4(a, b, c, d);
  } else {
    uint2 y;
    y.x = pack_bf16(a, b);
    y.y = pack_bf16(c, d);
    *reinterpret_cast<uint2*>((unsigned short*)out + at) = y;
  }
}

#define PAGED_ABSENT (-1.0f)

// Parts of a row, B at a time, added to (M, L, a): their maxima, sums and results
// are all on the way at once, the first maximum is not waited for before the first
// result is fetched. A merge is a chain of this and, in a kernel of its own, a launch:
// 32 rows x 16 heads, up to four parts 4.67 -> 4.07 us, 17 k rows of three parts 6.55 ->
// 5.95; by eights where there is room for more than four.
// ml(p), o(p): maximum and sum, and four results of part p. A part without
// keys has written no results and the sum PAGED_ABSENT: any other sum, NaN
// among them, counts.
template <int B, class Ml, class O>
XLLM_DEV void paged_add_parts(const Ml& ml, const O& o, int parts, float& M,
                              float& L, float (&a)[4]) {
  for (int p0 = 0; p0 < parts; p0 += B) {
    float2 z[B];
    float4 y[B];
#pragma unroll
    for (int k = 0; k < B; k++) {
      const int p = min(p0 + k, parts - 1);
      z[k] = ml(p);
      y[k] = o(p);
    }
    float top = M;
#pragma unroll
    for (int k = 0; k < B; k++) {
      if (p0 + k >= parts) z[k].y = PAGED_ABSENT;
      top = fmaxf(top, z[k].x);
    }
    if (top == -INFINITY) top = 0.0f;
    const float keep = __builtin_amdgcn_exp2f(M - top);
    M = top;
    L *= keep;
#pragma unroll
    for (int c = 0; c < 4; c++) a[c] *= keep;
#pragma unroll
    for (int k = 0; k < B; k++) {
      const bool on = !(z[k].y < 0.0f);
      const float w = on ? __builtin_amdgcn_exp2f(z[k].x - M) : 0.0f;
      L += on ? z[k].y * w : 0.0f;
      a[0] += on ? y[k].x * w : 0.0f; a[1] += on ? y[k].y * w : 0.0f;
      a[2] += on ? y[k].z * w : 0.0f; a[3] += on ? y[k].w * w : 0.0f;
    }
  }
}

// ---- the last of a unit's workgroups merges ------------------------------------
// A unit is what is split into parts. Its workgroups count themselves when their parts
// are in memory, and the one that finds all others counted merges: no second launch,
// which cost 4 to 5 us of which two thirds were its start and the end of the kernel
// before it.
//   The counters are scratch like the parts, which nobody has cleared: a launch for that
// would cost what the merge's did, and counters kept from call to call would have to
// know of streams, threads and captured graphs. Instead each call has a tag of 56 random
// bits, and whoever finds another value in a counter than its call's tag and a count
// puts the tag and no count there: before its own part is counted, and only if the
// counter still holds what it found. The last one sets it back, so a captured call finds
// no count of its last replay. What lay there before would have to agree in 56 random
// bits to pass for a count.
//   Parts and counts pass between XCDs, whose L2s do not see each other's lines: parts
// are stored and loaded past them (mr_store_far), a workgroup counts itself when all of
// its waves have waited for their stores, counts are atomics at device scope.
struct PagedMeet {
  unsigned long long* count = nullptr;   // [units]
  unsigned long long tag = 0;            // low 8 bits: none
};
typedef unsigned long long u64;
// by one thread of a workgroup, before it counts its part: at, its unit's counter
XLLM_DEV void paged_open(u64* at, u64 seen, u64 tag) {
  if (((seen ^ tag) >> 8) != 0)
    __hip_atomic_compare_exchange_strong(at, &seen, tag, __ATOMIC_RELAXED,
                                         __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
}
XLLM_DEV u64 paged_seen(u64* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// by all of its threads, with their stores behind them: whether it is the last of `parts`.
// last: LDS that nothing else is in
XLLM_DEV bool paged_last(u64* at, int parts, int* last) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const u64 old = __hip_atomic_fetch_add(at, 1ull, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    const bool all = (int)(old & 255) == parts - 1;
    *last = all;
    if (all)
      __hip_atomic_store(at, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return *last != 0;
}
// A call's counters, behind its parts: scratch is rows * parts * (D + 2) + 2 * units floats
inline PagedMeet paged_meet(float* ws_ml, long rows, int parts) {
  static std::atomic<u64> calls{[] {
    std::random_device r;
    return (u64)r() << 32 | r();
  }()};
  u64 z = calls.fetch_add(0x9e3779b97f4a7c15ull, std::memory_order_relaxed);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;   // splitmix64 (Steele et al. 2014)
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return {reinterpret_cast<u64*>(ws_ml + 2 * rows * parts), (z ^ (z >> 31)) << 8};
}

// Tiles of kt keys that a prompt of `keys` of them walks at most
template <bool MORE>
XLLM_DEV int paged_walk(const PagedMore& x, int keys, int kt) {
  const int n = (max(keys, 0) + kt - 1) / kt;
  return MORE && x.window > 0 ? min(n, (x.window + x.keep_first) / kt + 3) : n;
}
// Equal parts of a single prompt's rows, of at least four tiles
template <bool MORE>
XLLM_DEV int paged_equal(const PagedMore& x, int keys, int kt, int most) {
  return max(min((paged_walk<MORE>(x, keys, kt) + 3) / 4, most), 1);
}

// out[row] = sum_p o[row][p] 2^(m_p - M) / sum_p l_p 2^(m_p - M): D/4 lanes per
// row, four columns each. Rows are those of n_seqs prompts; tokens outside of all of
// them have no parts and stay as they are, rows with one part are there. ws_at: slot of
// a row's first part, parts; the others follow it. Of a single prompt (ONE) they are
// counted, the same for all: fetched, and with divisions of 64 bits, a merge of 16 parts
// took 5.0 us, 4.1 so (before there were places to look up 3.9). ROWS: of a row tile; rows
// are those of a few turns of the CUs.
template <int D, bool MORE, int ROWS, int KT, bool ONE>
__global__ __launch_bounds__(256) void paged_attn_merge_kernel(
    void* __restrict__ out, const float* __restrict__ ws_o,
    const float* __restrict__ ws_ml, const int2* __restrict__ ws_at,
    const int n_qheads, const int G, const long out_stride, const unsigned rows,
    const PagedMore x, const int* __restrict__ cu_q,
    const int* __restrict__ seq_lens, const int n_seqs, const int n_kv,
    const int most) {
  constexpr int LPR = D / 4;
  const unsigned row = (blockIdx.x * 256u + threadIdx.x) / LPR;
  const int col = (threadIdx.x % LPR) * 4;
  if (row >= rows) return;
  // all of it at once: what one wait is for does not wait for another
  const int q0 = cu_q[0], q1 = cu_q[n_seqs], keys = seq_lens[0];
  const int tok = row / n_qheads, head = row - tok * n_qheads;
  int slot, parts;
  if (ONE) {                                     // units: the last row tile's come first
    const int nt = ((q1 - q0) * G + ROWS - 1) / ROWS;
    const int kvh = head / G, rho = (tok - q0) * G + head - kvh * G;
    parts = paged_equal<MORE>(x, keys, KT, most);
    slot = (((nt - 1 - rho / ROWS) * n_kv + kvh) * ROWS + rho % ROWS) * parts;
  } else {
    const int2 at = ws_at[row];
    slot = at.x;
    parts = at.y;
  }
  if (tok < q0 || tok >= q1 || parts <= 1) return;
  const bool sink = MORE && x.sink != nullptr;
  float M = sink ? x.sink[head] * 1.4426950408889634f : -INFINITY;
  float L = sink ? 1.0f : 0.0f;
  float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const float2* ml = reinterpret_cast<const float2*>(ws_ml) + slot;
  const float* o = ws_o + (long)slot * D + col;
  auto ml_of = [&](int p) { return ml[p]; };
  auto o_of = [&](int p) {
    return *reinterpret_cast<const float4*>(o + p * D);
  };
  if (parts <= 4) paged_add_parts<4>(ml_of, o_of, parts, M, L, a);
  else paged_add_parts<8>(ml_of, o_of, parts, M, L, a);
  const float inv = L != 0.0f ? 1.0f / L : 0.0f;
  paged_put<MORE>(x, out, (long)tok * out_stride + (long)head * D + col, a[0] * inv,
                  a[1] * inv, a[2] * inv, a[3] * inv);
}

template <int D, bool MORE, int ROWS, int KT>
inline void paged_merge(void* out, const float* ws_o, const float* ws_ml,
                        const int2* ws_at, int n_qheads,
                        long out_stride, long rows, const PagedMore& x,
                        hipStream_t stream, const int* cu_q, const int* seq_lens,
                        int n_seqs, int n_kv, int most) {
  auto go = n_seqs == 1 ? paged_attn_merge_kernel<D, MORE, ROWS, KT, true>
                        : paged_attn_merge_kernel<D, MORE, ROWS, KT, false>;
  hipLaunchKernelGGL(go, dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0,
                     stream, out, ws_o, ws_ml, ws_at, n_qheads, n_qheads / n_kv,
                     out_stride, (unsigned)rows, x, cu_q, seq_lens, n_seqs, n_kv, most);
}

}  // namespace xllm
