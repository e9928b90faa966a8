// Soft-capped, windowed and sink attention in bf16 over 16-token pages, key and
// value width 64 or 128: the kernels of the dense decoders (../ops/paged_rows.h,
// ../ops/paged_stream.h) with their options, the softmax weights in 32 bits.
// Other widths and pages: capped_attn_mfma.hip.
#include "../ops/paged_short.h"
#include "../ops/paged_stream.h"

namespace xllm {
namespace hyb {

static PagedMore more_of(bool out_f32, float cap, int window, const float* sink,
                         int keep_first, const float* head_scale,
                         bool chunked) {
  PagedMore x;
  x.out_f32 = out_f32; x.cap = cap; x.window = window; x.sink = sink;
  x.keep_first = keep_first; x.head_scale = head_scale; x.chunked = chunked;
  return x;
}

// pages that a window lets a row see
static long seen_pages(long max_blocks, int window, int keep_first) {
  return window <= 0 ? max_blocks
      : std::min<long>(max_blocks,
                       (window + 15) / 16 + (keep_first + 15) / 16 + 2);
}

// Floats of scratch that a call asks for. cu_q null: decoded rows.
long paged_attn_scratch(bool decode, long tokens, int n_seqs, int heads, int n_kv,
                        int D, long max_blocks, int window, int keep_first,
                        bool capped) {
  if (tokens == 0 || n_seqs <= 0) return 0;
  max_blocks = seen_pages(max_blocks, window, keep_first);
  if (!decode)
    return paged_prompts(tokens, n_seqs, heads / n_kv, n_kv, D, max_blocks, 3,
                         true).scratch;
  const int parts =
      paged_stream_split(n_seqs, n_kv, max_blocks, true, capped).parts;
  return parts > 1 ? tokens * heads * parts * (D + 2) + 2L * n_seqs * n_kv : 0;
}

// Whether the kernels of capped_attn_mfma.hip are faster: they have 16 rows a wave
// and 32 keys a tile, so that one tile is done in half the time, but move four times
// as much through LDS, do not split the keys of prompts and look for a row tile's
// sequence one by one.
//   Decode, by the keys a row sees, us there | here: 16 or 32 5.6 | 6.3 (4 query heads
// a key head), 5.7 | 7.5 (16), 6.0 | 9.0 (32); 64 7.4 | 5.8, 7.2 | 6.8, 7.8 | 8.6; 300
// 11.4 | 8.5. The merge of the waves' results grows with the heads: above 16 a key
// head, for 2 pairs, 300 keys in tables of 4096 9.7 | 11.1, windows of 512 11.1 |
// 12.9 (16 heads 10.6 | 11.3), for 16 pairs 21.6 | 13.6.
//   Prompts, by the keys from the first to the last one of a row tile and by the
// number of row tiles: window 16, 64-wide heads, 256 tokens 7.2 | 9.9, 64 sequences of
// 128 56 | 39; window 512, 256 tokens 36 | 19; 128-wide, window 16 9.2 | 12.7, 64 of one
// head 16.8 | 17.8, 128 26 | 19, window 16 over 260 x 4 row tiles 24.6 | 22.1. In between
// a fit to 1370 timed calls of each kind decides, of which 70 to 130 take over 5 %
// longer than by the other kernels, one a third.
bool paged_attn_small(bool decode, long tokens, int n_seqs, int heads, int n_kv,
                      int D, long max_blocks, int window, int keep_first,
                      bool capped) {
  const long keys = max_blocks * 16, G = heads / n_kv;
  if (decode) {
    const long walk = window > 0 ? std::min<long>(keys, window) : keys;
    const long pairs = (long)n_seqs * n_kv;
    return walk <= 32 || (G > 16 && (walk <= 64 || (pairs <= 8 && walk <= 4096))) ||
           (G > 8 && pairs <= 16 && window > 256 && walk <= 1024);
  }
  // us: a + b * tiles of a walk, more where row tiles wait for others
  struct Fit { double a, b, wgs; };
  static const Fit there[2][2] = {{{4.8, 1.56, 350}, {5.1, 1.85, 340}},
                                  {{5.7, 2.45, 300}, {5.9, 2.73, 300}}};
  static const Fit here[2][2] = {{{7.1, 1.50, 190}, {8.1, 2.41, 240}},
                                 {{8.6, 2.10, 150}, {9.6, 3.01, 180}}};
  auto walk = [&](long rows) {
    const long span = std::max<long>(1, std::min<long>(tokens, rows / G));
    return (double)(window > 0 ? std::min<long>(keys, window + span + keep_first)
                               : keys);
  };
  auto time = [&](const Fit& f, int rows, int tile) {
    const double wgs = ((double)tokens * G / rows + n_seqs) * n_kv;
    return f.a + f.b * walk(rows) / tile * std::max(1.0, wgs / f.wgs);
  };
  return walk(64) <= 400 &&
         time(there[D == 128][capped], 64, 32) + 0.15 * n_seqs <
             time(here[D == 128][capped], 128, 64);
}

// out [tokens, heads * D] rows of out_stride, fp32 or bf16; q rows, caches and
// out 16 B aligned (a bf16 out 8 B); decode: at most 32 heads per key head
void launch_paged_attn(void* out, long out_stride, bool out_f32, float* ws,
                       const unsigned short* q,
                       const unsigned short* k_cache,
                       const unsigned short* v_cache, const int* block_tables,
                       const int* cu_q, const int* seq_lens, long tokens,
                       int n_seqs, int heads, int n_kv, int D, int max_blocks,
                       float scale, float cap, long q_stride, int window, const float* sink, int keep_first,
                       const float* head_scale, bool chunked, hipStream_t st) {
  const PagedMore x =
      more_of(out_f32, cap, window, sink, keep_first, head_scale, chunked);
  if (tokens == 0 || n_seqs <= 0) return;
  const long seen = seen_pages(max_blocks, window, keep_first);
  if (cu_q == nullptr) {
    auto go = D == 128 ? paged_stream<128, 3, true> : paged_stream<64, 3, true>;
    const PagedSplit split = paged_stream_split(n_seqs, n_kv, seen, true, cap > 0);
    go(out, ws, ws + tokens * heads * split.parts * D, q, k_cache, v_cache,
       block_tables, seq_lens, n_seqs, scale, heads, n_kv, max_blocks, q_stride,
       out_stride, split, x, st);
    return;
  }
  const PagedPrompts p =
      paged_prompts(tokens, n_seqs, heads / n_kv, n_kv, D, seen, 3, true);
  if (p.few) {
    auto go = D == 128 ? paged_short<128, 3, true> : paged_short<64, 3, true>;
    go(out, q, k_cache, v_cache, block_tables, cu_q, seq_lens, tokens, n_seqs,
       scale, heads, n_kv, max_blocks, q_stride, out_stride, x, PagedAhead{}, st);
    return;
  }
  auto go = D == 128 ? paged_rows<128, 3, true> : paged_rows<64, 3, true>;
  go(out, ws, q, k_cache, v_cache, block_tables, cu_q, seq_lens, tokens, n_seqs,
     scale, heads, n_kv, max_blocks, q_stride, out_stride, p, x,
     PagedAhead{}, st);
}

}  // namespace hyb
}  // namespace xllm
