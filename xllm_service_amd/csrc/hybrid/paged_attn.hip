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

// Whether the kernels of capped_attn_mfma.hip are faster: they have 16 rows a wave and 32
// keys a tile, so that one tile is done in half the time, but move four times as much
// through LDS, do not split the keys of prompts and look for a row tile's sequence one by
// one. They are where one tile holds all keys. Time there over that here, 1270 drawn calls:
//   Prompts, by the keys from the first to the last one of a row tile and by the workgroups
// here: up to 32 keys 0.91 (up to 99 workgroups), 1.07 (255), capped 0.85, 0.96; 33 to 48 1.06,
// 1.17, capped 0.97, 1.08; then 1.16 to 2.4. (A fit to calls of both before few rows' keys
// were shared by waves sent 179 of 600 there, of which 77 took over 5% longer.)
//   Decode, 128 wide, by the keys a row sees: tables of up to 32 keys 0.97, 0.87 (9 to 16
// heads a key head), 0.72 (more); windows as small in longer ones lie in two tiles, 1.31, 1.17,
// 0.96; 33 to 64 keys 1.27, 1.19, 0.97; 65 to 128 1.89, 1.78, 1.50; more 1.6, 1.3, and 0.90 for
// up to eight pairs of sequence and key head (their merge of waves' results is longest
// here), 1.36 for many. 64 wide 1.1 to 2.2.
bool paged_attn_small(bool decode, long tokens, int n_seqs, int heads, int n_kv,
                      int D, long max_blocks, int window, int keep_first,
                      bool capped) {
  const long keys = max_blocks * 16, G = heads / n_kv;
  if (keys == 0) return true;          // tables without columns: not read there
  if (decode) {
    const long walk = window > 0 ? std::min<long>(keys, window) : keys;
    const long pairs = (long)n_seqs * n_kv;
    return D == 128 &&
           (keys <= 32 || (G > 16 && (walk <= 64 || (pairs <= 8 && walk > 128 &&
                                                     walk <= 4096))));
  }
  const long span = std::max<long>(1, std::min<long>(tokens, 64 / G));
  const long walk = window > 0 ? std::min<long>(keys, window + span + keep_first)
                               : keys;
  const long wgs = (tokens * G / 128 + n_seqs) * n_kv;
  return capped ? wgs < 256 && walk <= (D == 128 && wgs < 100 ? 63 : 32)
                : wgs < 100 && walk <= 32;
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
