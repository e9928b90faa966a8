// Soft-capped, windowed and sink attention in bf16 over 16-token pages, key and
// value width 64 or 128: the kernels of the dense decoders (../ops/paged_rows.h,
// ../ops/paged_stream.h) with their options, the softmax weights in 32 bits.
// Other widths and pages: capped_attn_mfma.hip.
#include "../ops/paged_rows.h"
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

// Room for parts the keys are split into. cu_q null: decoded rows.
int paged_attn_parts(bool decode, long tokens, int n_seqs, int heads, int n_kv,
                     long max_blocks, int window, int keep_first, bool capped) {
  max_blocks = seen_pages(max_blocks, window, keep_first);
  return decode ? paged_stream_split(n_seqs, n_kv, max_blocks, capped).parts
                : paged_rows_parts(tokens, n_seqs, heads / n_kv, n_kv,
                                   max_blocks, 3);
}

// out [tokens, heads * D] rows of out_stride, fp32 or bf16; q rows, caches and
// out 16 B aligned (a bf16 out 8 B); decode: at most 32 heads per key head
void launch_paged_attn(void* out, long out_stride, bool out_f32, float* ws_o,
                       float* ws_ml, const unsigned short* q,
                       const unsigned short* k_cache,
                       const unsigned short* v_cache, const int* block_tables,
                       const int* cu_q, const int* seq_lens, long tokens,
                       int n_seqs, int heads, int n_kv, int D, int max_blocks,
                       float scale, float cap, long q_stride, int n_part,
                       int window, const float* sink, int keep_first,
                       const float* head_scale, bool chunked, hipStream_t st) {
  const PagedMore x =
      more_of(out_f32, cap, window, sink, keep_first, head_scale, chunked);
  if (cu_q == nullptr) {
    auto go = D == 128 ? paged_stream<128, 3, true> : paged_stream<64, 3, true>;
    go(out, ws_o, ws_ml, q, k_cache, v_cache, block_tables, seq_lens, n_seqs,
       scale, heads, n_kv, max_blocks, q_stride, out_stride,
       paged_stream_split(n_seqs, n_kv,
                          seen_pages(max_blocks, window, keep_first), cap > 0),
       x, st);
  } else {
    auto go = D == 128 ? paged_rows<128, 3, true> : paged_rows<64, 3, true>;
    go(out, ws_o, ws_ml, q, k_cache, v_cache, block_tables, cu_q, seq_lens,
       tokens, n_seqs, scale, heads, n_kv, max_blocks, q_stride, out_stride,
       n_part, x, st);
  }
}

}  // namespace hyb
}  // namespace xllm
