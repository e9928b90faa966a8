// Paged attention of decoded rows for the dense decoders: bf16 in and out (64-
// and 128-wide heads: paged_stream.h, with its reasons).
//
// Parity: reference engine's paged-attention decode.
#include "paged_stream.h"

namespace xllm {

// ---------------- other head widths: shuffle-reduce design -------------------
// (and 64- and 128-wide heads at addresses that are not multiples of 16 B, which
// loads straight to LDS ask for)
XLLM_DEV ushort8_t pa_eight(const unsigned short* p) {   // any alignment
  ushort8_t v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
template <int G>
__global__ __launch_bounds__(256) void paged_attn_decode_small_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ q,
    const unsigned short* __restrict__ k_cache,
    const unsigned short* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ seq_lens,
    const float scale, const int n_kv_heads, const int D,
    const int max_blocks_per_seq, const long q_stride, const long out_stride) {
  const int seq = blockIdx.x / n_kv_heads;
  const int kvh = blockIdx.x % n_kv_heads;
  const int n_qheads = n_kv_heads * G;
  const int seq_len = seq_lens[seq];
  const int n_blocks = (seq_len + PA_BS - 1) / PA_BS;
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int tg = lane >> 4;
  const int d8 = lane & 15;
  const int dvalid = (8 * d8) < D;

  float qf[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const long qoff = (long)seq * q_stride + (long)(kvh * G + g) * D + 8 * d8;
    if (dvalid) {
      ushort8_t v = pa_eight(q + qoff);
#pragma unroll
      for (int j = 0; j < 8; j++) qf[g][j] = bf16_to_f32(v.x[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) qf[g][j] = 0.0f;
    }
  }
  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    m[g] = -INFINITY; l[g] = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) acc[g][j] = 0.0f;
  }
  const int* btab = block_tables + (long)seq * max_blocks_per_seq;
  const long head_stride = (long)PA_BS * D;
  for (int bi = wid; bi < n_blocks; bi += 4) {
    const long base = ((long)btab[bi] * n_kv_heads + kvh) * head_stride;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int t = j * 4 + tg;
      const int tok = bi * PA_BS + t;
      if (tok >= seq_len) continue;
      const long roff = base + (long)t * D + 8 * d8;
      float kf[8], vf[8];
      if (dvalid) {
        ushort8_t k8 = pa_eight(k_cache + roff);
        ushort8_t v8 = pa_eight(v_cache + roff);
#pragma unroll
        for (int u = 0; u < 8; u++) { kf[u] = bf16_to_f32(k8.x[u]); vf[u] = bf16_to_f32(v8.x[u]); }
      } else {
#pragma unroll
        for (int u = 0; u < 8; u++) { kf[u] = 0.0f; vf[u] = 0.0f; }
      }
#pragma unroll
      for (int g = 0; g < G; g++) {
        float s = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) s += qf[g][u] * kf[u];
        s = group_reduce_sum<16>(s) * scale;
        const float m_new = fmaxf(m[g], s);
        const float a = __expf(m[g] - m_new);
        const float p = __expf(s - m_new);
        m[g] = m_new;
        l[g] = l[g] * a + p;
#pragma unroll
        for (int u = 0; u < 8; u++) acc[g][u] = acc[g][u] * a + p * vf[u];
      }
    }
  }
  __shared__ float ml[16][G][2];
  __shared__ float accs[16][G][16][8];
  const int part = wid * 4 + tg;
  if (d8 == 0) {
#pragma unroll
    for (int g = 0; g < G; g++) { ml[part][g][0] = m[g]; ml[part][g][1] = l[g]; }
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
#pragma unroll
    for (int u = 0; u < 8; u++) accs[part][g][d8][u] = acc[g][u];
  }
  __syncthreads();
  for (int g = wid; g < G; g += 4) {
    float m_star = -INFINITY;
#pragma unroll
    for (int p = 0; p < 16; p++) m_star = fmaxf(m_star, ml[p][g][0]);
    float l_tot = 0.0f, o0 = 0.0f, o1 = 0.0f;
    const int pd8 = lane >> 2;
    const int pu = (2 * lane) & 7;
#pragma unroll
    for (int p = 0; p < 16; p++) {
      const float mw = ml[p][g][0];
      const float w = (mw == -INFINITY) ? 0.0f : __expf(mw - m_star);
      l_tot += w * ml[p][g][1];
      o0 += w * accs[p][g][pd8][pu];
      o1 += w * accs[p][g][pd8][pu + 1];
    }
    const float inv = (l_tot > 0.0f) ? 1.0f / l_tot : 0.0f;
    if (2 * lane < D) {
      const long ooff = (long)seq * out_stride + (long)(kvh * G + g) * D + 2 * lane;
      out[ooff] = f32_to_bf16(o0 * inv);
      out[ooff + 1] = f32_to_bf16(o1 * inv);
    }
  }
}

// 64-wide heads had one workgroup per pair and no merge before they were streamed
// (by the shuffle kernel above), so the split of the 128-wide ones does not pay
// for many pairs: 128 sequences of 12 heads, 64 keys each in tables of 8192,
// shuffle 7.9 | split 17.1 | whole 9.2 us, 500 keys 35 | 38.5 | 32. From 768 pairs on
// workgroups of two waves, twice as many at a time: 64 keys 9.2 -> 6.8, 16 8.0 -> 5.9
// (384 pairs of 500 keys 11.8 -> 15.7, so not there).
//   Few pairs: as for 128-wide heads. 86 to 192, whole | by 16 tiles, at most four: 8
// sequences of 12 heads, 1000 keys 13.1 | 11.1, 2000 22.1 | 15.5, 0.1-2 k 17.6 | 10.3, but 600
// 8.9 | 9.1; 16 of 2000 25.6 | 24.2, 0.1-2 k 19.8 | 18.0, but 1300 19.1 | 19.9; 21 of 2000 27.5 |
// 31.4.
//   128-wide heads: two waves only where tables have few tiles, of which four leave
// waves idle that hold LDS (32 key heads, 32 x 16 keys 10.1 -> 8.4). In wide tables long
// sequences may be there, which two waves walk more slowly (30 x 0.1-3.6 k, 32 key heads
// 113 -> 123; 69 x 7.0-7.8 k, 8 key heads 311 -> 336); 16 keys in tables of 4096 stay
// at 10.3.
static PagedSplit decode_split(long num_seqs, int n_kv_heads, int D,
                               long max_blocks) {
  const long units = num_seqs * n_kv_heads;
  PagedSplit x;
  if (D == 64 && units >= 86) {
    if (units >= 768) x.waves = 2;
    if (units > 192) return x;
    x.per = 16;
    x.least = units <= 128 ? 24 : 48;
    x.parts = (int)std::min<long>(4, std::max<long>(1, (max_blocks + 31) / 32));
    return x;
  }
  x = paged_stream_split(num_seqs, n_kv_heads, max_blocks);
  if (max_blocks <= 2 || (units >= 768 && max_blocks <= 16)) x.waves = 2;
  return x;
}
// Tables of a page or of a few, one or two query heads per key head: the shuffle
// kernel, whose chain is shorter. One page, 12 heads x 16 sequences 3.4-4.5 | 4.3 us,
// x 128 3.9-5.2 | 5.9; four pages, x 32 4.8 | 5.2.
static bool decode_tiny(long units, int G, int D, long max_blocks) {
  return D == 64 && G <= 2 &&
         (max_blocks <= 1 || (max_blocks <= 4 && units >= 300 && units < 768));
}
int paged_attn_decode_parts(int num_seqs, int n_kv_heads, int D,
                            int max_blocks) {
  return decode_split(num_seqs, n_kv_heads, D, max_blocks).parts;
}

// streamed: rows of q and the caches on 16 B, of out on 8 B, and heads 64 or 128
// wide; ws_o, ws_ml: room for paged_attn_decode_parts() results per row
void launch_paged_attn_decode(unsigned short* out, const unsigned short* q,
                              const unsigned short* k_cache,
                              const unsigned short* v_cache,
                              const int* block_tables, const int* seq_lens,
                              float* ws_ml, float* ws_o, float scale,
                              int num_seqs, int n_qheads, int n_kv_heads, int D,
                              int max_blocks_per_seq, long q_stride,
                              long out_stride, bool streamed,
                              hipStream_t stream) {
  const int G = n_qheads / n_kv_heads;
  if (num_seqs == 0) return;
  if (!streamed ||
      decode_tiny((long)num_seqs * n_kv_heads, G, D, max_blocks_per_seq)) {
    const dim3 grid(num_seqs * n_kv_heads), block(256);
#define PA_SMALL(GV)                                                           \
  hipLaunchKernelGGL((paged_attn_decode_small_kernel<GV>), grid, block, 0,     \
                     stream, out, q, k_cache, v_cache, block_tables, seq_lens, \
                     scale, n_kv_heads, D, max_blocks_per_seq, q_stride,       \
                     out_stride)
    switch (G) {
      case 1: PA_SMALL(1); break;
      case 2: PA_SMALL(2); break;
      case 3: PA_SMALL(3); break;
      case 4: PA_SMALL(4); break;
      case 5: PA_SMALL(5); break;
      case 6: PA_SMALL(6); break;
      case 7: PA_SMALL(7); break;
      case 8: PA_SMALL(8); break;
      default: break;  // validated host-side
    }
#undef PA_SMALL
    return;
  }
  // 64-wide heads have 32-bit weights, as every other width but 128, whose
  // weights have 16 (G is at most 8)
  auto go = D == 128 ? paged_stream<128, 2, false> : paged_stream<64, 3, false>;
  go(out, ws_o, ws_ml, q, k_cache, v_cache, block_tables, seq_lens, num_seqs,
     scale, n_qheads, n_kv_heads, max_blocks_per_seq, q_stride, out_stride,
     decode_split(num_seqs, n_kv_heads, D, max_blocks_per_seq), PagedMore{},
     stream);
}

}  // namespace xllm
