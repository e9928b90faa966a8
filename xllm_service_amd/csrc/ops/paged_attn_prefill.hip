// Paged attention of prompt rows for the dense decoders: bf16 in and out, causal
// (kernels and their reasons: paged_rows.h, paged_long.h, paged_short.h).
//
// Parity: reference engine's paged-attention prefill.
#include "paged_long.h"
#include "paged_short.h"

namespace xllm {

static PagedPrompts prompts(long tokens, int n_seqs, int G, int n_kv, int D,
                            int max_blocks) {
  // 64-wide heads ran on fp32 weights before they had a kernel and still do
  return paged_prompts(tokens, n_seqs, G, n_kv, D, max_blocks, D == 128 ? 1 : 3,
                       false);
}
// floats of scratch that a call asks for
long paged_attn_prefill_scratch(long tokens, int n_seqs, int G, int n_kv, int D,
                                int max_blocks) {
  if (tokens == 0 || n_seqs <= 0) return 0;
  return prompts(tokens, n_seqs, G, n_kv, D, max_blocks).scratch;
}

// ahead: four pieces of memory that is read next, or null; streamed: bytes that are
// read before them
void launch_paged_attn_prefill(unsigned short* out, float* ws,
                               const unsigned short* q,
                               const unsigned short* k_cache,
                               const unsigned short* v_cache,
                               const int* block_tables, const int* cu_q,
                               const int* seq_lens, long tokens, int n_seqs,
                               float scale, int n_qheads, int n_kv, int D,
                               int max_blocks, long q_stride, long out_stride,
                               const void* const* ahead, const long* ahead_bytes,
                               long streamed, hipStream_t stream) {
  if (tokens == 0 || n_seqs <= 0) return;
  const int G = n_qheads / n_kv;
  const PagedPrompts p = prompts(tokens, n_seqs, G, n_kv, D, max_blocks);
  if (p.few) {
    auto go = D == 128 ? paged_short<128, 1, false> : paged_short<64, 3, false>;
    const PagedAhead a =
        paged_ahead(paged_rows_tiles<PS_ROWS>(tokens, n_seqs, G) * n_kv,
                    max_blocks * (long)PF_BS, ahead, ahead_bytes, streamed);
    go(out, q, k_cache, v_cache, block_tables, cu_q, seq_lens, tokens, n_seqs,
       scale, n_qheads, n_kv, max_blocks, q_stride, out_stride, PagedMore{}, a,
       stream);
    return;
  }
  if (D == 128 && p.least == 0 &&
      paged_long_takes(tokens, n_seqs, G, n_kv, max_blocks)) {
    paged_long(out, q, k_cache, v_cache, block_tables, cu_q, seq_lens, tokens,
               n_seqs, scale, n_qheads, n_kv, max_blocks, q_stride, out_stride,
               stream);
    return;
  }
  const PagedAhead a =
      paged_ahead(paged_rows_wgs(p, tokens, n_seqs, G, n_kv),
                  max_blocks * (long)PF_BS, ahead, ahead_bytes, streamed);
  auto go = D == 128 ? paged_rows<128, 1, false> : paged_rows<64, 3, false>;
  go(out, ws, q, k_cache, v_cache, block_tables, cu_q, seq_lens, tokens, n_seqs,
     scale, n_qheads, n_kv, max_blocks, q_stride, out_stride, p, PagedMore{},
     a, stream);
}

// ---------------------------------------------------------------------------------
// Probe of the 16x16x32 fragments, A[l&15][8 (l>>4) + j], B[8 (l>>4) + j][l&15],
// C[4 (l>>4) + r][l&15], which linear.hip's stream kernel and the 16-row kernels of
// ../hybrid rely on (the 32x32x16 ones of this directory: mfma_rows.h):
// tests/test_gpu_ops.py compares it with torch.matmul on random data.
__global__ void mfma_probe_kernel(float* __restrict__ c,
                                  const unsigned short* __restrict__ a,
                                  const unsigned short* __restrict__ b) {
  const int lane = threadIdx.x & 63;
  const int frow = lane & 15;
  const int fcol8 = (lane >> 4) * 8;
  bf16x8 af, bf;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    af[j] = (short)a[frow * 32 + fcol8 + j];   // A[frow][fcol8+j]
    bf[j] = (short)b[(fcol8 + j) * 16 + frow]; // B[fcol8+j][frow]
  }
  f32x4 acc = {0, 0, 0, 0};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; r++) c[((lane >> 4) * 4 + r) * 16 + frow] = acc[r];
}

void launch_mfma_probe(float* c, const unsigned short* a,
                       const unsigned short* b, hipStream_t stream) {
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, stream, c, a, b);
}

}  // namespace xllm
