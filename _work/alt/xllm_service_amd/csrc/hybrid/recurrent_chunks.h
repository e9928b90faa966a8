// What the chunked linear recurrences share: the numbering of a batch's chunks
// and the pass from chunk to chunk.
#pragma once
#include "hybrid_common.h"

namespace xllm {
namespace hyb {

// Chunk number b of the batch -> sequence, its chunk, first token, length. The
// chunks of C tokens are numbered through the sequences without gaps.
template <int C>
XLLM_DEV bool chunk_locate(int b, const int* cu_q, int n_seqs, int* s, int* c,
                           int* t0, int* len) {
  int acc = 0;
  for (int i = 0; i < n_seqs; ++i) {
    const int a = cu_q[i], e = cu_q[i + 1];
    const int nc = (e - a + C - 1) / C;
    if (b < acc + nc) {
      *s = i; *c = b - acc;
      *t0 = a + *c * C;
      *len = min(C, e - *t0);
      return true;
    }
    acc += nc;
  }
  return false;
}

// One thread per (sequence, state element): from what every chunk adds to the
// state (ws, one record per chunk) to the state BEFORE each chunk, in its
// place; the last state goes to the sequence's slot. One decay per head.
template <int C>
__global__ void chunk_scan_kernel(float* __restrict__ ws,
                                  float* __restrict__ state,
                                  const float* __restrict__ decay,
                                  const int* __restrict__ slots,
                                  const int* __restrict__ cu_q,
                                  const int* __restrict__ ctx_lens, int heads,
                                  long per_head, bool store_idle) {
  const int s = blockIdx.y;
  const long per_seq = per_head * heads;
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= per_seq) return;
  long base = 0;
  for (int i = 0; i < s; ++i) base += (cu_q[i + 1] - cu_q[i] + C - 1) / C;
  const int qlen = cu_q[s + 1] - cu_q[s];
  if (qlen <= 0 && !store_idle) return;
  const int full = qlen / C, rest = qlen - full * C;
  const int slot = slots[s];
  const float a = decay[(int)(e / per_head)];
  float S = (slot >= 0 && ctx_lens[s] > 0) ? state[slot * per_seq + e] : 0.f;
  const float a_full = powf(a, (float)C);
  float* w = ws + base * per_seq + e;
  constexpr int U = 8;                    // records in flight
  int c = 0;
  for (; c + U <= full; c += U) {
    float x[U];
#pragma unroll
    for (int i = 0; i < U; ++i) x[i] = w[(c + i) * per_seq];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      w[(c + i) * per_seq] = S;
      S = a_full * S + x[i];
    }
  }
  for (; c < full; ++c) {
    const float x = w[c * per_seq];
    w[c * per_seq] = S;
    S = a_full * S + x;
  }
  if (rest) {
    const float x = w[c * per_seq];
    w[c * per_seq] = S;
    S = powf(a, (float)rest) * S + x;
  }
  if (slot >= 0) state[slot * per_seq + e] = S;
}

}  // namespace hyb
}  // namespace xllm
