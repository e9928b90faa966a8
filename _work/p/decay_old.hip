// Decayed linear attention of prompt rows in bf16 on the matrix pipe.
//
//   S_t = a_h S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t      (S [D, V], fp32)
//
// with q, k, v = silu(projection), rounded to bf16. Because the decay is one
// number per head, a chunk of 128 tokens with the state S before it is
//   O = diag(a^(i+1)) Q S + ((Q K^T) * M) V,   M_ij = a^(i-j) for j <= i
//   S <- a^len S + sum_j a^(len-1-j) k_j v_j^T
// Q, K and V are bf16 values, so Q K^T is one bf16 product with fp32 sums;
// what is fp32 (the weighted scores, the weighted keys, the state) is split
// exactly into three bf16 terms (8 + 8 + 8 mantissa bits) with a product each:
// 32-bit factors at 3/16 of the cost of fp32 products.
//
//   sum   what every (chunk, head) adds to the state, all chunks at once
//   scan  chunk after chunk per state element (recurrent_chunks.h)
//   out   the outputs of every (chunk, head)
// Batches whose sequences all fit one chunk need no scratch and no scan: out
// reads the slots, then sum moves them.
//
// Chunks of 128 tokens halve the scratch traffic of 64 (a record is a whole
// state per head), and the products within a chunk they add are cheap.
//
// Measured, 3 prompts of 853-1657 tokens, 16 heads of 128 x 128: sum 20 us, scan
// 15 us (70 MB), out 31 us; 665 us as a recurrence on the vector unit, two
// passes and a scan. out and sum run one round of workgroups whose phases
// (fetch, activate, split, multiply) follow each other; two share a CU.
#include "../ops/mfma_rows.h"
#include "recurrent_chunks.h"

namespace xllm {
namespace hyb {

constexpr int DM_C = 128;      // tokens per chunk

struct DMArgs {
  float* out;                  // [T, heads, V]
  const unsigned short *q, *k, *v;
  long q_stride, k_stride, v_stride;
  const float* decay;
  float* state;                // [slots, heads, D, V]
  float* ws;                   // [chunks, heads, D, V]; null: one chunk each
  const int *slots, *cu_q, *ctx_lens;
  int n_seqs, heads;
};

// the workgroup's sequence and tokens
XLLM_DEV bool dm_locate(const DMArgs& P, int* s, int* c, int* t0, int* len) {
  if (P.ws != nullptr)
    return chunk_locate<DM_C>(blockIdx.x, P.cu_q, P.n_seqs, s, c, t0, len);
  *s = blockIdx.x; *c = 0;
  *t0 = P.cu_q[*s];
  *len = min(DM_C, P.cu_q[*s + 1] - *t0);
  return true;
}

struct alignas(16) dm_u4 { unsigned x[4]; };

// 8 neighbouring activations, packed. x / (1 + e^-x) with v_rcp and one Newton
// step in place of a division: half its instructions, and the same bf16 for
// every bf16 input. The denominator is 2^-24 of itself: the reciprocal of 1e38
// would be below what v_rcp returns.
XLLM_DEV dm_u4 dm_act(const unsigned short* p) {
  constexpr float s = 0x1p-24f;
  const ushort8_t x = *reinterpret_cast<const ushort8_t*>(p);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float z = bf16_to_f32(x.x[j]);
    const float d = fmaf(__expf(-z), s, s);       // infinite below -88.7: r = 0
    const float r = __builtin_amdgcn_rcpf(d);
    v[j] = z * (s * fmaf(fmaf(-fminf(d, 3e38f), r, 1.0f), r, r));
  }
  dm_u4 y;
#pragma unroll
  for (int j = 0; j < 4; ++j) y.x[j] = pack_bf16(v[2 * j], v[2 * j + 1]);
  return y;
}
// not zero where one of the two bf16 numbers is infinite or NaN
XLLM_DEV unsigned dm_odd(unsigned u) {
  return ((u & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
}
// v's three bf16 terms to the images at dst, dst + step, dst + 2 step
XLLM_DEV void dm_split(float v[8], unsigned short* dst, int step) {
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    dm_u4 y;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      y.x[j] = pack_bf16(v[2 * j], v[2 * j + 1]);
      drop_bf16(v[2 * j], v[2 * j + 1], y.x[j]);
    }
    *reinterpret_cast<dm_u4*>(dst + t * step) = y;
  }
}
// a^n by squaring in 64 bits: rounded once
XLLM_DEV float dm_pow(float a, int n) {
  double r = 1.0, b = (double)a;
#pragma unroll
  for (int i = 0; i < 8; ++i) {                   // n <= 255
    if ((n >> i) & 1) r *= b;
    b *= b;
  }
  return (float)r;
}

// ---- sum: U[d][e] = sum_j a^(len-1-j) k_j[d] v_j[e] ---------------------------
// A wave owns a quarter of the D x V sums; 64 tokens are staged at a time, the
// weighted keys as three images.
template <int D, int V>
__global__ void __launch_bounds__(256, 2) decay_sum_mfma_kernel(DMArgs P) {
  constexpr int ST = 64;
  constexpr int DT = D / 64, VT = V / 64;         // 32-wide tiles of a wave
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[3 * ST * D + ST * V];
  __shared__ float pw[DM_C + 1];
  int s, c, t0, len;
  if (!dm_locate(P, &s, &c, &t0, &len)) return;
  const int hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int h = lane >> 5, n = lane & 31;
  const float a = P.decay[hd];
  if (tid <= DM_C) pw[tid] = dm_pow(a, tid);
  unsigned short* ks = lds;
  unsigned short* vs = lds + 3 * ST * D;
  // products of the leading terms and those of the other two, summed apart:
  // adding the small ones to the large sum would round it three times as often
  f32x16 acc[2][DT][VT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < VT; ++j) acc[0][i][j] = acc[1][i][j] = mr_zero();
  const int kbase = mr_col_base<D>(lane), vbase = mr_col_base<V>(lane);
  const int d0 = (w & 1) * DT, e0 = (w >> 1) * VT;   // first tiles

  for (int b0 = 0; b0 < len; b0 += ST) {
    __syncthreads();                              // also: pw is there
#pragma unroll
    for (int i = 0; i < ST * (D / 8) / 256; ++i) {
      const int idx = tid + i * 256, r = idx / (D / 8), ch = idx % (D / 8);
      float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (b0 + r < len) {
        const dm_u4 y =
            dm_act(P.k + (long)(t0 + b0 + r) * P.k_stride + hd * D + ch * 8);
        const float wgt = pw[len - 1 - b0 - r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[2 * j] = __uint_as_float(y.x[j] << 16) * wgt;
          x[2 * j + 1] = __uint_as_float(y.x[j] & 0xffff0000u) * wgt;
        }
      }
      dm_split(x, ks + r * D + ((ch ^ mr_swz_cols<D>(r)) << 3), ST * D);
    }
#pragma unroll
    for (int i = 0; i < ST * (V / 8) / 256; ++i) {
      const int idx = tid + i * 256, r = idx / (V / 8), ch = idx % (V / 8);
      dm_u4 y = {{0u, 0u, 0u, 0u}};
      if (b0 + r < len)
        y = dm_act(P.v + (long)(t0 + b0 + r) * P.v_stride + hd * V + ch * 8);
      *reinterpret_cast<dm_u4*>(vs + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3)) =
          y;
    }
    __syncthreads();
#pragma unroll
    for (int st = 0; st < ST / 16; ++st) {
      bf16x8 b[VT];
#pragma unroll
      for (int j = 0; j < VT; ++j)
        b[j] = mr_cols<V>((const lds_u16*)vs + (vbase ^ ((e0 + j) << 5)) +
                          st * 16 * V);
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const bf16x8 x = mr_cols<D>((const lds_u16*)ks + t * ST * D +
                                      (kbase ^ ((d0 + i) << 5)) + st * 16 * D);
#pragma unroll
          for (int j = 0; j < VT; ++j)
            acc[t > 0][i][j] = mr_mma(x, b[j], acc[t > 0][i][j]);
        }
    }
  }
  float* dst;
  bool add = false;                               // to what is there,
  float keep = 0.f;                               // by this factor
  if (P.ws != nullptr) {
    dst = P.ws + ((long)blockIdx.x * P.heads + hd) * (D * V);
  } else {
    const int slot = P.slots[s];
    if (slot < 0) return;
    dst = P.state + ((long)slot * P.heads + hd) * (D * V);
    add = P.ctx_lens[s] > 0;
    // no new tokens: a carried state stays (and no barrier has made pw visible)
    if (add && len <= 0) return;
    if (add) keep = pw[len];
  }
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = (d0 + i) * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        float* p = dst + d * V + (e0 + j) * 32 + n;
        const float u = acc[0][i][j][r] + acc[1][i][j][r];
        *p = add ? keep * *p + u : u;
      }
}

// ---- out ------------------------------------------------------------------------
// A wave owns 32 queries. O^T = S^T Q^T with the state staged as three images of
// 64 rows at a time, faded, then the tiles of 32 keys up to its own.
template <int D, int V>
__global__ void __launch_bounds__(256, 2) decay_out_mfma_kernel(DMArgs P) {
  constexpr int KS = D / 16, VT = V / 32;
  constexpr int KV = DM_C * (D + V), SI = 3 * 64 * V;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[KV > SI ? KV : SI];
  __shared__ float pw[DM_C + 1];
  __shared__ int lost[V];      // first token with a non-finite value, if any has
  int s, c, t0, len;
  if (!dm_locate(P, &s, &c, &t0, &len)) return;
  const int hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31;
  if (tid <= DM_C) pw[tid] = dm_pow(P.decay[hd], tid);
  const int qi = w * 32 + n;
  const bool on = w * 32 < len;
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (qi < len)
      qf[ks] = __builtin_bit_cast(
          bf16x8, dm_act(P.q + (long)(t0 + qi) * P.q_stride + hd * D + ks * 16 +
                         h * 8));
  }
  // Apart as above, and the leading products of four steps (of two within the
  // chunk) are summed before they meet the large sum, which then is rounded 6
  // times instead of 16. Error against 64 bits, 3 prompts of 853-1657 tokens:
  // 8.2e-8 -> 6.7e-8 (the recurrence: 7.1e-8), for 3 us of 71.
  f32x16 acc[2][VT];
#pragma unroll
  for (int j = 0; j < VT; ++j) acc[0][j] = acc[1][j] = mr_zero();
  const int vbase = mr_col_base<V>(lane);

  // ---- through the state before the chunk ------------------------------------
  const int slot = P.slots[s];
  const bool carried = slot >= 0 && P.ctx_lens[s] > 0;
  if (c > 0 || carried) {                         // uniform
    const float* S =
        (P.ws != nullptr
             ? P.ws + ((long)blockIdx.x * P.heads + hd) * (D * V)
             : P.state + ((long)slot * P.heads + hd) * (D * V));
#pragma unroll
    for (int d0 = 0; d0 < D; d0 += 64) {
      if (d0) __syncthreads();
#pragma unroll
      for (int i = 0; i < 64 * (V / 8) / 256; ++i) {
        const int idx = tid + i * 256, r = idx / (V / 8), ch = idx % (V / 8);
        float x[8];
        Quad<float>::ld(S + (d0 + r) * V + ch * 8, x);
        Quad<float>::ld(S + (d0 + r) * V + ch * 8 + 4, x + 4);
        dm_split(x, lds + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3), 64 * V);
      }
      __syncthreads();
      if (!on) continue;
#pragma unroll
      for (int j = 0; j < VT; ++j) {
        f32x16 z = mr_zero();
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const bf16x8 x =
                mr_cols<V>((const lds_u16*)lds + t * 64 * V +
                           (vbase ^ (j << 5)) + st * 16 * V);
            if (t == 0) z = mr_mma(x, qf[d0 / 16 + st], z);
            else acc[1][j] = mr_mma(x, qf[d0 / 16 + st], acc[1][j]);
          }
        acc[0][j] += z;
      }
    }
    __syncthreads();                              // also: pw is there
    const float fade = pw[min(qi, DM_C - 1) + 1];
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[0][j][r] *= fade;
        acc[1][j][r] *= fade;
      }
  }

  // ---- within the chunk --------------------------------------------------------
  unsigned short* ks_ = lds;
  unsigned short* vs = lds + DM_C * D;
#pragma unroll 4
  for (int i = 0; i < DM_C * (D / 8) / 256; ++i) {
    const int idx = tid + i * 256, r = idx / (D / 8), ch = idx % (D / 8);
    dm_u4 y = {{0u, 0u, 0u, 0u}};
    if (r < len) y = dm_act(P.k + (long)(t0 + r) * P.k_stride + hd * D + ch * 8);
    *reinterpret_cast<dm_u4*>(ks_ + r * D + ((ch ^ mr_swz_rows<D>(r)) << 3)) =
        y;
  }
  unsigned odd = 0u;
#pragma unroll 4
  for (int i = 0; i < DM_C * (V / 8) / 256; ++i) {
    const int idx = tid + i * 256, r = idx / (V / 8), ch = idx % (V / 8);
    dm_u4 y = {{0u, 0u, 0u, 0u}};
    if (r < len) y = dm_act(P.v + (long)(t0 + r) * P.v_stride + hd * V + ch * 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) odd |= dm_odd(y.x[j]);
    *reinterpret_cast<dm_u4*>(vs + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3)) = y;
  }
  // A weight of zero keeps a key out of a row unless its value is not finite: the
  // products see zero instead, and rows from that token on are NaN at the end.
  const bool any_lost = __syncthreads_or(odd != 0u);
  if (any_lost) {
    for (int i = tid; i < V; i += 256) lost[i] = DM_C;
    __syncthreads();
    for (int i = tid; i < DM_C * V; i += 256) {
      const int r = i / V, e = i % V;
      unsigned short* x = vs + r * V + (((e >> 3) ^ mr_swz_cols<V>(r)) << 3) +
                          (e & 7);
      if (dm_odd(*x) == 0u) continue;
      *x = 0;
      atomicMin(lost + e, r);
    }
    __syncthreads();
  }
  if (!on) return;
  const int kbase = mr_row_base<D>(lane);
  for (int kt = 0; kt <= w; ++kt) {
    f32x16 z = mr_zero();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      z = mr_mma(*reinterpret_cast<const lds_bf16x8*>(
                     (const lds_u16*)ks_ + (kbase ^ (ks << 4)) + kt * 32 * D),
                 qf[ks], z);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int back = qi - kt * 32 - mr_key_of(r, h);
      z[r] = back >= 0 ? z[r] * pw[max(back, 0)] : 0.f;
    }
    bf16x8 p[3][2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      float x = z[r], y = z[r + 1];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const unsigned u = pack_bf16(x, y);
        reinterpret_cast<unsigned*>(&p[t][r >> 3])[(r & 7) >> 1] = u;
        drop_bf16(x, y, u);
      }
    }
#pragma unroll
    for (int j = 0; j < VT; ++j) {
      f32x16 y = mr_zero();
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 x = mr_cols<V>((const lds_u16*)vs + (vbase ^ (j << 5)) +
                                    (kt * 32 + st * 16) * V);
        y = mr_mma(x, p[0][st], y);
#pragma unroll
        for (int t = 1; t < 3; ++t) acc[1][j] = mr_mma(x, p[t][st], acc[1][j]);
      }
      acc[0][j] += y;
    }
  }
  if (qi >= len) return;
  if (any_lost) {
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (lost[j * 32 + 8 * (r >> 2) + 4 * h + (r & 3)] <= qi)
          acc[0][j][r] = NAN;
  }
  float* o = P.out + ((long)(t0 + qi) * P.heads + hd) * V + 4 * h;
#pragma unroll
  for (int j = 0; j < VT; ++j)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<float4*>(o + j * 32 + 2 * r) = make_float4(
          acc[0][j][r] + acc[1][j][r], acc[0][j][r + 1] + acc[1][j][r + 1],
          acc[0][j][r + 2] + acc[1][j][r + 2],
          acc[0][j][r + 3] + acc[1][j][r + 3]);
}

// records of scratch for a batch of prompt rows
long decay_attn_mfma_chunks(long tokens, long n_seqs) {
  return tokens / DM_C + n_seqs;
}
int decay_attn_mfma_chunk() { return DM_C; }

// Whether a batch is too short for this form: a sequence of a few tokens costs it
// nearly as much as one of 32 (both passes move the whole state through LDS), where
// the recurrence of decay_attn.hip walks token by token, one workgroup per 16
// columns of a state, whose rate falls once they fill the chip. Measured (us, the
// recurrence | here), 128 x 128, 8 states: 2 tokens 5.8 | 24, 16 16.8 | 24.6, 24 23.3 |
// 25.6, 32 29.6 | 25.9; 256 states: 8 22.6 | 26.7, 12 28.7 | 26.7; 1024: 8 68 | 82, 12
// 88 | 82. 64 x 64, 8 states: 8 8.6 | 12.0, 14 12.2 | 12.1; 512: 4 13.4 | 14.0, 6 16.3 |
// 13.9. 64 x 128, 64: 16 14.2 | 16.6, 20 17.1 | 17.2; 128 x 64, 256: 10 16.3 | 18.4, 14
// 20.2 | 18.4.
bool decay_attn_short(long longest, long states, int D, int V) {
  const int most = D != V ? 16 : D == 128 ? 24 : 12;   // tokens, few workgroups
  const long wgs = states * (V / 16);
  const int tenths = wgs <= 512 ? 10 : wgs <= 1024 ? 8 : wgs <= 1536 ? 6
                     : wgs <= 2048 ? 4 : D == 64 ? 3 : V == 64 ? 6 : 4;
  return longest * 10 <= most * tenths;
}

// D, V in {64, 128}; rows 16 B aligned. ws null: no sequence has more than
// DM_C tokens.
void launch_decay_attn_mfma(float* out, const unsigned short* q,
                            const unsigned short* k, const unsigned short* v,
                            const float* decay, float* state, const int* slots,
                            const int* cu_q, const int* ctx_lens, long tokens,
                            int n_seqs, int heads, int D, int V, long q_stride,
                            long k_stride, long v_stride, float* ws,
                            hipStream_t st) {
  if (n_seqs == 0) return;
  const DMArgs P = {out, q, k, v, q_stride, k_stride, v_stride, decay, state,
                    ws, slots, cu_q, ctx_lens, n_seqs, heads};
  const dim3 grid(
      (unsigned)(ws ? decay_attn_mfma_chunks(tokens, n_seqs) : n_seqs), heads);
#define DM_SUM(DD, VV)                                                        \
  hipLaunchKernelGGL((decay_sum_mfma_kernel<DD, VV>), grid, dim3(256), 0, st, P)
#define DM_OUT(DD, VV)                                                        \
  hipLaunchKernelGGL((decay_out_mfma_kernel<DD, VV>), grid, dim3(256), 0, st, P)
#define DM_BY_SIZE(CALL)                                                      \
  do {                                                                        \
    if (D == 128) { if (V == 128) CALL(128, 128); else CALL(128, 64); }       \
    else { if (V == 128) CALL(64, 128); else CALL(64, 64); }                  \
  } while (0)
  if (ws == nullptr) {
    DM_BY_SIZE(DM_OUT);
    DM_BY_SIZE(DM_SUM);
    return;
  }
  DM_BY_SIZE(DM_SUM);
  const long per_head = (long)D * V, per_seq = per_head * heads;
  hipLaunchKernelGGL((chunk_scan_kernel<DM_C>),
                     dim3((unsigned)((per_seq + 255) / 256), n_seqs),
                     dim3(256), 0, st, ws, state, decay, slots, cu_q, ctx_lens,
                     heads, per_head, true);
  DM_BY_SIZE(DM_OUT);
#undef DM_BY_SIZE
#undef DM_OUT
#undef DM_SUM
}

}  // namespace hyb
}  // namespace xllm
