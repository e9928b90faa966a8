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
//   walk  both, by workgroups that follow a sequence, or one of up to four groups of its
//         chunks: many sequences, or few chunks
//   out   the outputs of every (chunk, head), by four waves or by sixteen
// Batches whose sequences all fit one chunk need no scratch and no scan: out
// reads the slots and moves them too, or sum does afterwards.
//
// Chunks of 128 tokens halve the scratch traffic of 64 (a record is a whole
// state per head), and the products within a chunk they add are cheap.
//
// Measured, 3 prompts of 853-1657 tokens, 16 heads of 128 x 128: sum 18.7 us (64 MB),
// scan 14.4 (70 MB, the rate of a copy), out 30.6 (111 MB); 665 us as a recurrence on
// the vector unit, two passes and a scan. out and sum run one round of workgroups whose
// phases (activate, split, multiply) follow each other, two to a CU, and are bound by
// the vector unit: activations and splits. What a phase reads is fetched during the one
// before it: 68.0 -> 61.9 us in all. One wave issues a vector instruction in 6 cycles, two
// of a SIMD in 3 each: a workgroup alone on a CU takes as long as two, 19 us of out for
// 160 of them, hence the kernels of 8 and 16 waves for small batches.
#include "../ops/mfma_rows.h"
#include "recurrent_chunks.h"

namespace xllm {
namespace hyb {

constexpr int DM_C = 128;      // tokens per chunk
constexpr int DM_LATE = 4;     // ... at most that join the state one by one

struct DMArgs {
  float* out;                  // [T, heads, V]
  const unsigned short *q, *k, *v;
  long q_stride, k_stride, v_stride;
  const float* decay;
  float* state;                // [slots, heads, D, V]
  float* ws;                   // [chunks, heads, D, V]; null: one chunk each
  const int *slots, *cu_q, *ctx_lens;
  int n_seqs, heads;
  int groups;                  // that walk cuts a sequence's chunks into (DMGroups)
  long tail;                   // records of ws before the last groups' sums
};

// Where walk has more than one group to a sequence, of `size` chunks each, all but the
// first start from nothing: what group i adds by its end lies in the record of the chunk
// after it, which needs none of its own, the last one's in the tail. Chunk c's state
// before it is then its record's, of its own group, and the start of that faded.
struct DMGroups {
  int chunks, size, count;
  XLLM_DEV DMGroups(const DMArgs& P, int len) {
    chunks = (len + DM_C - 1) / DM_C;
    size = max((chunks + P.groups - 1) / P.groups, 1);
    count = max((chunks + size - 1) / size, 1);
  }
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

XLLM_DEV ushort8_t dm_row(const unsigned short* p) {
  return *reinterpret_cast<const ushort8_t*>(p);
}
// 8 neighbouring activations, packed. x / (1 + e^-x) with v_rcp in place of a
// division. The denominator is 2^-24 of itself: the reciprocal of 1e38 would be below
// what v_rcp returns. Its 1 is a step of 2^-23 larger: what v_rcp and v_exp return is
// then rounded to the bf16 number that the division gives for every bf16 input (without
// it for all but one; e^-x from a log2(e) up to 5 steps smaller or 2 larger changes
// none, so this is no close call). A Newton step on the reciprocal, which does that too,
// costs 2.3 us of 70.
XLLM_DEV dm_u4 dm_act(const ushort8_t& x) {
  constexpr float s = 0x1p-24f, one = s * (1.0f + 0x1p-23f);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float z = bf16_to_f32(x.x[j]);
    const float d = fmaf(__expf(-z), s, one);     // infinite below -88.7: 0
    v[j] = z * (s * __builtin_amdgcn_rcpf(d));
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

// a^n, rounded once, and finite: a state's zeros stay zero
XLLM_DEV float dm_pow_far(float a, int n) {
  double r = 1.0, b = (double)a;
  for (; n > 0; n >>= 1) {
    if (n & 1) r *= b;
    b *= b;
  }
  return fminf((float)r, 3.4028235e38f);
}

// A state's last tokens. They weigh most, and the matrix pipe cuts off what the products
// of 16 tokens have below the last bit of the largest. So some of them are left out of its
// sums (their weights are zero) and join one by one with a rounding each, as in the
// recurrence: all of up to four, else two below a decay of 3/4 and one below 0.9. Errors
// of states against 64 bits, 1e-8, fresh ones, without that | with it | the recurrence:
// heads of 0.75 to 0.996, 3 tokens 3.3 | 3.1 | 3.1, 6 3.8 | 3.8 | 4.4; of 0.3 to 0.7, 6
// tokens 3.8 | 3.0 | 3.0, 16 4.8 | 3.2 | 3.0. It takes 0.3 to 0.5 us of 6 to 11.
struct DMLate {
  float a;
  int from, end, len;          // the first one; the token as of which the others weigh
  XLLM_DEV DMLate(float decay, int n) {
    a = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(decay)));
    len = n;
    from = n <= DM_LATE ? 0 : n - (a < 0.75f ? 2 : a < 0.9f ? 1 : 0);
    end = min(from, n - 1);
  }
  XLLM_DEV int place(int r) const { return r - len + DM_LATE; }
  // acc: what the pipe has summed, leading and other terms; x: the state before, faded by
  // `fade`; k, v: of the last tokens, of this lane's key and value column
  XLLM_DEV void join(f32x16 (&acc)[2], const float (&x)[16], float fade,
                     const unsigned short (&k)[DM_LATE], const unsigned short (&v)[DM_LATE],
                     int h) const {
    const float by =
        __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(fade)));
    const bool alone = from == 0;                  // uniform, as all below
    if (alone) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][r] = x[r];
    } else if (by < 0.5f) {                        // a state that has faded meets the
#pragma unroll
      for (int r = 0; r < 16; ++r)                 // small terms, another one their sum
        acc[0][r] = fmaf(by, x[r], acc[1][r]) + acc[0][r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[0][r] = fmaf(by, x[r], acc[0][r] + acc[1][r]);
    }
#pragma unroll
    for (int i = 0; i < DM_LATE; ++i) {
      if (i < place(from)) continue;               // uniform
      // one product an entry, exact: the step's other 15 tokens are zeros
      bf16x8 a16 = {0, 0, 0, 0, 0, 0, 0, 0}, b16 = a16;
      a16[0] = h ? (short)0 : (short)k[i];
      b16[0] = h ? (short)0 : (short)v[i];
      const f32x16 z = mr_mma(a16, b16, mr_zero());
      const float keep = alone || i > place(from) ? a : 1.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][r] = fmaf(keep, acc[0][r], z[r]);
    }
  }
};

// ---- sum: U[d][e] = sum_j a^(len-1-j) k_j[d] v_j[e] ---------------------------
// A wave owns a quarter of the D x V sums; 64 tokens are staged at a time, the
// weighted keys as three images.
//   ONE: each sequence is one chunk, whose sum goes to its slot (DMLate).
template <int D, int V, bool ONE>
__global__ void __launch_bounds__(256, 2) decay_sum_mfma_kernel(DMArgs P) {
  constexpr int ST = 64;
  constexpr int DT = D / 64, VT = V / 64;         // 32-wide tiles of a wave
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[3 * ST * D + ST * V + (ONE ? DM_LATE * (D + V) : 0)];
  unsigned short* newest = lds + 3 * ST * D + ST * V;     // keys, values, with ONE
  __shared__ float pw[DM_C + 1];
  int s, c, t0, len;
  if (!dm_locate(P, &s, &c, &t0, &len)) return;
  const int hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int h = lane >> 5, n = lane & 31;
  const float a = P.decay[hd];
  const DMLate late(a, len);
  const int sum_to = ONE ? late.from : len;      // tokens that the pipe sums
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

  constexpr int KI = ST * (D / 8) / 256, VI = ST * (V / 8) / 256;
  ushort8_t kr[KI], vr[VI];
  auto fetch = [&](int b0) {                      // rows past the end: the last
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int idx = tid + i * 256, r = min(b0 + idx / (D / 8), len - 1);
      kr[i] = dm_row(P.k + (long)(t0 + r) * P.k_stride + hd * D +
                     idx % (D / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int idx = tid + i * 256, r = min(b0 + idx / (V / 8), len - 1);
      vr[i] = dm_row(P.v + (long)(t0 + r) * P.v_stride + hd * V +
                     idx % (V / 8) * 8);
    }
  };
  if (len > 0) fetch(0);
  for (int b0 = 0; b0 < len; b0 += ST) {
    __syncthreads();                              // also: pw is there
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int idx = tid + i * 256, r = idx / (D / 8), ch = idx % (D / 8);
      float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (ONE && b0 + r >= sum_to && b0 + r < len)
        *reinterpret_cast<dm_u4*>(newest + late.place(b0 + r) * D + ch * 8) = dm_act(kr[i]);
      if (b0 + r < sum_to) {
        const dm_u4 y = dm_act(kr[i]);
        const float wgt = pw[(ONE ? late.end : len - 1) - b0 - r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[2 * j] = __uint_as_float(y.x[j] << 16) * wgt;
          x[2 * j + 1] = __uint_as_float(y.x[j] & 0xffff0000u) * wgt;
        }
      }
      dm_split(x, ks + r * D + ((ch ^ mr_swz_cols<D>(r)) << 3), ST * D);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int idx = tid + i * 256, r = idx / (V / 8), ch = idx % (V / 8);
      dm_u4 y = {{0u, 0u, 0u, 0u}};
      if (b0 + r < len) y = dm_act(vr[i]);
      if (ONE && b0 + r >= sum_to && b0 + r < len)
        *reinterpret_cast<dm_u4*>(newest + DM_LATE * D + late.place(b0 + r) * V + ch * 8) = y;
      *reinterpret_cast<dm_u4*>(vs + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3)) =
          y;
    }
    __syncthreads();
    if (b0 + ST < len) fetch(b0 + ST);            // beside the products
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
  bool carried = false;
  if constexpr (!ONE) {
    dst = P.ws + ((long)blockIdx.x * P.heads + hd) * (D * V);
  } else {
    const int slot = P.slots[s];
    if (slot < 0) return;
    dst = P.state + ((long)slot * P.heads + hd) * (D * V);
    carried = P.ctx_lens[s] > 0;
    // no new tokens: a carried state stays (and no barrier has made pw visible)
    if (carried && len <= 0) return;
  }
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < VT; ++j) {
      float* p = dst + ((d0 + i) * 32 + 4 * h) * V + (e0 + j) * 32 + n;
      f32x16 u[2] = {acc[0][i][j], acc[1][i][j]};
      if constexpr (ONE) {
        // all of it on the way before the first is stored, which might be another's place
        float x[16];
        unsigned short late_k[DM_LATE], late_v[DM_LATE];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          x[r] = carried ? p[(8 * (r >> 2) + (r & 3)) * V] : 0.f;
        if (len > 0) {
#pragma unroll
          for (int t = 0; t < DM_LATE; ++t) {
            late_k[t] = newest[t * D + (d0 + i) * 32 + n];
            late_v[t] = newest[DM_LATE * D + t * V + (e0 + j) * 32 + n];
          }
          late.join(u, x, carried ? pw[late.end + 1] : 0.f, late_k, late_v, h);
        }
      } else {
        u[0] += u[1];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) p[(8 * (r >> 2) + (r & 3)) * V] = u[0][r];
    }
}

// ---- walk: a state from chunk to chunk --------------------------------------------
// A workgroup (8 waves) owns 64 x 64 entries of one (sequence, head)'s state and walks its
// chunks: the state before each goes to the chunk's record, the last one to the slot. A
// wave makes 32 x 32 of what a chunk adds from half of its tokens; two waves swap halves
// of their sums and keep half of the state each. 64 tokens are staged at a time, a 16 B
// piece of both a thread, into one of two buffers while the other one is multiplied.
//   A chunk takes 2.9 us, most of it activations and splits (each key and value is
// activated for two slices), whatever the number of sequences up to two workgroups a CU;
// in return records go out once and never come back to be summed. Us in all, sum and scan
// | walk: 2 prompts of 164-341 tokens, 32 heads 39.1 | 25.6, 8 of 197-471 114 | 90, 6 of
// 449-912 154 | 126, 30 of 200-300 353 | 229; but 3 of 700-2000, 16 heads 65 | 76.
//   Few sequences leave CUs idle and are long chains, so their chunks are cut into groups
// that are walked side by side (DMGroups; figures at decay_attn_mfma_groups): 800 tokens of
// 16 heads 34.7 -> 29.5 in all. Errors against 64 bits of seven such batches: 6.1e-8 -> 6.0e-8,
// states 5.9e-8 -> 5.2e-8.
template <int D, int V>
__global__ void __launch_bounds__(512, 4) decay_walk_mfma_kernel(DMArgs P) {
  constexpr int ST = 64, IMG = ST * 64, BUF = 4 * IMG;     // three of keys, one of values
  constexpr int SL = (D / 64) * (V / 64);
  // one object: its end swaps the sums
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[2 * BUF + 8 * 2 * 64 * 8];
  typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f4;
  f4* swap = reinterpret_cast<f4*>(lds + 2 * BUF);         // [wave][2][lane]
  // slices of a state on one XCD: they read the same rows
  const int in_group = gridDim.x / P.groups;
  const int group = blockIdx.x / in_group, b = blockIdx.x - group * in_group;
  const int sl = b / 8 % SL;
  const int sh = b / (8 * SL) * 8 + b % 8;
  if (sh >= P.n_seqs * P.heads) return;
  const int s = sh / P.heads, hd = sh - s * P.heads;
  const int d0 = sl % (D / 64) * 64, e0 = sl / (D / 64) * 64;
  const int all = P.cu_q[s + 1] - P.cu_q[s];
  const DMGroups of(P, all);
  if (group >= of.count) return;
  const bool final = group == of.count - 1;
  const int c0 = group * of.size;                          // its first chunk
  const int t0 = P.cu_q[s] + c0 * DM_C;
  const int len = final ? all - c0 * DM_C : of.size * DM_C;
  const int slot = P.slots[s];
  const bool carried = group == 0 && slot >= 0 && P.ctx_lens[s] > 0;
  const int chunks = (len + DM_C - 1) / DM_C;
  const int last = len - (chunks - 1) * DM_C;              // tokens of the last one
  long rec = c0;                                           // its first record
  for (int i = 0; i < s; ++i)
    rec += (P.cu_q[i + 1] - P.cu_q[i] + DM_C - 1) / DM_C;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31;
  const int dt = w & 1, et = w >> 1 & 1, half = w >> 2;
  const int r = tid >> 3, ch = tid & 7;                    // of its pieces

  // pieces of two chunks on their way
  ushort8_t kr[2][2], vr[2][2];
  auto fetch = [&](int c, int p, ushort8_t& k, ushort8_t& v) {
    const long t = t0 + min(c * DM_C + p * ST + r, len - 1);
    k = dm_row(P.k + t * P.k_stride + hd * D + d0 + ch * 8);
    v = dm_row(P.v + t * P.v_stride + hd * V + e0 + ch * 8);
  };
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int p = 0; p < 2; ++p)
      if (c < chunks) fetch(c, p, kr[c][p], vr[c][p]);
  // this wave's half of the 32 x 32: registers 8 half .. of a product's
  long at[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    at[i] = (long)(d0 + dt * 32 + 16 * half + 8 * i + 4 * h) * V + e0 + et * 32 + n;
  float S[8];
  float* st = P.state + ((long)max(slot, 0) * P.heads + hd) * (D * V);
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = carried ? st[at[i >> 2] + (i & 3) * V] : 0.f;
  // weights of this thread's token in either half of a whole chunk, and of the last
  const float a = P.decay[hd];
  float whole[2] = {0.f, 0.f}, keep = 0.f;
  if (chunks > 1) {
    whole[0] = dm_pow(a, DM_C - 1 - r);
    whole[1] = dm_pow(a, ST - 1 - r);
    keep = dm_pow(a, DM_C);
  }
  const float rest[2] = {dm_pow(a, max(last - 1 - r, 0)),
                         dm_pow(a, max(last - ST - 1 - r, 0))};
  const float keep_last = dm_pow(a, max(last, 0));
  auto stage = [&](int c, int p, const ushort8_t& k, const ushort8_t& v) {
    const bool end = c == chunks - 1;
    const bool in = !end || p * ST + r < last;
    unsigned short* ks = lds + p * BUF;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    dm_u4 y = {{0u, 0u, 0u, 0u}};
    if (in) {
      const dm_u4 z = dm_act(k);
      const float wgt = end ? rest[p] : whole[p];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[2 * j] = __uint_as_float(z.x[j] << 16) * wgt;
        x[2 * j + 1] = __uint_as_float(z.x[j] & 0xffff0000u) * wgt;
      }
      y = dm_act(v);
    }
    const int to = r * 64 + ((ch ^ mr_swz_cols<64>(r)) << 3);
    dm_split(x, ks + to, IMG);
    *reinterpret_cast<dm_u4*>(ks + 3 * IMG + to) = y;
  };
  const int base = mr_col_base<64>(lane) + half * 32 * 64;
  // leading and other terms apart, as in sum
  f32x16 acc[2];
  auto multiply = [&](int p) {
    const lds_u16* ks = (const lds_u16*)lds + p * BUF;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const bf16x8 b = mr_cols<64>(ks + 3 * IMG + (base ^ (et << 5)) + k * 16 * 64);
#pragma unroll
      for (int t = 0; t < 3; ++t)
        acc[t > 0] = mr_mma(
            mr_cols<64>(ks + t * IMG + (base ^ (dt << 5)) + k * 16 * 64), b,
            acc[t > 0]);
    }
  };
  auto chunk = [&](int c, ushort8_t (&k)[2], ushort8_t (&v)[2], ushort8_t& k_next,
                   ushort8_t& v_next) {
    acc[0] = acc[1] = mr_zero();
    multiply(0);
    const bool two = c < chunks - 1 || last > ST;  // halves of the chunk, uniform
    if (two) stage(c, 1, k[1], v[1]);
    if (c + 2 < chunks) {
      fetch(c + 2, 0, k[0], v[0]);
      fetch(c + 2, 1, k[1], v[1]);
    }
    __syncthreads();
    if (two) multiply(1);
    if (c + 1 < chunks) stage(c + 1, 0, k_next, v_next);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f4 z;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int x = 4 * i + j;
        z[j] = half ? acc[0][x] + acc[1][x] : acc[0][8 + x] + acc[1][8 + x];
      }
      swap[(w * 2 + i) * 64 + lane] = z;
    }
    __syncthreads();
    float* to = P.ws + ((rec + c) * P.heads + hd) * (D * V);
    const bool store = c > 0 || carried;
    const float by = c == chunks - 1 ? keep_last : keep;
    // z: the other half's. What weighs little comes first, so that most sums are not
    // rounded against what is large: small terms, a state that has faded, earlier tokens.
    // A state that has not is what is large. (Error of states of 130-1000 tokens against
    // 64 bits, by sum and scan | here before | now: decays of 0.3 to 0.97 5.03e-8 | 5.25 |
    // 4.95, of 0.3 to 0.7 4.73 | 5.12 | 4.91, of 0.75 to 0.996 5.9 | 5.6 | 5.6.)
    const bool faded = __builtin_amdgcn_readfirstlane(by < 0.5f);
    // whether the chunk's last 32 tokens are this wave's
    const bool latest = half == (c == chunks - 1 ? (last - 1) >> 5 & 1 : 1);
    auto join = [&](auto second) {
      constexpr int o = second.value ? 8 : 0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const f4 z = swap[((w ^ 4) * 2 + i) * 64 + lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int x = 4 * i + j;
          const float lead = acc[0][o + x], u = acc[1][o + x];
          if (store) to[at[i] + j * V] = S[x];
          if (faded) {
            const float y = fmaf(by, S[x], u);
            S[x] = latest ? (y + z[j]) + lead : (y + lead) + z[j];
          } else {
            S[x] = fmaf(by, S[x], (lead + u) + z[j]);
          }
        }
      }
    };
    if (half) join(std::true_type{});              // uniform
    else join(std::false_type{});
  };
  if (chunks > 0) stage(0, 0, kr[0][0], vr[0][0]);
  __syncthreads();
  for (int c = 0; c < chunks; c += 2) {
    chunk(c, kr[0], vr[0], kr[1][0], vr[1][0]);
    if (c + 1 < chunks) chunk(c + 1, kr[1], vr[1], kr[0][0], vr[0][0]);
  }
  if (!final) {
    st = P.ws + ((rec + chunks) * P.heads + hd) * (D * V);
  } else {
    if (slot < 0 || (len <= 0 && carried)) return;         // nothing to keep, or as it is
    if (group > 0) st = P.ws + ((P.tail + s) * P.heads + hd) * (D * V);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) st[at[i >> 2] + (i & 3) * V] = S[i];
}

// A sequence's last state, where walk had groups of it: by workgroups of `out` past its
// heads, which nothing there waits for
template <int D, int V, int NT>
XLLM_DEV void dm_last_state(const DMArgs& P) {
  const long unit = (long)(blockIdx.y - P.heads) * gridDim.x + blockIdx.x;
  if (unit >= (long)P.n_seqs * P.heads) return;
  const int s = (int)(unit / P.heads), hd = (int)(unit - (long)s * P.heads);
  const int len = P.cu_q[s + 1] - P.cu_q[s], slot = P.slots[s];
  const DMGroups of(P, len);
  if (of.count < 2 || slot < 0) return;           // it is there
  long rec = 0;
  for (int i = 0; i < s; ++i)
    rec += (P.cu_q[i + 1] - P.cu_q[i] + DM_C - 1) / DM_C;
  const float a = P.decay[hd], by = dm_pow_far(a, of.size * DM_C);
  const float by_last = dm_pow_far(a, len - (of.count - 1) * of.size * DM_C);
  const long step = (long)of.size * P.heads * (D * V);
  const float* first = P.ws + ((rec + of.size) * P.heads + hd) * (D * V);
  const float* tail = P.ws + ((P.tail + s) * P.heads + hd) * (D * V);
  float* to = P.state + ((long)slot * P.heads + hd) * (D * V);
#pragma unroll 4
  for (int i = threadIdx.x * 4; i < D * V; i += NT * 4) {
    float S[4], x[4], y[4];
    Quad<float>::ld(first + i, S);
    Quad<float>::ld(tail + i, y);
    for (int g = 1; g + 1 < of.count; ++g) {
      Quad<float>::ld(first + g * step + i, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) S[e] = fmaf(by, S[e], x[e]);
    }
    *reinterpret_cast<float4*>(to + i) =
        make_float4(fmaf(by_last, S[0], y[0]), fmaf(by_last, S[1], y[1]),
                    fmaf(by_last, S[2], y[2]), fmaf(by_last, S[3], y[3]));
  }
}
// What a chunk's state before it is made of
struct DMStart {
  const float *own, *first;    // its record or slot, null: nothing; the first group's end
  long step;                   // from one group's end to the next one's
  int more;                    // groups between the first one and its own
  float by, fade;              // over a group, and since its own began
  template <int DV>
  XLLM_DEV void init(const DMArgs& P, int s, int c, int hd, const float* S) {
    const DMGroups of(P, P.cu_q[s + 1] - P.cu_q[s]);
    const int g = c / of.size, in = c - g * of.size;
    if (g == 0) return;
    const float a = P.decay[hd];
    more = g - 1;
    step = (long)of.size * P.heads * DV;
    first = S - (long)(c - of.size) * P.heads * DV;
    if (in == 0) own = nullptr;
    by = more > 0 ? dm_pow_far(a, of.size * DM_C) : 0.f;
    fade = dm_pow_far(a, in * DM_C);
  }
  // x: its own 8 entries from `at` on, y: the first group's end
  XLLM_DEV void ask(long at, float (&x)[8]) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.f;
    if (own == nullptr) return;                   // uniform
    Quad<float>::ld(own + at, x);
    Quad<float>::ld(own + at + 4, x + 4);
  }
  XLLM_DEV void ask_first(long at, float (&y)[8]) const {
    Quad<float>::ld(first + at, y);
    Quad<float>::ld(first + at + 4, y + 4);
  }
  XLLM_DEV void join(long at, float (&x)[8], float (&y)[8]) const {
    for (int g = 1; g <= more; ++g) {
      float z[8];
      Quad<float>::ld(first + g * step + at, z);
      Quad<float>::ld(first + g * step + at + 4, z + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = fmaf(by, y[e], z[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = fmaf(fade, y[e], x[e]);
  }
};

// ---- out ------------------------------------------------------------------------
// A wave owns 32 queries. O^T = S^T Q^T with the state staged as three images of
// 64 rows at a time, faded, then the tiles of 32 keys up to its own.
template <int D, int V, bool GROUPS>
__global__ void __launch_bounds__(256, 2) decay_out_mfma_kernel(DMArgs P) {
  constexpr int KS = D / 16, VT = V / 32;
  constexpr int KV = DM_C * (D + V), SI = 3 * 64 * V;
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[KV > SI ? KV : SI];
  __shared__ float pw[DM_C + 1];
  __shared__ int lost[V];      // first token with a non-finite value, if any has
  int s, c, t0, len;
  if (GROUPS && (int)blockIdx.y >= P.heads) return dm_last_state<D, V, 256>(P);
  if (!dm_locate(P, &s, &c, &t0, &len)) return;
  const int hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31;
  if (tid <= DM_C) pw[tid] = dm_pow(P.decay[hd], tid);
  const int qi = w * 32 + n;
  const bool on = w * 32 < len;
  // half of the state before the chunk, on its way while what comes before it
  // is made
  const int slot = P.slots[s];
  const bool carried = slot >= 0 && P.ctx_lens[s] > 0;
  const bool before = c > 0 || carried;           // uniform
  const float* S =
      (P.ws != nullptr
           ? P.ws + ((long)blockIdx.x * P.heads + hd) * (D * V)
           : P.state + ((long)max(slot, 0) * P.heads + hd) * (D * V));
  constexpr int SN = 64 * (V / 8) / 256;
  DMStart start = {S, nullptr, 0, 0, 0.f, 0.f};
  if constexpr (GROUPS) start.init<D * V>(P, s, c, hd, S);
  float sr[SN][8];
  auto fetch_state = [&](int d0) {
#pragma unroll
    for (int i = 0; i < SN; ++i) start.ask(d0 * V + (tid + i * 256) * 8, sr[i]);
  };
  bf16x8 qf[KS];
  {
    ushort8_t qr[KS];
    const unsigned short* p = P.q + (long)(t0 + min(qi, len - 1)) * P.q_stride +
                              hd * D + h * 8;
    if (len > 0) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qr[ks] = dm_row(p + ks * 16);
    }
    if (before) fetch_state(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (qi < len) qf[ks] = __builtin_bit_cast(bf16x8, dm_act(qr[ks]));
    }
  }
  // Apart as above, and the leading products of four steps (of two within the
  // chunk) are summed before they meet the large sum, which then is rounded 6
  // times instead of 16. Error against 64 bits, 3 prompts of 853-1657 tokens:
  // 8.2e-8 -> 6.7e-8 (the recurrence: 7.1e-8), for 3 us.
  f32x16 acc[2][VT];
#pragma unroll
  for (int j = 0; j < VT; ++j) acc[0][j] = acc[1][j] = mr_zero();
  const int vbase = mr_col_base<V>(lane);

  // K, then V: batches of four pieces a lane, one on its way while another one is
  // activated
  constexpr int NB = DM_C * (D / 8 + V / 8) / 1024;
  ushort8_t raw[2][4];
  auto fetch = [&](int b) {
    const bool key = b < DM_C * (D / 8) / 1024;
    const int W = key ? D : V;
    const unsigned short* p = key ? P.k : P.v;
    const long stride = key ? P.k_stride : P.v_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + (b * 4 + i) * 256 - (key ? 0 : DM_C * (D / 8));
      const int r = min(idx / (W / 8), len - 1);  // rows past the end: the last
      raw[b & 1][i] =
          dm_row(p + (long)(t0 + r) * stride + hd * W + idx % (W / 8) * 8);
    }
  };

  // ---- through the state before the chunk ------------------------------------
  if (before) {
#pragma unroll
    for (int d0 = 0; d0 < D; d0 += 64) {
      if (start.first != nullptr) {
        float y[SN][8];
#pragma unroll
        for (int i = 0; i < SN; ++i)
          start.ask_first(d0 * V + (tid + i * 256) * 8, y[i]);
#pragma unroll
        for (int i = 0; i < SN; ++i)
          start.join(d0 * V + (tid + i * 256) * 8, sr[i], y[i]);
      }
      if (d0) __syncthreads();
#pragma unroll
      for (int i = 0; i < SN; ++i) {
        const int idx = tid + i * 256, r = idx / (V / 8), ch = idx % (V / 8);
        dm_split(sr[i], lds + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3), 64 * V);
      }
      if (d0 + 64 < D) fetch_state(d0 + 64);
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
    if (len > 0) fetch(0);
    __syncthreads();                              // also: pw is there
    const float fade = pw[min(qi, DM_C - 1) + 1];
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[0][j][r] *= fade;
        acc[1][j][r] *= fade;
      }
  } else if (len > 0) {
    fetch(0);
  }
  if (len <= 0) return;                           // uniform

  // ---- within the chunk --------------------------------------------------------
  unsigned short* ks_ = lds;
  unsigned short* vs = lds + DM_C * D;
  unsigned odd = 0u;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (b + 1 < NB) fetch(b + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool key = b < DM_C * (D / 8) / 1024;
      const int W = key ? D : V;
      const int idx = tid + (b * 4 + i) * 256 - (key ? 0 : DM_C * (D / 8));
      const int r = idx / (W / 8), ch = idx % (W / 8);
      dm_u4 y = {{0u, 0u, 0u, 0u}};
      if (r < len) y = dm_act(raw[b & 1][i]);
      if (key) {
        *reinterpret_cast<dm_u4*>(ks_ + r * D +
                                  ((ch ^ mr_swz_rows<D>(r)) << 3)) = y;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) odd |= dm_odd(y.x[j]);
        *reinterpret_cast<dm_u4*>(vs + r * V +
                                  ((ch ^ mr_swz_cols<V>(r)) << 3)) = y;
      }
    }
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
    // 128 wide keys in two chains, as in the kernel of 8 and 16 waves, where there are
    // registers for both: scores of one, over 64-wide values, made outputs of 4 to 9
    // tokens 6.4e-8 off, 5.7e-8 by the recurrence
    constexpr int CHAINS = D == 128 && V == 64 ? 2 : 1;
    f32x16 zs[CHAINS];
#pragma unroll
    for (int i = 0; i < CHAINS; ++i) zs[i] = mr_zero();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      zs[ks % CHAINS] = mr_mma(
          *reinterpret_cast<const lds_bf16x8*>(
              (const lds_u16*)ks_ + (kbase ^ (ks << 4)) + kt * 32 * D),
          qf[ks], zs[ks % CHAINS]);
    f32x16 z = zs[0];
    if constexpr (CHAINS > 1) z += zs[CHAINS - 1];
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

// ---- out, few workgroups ---------------------------------------------------------
// A workgroup (16 waves, 8 of 64 values, a CU to itself) owns a (chunk, head); a wave 32
// queries by 32 values, sums in 32 registers. All that it reads is asked for at once;
// then the state's three images and the queries go to LDS and meet there, keys and values
// are activated in registers meanwhile and take the images' place. Each weighted tile of
// scores is made once, by one of the waves that want it, and passed on through LDS: 16 B a
// lane, as the products take it.
//   Up to a workgroup for each CU it takes 14 us for 19 of the four waves' kernel (2
// prompts of 164-341 tokens, 32 heads, 30.3 -> 25.6 in all): all it reads comes at the rate
// of a CU (160 KB, 2 us), then a SIMD has four waves to issue from. Beyond that nothing
// is read while it computes, and two workgroups a CU are faster: 528 of them 31 | 36.
//   LAST: each sequence is one chunk, whose workgroup then moves its state too: the keys lie
// in LDS, are weighted and split in place of queries, keys and weights, and a wave has 32 x
// 32 of the state. A kernel of its own would start over, fetch and activate again; figures
// at decay_attn_one.
template <int D, int V, bool GROUPS, bool LAST>
__global__ void __launch_bounds__(32 * V / 4) decay_out_wide_kernel(DMArgs P) {
  constexpr int NV = V / 32, NT = 256 * NV;       // column tiles, threads
  constexpr int KS = D / 16;
  constexpr int QP = DM_C * D / 8 / NT, VP = DM_C * V / 8 / NT;   // pieces of a thread
  constexpr int SP = D * V / 8 / NT;
  // queries | state, then keys, weights, values | powers, first lost token of a column
  constexpr int IMG = D * V, KEYS = DM_C * D, WGTS = KEYS + DM_C * D,
                TILE = 3 * 2 * 64 * 8, VALS = WGTS + 10 * TILE;
  constexpr int END = (KEYS + 3 * IMG > VALS + DM_C * V ? KEYS + 3 * IMG
                                                        : VALS + DM_C * V);
  __shared__ __attribute__((aligned(1024))) unsigned short
      lds[END + 2 * (DM_C + 4) + 2 * V];
  float* pw = reinterpret_cast<float*>(lds + END);
  int* lost = reinterpret_cast<int*>(lds + END + 2 * (DM_C + 4));
  int s, c, t0, len;
  if (GROUPS && (int)blockIdx.y >= P.heads) return dm_last_state<D, V, NT>(P);
  if (!dm_locate(P, &s, &c, &t0, &len)) return;
  const int hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int slot = P.slots[s];
  const bool carried = slot >= 0 && P.ctx_lens[s] > 0;
  float* kept = P.state + ((long)max(slot, 0) * P.heads + hd) * (D * V);
  if (len <= 0) {
    if (LAST && slot >= 0 && !carried)            // a new state, of no tokens
      for (int i = tid * 4; i < D * V; i += NT * 4)
        *reinterpret_cast<float4*>(kept + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a SIMD's waves have different queries: later ones meet more keys
  const int vt = w >> 2, qt = (w + vt) & 3;
  const DMLate late(LAST ? P.decay[hd] : 0.f, len);
  const int h = lane >> 5, n = lane & 31;
  const bool before = c > 0 || carried;           // uniform
  const float* S = (P.ws != nullptr
                        ? P.ws + ((long)blockIdx.x * P.heads + hd) * (D * V) : kept);
  auto row_of = [&](int idx, int W) { return min(idx / (W / 8), len - 1); };
  DMStart start = {S, nullptr, 0, 0, 0.f, 0.f};
  if constexpr (GROUPS) start.init<D * V>(P, s, c, hd, S);
  ushort8_t qr[QP], kr[QP], vr[VP];
  float sr[SP][8], sy[SP][8];
#pragma unroll
  for (int i = 0; i < QP; ++i) {
    const int idx = tid + i * NT;
    qr[i] = dm_row(P.q + (long)(t0 + row_of(idx, D)) * P.q_stride + hd * D +
                   idx % (D / 8) * 8);
  }
  if (before) {
#pragma unroll
    for (int i = 0; i < SP; ++i) start.ask((tid + i * NT) * 8, sr[i]);
  }
  if (start.first != nullptr) {
#pragma unroll
    for (int i = 0; i < SP; ++i) start.ask_first((tid + i * NT) * 8, sy[i]);
  }
#pragma unroll
  for (int i = 0; i < QP; ++i) {
    const int idx = tid + i * NT;
    kr[i] = dm_row(P.k + (long)(t0 + row_of(idx, D)) * P.k_stride + hd * D +
                   idx % (D / 8) * 8);
  }
#pragma unroll
  for (int i = 0; i < VP; ++i) {
    const int idx = tid + i * NT;
    vr[i] = dm_row(P.v + (long)(t0 + row_of(idx, V)) * P.v_stride + hd * V +
                   idx % (V / 8) * 8);
  }
  if (tid <= DM_C) pw[tid] = dm_pow(P.decay[hd], tid);
#pragma unroll
  for (int i = 0; i < QP; ++i) {
    const int idx = tid + i * NT, r = idx / (D / 8), ch = idx % (D / 8);
    dm_u4 y = {{0u, 0u, 0u, 0u}};
    if (r < len) y = dm_act(qr[i]);
    *reinterpret_cast<dm_u4*>(lds + r * D + ((ch ^ mr_swz_rows<D>(r)) << 3)) = y;
  }
  if (before) {
#pragma unroll
    for (int i = 0; i < SP; ++i) {
      const int idx = tid + i * NT, r = idx / (V / 8), ch = idx % (V / 8);
      if (start.first != nullptr) start.join(idx * 8, sr[i], sy[i]);
      dm_split(sr[i], lds + KEYS + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3), IMG);
    }
  }
  __syncthreads();
  const bool on = qt * 32 < len;                  // uniform in a wave
  const int qi = qt * 32 + n;
  const int rbase = mr_row_base<D>(lane), vbase = mr_col_base<V>(lane) ^ (vt << 5);
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = *reinterpret_cast<const lds_bf16x8*>(
        (const lds_u16*)lds + qi * D + (((2 * ks + h) ^ mr_swz_rows<D>(qi)) << 3));
  // Products of the leading terms and those of the other two are summed apart, and the
  // leading ones of four steps (of two within the chunk) before they meet the large sum,
  // which then is rounded 6 times instead of 16. Error against 64 bits, 3 prompts of
  // 853-1657 tokens: 8.2e-8 -> 6.7e-8 (the recurrence: 7.1e-8).
  f32x16 acc[2] = {mr_zero(), mr_zero()};

  // ---- through the state before the chunk ------------------------------------
  if (before && on) {
#pragma unroll
    for (int d0 = 0; d0 < D; d0 += 64) {
      f32x16 z = mr_zero();
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const bf16x8 x = mr_cols<V>((const lds_u16*)lds + KEYS + t * IMG +
                                      (d0 + st * 16) * V + vbase);
          if (t == 0) z = mr_mma(x, qf[d0 / 16 + st], z);
          else acc[1] = mr_mma(x, qf[d0 / 16 + st], acc[1]);
        }
      acc[0] += z;
    }
    const float fade = pw[min(qi, DM_C - 1) + 1];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[0][r] *= fade;
      acc[1][r] *= fade;
    }
  }
  // ---- within the chunk --------------------------------------------------------
  unsigned odd = 0u;
  dm_u4 ka[QP], va[VP];
#pragma unroll
  for (int i = 0; i < QP; ++i) {
    ka[i] = dm_u4{{0u, 0u, 0u, 0u}};
    if ((tid + i * NT) / (D / 8) < len) ka[i] = dm_act(kr[i]);
  }
#pragma unroll
  for (int i = 0; i < VP; ++i) {
    va[i] = dm_u4{{0u, 0u, 0u, 0u}};
    if ((tid + i * NT) / (V / 8) < len) va[i] = dm_act(vr[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) odd |= dm_odd(va[i].x[j]);
  }
  if (before) __syncthreads();                    // the images are read
  unsigned short* vs = lds + VALS;
#pragma unroll
  for (int i = 0; i < QP; ++i) {
    const int idx = tid + i * NT, r = idx / (D / 8), ch = idx % (D / 8);
    *reinterpret_cast<dm_u4*>(lds + KEYS + r * D +
                              ((ch ^ mr_swz_rows<D>(r)) << 3)) = ka[i];
  }
#pragma unroll
  for (int i = 0; i < VP; ++i) {
    const int idx = tid + i * NT, r = idx / (V / 8), ch = idx % (V / 8);
    *reinterpret_cast<dm_u4*>(vs + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3)) = va[i];
  }
  // A weight of zero keeps a key out of a row unless its value is not finite: the
  // products see zero instead, and rows from that token on are NaN at the end.
  const bool any_lost = __syncthreads_or(odd != 0u);
  if (any_lost) {
    for (int i = tid; i < V; i += NT) lost[i] = DM_C;
    __syncthreads();
    for (int i = tid; i < DM_C * V; i += NT) {
      const int r = i / V, e = i % V;
      unsigned short* x = vs + r * V + (((e >> 3) ^ mr_swz_cols<V>(r)) << 3) +
                          (e & 7);
      if (dm_odd(*x) == 0u) continue;
      *x = 0;
      atomicMin(lost + e, r);
    }
    __syncthreads();
  }
  // the weights of keys 32 kt .. for queries 32 qt ..: tile qt (qt + 1) / 2 + kt
  typedef __attribute__((address_space(3))) bf16x8 lds_frag;
  lds_frag* wt = (lds_frag*)((lds_u16*)lds + WGTS) + qt * (qt + 1) / 2 * 6 * 64 + lane;
  if (on) {
    for (int kt = vt; kt <= qt; kt += NV) {
      // in two chains: a chunk of 16 tokens is no less precise than the recurrence
      f32x16 z = mr_zero(), z1 = mr_zero();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8 x = *reinterpret_cast<const lds_bf16x8*>(
            (const lds_u16*)lds + KEYS + (rbase ^ (ks << 4)) + kt * 32 * D);
        if (ks % 2 == 0) z = mr_mma(x, qf[ks], z);
        else z1 = mr_mma(x, qf[ks], z1);
      }
      z += z1;
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
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int st = 0; st < 2; ++st) wt[(kt * 6 + t * 2 + st) * 64] = p[t][st];
    }
  }
  __syncthreads();
  auto outputs = [&] {
    for (int kt = 0; kt <= qt; ++kt) {
      f32x16 y = mr_zero();
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 x =
            mr_cols<V>((const lds_u16*)vs + vbase + (kt * 32 + st * 16) * V);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const bf16x8 p = wt[(kt * 6 + t * 2 + st) * 64];
          if (t == 0) y = mr_mma(x, p, y);
          else acc[1] = mr_mma(x, p, acc[1]);
        }
      }
      // the nearest keys weigh most: what is small meets what they do not add to
      if (kt == qt) acc[0] += acc[1];
      acc[0] += y;
    }
    if (qi >= len) return;
    if (any_lost) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (lost[vt * 32 + 8 * (r >> 2) + 4 * h + (r & 3)] <= qi) acc[0][r] = NAN;
    }
    float* o = P.out + ((long)(t0 + qi) * P.heads + hd) * V + vt * 32 + 4 * h;
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<float4*>(o + 2 * r) =
          make_float4(acc[0][r], acc[0][r + 1], acc[0][r + 2], acc[0][r + 3]);
  };
  if (on) outputs();
  if constexpr (LAST) {
    if (slot < 0) return;                         // uniform
    // ---- the state: this wave's 32 keys' columns (dt) by 32 values' -------------
    const int dt = w & 3;
    const bool mine = dt < D / 32;
    float* st = kept + (long)(dt * 32 + 4 * h) * V + vt * 32 + n;
    float x0[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      x0[r] = carried && mine ? st[(8 * (r >> 2) + (r & 3)) * V] : 0.f;
    const float by = carried ? pw[late.end + 1] : 0.f;
    unsigned short late_k[DM_LATE], late_v[DM_LATE];
#pragma unroll
    for (int i = 0; i < DM_LATE; ++i) {
      const int t = max(len - DM_LATE + i, 0), d = (dt & (D / 32 - 1)) * 32 + n;
      late_k[i] = lds[KEYS + t * D + (((d >> 3) ^ mr_swz_rows<D>(t)) << 3) + (d & 7)];
    }
    __syncthreads();                              // weights and values are read
    // a row's pieces are a wave's, which has read them all when it writes the first
#pragma unroll
    for (int i = 0; i < QP; ++i) {
      const int idx = tid + i * NT, r = idx / (D / 8), ch = idx % (D / 8);
      const dm_u4 z = *reinterpret_cast<const dm_u4*>(
          lds + KEYS + r * D + ((ch ^ mr_swz_rows<D>(r)) << 3));
      float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (r < late.from) {
        const float wgt = pw[late.end - r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[2 * j] = __uint_as_float(z.x[j] << 16) * wgt;
          x[2 * j + 1] = __uint_as_float(z.x[j] & 0xffff0000u) * wgt;
        }
      }
      dm_split(x, lds + r * D + ((ch ^ mr_swz_cols<D>(r)) << 3), DM_C * D);
    }
    if (any_lost) {                               // values as they were
      for (int i = tid; i < DM_C * V / 8; i += NT) {
        const int r = i / (V / 8), ch = i % (V / 8);
        dm_u4 y = {{0u, 0u, 0u, 0u}};
        if (r < len)
          y = dm_act(dm_row(P.v + (long)(t0 + r) * P.v_stride + hd * V + ch * 8));
        *reinterpret_cast<dm_u4*>(vs + r * V + ((ch ^ mr_swz_cols<V>(r)) << 3)) = y;
      }
    }
    __syncthreads();
    if (!mine) return;
    const int cbase = mr_col_base<D>(lane) ^ (dt << 5);
#pragma unroll
    for (int i = 0; i < DM_LATE; ++i) {
      const int t = max(len - DM_LATE + i, 0), e = vt * 32 + n;
      late_v[i] = vs[t * V + (((e >> 3) ^ mr_swz_cols<V>(t)) << 3) + (e & 7)];
    }
    acc[0] = acc[1] = mr_zero();
    // leading and other terms apart, without the late tokens
#pragma unroll 4
    for (int k = 0; k < len; k += 16) {
      const bf16x8 y = mr_cols<V>((const lds_u16*)vs + vbase + k * V);
#pragma unroll
      for (int t = 0; t < 3; ++t)
        acc[t > 0] = mr_mma(mr_cols<D>((const lds_u16*)lds + t * DM_C * D + k * D + cbase),
                            y, acc[t > 0]);
    }
    late.join(acc, x0, by, late_k, late_v, h);
#pragma unroll
    for (int r = 0; r < 16; ++r) st[(8 * (r >> 2) + (r & 3)) * V] = acc[0][r];
  }
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
// recurrence | here, tokens), fresh, continued: 128 x 128, 16 states: 6 8.1 9.0 | 7.9 10.3, 8
// 9.7 10.6 | 8.6 10.2; 64: 5 8.8 9.5 | 8.5 10.8, 7 10.2 11.1 | 8.6 10.7; 128: 5 10.4 12.4 |
// 9.4 11.6; 256: 4 14.8 19.0 | 10.7 14.7; fresh ones, 1024: 2 27.3 | 34.2, 4 37.2 | 34.3. 64 x
// 64, 64 states: 6 7.5 7.7 | 7.3 7.5; 256: 4 7.6 9.1 | 7.4 8.1, 5 8.8 10.0 | 7.6 8.0; 1024: 2
// 15.3 | 16.7, 3 17.2 | 16.8. 64 x 128, 256: 4 11.9 14.8 | 8.4 9.5; 128 x 64, 256: 4 9.2 10.9 |
// 9.0 10.9, 6 11.3 13.1 | 9.0 11.0; 1024: 4 22.9 | 25.6, 6 28.9 | 25.6. Whatever the
// length, outputs and states are no further off 64 bits here (DMLate), heads of 0.75 to
// 0.996 or of 0.5 to 0.996 (184 sizes, parts of the recurrence's: 0.88 and 0.82, at most
// 1.01); where all of them decay to 0.7 or less within a token, states 1.03, at most 1.09.
bool decay_attn_short(long longest, long states, int D, int V) {
  const long wgs = states * (V / 16);
  const int most = wgs <= 128 ? 7 : wgs <= 512 ? 6                    // tokens
                   : wgs <= 2048 ? (D == 128 || wgs <= 1024 ? 4 : 3)
                   : D == 128 ? 3 : 2;
  return longest <= most;
}

// Groups of chunks that walk, in the place of sum and scan, cuts a sequence into; 0: sum
// and scan. Walk's time is 3 us and 2.9 a chunk of the longest sequence's groups, more with
// two workgroups on a CU; theirs a start and so much for each (chunk, head). Measured
// (us, both kernels' | chunks of the longest, units), 128 x 128: 15 | 3, 48; 17 | 4, 128;
// 27 | 5, 480; 30 | 13, 528; 38 | 8, 1024; 45 | 13, 1056; 51 | 7, 1150. 64 x 128 and back:
// 12 | 4, 68; 15 | 5, 144; 17 | 3, 192; 22 | 4, 368; 27 | 3, 496. 64 x 64: 10 | 3, 48; 12 |
// 3, 176; 18 | 5, 448; 22 | 6, 928.
//   More than one group leaves `out` more to read, a record for each group before a
// chunk's, and the last states to make: 0.6 us and 4.5 ns a unit for each, 9 ns by four
// waves, which have no registers left for it (1200, 1300 and 1323 tokens of 16 heads: 66.0
// by sum and scan, 71.8 | 72.1 | 73.3 by groups; 2 of 1000, 32 heads, 69.9 | 71.1). 4 more where
// workgroups of 16 waves, one to a CU, leave none free for those. Us in all, 128 x 128, sum
// and scan | one group | two | three | four: 16 heads, 300 tokens 29.6 | 25.4 | 23.4 | 21.2 |
// 21.2, 500 30.3 | 29.7 | 24.7 | 24.8 | 23.7, 800 34.7 | 39.4 | 33.3 | 31.2 | 29.5, 1200 37.0 |
// 50.1 | 38.8 | 36.0 | 34.8, but 2000 40.5 | 72.2 | 53.6 | 48.9 | 45.7; 2 x 500-900 39.0 | 39.7 |
// 34.7 | 34.6 | 34.5, 4 x 500-1200 60.0 | 59.2 | 56.8 | 57.7 | 60.8; 32 heads, 400 35.1 | 30.5 |
// 27.2 | 27.3 | 28.7, but 1000 40.5 | 48.8 | 42.1 | 43.6 | 43.3.
int decay_attn_mfma_groups(long longest, long tokens, int n_seqs, int heads, int D,
                           int V) {
  const long chunks = (longest + DM_C - 1) / DM_C, chains = (long)n_seqs * heads;
  if (chunks <= 1) return 0;
  const long units = (2 * tokens / DM_C + n_seqs) * heads / 2;
  const long there = D + V == 256 ? 14000 + 30 * units
                     : D + V == 192 ? 9000 + 40 * units : 8500 + 18 * units;   // ns
  if (D + V < 256) return 3000 + 2900 * chunks < there;
  const long grid = decay_attn_mfma_chunks(tokens, n_seqs) * heads;
  const long crowd = grid <= 256 && grid + chains > 256 ? 4000 : 0;
  auto cost = [&](long g) {
    const long wgs = 4 * chains * g;
    const long chunk = wgs <= 256 ? 2900 : wgs <= 512 ? 2200 + wgs * 3 : wgs * 7;
    return 3000 + (chunks + g - 1) / g * chunk +
           (g > 1 ? crowd + (g - 1) * (600 + units * (grid <= 256 ? 9 : 18) / 2) : 0);
  };
  // not for a little: 5 of 365 to 850 tokens 60.7 by sum and scan, 63.2 by one group
  long at = cost(1) < there - there / 16, best = at ? cost(1) : there;
  best -= best / 8;
  for (int g = 2; g <= 4 && g <= chunks; ++g)
    if (cost(g) < best) best = cost(g), at = g;
  return (int)at;
}

// Whether out moves the states of sequences of a chunk each, in workgroups of 16 or 8
// waves. Instead: out by four waves (beyond 256 states) and sum. Measured (us, two kernels |
// one; fresh, continued; states), 128 x 128: 64 tokens 64 17.8 28.1 | 11.0 13.8, 272 26.5
// 33.8 | 23.2 29.7, 1024 59.4 81.2 | 53.4 76.8, 4096 207 293 | 184 255, 20 tokens 272 19.2
// 24.8 | 17.9 24.1, 4096 142 230 | 141 191. 64 x 128: 128 tokens 280 29.4 33.6 | 27.8 31.9,
// 4096 241 292 | 223 268, 40 tokens 800 32.7 42.3 | 31.9 39.5, 20 tokens 1024 27.4 38.0 | 28.0
// 35.2, 4096 93 136 | 104 131. 128 x 64: 128 tokens 280 30.7 34.1 | 27.8 33.1, 448 33.5 38.4 |
// 30.3 36.7, 520 42.8 49.7 | 41.3 49.7, 20 tokens 320 15.8 18.5 | 16.0 19.6. 64 x 64: 128
// tokens 256 18.0 20.7 | 13.1 15.6, 320 22.2 24.4 | 22.0 24.8, 768 32.4 36.9 | 34.3 39.4.
static bool decay_attn_one(long longest, long states, int D, int V) {
  if (states <= 256 || (D == 128 && V == 128)) return true;
  if (V == 128) return states <= 512 || longest > 32;
  return D == 128 && states <= 448 && longest > 32;
}

// How a batch of prompt rows goes: groups of chunks that are walked (0: sum and scan, if
// any has more than a chunk); whether out moves the states of a chunk each; whether its
// workgroups have 8 or 16 waves.
void decay_attn_mfma_way(long longest, long tokens, int n_seqs, int heads, int D, int V,
                         int* groups, bool* one, bool* wide) {
  *groups = decay_attn_mfma_groups(longest, tokens, n_seqs, heads, D, V);
  *one = longest <= DM_C && decay_attn_one(longest, (long)n_seqs * heads, D, V);
  const long units =
      (longest > DM_C ? decay_attn_mfma_chunks(tokens, n_seqs) : n_seqs) * heads;
  *wide = *one || units <= 256;
}

// D, V in {64, 128}; rows 16 B aligned. ws null: no sequence has more than
// DM_C tokens. longest: tokens of a sequence at most
void launch_decay_attn_mfma(float* out, const unsigned short* q,
                            const unsigned short* k, const unsigned short* v,
                            const float* decay, float* state, const int* slots,
                            const int* cu_q, const int* ctx_lens, long tokens,
                            int n_seqs, int heads, int D, int V, long q_stride,
                            long k_stride, long v_stride, float* ws,
                            long longest, hipStream_t st) {
  if (n_seqs == 0) return;
  int groups;
  bool one, wide;
  decay_attn_mfma_way(longest, tokens, n_seqs, heads, D, V, &groups, &one, &wide);
  const DMArgs P = {out, q, k, v, q_stride, k_stride, v_stride, decay, state,
                    ws, slots, cu_q, ctx_lens, n_seqs, heads,
                    std::max(groups, 1),
                    decay_attn_mfma_chunks(tokens, n_seqs)};
  const dim3 grid(
      (unsigned)(ws ? decay_attn_mfma_chunks(tokens, n_seqs) : n_seqs), heads);
  // with those that make the last states (dm_last_state)
  const dim3 grid_out(
      grid.x, heads + (groups > 1 ? (n_seqs * heads + grid.x - 1) / grid.x : 0));
#define DM_SUM_(DD, VV, ONE)                                                  \
  hipLaunchKernelGGL((decay_sum_mfma_kernel<DD, VV, ONE>), grid, dim3(256), 0, st, P)
#define DM_SUM(DD, VV) DM_SUM_(DD, VV, false)
// (128 x 128: decay_attn_one)
#define DM_SUM_ONE(DD, VV)                                                    \
  do {                                                                        \
    if constexpr (DD + VV < 256) DM_SUM_(DD, VV, true);                       \
  } while (0)
#define DM_WALK(DD, VV)                                                       \
  hipLaunchKernelGGL((decay_walk_mfma_kernel<DD, VV>),                        \
                     dim3((unsigned)(((long)n_seqs * heads + 7) / 8 * 8 *     \
                                     (DD / 64) * (VV / 64) * P.groups)),       \
                     dim3(512), 0, st, P)
#define DM_WIDE(DD, VV, GROUPS, LAST)                                         \
  hipLaunchKernelGGL((decay_out_wide_kernel<DD, VV, GROUPS, LAST>), grid_out, \
                     dim3(8 * VV), 0, st, P)
#define DM_OUT_(DD, VV, GROUPS)                                               \
  do {                                                                        \
    if (wide)                                                                 \
      DM_WIDE(DD, VV, GROUPS, false);                                         \
    else                                                                      \
      hipLaunchKernelGGL((decay_out_mfma_kernel<DD, VV, GROUPS>), grid_out,   \
                         dim3(256), 0, st, P);                                \
  } while (0)
#define DM_OUT(DD, VV) DM_OUT_(DD, VV, false)
#define DM_BY_SIZE(CALL)                                                      \
  do {                                                                        \
    if (D == 128) { if (V == 128) CALL(128, 128); else CALL(128, 64); }       \
    else { if (V == 128) CALL(64, 128); else CALL(64, 64); }                  \
  } while (0)
#define DM_ALL(DD, VV) DM_WIDE(DD, VV, false, true)
  if (ws == nullptr) {                            // a chunk each
    if (one) {
      DM_BY_SIZE(DM_ALL);
    } else {
      DM_BY_SIZE(DM_OUT);
      DM_BY_SIZE(DM_SUM_ONE);
    }
    return;
  }
  if (groups > 0) {
    DM_BY_SIZE(DM_WALK);
  } else {
    DM_BY_SIZE(DM_SUM);
    const long per_head = (long)D * V, per_seq = per_head * heads;
    hipLaunchKernelGGL((chunk_scan_kernel<DM_C>),
                       dim3((unsigned)((per_seq + 255) / 256), n_seqs),
                       dim3(256), 0, st, ws, state, decay, slots, cu_q, ctx_lens,
                       heads, per_head, true);
  }
  if (groups > 1) DM_OUT_(128, 128, true);       // the only ones with groups
  else DM_BY_SIZE(DM_OUT);
#undef DM_BY_SIZE
#undef DM_OUT
#undef DM_ALL
#undef DM_WIDE
#undef DM_OUT_
#undef DM_WALK
#undef DM_SUM
#undef DM_SUM_ONE
#undef DM_SUM_
}

}  // namespace hyb
}  // namespace xllm
