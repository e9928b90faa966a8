// Helpers of the kernels built on v_mfma_f32_32x32x16_bf16 (gfx950).
//
// Fragments (lane l, h = l >> 5):
//   A[l&31][h*8 + j], B[h*8 + j][l&31], C[8*(r>>2) + 4h + (r&3)][l&31]
//
// A product S^T = K Q^T leaves 16 entries of ONE query's row in a lane. Feeding
// key mr_key(m) as A row m makes those the keys 16t + 8h + 0..7 (t = r >> 3)
// that the B operand of step t of the next product O^T += V^T P^T wants of that
// lane, so P stays where it is.
//
// LDS images are row-major [row][W] with the 16 B chunks of a row permuted by
// the row: chunk c sits at c ^ mr_swz_rows(row) where rows are read whole (A
// rows, ds_read_b128), at c ^ mr_swz_cols(row) where columns are
// (ds_read_b64_tr_b16). Either way the lanes that share an LDS cycle touch
// every bank once, without padding.
#pragma once
#include "common.h"

namespace xllm {

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bfx2;
typedef __attribute__((ext_vector_type(2))) float fx2;

typedef __attribute__((address_space(3))) unsigned short lds_u16;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;

// larger / sum of a lane's and its partner's (l ^ 32) value
XLLM_DEV float pair_max(float v) {
  const unsigned u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
XLLM_DEV float pair_sum(float v) {
  const unsigned u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// two fp32 rounded to bf16 (nearest even), the first in the low half
XLLM_DEV unsigned pack_bf16(float a, float b) {
  const fx2 f = {a, b};
  const bfx2 x = __builtin_convertvector(f, bfx2);
  return __builtin_bit_cast(unsigned, x);
}
// a, b <- what the packed pair leaves of them (exact)
XLLM_DEV void drop_bf16(float& a, float& b, unsigned u) {
  a -= __uint_as_float(u << 16);
  b -= __uint_as_float(u & 0xffff0000u);
}

// key that A row m stands for
XLLM_DEV int mr_key(int m) {
  return ((m >> 4) << 4) | (((m >> 2) & 1) << 3) | (((m >> 3) & 1) << 2) |
         (m & 3);
}
// key of C register r, lane half h, within the 32 keys
XLLM_DEV int mr_key_of(int r, int h) {
  return 16 * (r >> 3) + 8 * h + 4 * ((r >> 2) & 1) + (r & 3);
}
template <int W> XLLM_DEV int mr_swz_rows(int row) {
  static_assert(W == 64 || W == 128, "");
  return W == 128 ? row & 15 : (row >> 1) & 7;
}
template <int W> XLLM_DEV int mr_swz_cols(int row) {
  static_assert(W == 64 || W == 128, "");
  return W == 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2;
}
// Row reads: element offset of chunk h of A row c32; step ks: ^ (ks << 4), 32
// rows on: + 32 * W
template <int W> XLLM_DEV int mr_row_base(int lane) {
  const int km = mr_key(lane & 31);
  return km * W + (((lane >> 5) ^ mr_swz_rows<W>(km)) << 3);
}
// Column reads: column tile ct (32 wide): ^ (ct << 5), 16 rows on: + 16 * W
template <int W> XLLM_DEV int mr_col_base(int lane) {
  const int i = lane & 15, row = 8 * (lane >> 5) + (i >> 2);
  return row * W + ((lane >> 4) & 1) * 16 + (i & 3) * 4 +
         (mr_swz_cols<W>(row) << 3);
}
// 8 rows (of 16 from the base on) of one column: an A or a B operand
template <int W> XLLM_DEV bf16x8 mr_cols(const lds_u16* p) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
  const s16x4 hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * W));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// The same where the caller has waited for what it reads: through a pointer without
// alias information the compiler waits for all loads to LDS first.
template <int W>
XLLM_DEV bf16x8 mr_cols_own(const lds_u16* __restrict__ p) {
  return mr_cols<W>(p);
}
// `bytes` of memory for loads to LDS. Those through global addresses are flat
// instructions to the compiler, which from then on lets no LDS read pass another:
// every use of one waits for all.
XLLM_DEV __amdgpu_buffer_rsrc_t mr_buffer(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}
// 16 bytes per lane, in lane order from dst on; zeros from out of the bounds
XLLM_DEV void mr_to_lds(__amdgpu_buffer_rsrc_t src, unsigned off,
                        unsigned short* dst, unsigned base = 0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_void*)dst, 16, off, base,
                                           0, 0);
}
// the same to registers
XLLM_DEV uint4 mr_load(__amdgpu_buffer_rsrc_t src, unsigned off) {
  typedef __attribute__((ext_vector_type(4))) unsigned u4;
  const u4 v = __builtin_amdgcn_raw_buffer_load_b128(src, off, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}
XLLM_DEV f32x16 mr_zero() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = 0.0f;
  return z;
}
XLLM_DEV f32x16 mr_mma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace xllm
