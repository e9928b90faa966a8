// Fused rotary position embedding (RoPE) for MI355X (gfx950).
//
// NeoX / Llama "rotate-half" layout, applied in-place to q and k, which may
// be strided row views into a fused qkv projection output (no host-side
// .contiguous() copies). One 64-lane wave per (token, head) pair; the grid
// is sized by total wave-work so decode batches fill the chip.
//
// cos/sin precomputed host-side as f32 [max_pos, rot_dim] (first half cos):
// on-device trig would turn this memory-bound op VALU-bound (guide App. B).
//
// Parity: the reference engine's fused RoPE.
#include "common.h"

namespace xllm {

__global__ void rope_kernel(
    unsigned short* __restrict__ q,      // [T, n_qheads, D] rows stride q_stride
    unsigned short* __restrict__ k,      // [T, n_kheads, D] rows stride k_stride
    const long* __restrict__ positions,  // [T]
    const float* __restrict__ cos_sin,   // [max_pos, rot_dim]
    const int n_qheads, const int n_kheads,
    const int head_dim, const int rot_dim,
    const long q_stride, const long k_stride,
    const int T) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int waves_per_block = blockDim.x >> 6;
  const int total_heads = n_qheads + n_kheads;
  const long total_work = (long)T * total_heads;
  const int half = rot_dim / 2;

  for (long wk = blockIdx.x * (long)waves_per_block + wid; wk < total_work;
       wk += (long)gridDim.x * waves_per_block) {
    const int token = (int)(wk / total_heads);
    const int h = (int)(wk % total_heads);
    unsigned short* base =
        (h < n_qheads) ? q + token * q_stride + (long)h * head_dim
                       : k + token * k_stride + (long)(h - n_qheads) * head_dim;
    const float* cs = cos_sin + positions[token] * rot_dim;
    for (int i = lane; i < half; i += 64) {
      const float c = cs[i];
      const float s = cs[half + i];
      const float x1 = bf16_to_f32(base[i]);
      const float x2 = bf16_to_f32(base[i + half]);
      base[i] = f32_to_bf16(x1 * c - x2 * s);
      base[i + half] = f32_to_bf16(x2 * c + x1 * s);
    }
  }
}

void launch_rope(unsigned short* q, unsigned short* k, const long* positions,
                 const float* cos_sin, int T, int n_qheads, int n_kheads,
                 int head_dim, int rot_dim, long q_stride, long k_stride,
                 hipStream_t stream) {
  const long waves = (long)T * (n_qheads + n_kheads);
  long g = (waves + 3) / 4;  // 4 waves per 256-thread block
  if (g > 2048) g = 2048;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(rope_kernel, dim3((unsigned)g), dim3(256), 0, stream, q,
                     k, positions, cos_sin, n_qheads, n_kheads, head_dim,
                     rot_dim, q_stride, k_stride, T);
}

// Fused RoPE + KV-cache scatter: one pass ropes q in place, ropes k and
// writes it straight into the paged cache together with v (replaces the
// separate rope + reshape_and_cache launches and k's LDS->HBM round trip).
__global__ void fused_rope_cache_kernel(
    unsigned short* __restrict__ q,            // [T, n_q, D] strided rows
    const unsigned short* __restrict__ k,      // [T, n_kv, D] strided rows
    const unsigned short* __restrict__ v,      // [T, n_kv, D] strided rows
    unsigned short* __restrict__ k_cache,      // [blocks, n_kv, bs, D]
    unsigned short* __restrict__ v_cache,
    const long* __restrict__ positions,  // [T], or [3, T] when ms0 > 0
    const long* __restrict__ slot_mapping,     // [T] (-1 = skip cache write)
    const float* __restrict__ cos_sin,         // [max_pos, rot]
    const int n_q, const int n_kv, const int D, const int rot,
    const long q_stride, const long kv_stride, const int block_size,
    const int T,
    // M-RoPE (Qwen2-VL): cumulative frequency-section bounds; freq i takes
    // its position from row 0 (i < ms0: temporal), 1 (i < ms1: height) or
    // 2 (width) of the [3, T] positions. ms0 == 0 disables (1-D rope).
    const int ms0, const int ms1) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int wpb = blockDim.x >> 6;
  const int total_heads = n_q + 2 * n_kv;  // q-rope | k-rope+store | v-store
  const long total_work = (long)T * total_heads;
  const int half = rot / 2;

  for (long wk = blockIdx.x * (long)wpb + wid; wk < total_work;
       wk += (long)gridDim.x * wpb) {
    const int token = (int)(wk / total_heads);
    const int h = (int)(wk % total_heads);
    const long slot = slot_mapping[token];
    const float* cs = cos_sin + positions[token] * rot;
    auto cs_at = [&](int i) -> const float* {
      if (ms0 == 0) return cs;
      const int sec = i < ms0 ? 0 : (i < ms1 ? 1 : 2);
      return cos_sin + positions[(long)sec * T + token] * rot;
    };
    if (h < n_q) {                       // rope q in place
      unsigned short* base = q + token * q_stride + (long)h * D;
      for (int i = lane; i < half; i += 64) {
        const float* cf = cs_at(i);
        const float c = cf[i], s = cf[half + i];
        const float x1 = bf16_to_f32(base[i]);
        const float x2 = bf16_to_f32(base[i + half]);
        base[i] = f32_to_bf16(x1 * c - x2 * s);
        base[i + half] = f32_to_bf16(x2 * c + x1 * s);
      }
    } else if (h < n_q + n_kv) {         // rope k -> cache
      if (slot < 0) continue;
      const int kh = h - n_q;
      const unsigned short* src = k + token * kv_stride + (long)kh * D;
      unsigned short* dst =
          k_cache + (((slot / block_size) * n_kv + kh) * block_size +
                     slot % block_size) * (long)D;
      for (int i = lane; i < half; i += 64) {
        const float* cf = cs_at(i);
        const float c = cf[i], s = cf[half + i];
        const float x1 = bf16_to_f32(src[i]);
        const float x2 = bf16_to_f32(src[i + half]);
        dst[i] = f32_to_bf16(x1 * c - x2 * s);
        dst[i + half] = f32_to_bf16(x2 * c + x1 * s);
      }
      for (int i = rot + lane; i < D; i += 64) dst[i] = src[i];
    } else {                             // copy v -> cache (16 B vectors)
      if (slot < 0) continue;
      const int vh = h - n_q - n_kv;
      const unsigned short* src = v + token * kv_stride + (long)vh * D;
      unsigned short* dst =
          v_cache + (((slot / block_size) * n_kv + vh) * block_size +
                     slot % block_size) * (long)D;
      for (int i = lane * 8; i < D; i += 64 * 8)
        *reinterpret_cast<ushort8_t*>(dst + i) =
            *reinterpret_cast<const ushort8_t*>(src + i);
    }
  }
}

// The same where whole heads are rotated and everything is in steps of eight: a lane
// has eight pairs, 16 B each, and its loads do not wait for each other (but for
// cos and sin, which the position leads to). One token per row of workgroups, which
// are no larger than its lanes.
// 32/8 heads of 128, (one pair per lane, a wave per head and token) -> here: 8192
// tokens 92.8 -> 33.4 us, 2048 27.1 -> 8.3, 300 5.10 -> 3.13, 128 3.36 -> 2.67 (an empty
// launch: 2.0). That kernel stays for partial rotary, for rows that are not aligned
// and for few tokens.
__global__ void fused_rope_cache8_kernel(
    unsigned short* __restrict__ q, const unsigned short* __restrict__ k,
    const unsigned short* __restrict__ v, unsigned short* __restrict__ k_cache,
    unsigned short* __restrict__ v_cache, const long* __restrict__ positions,
    const long* __restrict__ slot_mapping, const float* __restrict__ cos_sin,
    const int n_q, const int n_kv, const int D, const long q_stride,
    const long kv_stride, const int block_size, const int T, const int ms0,
    const int ms1) {
  const long token = blockIdx.x;
  long pos = positions[token];
  const long slot = slot_mapping[token];
  const unsigned half = D / 2, lanes = half / 8;    // lanes of a head
  const unsigned at = blockIdx.y * blockDim.x + threadIdx.x;
  const int h = at / lanes, i = (at - h * lanes) * 8;
  if (h >= n_q + 2 * n_kv) return;
  const int kvh = h - n_q < n_kv ? h - n_q : h - n_q - n_kv;
  const bool is_q = h < n_q, is_v = h >= n_q + n_kv;
  const unsigned short* src =
      is_q ? q + token * q_stride + (long)h * D
           : (is_v ? v : k) + token * kv_stride + (long)kvh * D;
  ushort8_t a = *reinterpret_cast<const ushort8_t*>(src + i);
  ushort8_t b = *reinterpret_cast<const ushort8_t*>(src + i + half);
  if (ms0 != 0 && i >= ms0) pos = positions[(i < ms1 ? 1L : 2L) * T + token];
  const float* cs = cos_sin + pos * D + i;
  if (!is_v) {
    float c[8], s[8];
#pragma unroll
    for (int j = 0; j < 8; j += 4) {
      const float4 cv = *reinterpret_cast<const float4*>(cs + j);
      const float4 sv = *reinterpret_cast<const float4*>(cs + half + j);
      c[j] = cv.x, c[j + 1] = cv.y, c[j + 2] = cv.z, c[j + 3] = cv.w;
      s[j] = sv.x, s[j + 1] = sv.y, s[j + 2] = sv.z, s[j + 3] = sv.w;
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float x1 = bf16_to_f32(a.x[j]), x2 = bf16_to_f32(b.x[j]);
      a.x[j] = f32_to_bf16(x1 * c[j] - x2 * s[j]);
      b.x[j] = f32_to_bf16(x2 * c[j] + x1 * s[j]);
    }
  }
  unsigned short* dst;
  if (is_q) {
    dst = q + token * q_stride + (long)h * D;
  } else {
    if (slot < 0) return;
    const long blk = slot >> 31 == 0 ? (unsigned)slot / (unsigned)block_size
                                     : slot / block_size;
    dst = (is_v ? v_cache : k_cache) +
          ((blk * n_kv + kvh) * block_size + (slot - blk * block_size)) *
              (long)D;
  }
  *reinterpret_cast<ushort8_t*>(dst + i) = a;
  *reinterpret_cast<ushort8_t*>(dst + i + half) = b;
}

void launch_fused_rope_cache(unsigned short* q, const unsigned short* k,
                             const unsigned short* v, unsigned short* k_cache,
                             unsigned short* v_cache, const long* positions,
                             const long* slot_mapping, const float* cos_sin,
                             int T, int n_q, int n_kv, int D, int rot,
                             long q_stride, long kv_stride, int block_size,
                             int ms0, int ms1, hipStream_t stream) {
  // 16 B accesses of q, k, v, the caches and the table; rows of the M-RoPE
  // sections in steps of eight. Few lanes stay with the other kernel, which finds
  // its place without a division: 3 heads of 64, 1000 tokens 3.0 | 3.3 us here, 48
  // heads of 80, 8 tokens 2.6 | 2.8, 32 2.7 | 2.9, 64 3.0 | 2.9.
  const auto on16 = [](const void* p) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0;
  };
  const int lanes = (n_q + 2 * n_kv) * (D / 16);       // of a token
  if ((long)T * lanes >= 16384 && rot == D && D % 16 == 0 && q_stride % 8 == 0 &&
      kv_stride % 8 == 0 && ms0 % 8 == 0 && ms1 % 8 == 0 && on16(q) &&
      on16(k) && on16(v) && on16(k_cache) && on16(v_cache) && on16(cos_sin)) {
    const int wg = lanes < 256 ? (lanes + 63) / 64 * 64 : 256;
    const dim3 grid((unsigned)T, (unsigned)((lanes + wg - 1) / wg));
    hipLaunchKernelGGL(fused_rope_cache8_kernel, grid, dim3(wg), 0, stream, q,
                       k, v, k_cache, v_cache, positions, slot_mapping, cos_sin,
                       n_q, n_kv, D, q_stride, kv_stride, block_size, T, ms0,
                       ms1);
    return;
  }
  const long waves = (long)T * (n_q + 2 * n_kv);
  long g = (waves + 3) / 4;
  if (g > 2048) g = 2048;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(fused_rope_cache_kernel, dim3((unsigned)g), dim3(256), 0,
                     stream, q, k, v, k_cache, v_cache, positions,
                     slot_mapping, cos_sin, n_q, n_kv, D, rot, q_stride,
                     kv_stride, block_size, T, ms0, ms1);
}

}  // namespace xllm
