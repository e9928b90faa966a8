// Options of the products of linear.hip.
#pragma once

namespace xllm {

// What a product does with its rows on the way in and out, by bits of MODE.
// LN_SCALE: x holds the rows of an RMS norm without their factors, which come from the
// sums of their squares' parts: results times 1 / sqrt(sum / K + eps).
// LN_ADD: results join the residual before either is rounded; y gets the new residual times the norm's
// weights (the rows of the next product but for their factors), sums the squares of
// this tile's columns. So a norm needs no launch of its own between two products: 4.6 us
// of a decode step, 3.4 of a prompt's, for 1.5 more in the two products. 8 layers, 24
// rows of 4096: 701 -> 677 us, 300 of 2048 589 -> 563. Of the norm's and the gate's own
// roundings the residual's and the rows' are left, the sums' in between are not made:
// error against 64 bits 0.0189 -> 0.0158 and 0.0132 -> 0.0118.
// LN_ROPE, heads of 128: W = [queries | keys | values] by heads; y [M, queries] gets
// queries rotated by their rows' positions, the caches keys (rotated) and values. A
// tile has columns of one half of a head and their partners of the other one. A launch
// less, 4.0 us of 300 rows and 4.7 of 24, for 0.5 to 1.5 more in the product: 548 -> 526 us,
// 675 -> 657.
enum { LN_GATE = 1, LN_SCALE = 2, LN_ADD = 4, LN_ROPE = 8 };
constexpr int LN_HEAD = 128;
struct LinearEnds {
  const float* squares = nullptr;            // [M][n_squares]
  int n_squares = 0;                         // a multiple of 4, at most 256, 64 (tiles)
  float eps = 0.0f;
  unsigned short* residual = nullptr;        // [M, N]
  const unsigned short* norm = nullptr;      // [N]
  float* sums = nullptr;                     // [M][tiles of N]
  const long* positions = nullptr;           // [M]
  const long* slots = nullptr;               // [M], negative: no row in the caches
  const float* cos_sin = nullptr;            // [positions][64 cos, 64 sin]
  unsigned short* k_cache = nullptr;         // [blocks, n_kv, block, 128]
  unsigned short* v_cache = nullptr;
  int n_q = 0, n_kv = 0, block = 0;
};

}  // namespace xllm
