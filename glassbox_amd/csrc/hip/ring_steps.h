// The k-steps of the ring kernel (gemm_bf16.hip), where each begins in a slice of k and which half of it counts as zeros, and the
// heights of its tiles.
// Plain C++, without the device's headers, so that the arithmetic can be checked on the host for every slice.
#pragma once

namespace gb {

constexpr int RBK = 64;           // k of a k-step
constexpr int RING_K = 32;        // a slice is a whole number of these (a last k-step may be half of one)
constexpr int RING_MIN_K = 128;   // and the row it is cut from at least so long

constexpr int ring_steps(int K) { return (K + RBK - 1) / RBK; }

// Where a slice of K is an odd number of halves its last k-step begins 32 earlier, on what the step before has summed (or, in
// a slice of 32, on the slice before): that half counts as zeros.  A slice of 32 at the head of the row has nothing before it:
// its k-step begins with it, and the other half, which is the next slice's, counts as zeros.
constexpr int ring_step_at(int s, int K, bool head) {
  return s * RBK < K - RBK ? s * RBK : head && K < RBK ? 0 : K - RBK;
}
// 0 or 1, or -1 where the last k-step is whole
constexpr int ring_dead_half(int K, bool head) { return K % RBK == 0 ? -1 : head && K < RBK ? 1 : 0; }

// The heights of a product's tiles.  One workgroup fills a compute unit, so tiles go in rounds of 256, and a last round of few
// costs as much as a full one: 6,151 rows of 4,096 columns are 25 x 16 = 400 tiles of 256, two rounds of which a quarter is idle,
// but 30 x 16 = 480 of 192 and 224.  So the rows are dealt evenly to a number of tiles (two heights, 32 apart, the taller ones
// first), the number by an estimate of the rounds' times.  Measured (130 products of 500 to 8,192 rows, each with several
// numbers of tiles; within 5 % from a k of 2,048 on): a k-step of a round of n tiles of 32 h rows takes 0.0806 us (h + 1.5)
// (1 + 1.09 n / 256), the last factor being the clock, which falls as more compute units multiply; and a round 6 us of its own.
// us, tiles of 256 / these: 6,151 x 4,096 x 14,336 617 / 559, 6,151 x 6,144 x 4,096 260 / 237, 5,487 x 4,096 x 4,096 197 / 158,
// 2,048 x 6,144 x 2,048 46.7 / 44.3, 5,173 x 4,096 x 14,336 578 / 502.  The bits are the same: a cell's k-steps are.
struct RingRows {
  int height, tall, tiles;   // of 32 rows: the tall tiles; how many of them, the others being one less; all tiles
  float us;                  // the estimate
};
constexpr bool ring_has(int height) { return height >= 5 && height <= 8; }   // what the kernel is built for: 129 rows and more are dealt so
inline RingRows ring_rows(int M, int columns, int K) {
  const int rows = (M + 31) / 32;
  auto round_us = [&](int h, long long n) {
    return (float)((K + RBK - 1) / RBK) * 0.0806f * ((float)h + 1.5f) * (1.f + 1.09f * (float)n / 256.f) + 6.f;
  };
  RingRows best{};
  const int least = (rows + 7) / 8;   // (that many in any case; more only while they fit a grid's second dimension)
  for (int tiles = least; tiles <= least + 24 && (tiles == least || tiles <= 65535); ++tiles) {
    const int height = (rows + tiles - 1) / tiles, tall = rows - tiles * (height - 1);
    if (height < 5 && best.tiles) break;
    const long long all = (long long)tiles * columns, whole = all / 256, high = ((long long)tall * columns + 255) / 256;
    float us = (float)(high < whole ? high : whole) * round_us(height, 256) + (float)(high < whole ? whole - high : 0) * round_us(height - 1, 256);
    if (all % 256) us += round_us(high > whole ? height : height - 1, all % 256);
    if (best.tiles == 0 || us < best.us) best = {height, tall, tiles, us};
  }
  return best;
}

}  // namespace gb
