// The k-steps of the ring kernel (gemm_bf16.hip): where each begins in a slice of k and which half of it counts as zeros.
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

}  // namespace gb
