// 32-bit matrix product for the true 32-bit path: C[M,N] (+)= A[M,K] . W[N,K]^T with
// W in the nn.Linear layout [out, in] (crates/glassbox-core/src/kernels.rs:381,586).
// Fused multiply-adds of 32 bits throughout, on the vector units or in the matrix cores' 32-bit instruction: no mode of
// reduced precision.
//
// Every output cell is summed in one order, whatever kernel computes it and whatever else is
// in the batch: k is cut into slices of 64; a slice's products are added in ascending k by a
// chain of fused multiply-adds that starts from zero; the slices' sums are added in ascending
// order.  So a cell's bits do not depend on M, on the tile it falls in, or on which of the
// kernels ran.  The matrix cores keep to it: v_mfma_f32_32x32x2_f32 adds its two products one after the other, each
// fused and rounded as fmaf rounds it (denormals, infinities and NaN included: the tests compare bits), at twice the rate of the
// vector units.
//
//  * tiled (any sizes, in practice rows that are no 16-byte words): a 64 x 64 tile of C a workgroup, k in steps of 16
//    through LDS, a thread 4 x 4 cells; after every fourth step (a slice) the chain's sum goes into the cell's total.
//  * wide (prompts; rows of 16 bytes): a 128 x 128 tile a workgroup on the matrix cores, two k-steps of 32 in LDS, the
//    next one's operands on their way from memory; two workgroups a unit, so that one multiplies while the other waits
//    at its barrier (2,048 x 16,384 x 2,048: 1,210 us, 114 TFLOP/s; on the vector units, 128 x 64 tiles, 65 to 85).
//  * sliced (everything between): a 32 x 32 tile a workgroup, whose waves take slices of k in turn, so that a product of
//    few tiles walks k in a quarter or an eighth of the steps (200 x 960 x 2,560: 458 us in the tiled kernel's 60
//    workgroups, 24 here; 64 x 2,048 x 8,192: 565 in the skinny kernel, 65 here).
//  * skinny (a few rows of 16 bytes: a decode step): a workgroup owns 4, 8 or 16 rows of W and every lane one (slice, row)
//    pair: all of a workgroup's weights (64 KB) are on their way at once, a lane runs the chain for each row of A, and the
//    slices' sums meet in LDS, where one thread a cell adds them in order (1 x 960 x 2,560: 10.3 -> 5.5 us with whole lines
//    through LDS and 4 rows of W a workgroup instead of 8; 1 x 49,152 x 960 64 -> 41 with 16).
#include "common.h"

using namespace gb;

GB_DEFINE_LAST_ERROR

namespace {

constexpr int kSlice = 64;   // the summation order's slice of k: all four kernels keep to it

constexpr int BM = 64, BN = 64, BK = 16, TM = 4, TN = 4;
static_assert(kSlice % BK == 0, "a slice is whole steps of the tiled kernel");

__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w,
                                                       int ldw, float* __restrict__ c, int ldc, int M, int N, int K,
                                                       int accumulate) {
  __shared__ float As[BK][BM + 4];
  __shared__ float Ws[BK][BN + 4];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  float acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
    for (int j = 0; j < (BM * BK) / 256; ++j) {
      const int e = tid + 256 * j;
      const int r = e / BK, kk = e % BK;
      const int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
      As[kk][r] = (gm < M && gk < K) ? a[(size_t)gm * lda + gk] : 0.f;
      Ws[kk][r] = (gn < N && gk < K) ? w[(size_t)gn * ldw + gk] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float av[TM], wv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) av[i] = As[kk][ty * TM + i];
#pragma unroll
      for (int j = 0; j < TN; ++j) wv[j] = Ws[kk][tx * TN + j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    if ((k0 + BK) % kSlice == 0 || k0 + BK >= K) {   // a slice ends: its sum joins the total
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int gm = m0 + ty * TM + i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int gn = n0 + tx * TN + j;
      if (gn >= N) continue;
      float* dst = c + (size_t)gm * ldc + gn;
      *dst = accumulate ? *dst + total[i][j] : total[i][j];
    }
  }
}

// ---- matrix cores: v_mfma_f32_32x32x2_f32 --------------------------------------------------------------------
// An operand of the instruction is one float a lane: row lane % 32, k = lane / 32.  A lane here loads 16-byte words: of
// eight consecutive k of its row it has k = 4 (lane / 32) .. + 3, and pairs() turns the words into the four operands of
// k = (0, 1), (2, 3), (4, 5), (6, 7) by swapping half waves.
__device__ __forceinline__ void pairs(const f32x4& v, float (&p)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2]), __float_as_uint(v[3]), false, false);
  p[0] = __uint_as_float(a[0]);
  p[1] = __uint_as_float(b[0]);
  p[2] = __uint_as_float(a[1]);
  p[3] = __uint_as_float(b[1]);
}
__device__ __forceinline__ f32x16 mfma(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// row of the 32 x 32 tile that register r of a lane holds; its column is lane % 32
__device__ __forceinline__ int tile_row(int r, int lane) { return 8 * (r / 4) + 4 * (lane / 32) + r % 4; }

// wide: 128 x 128 of C a workgroup, a wave 64 x 64; k-steps of 32 through two buffers in LDS
constexpr int WM = 128, WN = 128, WK = 32;
constexpr int WS = WK + 4;   // floats a row of a k-step: 144 bytes, so that the rows of a wave's reads lie on other banks
static_assert(kSlice % WK == 0, "a slice is whole steps of the wide kernel");

__global__ __launch_bounds__(256, 2) void gemm_f32_wide_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w,
                                                            int ldw, float* __restrict__ c, int ldc, int M, int N, int K,
                                                            int accumulate) {
  __shared__ __attribute__((aligned(16))) float As[2][WM * WS];
  __shared__ __attribute__((aligned(16))) float Ws[2][WN * WS];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int wm = wave / 2 * 64, wn = wave % 2 * 64;
  const int m0 = blockIdx.y * WM, n0 = blockIdx.x * WN;
  // a thread brings word lc of the k-step's eight for rows lr, lr + 32, lr + 64 and lr + 96 of both operands
  const int lr = tid / 8, lc = tid % 8;
  f32x4 pa[4], pw[4];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int k0) {
    const int gk = k0 + 4 * lc;   // K is whole words: a word is inside k or outside
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int gm = m0 + lr + 32 * h, gn = n0 + lr + 32 * h;
      pa[h] = (gm < M && gk < K) ? *reinterpret_cast<const f32x4*>(a + (size_t)gm * lda + gk) : zero;
      pw[h] = (gn < N && gk < K) ? *reinterpret_cast<const f32x4*>(w + (size_t)gn * ldw + gk) : zero;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      *reinterpret_cast<f32x4*>(&As[buf][(lr + 32 * h) * WS + 4 * lc]) = pa[h];
      *reinterpret_cast<f32x4*>(&Ws[buf][(lr + 32 * h) * WS + 4 * lc]) = pw[h];
    }
  };
  f32x16 acc[2][2], total[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = total[i][j][r] = 0.f;

  const int steps = (K + WK - 1) / WK;
  const int read = (lane % 32) * WS + 4 * (lane / 32);
  fetch(0);
  stash(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int buf = s & 1;
    if (s + 1 < steps) fetch((s + 1) * WK);
#pragma unroll
    for (int kk = 0; kk < WK; kk += 8) {
      float av[2][4], wv[2][4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        pairs(*reinterpret_cast<const f32x4*>(&As[buf][(wm + 32 * i) * WS + read + kk]), av[i]);
        pairs(*reinterpret_cast<const f32x4*>(&Ws[buf][(wn + 32 * i) * WS + read + kk]), wv[i]);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma(av[i][q], wv[j][q], acc[i][j]);
    }
    if (((s + 1) * WK) % kSlice == 0 || s + 1 == steps) {   // a slice ends: its sum joins the total
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            total[i][j][r] += acc[i][j][r];
            acc[i][j][r] = 0.f;
          }
    }
    // the other half of LDS was last read a step ago, before the barrier that every thread has passed since
    if (s + 1 < steps) stash(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int gn = n0 + wn + 32 * j + lane % 32;
      if (gn >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = m0 + wm + 32 * i + tile_row(r, lane);
        if (gm >= M) continue;
        float* dst = c + (size_t)gm * ldc + gn;
        *dst = accumulate ? *dst + total[i][j][r] : total[i][j][r];
      }
    }
}

// sliced: 32 x 32 of C a workgroup, whose waves take the slices of k in turn; the slices' sums of a round meet in LDS,
// where one thread adds a cell's in order.  A wave brings its slice of both operands straight into LDS, whole rows of
// 256 bytes (word p of row r lies at position p ^ (r % 16), so that a read's 16 neighbouring rows spread over all
// banks): loaded by the lanes that multiply them, an instruction of a wave touches 32 bytes of 32 rows, 100 cycles each.
template <int NW>
__global__ __launch_bounds__(NW * kWave) void gemm_f32_sliced_kernel(const float* __restrict__ a, int lda,
                                                                     const float* __restrict__ w, int ldw,
                                                                     float* __restrict__ c, int ldc, int M, int N, int K,
                                                                     int accumulate) {
  constexpr int T = 32, CELLS = T * T / (NW * kWave);   // cells a thread adds up
  extern __shared__ __attribute__((aligned(16))) float smem[];   // a wave's slice [2][32][64], then the sums [NW][32 * 32]
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  float* own = smem + wave * (2 * T * kSlice);
  float* part = smem + NW * (2 * T * kSlice);
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int slices = (K + kSlice - 1) / kSlice;
  auto fetch = [&](int slice) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int row = (u % 8) * 4 + lane / 16;   // the first eight instructions bring A, the others W
      // (a word beyond k is replaced by zeros where it is read, a row beyond m or n goes nowhere: any address inside will do)
      const int k = slice * kSlice + 4 * ((lane % 16) ^ (row % 16));
      const float* from = (u < 8 ? a + (size_t)min(m0 + row, M - 1) * lda : w + (size_t)min(n0 + row, N - 1) * ldw) + (k < K ? k : 0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)(uintptr_t)from,
                                       (__attribute__((address_space(3))) uint32_t*)(uint32_t)(uintptr_t)(own + u * 256), 16, 0, 0);
    }
  };
  float total[CELLS];
#pragma unroll
  for (int e = 0; e < CELLS; ++e) total[e] = 0.f;
  if (wave < slices) fetch(wave);
  for (int s0 = 0; s0 < slices; s0 += NW) {
    const int slice = s0 + wave;
    if (slice < slices) {   // the same for a whole wave
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      f32x4 av[8], wv[8];
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      const int r = lane % 32;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int word = 2 * i + lane / 32;
        const bool in = slice * kSlice + 4 * word < K;
        const f32x4 x = *reinterpret_cast<const f32x4*>(own + r * kSlice + 4 * (word ^ (r % 16)));
        const f32x4 y = *reinterpret_cast<const f32x4*>(own + (T + r) * kSlice + 4 * (word ^ (r % 16)));
        av[i] = in ? x : zero;
        wv[i] = in ? y : zero;
      }
      // every operand is in registers: the next slice may come in under the products
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (slice + NW < slices) fetch(slice + NW);
      f32x16 acc;
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[q] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float x[4], y[4];
        pairs(av[i], x);
        pairs(wv[i], y);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = mfma(x[q], y[q], acc);
      }
#pragma unroll
      for (int q = 0; q < 16; ++q) part[wave * (T * T) + tile_row(q, lane) * T + lane % 32] = acc[q];
    }
    // (the sums must be there; the loads that are on their way need not)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int count = min(NW, slices - s0);
#pragma unroll
    for (int e = 0; e < CELLS; ++e) {
      float v[NW];
#pragma unroll
      for (int q = 0; q < NW; ++q) v[q] = q < count ? part[q * (T * T) + tid + e * NW * kWave] : 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q)
        if (q < count) total[e] += v[q];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
#pragma unroll
  for (int e = 0; e < CELLS; ++e) {
    const int cell = tid + e * NW * kWave;
    const int cm = m0 + cell / T, cn = n0 + cell % T;
    if (cm < M && cn < N) {
      float* dst = c + (size_t)cm * ldc + cn;
      *dst = accumulate ? *dst + total[e] : total[e];
    }
  }
}

template <int NW>
int launch_sliced(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K, int accumulate,
                  hipStream_t stream) {
  const dim3 grid((N + 31) / 32, (M + 31) / 32);
  GB_REQUIRE(grid.y <= 65535, "gemm_f32: M=%d needs more than 65535 row tiles", M);
  hipLaunchKernelGGL(gemm_f32_sliced_kernel<NW>, grid, dim3(NW * kWave), NW * (2 * 32 * kSlice + 32 * 32) * 4, stream, a, lda, w,
                     ldw, c, ldc, M, N, K, accumulate);
  return launched("gemm_f32 (sliced)");
}

// The wide kernel from so many of its tiles on: with fewer, units are idle while a tile walks all of k (us, wide / sliced:
// 160 tiles, 400 x 5,120 x 960, 88 / 71; 200 tiles, 600 rows, 89 / 92; 256 tiles, 2,048 x 2,048 x 8,192, 711 / 912).
constexpr int kWideMinTiles = 192;
// And from so many rows on: a single row tile of 128 rows that is half empty takes as long as a full one (49,152 x 2,048 at 3,
// 33 and 64 rows 306, 308 and 310 / sliced 107, 204 and 210; at 65 and 97 rows 309 and 310 / 309 and 409).
constexpr int kWideMinRows = 65;
// Up to so many tiles a unit has one workgroup of the sliced kernel at most: eight waves then walk k in half the rounds
// (200 x 960 x 2,560 29.7 -> 23.6 us).  With more, two workgroups of four waves share a unit, one's loads on their way
// under the other's products (2,048 x 960 x 960 69.7 -> 64.0).
constexpr int kFewTiles = 256;

// ---- skinny: R rows of W a workgroup, a lane a (slice, row) pair ------------------------------------------
// What a lane multiplies lies 256 bytes from what its neighbour does: loaded into registers by the lane itself, an
// instruction of a wave would touch 64 lines of memory, each again by seven more.  So W goes through LDS: a wave's
// instruction brings four slices of a row (a kilobyte in a run) straight into LDS, where a lane reads its own slice.
// Word p of the slice of pair t lies at position p ^ (t % 16), so that the reads of 16 neighbouring lanes spread over all banks.
constexpr int SV = kSlice / 4;    // 16-byte words a slice of one row

// What the skinny kernel may do besides the product, for a step of one or two rows (a decode step of the 32-bit path, whose
// kernels are so short that what lies between them counts).  The bits are those of the kernels that each does by itself: the
// expressions and the order of every sum are shared with them (common.h).
//  * NORM: A is the residual, and the rows that are multiplied are its RMS norm's (gb_rmsnorm): in every workgroup a fifth wave,
//    which asks for none of W and so need not wait for it, norms them into LDS while W is on its way.
//  * EPI_UNIT: W stacks gate rows over as many up rows; C holds silu(gate) * up (gb_silu_mul).  A workgroup owns R / 2 gate rows
//    and the up rows that go with them.
//  * EPI_HEADS: W stacks nh query heads, nkv key heads and nkv value heads of hd rows; queries and keys are turned by
//    their position's angles, and keys and values also go to their places in the pages (gb_rope_store).  A workgroup owns
//    R / 2 pairs (i, i + hd / 2) of coordinates.
// us, replayed from a graph over weights that no cache holds, each kernel by itself / in one, a row of 960: norm, product by 5,120
// rows and unit 12.7 / 8.9 (the product alone 8.2); norm, product by 1,600 rows, rotation and cache write 8.9 / 6.2 (4.2); a row
// of 576: 8.7 / 6.0 (4.7), 8.1 / 5.7 (3.6); of 2,048: 33.9 / 31.5 (29.1), 19.2 / 13.6 (13.5).
enum : int { EPI_PLAIN = 0, EPI_UNIT = 2, EPI_HEADS = 3 };
constexpr int kStepMaxRows = 2;
struct StepExtras {
  const float* gamma;   // of the norm, with NORM
  float eps;
  const float* cosv;    // [M][hd / 2], or null: nothing is turned
  const float* sinv;
  const int32_t* slots;   // [M], or null: nothing is stored
  float* k_pages;
  float* v_pages;
  int nh, nkv, hd, page_size;
  float per_half;   // 2 / hd, and page_size as a shift (-1: no power of two): the kernel has no time for divisions
  int page_shift;
};

constexpr int kNormedFloats = 2560;   // of the rows that a workgroup norms (step_takes)

// Wave `NV` times norm_threads' worth: one wave norms MT rows of K numbers into LDS; a lane stands for threads lane, lane + 64, ...
// of the NV waves of the norm's own kernel.  Word p of slice t of a row lies at position p ^ (t % 16), for the reads of 16 lanes
// on as many slices.
template <int MT, int NV>
__device__ __forceinline__ void norm_rows(const float* __restrict__ a, int lda, const float* __restrict__ gamma, float eps, int M, int K,
                                          int lane, int slices, float* rows) {
  constexpr int NW = kNormedFloats / 4 / kWave / MT;   // words a lane
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 x[MT][NW], g[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {   // (a word beyond k: the first one, not used)
    const int k = 4 * (lane + kWave * i), from = k < K ? k : 0;
    g[i] = *reinterpret_cast<const f32x4*>(gamma + from);
#pragma unroll
    for (int m = 0; m < MT; ++m) x[m][i] = *reinterpret_cast<const f32x4*>(a + (size_t)min(m, M - 1) * lda + from);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float total = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      constexpr int OWN = (NW + NV - 1) / NV < 1 ? 1 : (NW + NV - 1) / NV;
      f32x4 own[OWN];
#pragma unroll
      for (int j = 0; j < OWN; ++j) {
        const int i = v + j * NV;
        own[j] = i < NW && 4 * (lane + kWave * i) < K ? x[m][i < NW ? i : 0] : zero;
      }
      total += wave_sum(norm_squares(own));
    }
    const float s = norm_scale(total, K, eps);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int word = lane + kWave * i, t = word / SV, p = word % SV;
      if (4 * word < K) {
        f32x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = g[i][e] * (x[m][i][e] * s);
        *reinterpret_cast<f32x4*>(rows + ((size_t)m * slices + t) * kSlice + 4 * (p ^ (t % 16))) = h;
      }
    }
  }
}

template <int MT, int R, int EPI, bool NORM>   // rows of A a pass (the step's rows go MT at a time); rows of W a workgroup
__global__ __launch_bounds__(NORM ? 256 + kWave : 256, NORM ? 4 : 1)   // (five waves: two workgroups a unit fit with four a SIMD)
void gemm_f32_skinny_kernel(const float* __restrict__ a, int lda,
                                                              const float* __restrict__ w, int ldw,
                                                              float* __restrict__ c, int ldc, int M, int N, int K,
                                                              int accumulate, StepExtras ex) {
  constexpr int SG = 256 / R;   // slices in flight a workgroup
  extern __shared__ __attribute__((aligned(16))) float wl[];   // [R][SG][64], then part [SG][R][MT], then with NORM the rows [MT][slices][64]
  float* part = wl + 256 * kSlice;
  float* rows = part + 256 * MT;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const bool works = !NORM || wave < 256 / kWave;   // (else: the wave that norms)
  const int r = tid % R, sl = tid / R;
  const int n0 = blockIdx.x * R;
  const int slices = (K + kSlice - 1) / kSlice;
  // the thread that adds the slices of cell (row cm of the pass, column cr)
  const int cr = tid % R, cm = tid / R;
  // the row of W behind row t of the workgroup's (beyond the last: that one again)
  const int half = EPI == EPI_HEADS ? ex.hd / 2 : N / 2;
  auto head_of = [&](int p) { return (int)(((float)p + 0.5f) * ex.per_half); };   // p / half, exact below 2^21 pairs
  auto w_row = [&](int t) -> int {
    if constexpr (EPI == EPI_PLAIN) return min(n0 + t, N - 1);
    const int pair = min(n0 / 2 + t % (R / 2), N / 2 - 1);
    return (EPI == EPI_HEADS ? pair + head_of(pair) * half : pair) + (t >= R / 2 ? half : 0);   // (a head's rows are twice its pairs)
  };
  // with EPI_HEADS the pair that a thread finishes
  const int pair = n0 / 2 + cr;
  const int head = EPI == EPI_HEADS ? head_of(pair) : 0, at = EPI == EPI_HEADS ? pair - head * half : 0;
  const bool finishes = EPI != EPI_PLAIN && cm < MT && cm < M && cr < R / 2 && pair < N / 2;
  const bool is_value = EPI == EPI_HEADS && head >= ex.nh + ex.nkv;
  float cs = 1.f, sn = 0.f;
  int slot = -1;
  if (NORM && !works) {   // (NORM: one pass)
    switch (norm_threads(K) / kWave) {
      case 1: norm_rows<MT, 1>(a, lda, ex.gamma, ex.eps, M, K, lane, slices, rows); break;
      case 2: norm_rows<MT, 2>(a, lda, ex.gamma, ex.eps, M, K, lane, slices, rows); break;
      default: norm_rows<MT, 4>(a, lda, ex.gamma, ex.eps, M, K, lane, slices, rows);
    }
  }

  for (int m0 = 0; m0 < M; m0 += MT) {
    float total = 0.f, old = 0.f;
    const int gm = m0 + cm, gn = n0 + cr;
    const bool owns = EPI == EPI_PLAIN && cm < MT && gm < M && gn < N;
    for (int s0 = 0; s0 < slices; s0 += SG) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        // four slices of a row, which one wave brings: unit u of the wave's
        const int unit = wave * 16 + u, row = unit / (SG / 4), first = unit % (SG / 4) * 4;
        if (!works || s0 + first >= slices) continue;                      // the same for the whole wave
        const int mine = first + lane / 16;
        const int word = (lane % 16) ^ ((mine * R + row) % 16);
        // (a word beyond k or n is not used: any address inside W will do for it)
        const int k = (s0 + mine) * kSlice + 4 * word;
        const float* from = w + (size_t)w_row(row) * ldw + (k < K ? k : 0);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)(uintptr_t)from,
                                         (__attribute__((address_space(3))) uint32_t*)(uint32_t)(uintptr_t)(wl + unit * 256), 16, 0, 2);   // (nontemporal: read once)
      }
      // What the end will want from memory is asked for under W: a cell's old value; a pair's angle and its row's place in the pages.
      // (Not before W: the compiler would wait for it there.)
      if (EPI == EPI_PLAIN && accumulate && owns && s0 == 0) old = c[(size_t)gm * ldc + gn];
      if constexpr (EPI == EPI_HEADS) {
        if (finishes && s0 == 0) {
          if (ex.cosv && !is_value) {
            cs = ex.cosv[(size_t)cm * half + at];
            sn = ex.sinv[(size_t)cm * half + at];
          }
          if (ex.slots && head >= ex.nh) slot = ex.slots[cm];
        }
      }
      const int k0 = (s0 + sl) * kSlice;
      const bool live = works && k0 < K;
      // a single row of A is asked for before W has arrived
      constexpr bool EARLY = MT == 1 && !NORM;
      f32x4 x1[EARLY ? SV : 1];
      if constexpr (EARLY) {
#pragma unroll
        for (int i = 0; i < SV; ++i) {
          const int k = k0 + 4 * i;
          x1[i] = *reinterpret_cast<const f32x4*>(a + (size_t)m0 * lda + (k < K ? k : 0));
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      float acc[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = 0.f;
      if (live) {
        const float* own = wl + (r * SG + sl) * kSlice;
#pragma unroll
        for (int i = 0; i < SV; ++i) {
          const int k = k0 + 4 * i;
          if (k < K) {
            const f32x4 wv = *reinterpret_cast<const f32x4*>(own + 4 * (i ^ (tid % 16)));
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              if (MT == 1 || m0 + m < M) {
                f32x4 x;
                if constexpr (EARLY) x = x1[i];
                else if constexpr (NORM) x = *reinterpret_cast<const f32x4*>(rows + ((size_t)m * slices + s0 + sl) * kSlice + 4 * (i ^ ((s0 + sl) % 16)));
                else x = *reinterpret_cast<const f32x4*>(a + (size_t)(m0 + m) * lda + k);
                acc[m] = fmaf(x[0], wv[0], acc[m]);
                acc[m] = fmaf(x[1], wv[1], acc[m]);
                acc[m] = fmaf(x[2], wv[2], acc[m]);
                acc[m] = fmaf(x[3], wv[3], acc[m]);
              }
            }
          }
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (works) part[(sl * R + r) * MT + m] = acc[m];
      __syncthreads();
      if (cm < MT) {
        const int count = min(SG, slices - s0);
        for (int s = 0; s < count; s += 8) {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = part[(min(s + q, SG - 1) * R + cr) * MT + cm];
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (s + q < count) total += v[q];
        }
      }
      if (EPI != EPI_PLAIN || s0 + SG < slices || m0 + MT < M) __syncthreads();
    }
    if constexpr (EPI == EPI_PLAIN) {
      if (owns) c[(size_t)gm * ldc + gn] = accumulate ? old + total : total;
    } else {
      // the two rows of a pair meet (every thread has read the slices' sums)
      if (cm < MT) part[cm * R + cr] = total;
      __syncthreads();
      if (finishes) {   // (a launch has one pass)
        const float lo = total, hi = part[cm * R + cr + R / 2];
        if constexpr (EPI == EPI_UNIT) {
          c[(size_t)cm * ldc + pair] = silu_times(lo, hi);
        } else {
          const bool turns = ex.cosv && !is_value;
          const float y0 = turns ? turned_lo(lo, hi, cs, sn) : lo, y1 = turns ? turned_hi(lo, hi, cs, sn) : hi;
          float* row = c + (size_t)cm * ldc + (size_t)head * ex.hd;
          row[at] = y0;
          row[half + at] = y1;
          if (slot >= 0) {
            const int page = ex.page_shift >= 0 ? slot >> ex.page_shift : slot / ex.page_size, off = slot - page * ex.page_size, piece = key_piece(ex.hd);
            if (is_value) {
              float* to = ex.v_pages + ((size_t)page * ex.nkv + (head - ex.nh - ex.nkv)) * ex.hd * ex.page_size + off;
              to[(size_t)at * ex.page_size] = y0;
              to[(size_t)(half + at) * ex.page_size] = y1;
            } else {
              float* to = ex.k_pages + ((size_t)page * ex.nkv + (head - ex.nh)) * ex.page_size * ex.hd;
              to[key_offset(off, at, ex.page_size, piece)] = y0;
              to[key_offset(off, half + at, ex.page_size, piece)] = y1;
            }
          }
        }
      }
    }
  }
}

template <int MT, int R, int EPI = EPI_PLAIN, bool NORM = false>
void launch_skinny(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                        int accumulate, hipStream_t stream, const StepExtras& ex = StepExtras{}) {
  static_assert(MT * R <= 256, "one thread a cell of a pass");
  const size_t rows = NORM ? (size_t)MT * ((K + kSlice - 1) / kSlice) * kSlice : 0;
  hipLaunchKernelGGL((gemm_f32_skinny_kernel<MT, R, EPI, NORM>), dim3((N + R - 1) / R), dim3(NORM ? 256 + kWave : 256),
                     (256 * (kSlice + MT) + rows) * 4,
                     stream, a, lda, w, ldw, c, ldc, M, N, K, accumulate, ex);
}
constexpr int kSkinnyMaxRows = 64;   // in passes of eight; by itself (skinny_pays) it runs at up to eight
// Where the skinny kernel is the faster one (us, skinny / sliced, replayed from a graph over weights that no cache holds):
// up to 4 rows of narrow products (960 x 960 at 1 and 4 rows 4.2 and 8.5 / 9.8, 2,048 x 8,192 17 and 29 / 63), up to 6 where k
// is long (576 x 1,536 10.4 and 11.5 at 5 and 6 rows / 13.5, but 960 x 960 10.3 / 9.9), up to 8 where it is longer and the
// workgroups own 4 rows (2,048 x 8,192 48 / 64, 960 x 2,560 20.0 / 21.1, but 3,072 x 2,048 20.6 / 18.6); wide products
// read W at the memory's pace with 16 rows a workgroup, and the sums of more than two rows of A then take longer than the
// matrix cores (49,152 x 960 at 1, 2 and 4 rows 42, 50 and 68 / 54).
// Rows of W a workgroup: the fewest that leave a unit no more than two workgroups, which is what its LDS holds (one row of A,
// 4 / 8 / 16: 960 x 2,560 5.5 / 6.9 / 9.1, 2,304 x 576 6.3 / 4.9 / 4.7, 4,096 x 4,096 17.9 / 16.8 / 21.9, 5,120 x 960 10.5 / 9.2 /
// 8.3; four rows of A, 3,072 x 576 14.8 / 8.9 / 9.0).
constexpr int kTwoAUnit = 512, kNarrow = 8 * kTwoAUnit, kLongK = 1280, kLongerK = 2048;
inline bool skinny_pays(int M, int N, int K) {
  if (N > kNarrow) return M <= 2;
  return M <= 4 || (M <= 6 && K >= kLongK) || (M <= 8 && K >= kLongerK && N <= 4 * kTwoAUnit);
}

// A step's kernels in one: where the skinny kernel runs anyway, up to two rows; with the norm, as long as the rows that a
// workgroup norms for itself leave LDS for two workgroups a unit (160 KB: 2 x (64 for W, 2 for the sums, 10)), and not before very many
// rows of W of a short k, whose workgroups each wait for the norm and have little else to do (16,384 rows, us, apart / in one: k 256 with
// the unit 12.4 / 13.9, k 576 17.2 / 17.4, k 1,024 22.3 / 21.6; 8,192 rows of 256 8.7 / 6.0).
inline bool step_takes(int M, int N, int K, bool norm) {
  return M >= 1 && M <= kStepMaxRows && K % 4 == 0 && N % 2 == 0 && skinny_pays(M, N, K) &&
         (!norm || (M * ((K + kSlice - 1) / kSlice) * kSlice <= kNormedFloats && (K >= 512 || N <= 8192)));
}

inline bool words_of_16_bytes(const void* p, int ld) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 4 == 0; }

}  // namespace

// which = 0: the kernel the sizes call for; 1: the tiled kernel; 2: the skinny kernel; 3: the wide kernel; 4 and 5: the
// sliced kernel with four and eight waves (all but the tiled one refused where they do not apply).  All give the same
// bits; tests compare them.
extern "C" int gb_gemm_f32_by(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                              int accumulate, int which, hipStream_t stream) {
  GB_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  GB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: a leading dimension is shorter than its row (lda=%d ldw=%d ldc=%d)", lda, ldw, ldc);
  GB_REQUIRE(which >= 0 && which <= 5, "gemm_f32: no kernel %d", which);
  if (M == 0) return 0;
  const bool words = K % 4 == 0 && words_of_16_bytes(a, lda) && words_of_16_bytes(w, ldw);
  const bool skinny_fits = M <= kSkinnyMaxRows && words;
  GB_REQUIRE(which != 2 || skinny_fits, "gemm_f32: the skinny kernel takes at most %d rows of 16-byte words (M=%d K=%d)",
             kSkinnyMaxRows, M, K);
  if (which == 2 || (which == 0 && skinny_fits && skinny_pays(M, N, K))) {
#define GB_SKINNY(MT, R) launch_skinny<MT, R>(a, lda, w, ldw, c, ldc, M, N, K, accumulate, stream)
    if (N > kNarrow && M <= 1) GB_SKINNY(1, 16);
    else if (N > kNarrow && M <= 2) GB_SKINNY(2, 16);
    else if (N > 4 * kTwoAUnit) {
      if (M <= 1) GB_SKINNY(1, 8);
      else if (M <= 2) GB_SKINNY(2, 8);
      else if (M <= 4) GB_SKINNY(4, 8);
      else GB_SKINNY(8, 8);
    } else {
      if (M <= 1) GB_SKINNY(1, 4);
      else if (M <= 2) GB_SKINNY(2, 4);
      else if (M <= 4) GB_SKINNY(4, 4);
      else GB_SKINNY(8, 4);
    }
#undef GB_SKINNY
    return launched("gemm_f32 (skinny)");
  }
  GB_REQUIRE(which < 3 || words, "gemm_f32: the wide and the sliced kernel take rows of 16-byte words (K=%d lda=%d ldw=%d)", K, lda, ldw);
  const dim3 wide((N + WN - 1) / WN, (M + WM - 1) / WM);
  if (which == 3 || (which == 0 && words && M >= kWideMinRows && (long long)wide.x * wide.y >= kWideMinTiles)) {
    GB_REQUIRE(wide.y <= 65535, "gemm_f32: M=%d needs more than 65535 row tiles", M);
    hipLaunchKernelGGL(gemm_f32_wide_kernel, wide, dim3(256), 0, stream, a, lda, w, ldw, c, ldc, M, N, K, accumulate);
    return launched("gemm_f32 (wide)");
  }
  if (which >= 4 || (which == 0 && words)) {
    const bool few = (long long)((N + 31) / 32) * ((M + 31) / 32) <= kFewTiles;
    return which == 4 || (which == 0 && !few) ? launch_sliced<4>(a, lda, w, ldw, c, ldc, M, N, K, accumulate, stream)
                                              : launch_sliced<8>(a, lda, w, ldw, c, ldc, M, N, K, accumulate, stream);
  }
  const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  GB_REQUIRE(grid.y <= 65535, "gemm_f32: M=%d needs more than 65535 row tiles", M);
  hipLaunchKernelGGL(gemm_f32_kernel, grid, dim3(256), 0, stream, a, lda, w, ldw, c, ldc, M, N, K, accumulate);
  return launched("gemm_f32");
}

extern "C" int gb_gemm_f32(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                           int accumulate, hipStream_t stream) {
  return gb_gemm_f32_by(a, lda, w, ldw, c, ldc, M, N, K, accumulate, 0, stream);
}

// Whether gb_gemm_f32_step takes a product of M rows by N rows of W (with the norm before it).
extern "C" int gb_gemm_f32_step_takes(int M, int N, int K, int norm) { return step_takes(M, N, K, norm != 0) ? 1 : 0; }

// A product of one or two rows with what stands around it in a decode step, see StepExtras: gamma (or null): a is the
// residual and is normed first; epilogue 0 stores, 2 forms the gated unit of stacked gate and up rows (C is [M, N / 2]), 3 turns
// heads and writes the pages.  The bits are those of gb_rmsnorm, gb_gemm_f32, gb_silu_mul and gb_rope_store one after the other.
extern "C" int gb_gemm_f32_step(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                                const float* gamma, float eps, int epilogue, const float* cosv, const float* sinv,
                                const int32_t* slots, void* k_pages, void* v_pages, int nh, int nkv, int hd, int page_size,
                                hipStream_t stream) {
  GB_REQUIRE(N > 0 && K > 0 && step_takes(M, N, K, gamma != nullptr), "gemm_f32_step: not for M=%d N=%d K=%d", M, N, K);
  GB_REQUIRE(epilogue == EPI_PLAIN || epilogue == EPI_UNIT || epilogue == EPI_HEADS, "gemm_f32_step: unknown epilogue %d", epilogue);
  GB_REQUIRE(lda >= K && ldw >= K && ldc >= (epilogue == EPI_UNIT ? N / 2 : N), "gemm_f32_step: a leading dimension is shorter than its row (lda=%d ldw=%d ldc=%d)", lda, ldw, ldc);
  GB_REQUIRE(words_of_16_bytes(a, lda) && words_of_16_bytes(w, ldw) && (uintptr_t)gamma % 16 == 0, "gemm_f32_step: rows of 16-byte words");
  GB_REQUIRE(epilogue != EPI_HEADS || (hd >= 2 && hd % 2 == 0 && nh > 0 && nkv >= 0 && N == (nh + 2 * nkv) * hd && (cosv == nullptr) == (sinv == nullptr) &&
                                       (!slots || (nkv > 0 && k_pages && v_pages && page_size > 0))),
             "gemm_f32_step: N=%d is not (nh + 2 nkv) hd with nh=%d nkv=%d hd=%d, or pages or angles are missing", N, nh, nkv, hd);
  const StepExtras ex{gamma, eps, cosv, sinv, slots, (float*)k_pages, (float*)v_pages, nh, nkv, hd, page_size, hd > 0 ? 2.0f / (float)hd : 0.f,
                      page_size > 0 && (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1};
  if (!gamma && epilogue == EPI_PLAIN) return gb_gemm_f32(a, lda, w, ldw, c, ldc, M, N, K, 0, stream);
#define GB_STEP(MT, R, EPI)                                                                                                 \
  if (epilogue == EPI && (M <= 1) == (MT == 1) && R == (N > kNarrow ? 16 : N > 4 * kTwoAUnit ? 8 : 4)) {                      \
    if (gamma) launch_skinny<MT, R, EPI, true>(a, lda, w, ldw, c, ldc, M, N, K, 0, stream, ex);                             \
    else if constexpr (EPI != EPI_PLAIN) launch_skinny<MT, R, EPI, false>(a, lda, w, ldw, c, ldc, M, N, K, 0, stream, ex);  \
  }
#define GB_STEPS(EPI) GB_STEP(1, 4, EPI) GB_STEP(1, 8, EPI) GB_STEP(1, 16, EPI) GB_STEP(2, 4, EPI) GB_STEP(2, 8, EPI) GB_STEP(2, 16, EPI)
  GB_STEPS(EPI_PLAIN) GB_STEPS(EPI_UNIT) GB_STEPS(EPI_HEADS)
#undef GB_STEPS
#undef GB_STEP
  return launched("gemm_f32 (step)");
}

// the launches of a layer can be recorded and made again for the layers like it (common.h)
GB_TAPED(gb_gemm_f32_step)
GB_TAPED(gb_gemm_f32)
GB_TAPED(gb_gemm_f32_by)
