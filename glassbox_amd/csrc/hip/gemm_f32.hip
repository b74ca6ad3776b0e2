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

template <int MT, int R>   // rows of A a pass (the step's rows go MT at a time); rows of W a workgroup
__global__ __launch_bounds__(256) void gemm_f32_skinny_kernel(const float* __restrict__ a, int lda,
                                                              const float* __restrict__ w, int ldw,
                                                              float* __restrict__ c, int ldc, int M, int N, int K,
                                                              int accumulate) {
  constexpr int SG = 256 / R;   // slices in flight a workgroup
  extern __shared__ __attribute__((aligned(16))) float wl[];   // [R][SG][64], then part [SG][R][MT]
  float* part = wl + 256 * kSlice;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int r = tid % R, sl = tid / R;
  const int n0 = blockIdx.x * R;
  const int slices = (K + kSlice - 1) / kSlice;
  // the thread that adds the slices of cell (row cm of the pass, column cr)
  const int cr = tid % R, cm = tid / R;

  for (int m0 = 0; m0 < M; m0 += MT) {
    float total = 0.f;
    for (int s0 = 0; s0 < slices; s0 += SG) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        // four slices of a row, which one wave brings: unit u of the wave's
        const int unit = wave * 16 + u, row = unit / (SG / 4), first = unit % (SG / 4) * 4;
        if (s0 + first >= slices) continue;                                // the same for the whole wave
        const int mine = first + lane / 16;
        const int word = (lane % 16) ^ ((mine * R + row) % 16);
        // (a word beyond k or n is not used: any address inside W will do for it)
        const int k = (s0 + mine) * kSlice + 4 * word;
        const float* from = w + (size_t)min(n0 + row, N - 1) * ldw + (k < K ? k : 0);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)(uintptr_t)from,
                                         (__attribute__((address_space(3))) uint32_t*)(uint32_t)(uintptr_t)(wl + unit * 256), 16, 0, 0);
      }
      const int k0 = (s0 + sl) * kSlice;
      const bool live = k0 < K;
      // a single row of A is asked for before W has arrived
      f32x4 x1[MT == 1 ? SV : 1];
      if (MT == 1) {
#pragma unroll
        for (int i = 0; i < SV; ++i) {
          const int k = k0 + 4 * i;
          x1[MT == 1 ? i : 0] = *reinterpret_cast<const f32x4*>(a + (size_t)m0 * lda + (k < K ? k : 0));
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
                const f32x4 x = MT == 1 ? x1[MT == 1 ? i : 0] : *reinterpret_cast<const f32x4*>(a + (size_t)(m0 + m) * lda + k);
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
      for (int m = 0; m < MT; ++m) part[(sl * R + r) * MT + m] = acc[m];
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
      if (s0 + SG < slices || m0 + MT < M) __syncthreads();
    }
    const int gm = m0 + cm, gn = n0 + cr;
    if (cm < MT && gm < M && gn < N) {
      float* dst = c + (size_t)gm * ldc + gn;
      *dst = accumulate ? *dst + total : total;
    }
  }
}

template <int MT, int R>
void launch_skinny(const float* a, int lda, const float* w, int ldw, float* c, int ldc, int M, int N, int K,
                        int accumulate, hipStream_t stream) {
  static_assert(MT * R <= 256, "one thread a cell of a pass");
  hipLaunchKernelGGL((gemm_f32_skinny_kernel<MT, R>), dim3((N + R - 1) / R), dim3(256), 256 * (kSlice + MT) * 4, stream, a, lda,
                     w, ldw, c, ldc, M, N, K, accumulate);
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

// the launches of a layer can be recorded and made again for the layers like it (common.h)
GB_TAPED(gb_gemm_f32)
GB_TAPED(gb_gemm_f32_by)
