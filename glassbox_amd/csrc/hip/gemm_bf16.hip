// bfloat16 matrix products on the matrix cores (MFMA), 32-bit accumulation:
//   C[M,N] (+)= A[M,K] . W[N,K]^T,   W in the nn.Linear layout [out, in]
// (crates/glassbox-core/src/kernels.rs:381,586).  Both operands are contiguous along k, which
// is the layout MFMA operands want: every lane loads 8 consecutive k as one 16-byte word.
//
// Seven kernels:
//  * tiled  (M > 64, prompt portions): a workgroup of 2x2 waves, each wave a block of 2x2 or 2x1
//    v_mfma_f32_32x32x16_bf16 tiles (workgroup tile 128x128 or 128x64; 64 rows high where the taller tiles would be
//    few), operands staged through LDS in k-steps of 64 with two buffers; the SiLU-multiply of stacked gate/up rows
//    can be its epilogue.  Its workgroups can also divide k (split k: a second pass adds their sums in order).
//  * block  (some hundred rows): tiles of 64 to 256 rows by 64 to 128 columns, whichever move the fewest bytes, both operands
//    straight into LDS several k-steps ahead.
//  * ring   (257 rows and more, where its tiles of 256 columns by 128 to 256 rows are ahead): 2x2 waves, a wave up to 8x8
//    tiles of v_mfma_f32_16x16x32_bf16; operands go from memory straight into a ring of LDS buffers in k-steps of 64.
//  * skinny (17 to 64 rows, or up to 64 with the norm on the way; decoding): bound by reading W once.  A workgroup owns 16 or 32 rows of W (8 where the
//    rows of W are few); its
//    waves take interleaved 64-wide k blocks, stream W straight from memory into MFMA operands
//    (v_mfma_f32_16x16x32_bf16, W as the A operand so that the 16 rows fill the tile) and combine
//    through LDS in a fixed order; it can norm float32 rows on the way, apply the SiLU-multiply, or
//    (the QKV product) rotate the heads and write the key/value cache, or prepare the next norm where it adds
//    into the residual.
//  * held   (17 to 64 rows by many rows of W, decode steps of a busy server): a workgroup a compute unit holds the rows of
//    A in registers and streams tiles of W through LDS.
//  * few    (M <= 16, decode steps): 8 rows of W over two k ranges side by side in a tile, so that loads bring whole lines, all of
//    them asked for at once.  (folded: the same tiles with the norm on the way, up to 8 rows by few rows of W.)
// In all, every output cell is summed in an order fixed by the product's sizes (they choose the kernel and how it divides k), not by
// what its neighbours hold.  C is bfloat16 or float32; accumulation (+=) is into float32.
#include <type_traits>

#include "common.h"
#include "ring_steps.h"

using namespace gb;

GB_DEFINE_LAST_ERROR

namespace {

__device__ __forceinline__ bf16x8 load8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
// read once and not again in this kernel: the caches need not keep it
__device__ __forceinline__ bf16x8 load8_once(const bf16* p) { return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p)); }
__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (bf16)0.f;
  return z;
}

// The gated unit of an EPI_SILU_MUL product, with the numbers that a clamped unit changes:
// g' = min(g, limit), u' = clamp(u, -limit, limit), act = g' sigmoid(alpha g') (u' + plus).  As it stands here it is
// silu(g) u to the bit.
struct Glu {
  float limit = INFINITY;
  float alpha = 1.0f;
  float plus = 0.0f;
};
__device__ __forceinline__ float gated_unit(float g, float u, const Glu& p) {
  g = fminf(g, p.limit);
  u = fminf(fmaxf(u, -p.limit), p.limit);
  return g / (1.0f + __expf(-(p.alpha * g))) * (u + p.plus);
}

// A lane's 16 bytes, or zeros where it has nothing to read: then the address is one of zeros, so that a run of loads stays one
// stretch of code, which a branch round each of them would cut up.  (Named as global memory: of an address that is one of two the
// compiler cannot tell, and would wait for all loads where it needs the first.)  For kernels that ask for all they read at once;
// a long loop is faster with the branches (see gemm_skinny_kernel).
__device__ const bf16x8 kZeros = {};
__device__ __forceinline__ const bf16x8 __attribute__((address_space(1))) * or_zeros(bool ok, const bf16* p) {
  typedef const bf16x8 __attribute__((address_space(1))) * global_words;
  return ok ? (global_words)(uintptr_t)p : (global_words)(uintptr_t)&kZeros;
}

// What a product of at most 64 rows may do for the RMS norm that follows it or precedes it.
//  * emit (gemm_few_kernel for up to 16 rows, the skinny kernel beyond; accumulating into the float32 residual):
//    besides the new residual r it writes h[m, n] = bf16(gamma[n] * r[m, n]), the operand of the next product, and
//    for every tile of columns (8 or 16: gb_gemm_bf16_emit_parts says how many tiles) the sums over them of
//    r[m, n]^2 to ss[tile * stride + m]: the next norm's pass over the residual is done where the residual is made.
//    stride = parts_stride(M): 8 for up to 8 rows, 64 beyond.
//  * parts (the same two, and the held kernel): the rows of A are such an h; the product is scaled by
//    1 / sqrt(sum of the n_parts partial sums of row m / K + eps), added up in the order of the tiles.
__host__ __device__ __forceinline__ int parts_stride(int M) { return M <= 8 ? 8 : 64; }
struct NormExtras {
  const void* emit_gamma;
  int emit_gamma_f32;
  bf16* emit_h;
  int emit_ldh;
  float* emit_ss;
  const float* parts;
  int n_parts;
  Glu glu;   // the gated unit of an EPI_SILU_MUL product
};

// EPI_ROPE (gemm_few_kernel, the skinny and the held kernel; the QKV product of a decode step): W stacks nh query heads, nkv key heads
// and nkv value heads of hd rows each.  The product rotates query and key heads by the angles of each
// row's position (pairs (i, i + hd/2), crates/glassbox-core/src/model.rs:102-115) while the sums are
// still 32-bit, writes the stacked rows to C as usual, and the key and value heads straight into the
// cache pages at slots[m] (keys [page][kv head][hd / 8][slot][8], values [page][kv head][hd][slot]) if slots is
// given: the rotation kernel and its round trip through memory are not needed.
struct RopeExtras {
  const float* cosv;   // [M][hd/2], nullptr: no rotation
  const float* sinv;
  const int32_t* slots;  // [M], nullptr: nothing is stored
  bf16* k_pages;
  bf16* v_pages;
  int nh, nkv, hd, page_size;
  int three_halves;  // the launch gives a workgroup a tile and a half (see three_halves_tile), not two tiles
  float per_tile;    // 8 / hd: heads a tile of 8 rows (the kernel for up to 8 rows of A), and the page size as a shift
  int page_shift;    // (-1: no power of two)
};

// Tiles of the skinny kernel's rotating product, 8 pairs each, dealt a tile and a half to a workgroup: workgroup g
// takes tile 3g/2 whole and the first four pairs of the next (g even), or the last four pairs of tile (3g - 1)/2 and
// the next whole (g odd).  384 tiles (the 6,144 rows of a QKV product) then make 256 workgroups of equal work, one for
// every compute unit, where two tiles each would make 192.  [lo, hi): the pairs of tile rt that are the workgroup's.
__device__ __forceinline__ int three_halves_tile(int g, int rt, int* lo, int* hi) {
  *lo = (g & 1) && rt == 0 ? 4 : 0;
  *hi = !(g & 1) && rt == 1 ? 4 : 8;
  return ((g & 1) ? (3 * g - 1) / 2 : 3 * g / 2) + rt;
}

template <typename CT> __device__ __forceinline__ void store_c(CT* c, float v, int accumulate);
template <> __device__ __forceinline__ void store_c<float>(float* c, float v, int accumulate) { *c = accumulate ? *c + v : v; }
template <> __device__ __forceinline__ void store_c<bf16>(bf16* c, float v, int) { *c = (bf16)v; }

// ------------------------------------------------------------------------- tiled
// A workgroup of 2 x 2 waves; a wave owns WM x WN tiles of 32 x 32, so the workgroup's tile is
// (64 WM) x (64 WN).  Operands are staged through LDS in k-steps of 64, two buffers; rows are padded
// to 144 bytes so that the 16-byte operand reads of a wave spread over the banks.
//
// EPI_SILU_MUL (WN = 2): W stacks gate rows [0, N/2) over up rows [N/2, N).  Of a wave's two column
// tiles the first holds 32 gate columns and the second the 32 up columns that belong to them, so
// act = gate / (1 + exp(-gate)) * up (crates/glassbox-core/src/model.rs:336-340) is formed in
// registers and C is [M, N/2].
enum : int { EPI_STORE = 0, EPI_ACCUMULATE = 1, EPI_SILU_MUL = 2, EPI_ROPE = 3 };
constexpr int TBK = 64, TLD = TBK + 8;  // k-step; LDS row stride in elements (144 bytes)
constexpr int TCPR = TBK / 8;           // 16-byte chunks per row of a k-step
constexpr int TKS = TBK / 16;           // MFMA k-steps per LDS k-step

//
// GROUPED: the rows of A fall into groups that each have a W of their own (the tokens of an expert).  Row tile
// blockIdx.y is not rows [y BM, (y + 1) BM) but what grp.map says of it: three numbers a tile, the group (below zero: a
// tile that this launch does not need), the tile's first row and the end of its group's rows, which takes the place of M.
// The group's W begins grp.w_stride elements a group further on; with EPI_SILU_MUL its up rows lie grp.up_off rows
// behind its gate rows.  grp.rows, if given, names the row of A behind each row of the product.
struct Groups {
  const int32_t* map;
  const int32_t* rows;
  long long w_stride;
  int up_off;
  int slice_rows;   // rows of C a slice of k (the ring kernel's grouped form)
  const float* in_scale;   // with EPI_SILU_MUL, if given: what each row of A is multiplied by (both sums are, before the unit)
};

template <int WM, int WN, int DEPTH, int EPI, bool KFULL, typename CT, bool GROUPED = false>
__global__ __launch_bounds__(256, WN == 2 ? 2 : 1) void gemm_tiled_kernel(const bf16* __restrict__ a, int lda, const bf16* __restrict__ w,
                                                         int ldw, CT* __restrict__ c, int ldc, int M, int N, int K,
                                                         int k_slice, Groups grp, Glu glu) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  constexpr int CA = BM * TCPR / 256, CW = BN * TCPR / 256;  // chunks a thread moves per k-step
  if (k_slice > 0) {  // split k: workgroup z of a tile sums its own slice of k into its own copy of C
    const int z = blockIdx.z;
    a += (size_t)z * k_slice;
    w += (size_t)z * k_slice;
    c += (size_t)z * M * ldc;
    K = min(k_slice, K - z * k_slice);
  }
  __shared__ __attribute__((aligned(16))) bf16 As[2][BM][TLD];
  __shared__ __attribute__((aligned(16))) bf16 Ws[2][BN][TLD];
  constexpr bool SCALES = GROUPED && EPI == EPI_SILU_MUL;
  __shared__ float in_scale[SCALES ? BM : 1];   // the rows' factors (read behind the loop's barriers)
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / 2, wn = wave % 2;
  int m0 = blockIdx.y * BM;
  const int half = N / 2;  // EPI_SILU_MUL: number of gate rows
  int up_off = half;       // and how far behind its gate row an up row lies
  if constexpr (GROUPED) {
    const int32_t* tile = grp.map + 3 * blockIdx.y;
    const int group = tile[0];
    if (group < 0) return;
    m0 = tile[1];
    M = tile[2];
    w += (size_t)group * grp.w_stride;
    up_off = grp.up_off;
    if (SCALES && grp.in_scale && tid < BM) in_scale[tid] = grp.in_scale[min(m0 + tid, M - 1)];
  }
  // row of W behind row r of the workgroup's W tile (r = wn*32*WN + j*32 + column)
  auto w_row = [&](int r) -> int {
    if (EPI == EPI_SILU_MUL) {
      const int wv = r / 64, j = (r % 64) / 32, col = r % 32;
      const int n = blockIdx.x * 64 + wv * 32 + col;
      return n < half ? (j ? up_off + n : n) : -1;
    }
    const int n = blockIdx.x * BN + r;
    return n < N ? n : -1;
  };

  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // Chunks on their way from memory to LDS wait in registers, DEPTH k-steps' worth: a load has DEPTH
  // k-steps of arithmetic to arrive in before its registers are written to LDS.  Within a k-step the
  // LDS writes and the loads that refill their registers are spread over the first three of the four
  // MFMA steps, so that memory requests and arithmetic are issued side by side, not in bursts.
  // Rows beyond M or N are read from a row that exists (their results are never stored), so that the
  // loop has no branch around a load.
  constexpr int CT_ = CA + CW;
  bf16x8 held[DEPTH][CT_];
  const bf16* src[CT_];
#pragma unroll
  for (int ci = 0; ci < CT_; ++ci) {
    const int ch = tid + 256 * (ci < CA ? ci : ci - CA);
    if (ci < CA) {
      int row = min(m0 + ch / TCPR, M - 1);
      if constexpr (GROUPED) {
        if (grp.rows) row = grp.rows[row];
      }
      src[ci] = a + (size_t)row * lda + (ch % TCPR) * 8;
    } else {
      src[ci] = w + (size_t)max(w_row(ch / TCPR), 0) * ldw + (ch % TCPR) * 8;
    }
  }
  auto fetch = [&](int ci, int k0, auto set) {
    if constexpr (KFULL) {
      held[decltype(set)::value][ci] = load8(src[ci] + k0);
    } else {
      const int ch = tid + 256 * (ci < CA ? ci : ci - CA);
      held[decltype(set)::value][ci] = k0 + (ch % TCPR) * 8 < K ? load8(src[ci] + k0) : zero8();
    }
  };
  auto stash = [&](int ci, int buf, auto set) {
    const int ch = tid + 256 * (ci < CA ? ci : ci - CA);
    bf16* dst = ci < CA ? &As[buf][ch / TCPR][(ch % TCPR) * 8] : &Ws[buf][ch / TCPR][(ch % TCPR) * 8];
    *reinterpret_cast<bf16x8*>(dst) = held[decltype(set)::value][ci];
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  using Yes = std::true_type;
  using No = std::false_type;

  const int steps = (K + TBK - 1) / TBK;
  const int arow = wm * 32 * WM + lane % 32, wrow = wn * 32 * WN + lane % 32, koff = 8 * (lane / 32);
  bf16x8 fa[2][WM], fw[2][WN];  // operands of MFMA step ks+1 are read from LDS while the MFMAs of step ks run
  auto read_operands = [&](int buf, int kk, int into) {
#pragma unroll
    for (int i = 0; i < WM; ++i) fa[into][i] = *reinterpret_cast<const bf16x8*>(&As[buf][arow + i * 32][kk * 16 + koff]);
#pragma unroll
    for (int j = 0; j < WN; ++j) fw[into][j] = *reinterpret_cast<const bf16x8*>(&Ws[buf][wrow + j * 32][kk * 16 + koff]);
  };
  // k-step s is computed from LDS buffer s % 2.  Register set `other` holds k-step s + 1: it is written
  // to the other buffer (if there is a k-step s + 1: more), and loaded again with k-step s + 1 + DEPTH
  // (if there is one: refill).  The barrier stands before the last MFMA step: by then every wave has
  // written its part of k-step s + 1 and has read the last operands of k-step s, so the last MFMA
  // step can already read the first operands of k-step s + 1.
  static_assert(TKS == 4, "the schedule below is written for four MFMA steps per k-step");
  auto step = [&](int s, auto other, auto more, auto refill) {
    const int buf = s & 1;
#pragma unroll
    for (int ks = 0; ks < TKS; ++ks) {
      const int cur = ks & 1, nxt = cur ^ 1;
      if (ks + 1 < TKS)
        read_operands(buf, ks + 1, nxt);
      else if (decltype(more)::value)
        read_operands(buf ^ 1, 0, nxt);
      if (ks < 3) {
#pragma unroll
        for (int ci = ks; ci < CT_; ci += 3) {
          if (decltype(more)::value) stash(ci, buf ^ 1, other);
          if (decltype(refill)::value) fetch(ci, (s + 1 + DEPTH) * TBK, other);
        }
      }
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[cur][i], fw[cur][j], acc[i][j], 0, 0, 0);
      if (ks == 2) __syncthreads();
      __builtin_amdgcn_sched_barrier(0);  // each MFMA step keeps its share of the memory traffic
    }
  };

  auto any_step = [&](int s, auto other) {  // near the end fewer and fewer k-steps have something ahead of them
    if (s + 1 + DEPTH < steps)
      step(s, other, Yes{}, Yes{});
    else if (s + 1 < steps)
      step(s, other, Yes{}, No{});
    else
      step(s, other, No{}, No{});
  };
#pragma unroll
  for (int ci = 0; ci < CT_; ++ci) fetch(ci, 0, Set0{});
  if (DEPTH == 2 && steps > 1) {
#pragma unroll
    for (int ci = 0; ci < CT_; ++ci) fetch(ci, TBK, std::integral_constant<int, DEPTH - 1>{});
  }
#pragma unroll
  for (int ci = 0; ci < CT_; ++ci) stash(ci, 0, Set0{});
  if (steps > DEPTH) {
#pragma unroll
    for (int ci = 0; ci < CT_; ++ci) fetch(ci, DEPTH * TBK, Set0{});
  }
  __syncthreads();
  read_operands(0, 0, 0);
  int s = 0;
  if constexpr (DEPTH == 2) {
    for (; s + 4 < steps; s += 2) {  // both k-steps of a round have a k-step three ahead
      step(s, Set1{}, Yes{}, Yes{});
      step(s + 1, Set0{}, Yes{}, Yes{});
    }
    for (; s < steps; s += 2) {
      any_step(s, Set1{});
      if (s + 1 < steps) any_step(s + 1, Set0{});
    }
  } else {
    for (; s + 2 < steps; ++s) step(s, Set0{}, Yes{}, Yes{});
    for (; s < steps; ++s) any_step(s, Set0{});
  }

  // accumulator layout of a 32x32 tile: lane holds column lane%32, rows 8*(r/4) + 4*(lane/32) + r%4
  if (EPI == EPI_SILU_MUL) {
    const int gn = blockIdx.x * 64 + wn * 32 + lane % 32;
    if (gn >= half) return;
    const bool scaled = SCALES && grp.in_scale;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = m0 + wm * 32 * WM + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
        float g = acc[i][0][r], u = acc[i][WN - 1][r];
        if (SCALES && scaled) {
          const float s = in_scale[wm * 32 * WM + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4];
          g *= s, u *= s;
        }
        if (gm < M) c[(size_t)gm * ldc + gn] = (CT)gated_unit(g, u, glu);
      }
    return;
  }
  if constexpr (EPI == EPI_ACCUMULATE) {
    // a wave whose tiles lie wholly inside C reads all old values of a tile before it adds: behind the checks
    // below every read would wait for the one before it
    if (m0 + (wm + 1) * 32 * WM <= M && blockIdx.x * BN + (wn + 1) * 32 * WN <= N) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          CT* base = c + (size_t)(m0 + wm * 32 * WM + i * 32 + 4 * (lane / 32)) * ldc + blockIdx.x * BN + wn * 32 * WN + j * 32 + lane % 32;
          float old[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) old[r] = (float)base[(size_t)(8 * (r / 4) + r % 4) * ldc];
#pragma unroll
          for (int r = 0; r < 16; ++r) base[(size_t)(8 * (r / 4) + r % 4) * ldc] = (CT)(old[r] + acc[i][j][r]);
        }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = blockIdx.x * BN + wn * 32 * WN + j * 32 + lane % 32;
      if (gn >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = m0 + wm * 32 * WM + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
        if (gm < M) store_c<CT>(c + (size_t)gm * ldc + gn, acc[i][j][r], EPI == EPI_ACCUMULATE);
      }
    }
}

// Tile of the workgroup, bm x (64 wn), how many there are, and the depth of the register prefetch.  128 x 128 re-reads
// the operands least; 128 x 64 when that would leave compute units idle.  The wide tile's registers
// allow two workgroups a compute unit only with one k-step of prefetch, the narrow tile's with two.
// Tiles of 64 rows where those of 128 would leave a third of the compute units without a workgroup (the
// products of a narrow model at some hundred rows): a workgroup's time is its k-steps' arithmetic, and half the
// rows halve it.  A SiLU-multiply product, whose workgroups take 128 rows of W each, gains up to 300 workgroups
// (two of the smaller ones share a compute unit: gate/up of 256 rows on SmolLM2-1.7B shapes 34 -> 30 us, of 640 to
// 896 rows on SmolLM2-360M shapes 17 -> 14 and 24 -> 20 us; the other products lose from 168 on).
struct TiledGrid {
  int wn, depth, bm, cols, rows;   // cols x rows workgroups
  long long groups() const { return (long long)cols * rows; }
};
inline TiledGrid tiled_grid(int epi, int M, int N) {
  const long long blocks = (long long)((M + 127) / 128) * ((N + 127) / 128);
  TiledGrid g;
  g.wn = blocks < 384 ? 1 : 2;
  g.depth = g.wn == 1 ? 2 : 1;
  if (epi == EPI_SILU_MUL) g.wn = 2;  // a wave's two column tiles are gate and up
  const int cols = epi == EPI_SILU_MUL ? N / 2 : N, bn = epi == EPI_SILU_MUL ? 64 : 64 * g.wn;
  g.cols = (cols + bn - 1) / bn;
  const bool low = M > 64 && (long long)g.cols * ((M + 127) / 128) < (epi == EPI_SILU_MUL ? 300 : 168);
  g.bm = low ? 64 : 128;
  if (low) g.depth = g.wn == 1 ? 2 : 1;
  g.rows = (M + g.bm - 1) / g.bm;
  return g;
}

template <int EPI, typename CT>
int launch_tiled(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, hipStream_t stream,
                 Glu glu = Glu{}) {
  const TiledGrid g = tiled_grid(EPI, M, N);
  const int wn = g.wn, depth = g.depth;
  const bool low = g.bm == 64;
  const dim3 grid(g.cols, g.rows), block(256);
  GB_REQUIRE(grid.y <= 65535, "gemm_bf16: M=%d needs more than 65535 row tiles", M);
  const bool kfull = K % TBK == 0;  // then no load needs a check against K
#define GB_T(WM, B, D)                                                                                                      \
  if (wn == (B) && depth == (D)) {                                                                                          \
    if (kfull)                                                                                                              \
      hipLaunchKernelGGL((gemm_tiled_kernel<WM, (B), (D), EPI, true, CT>), grid, block, 0, stream, a, lda, w, ldw, c, ldc, M, \
                         N, K, 0, Groups{}, glu);                                                                                          \
    else                                                                                                                    \
      hipLaunchKernelGGL((gemm_tiled_kernel<WM, (B), (D), EPI, false, CT>), grid, block, 0, stream, a, lda, w, ldw, c, ldc,  \
                         M, N, K, 0, Groups{}, glu);                                                                                       \
  }
  if (low) {
    GB_T(1, 2, 1)
    if (EPI != EPI_SILU_MUL) { GB_T(1, (EPI == EPI_SILU_MUL ? 2 : 1), 2) }
  } else {
    GB_T(2, 2, 1) GB_T(2, 2, 2)
    if (EPI != EPI_SILU_MUL) { GB_T(2, (EPI == EPI_SILU_MUL ? 2 : 1), 1) GB_T(2, (EPI == EPI_SILU_MUL ? 2 : 1), 2) }
  }
#undef GB_T
  return launched("gemm_bf16 (tiled)");
}

// ------------------------------------------------------------------------- ring
// Large products (many rows, many tiles): a workgroup of 2 x 2 waves with a tile of 256 x 256, a wave 8 x 8 tiles of
// 16 x 16, whose sums fill the accumulation registers (one wave a SIMD); or of 256 columns and fewer rows, 32 H, where tiles
// of 256 would leave many compute units idle in a last round (ring_rows).  Operands go from memory straight into LDS
// (global_load_lds, 16 bytes a lane: a wave's instruction fills 1 KB of LDS in lane order, so the lane decides which
// piece of memory lands where), in k-steps of 64, so that an instruction brings eight whole lines of 128 bytes.  LDS, all
// of it, is a ring of five slots of 256 rows by 64 of k: A and W of the k-step that is multiplied, A and W of the next
// and A of the one after.  A row of a k-step is 128 bytes = 8 pieces; piece c of row r lies at position
// c ^ ((r >> 1) & 7), which spreads the 16-byte operand reads of 16 neighbouring rows over all banks.
//
// The matrix cores take W as their first operand and A as the second, so that a lane holds four neighbouring columns of a row of
// C: an epilogue of whole words.
//
// The compiler knows nothing of what those loads write, and left to itself it keeps neither the accumulators in place nor
// this order.  So the operand reads and the MFMAs are inline assembly, issued in the order written here (an operand read or a
// request to memory between MFMAs costs no cycle of theirs), and the waits are written by hand:
//   * lgkmcnt before the 64 MFMAs that use the operands (read among the 64 before them);
//   * the barrier of a k-step stands between its two blocks of 64 MFMAs.  Before it a wave waits for its last operand
//     reads of the k-step (lgkmcnt) and for its own loads of the next one (vmcnt: loads retire in order).  After it,
//     every wave's loads of the next k-step have landed, so its operands may be read (they arrive under the second
//     block), and every wave is done with this k-step's slots, so that W of k-step + 2 may overwrite its A, and A of
//     k-step + 3 its W (in the next k-step's first block).
//
// What bounds it: power and the way from memory.  Multiplying 8,192^3, the chip runs at 1.7 GHz, and all-zero operands take 640 us
// where random ones take 749; without requests to memory it would take 530.  The kernel before this one (eight waves of 128 x 64,
// 32 x 32 x 16 MFMAs, k-steps of 32, so that a request brought half lines: twice the requests to the second-level cache) kept
// the matrix cores busy for 71 % of the cycles.  us, before -> now, same box: 8,192^3 842 -> 749 (1,468 TFLOP/s);
// 6,151 x 28,672 x 4,096 with SiLU-multiply (another card) 1,283 -> 1,143; 6,151 x 4,096 x 14,336 676 -> 584.  Tried: the same with 32 x 32 x 16 MFMAs
// (8,192^3: 850 where this took 805); tiles dealt to the dies in squares (no gain).
constexpr int RING_SLOTS = 5;   // (RBK, a k-step, and what slices of k may be: ring_steps.h)
constexpr int RGM = 2, RGN = 2, RT = 8;                  // waves along m, n; 16 x 16 tiles of a wave along m and along n
constexpr int RBM = RGM * RT * 16, RBN = RGN * RT * 16;  // 256 x 256
constexpr int RL = RBM / 8 / (RGM * RGN);                // loads of a wave that bring its share of a slot
static_assert(RBM == RBN, "a slot of the ring holds either operand");
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

__device__ __forceinline__ bf16x8 lds_read16(uint32_t addr) {
  bf16x8 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr) : "memory");
  return v;
}
// waits until at most LEFT LDS reads are outstanding; the operands named become usable
template <int LEFT, int NA, int NB>
__device__ __forceinline__ void lds_wait(bf16x8 (&fa)[NA], bf16x8 (&fb)[NB]) {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(LEFT) : "memory");
#pragma unroll
  for (int i = 0; i < NA; ++i) asm volatile("" : "+v"(fa[i]));
#pragma unroll
  for (int j = 0; j < NB; ++j) asm volatile("" : "+v"(fb[j]));
}
// waits until at most LEFT of this wave's loads from memory are on their way (the counter's six bits lie in two
// places of the instruction's operand: bits 3:0 and 15:14; the other counters are left alone)
template <int LEFT> __device__ __forceinline__ void vm_wait() {
  static_assert(LEFT >= 0 && LEFT < 64, "the counter has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (LEFT & 15) | ((LEFT >> 4) << 14));
}

// four neighbouring columns of a row of C
template <typename CT> __device__ __forceinline__ void store_c4(CT* c, const f32x4& v);
template <> __device__ __forceinline__ void store_c4<float>(float* c, const f32x4& v) { *reinterpret_cast<f32x4*>(c) = v; }
template <> __device__ __forceinline__ void store_c4<bf16>(bf16* c, const f32x4& v) {
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = (bf16)v[r];
  *reinterpret_cast<bf16x4*>(c) = o;
}

// One tile of 32 H rows by 256 rows of W.  GROUPED: see the kernel.
template <int EPI, typename CT, bool GROUPED, int H>
__device__ __forceinline__ void ring_tile(bf16 (&ring)[RING_SLOTS][RBM * RBK], const bf16* __restrict__ a, int lda, const bf16* __restrict__ w,
                                          int ldw, CT* __restrict__ c, int ldc, int M, int N, int K, bool head, int bx, int m0,
                                          int up_off, const Groups& grp, const Glu& glu) {
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / RGN, wn = wave % RGN;
  const int half = N / 2;  // EPI_SILU_MUL: number of gate rows
  // row of W behind row r of the workgroup's W tile (r = wn * 128 + j * 16 + column); with EPI_SILU_MUL a wave's
  // even column tiles hold gate rows and the odd ones the up rows that belong to them
  auto w_row = [&](int r) -> int {
    if (EPI == EPI_SILU_MUL) {
      const int j = r % (RT * 16) / 16;
      const int n = bx * (RBN / 2) + r / (RT * 16) * (RT / 2 * 16) + j / 2 * 16 + r % 16;
      return n < half ? (j % 2 ? up_off + n : n) : 0;
    }
    return min(bx * RBN + r, N - 1);
  };
  // a wave's load instruction moves 8 rows x 8 pieces; rows beyond M or N are read from a row that exists
  const bf16* asrc[H];
  const bf16* wsrc[RL];
#pragma unroll
  for (int t = 0; t < H; ++t) {
    const int row = (wave * H + t) * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
    int arow = min(m0 + row, M - 1);
    if constexpr (GROUPED) {
      if (grp.rows) arow = grp.rows[arow];
    }
    asrc[t] = a + (size_t)arow * lda + piece * 8;
  }
#pragma unroll
  for (int t = 0; t < RL; ++t) {
    const int row = (wave * RL + t) * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
    wsrc[t] = w + (size_t)w_row(row) * ldw + piece * 8;
  }
  auto load_a = [&](int t, int slot, int k0) {
    __builtin_amdgcn_global_load_lds((glb_void*)(asrc[t] + k0), (lds_void*)&ring[slot][(wave * H + t) * 8 * RBK], 16, 0, 0);
  };
  auto load_w = [&](int t, int slot, int k0) {
    __builtin_amdgcn_global_load_lds((glb_void*)(wsrc[t] + k0), (lds_void*)&ring[slot][(wave * RL + t) * 8 * RBK], 16, 0, 0);
  };
  f32x4 acc[H][RT];
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  // operand of block kh (0, 1): row lane % 16 of a 16-row tile, piece 4 kh + lane / 16
  uint32_t off[2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) off[kh] = 2 * ((lane % 16) * RBK + (((4 * kh + lane / 16) ^ ((lane >> 1) & 7)) * 8));
  constexpr uint32_t SLOT = 2 * RBM * RBK, TILE = 2 * 16 * RBK;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)&ring[0][0];
  const uint32_t abase = base + wm * H * TILE, wbase = base + wn * RT * TILE;

  // GROUPED: a group's last tile may hold few rows: a wave leaves out the MFMAs of rows of 16 that lie beyond the group's end,
  // in its second half, between whose MFMAs nothing else stands: a branch each eight of them, which their time hides.  (us of
  // two experts of eight a token, 2,048 tokens, 4,096 units of 2,048, gate/up and down, traced: 159 and 113; a branch before
  // every MFMA 226 and 152; the kernel with k-steps of 32 175 and 112.)
  const int live = GROUPED ? __builtin_amdgcn_readfirstlane(min(max((M - m0 - wm * RT * 16 + 15) / 16, 0), RT)) : RT;

  // k-steps; the last may hold a half that counts as zeros
  const int steps = ring_steps(K), dead = ring_dead_half(K, head);
  auto k_of = [&](int s) { return ring_step_at(s, K, head); };
  bf16x8 fa[2][H], fw[2][RT];
  auto read_a = [&](int set, int t, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][t]) : "v"(addr), "n"(t * TILE) : "memory");
  };
  auto read_w = [&](int set, int t, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fw[set][t]) : "v"(addr), "n"(t * TILE) : "memory");
  };
  constexpr int LIVE_FROM = RT / 2;
  static_assert(RT == 8 && H >= 4 && H <= 8 && 2 * RT <= RT * LIVE_FROM / 2 && 4 * RL <= RT * LIVE_FROM,
                "the reads and the loads stand among the first half's MFMAs");
  // The 8 H MFMAs of operand set `set`; among them the reads of the other set from ra and rw, and (with `more`) a slot's
  // loads from memory: of A among those of set 0, of W among those of set 1.
  auto block = [&](auto which, uint32_t ra, uint32_t rw, bool more, int slot, int k0) {
    constexpr int set = decltype(which)::value;
#pragma unroll
    for (int at = 0; at < H * RT; ++at) {
      const int i = at / RT, j = (i & 1) ? RT - 1 - at % RT : at % RT;
      if constexpr (GROUPED) {
        if (i >= LIVE_FROM) {
          if (at % RT == 0)
            asm volatile(
                "s_cmp_le_i32 %17, %18\n\ts_cbranch_scc1 .Lbeyond%=\n\t"
                "v_mfma_f32_16x16x32_bf16 %0, %8, %16, %0\n\tv_mfma_f32_16x16x32_bf16 %1, %9, %16, %1\n\t"
                "v_mfma_f32_16x16x32_bf16 %2, %10, %16, %2\n\tv_mfma_f32_16x16x32_bf16 %3, %11, %16, %3\n\t"
                "v_mfma_f32_16x16x32_bf16 %4, %12, %16, %4\n\tv_mfma_f32_16x16x32_bf16 %5, %13, %16, %5\n\t"
                "v_mfma_f32_16x16x32_bf16 %6, %14, %16, %6\n\tv_mfma_f32_16x16x32_bf16 %7, %15, %16, %7\n.Lbeyond%=:"
                : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]),
                  "+a"(acc[i][6]), "+a"(acc[i][7])
                : "v"(fw[set][0]), "v"(fw[set][1]), "v"(fw[set][2]), "v"(fw[set][3]), "v"(fw[set][4]), "v"(fw[set][5]),
                  "v"(fw[set][6]), "v"(fw[set][7]), "v"(fa[set][i]), "s"(live), "n"(i) : "scc");
          continue;
        }
      }
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fw[set][j]), "v"(fa[set][i]));
      if (at % 2 == 0 && at / 2 < H) read_a(set ^ 1, at / 2, ra);
      else if (at % 2 == 0 && at / 2 < H + RT) read_w(set ^ 1, at / 2 - H, rw);
      else if (at % 4 == 1 && at / 4 < (set == 1 ? RL : H) && more) {
        if constexpr (set == 1) load_w(at / 4, slot, k0);
        else load_a(at / 4, slot, k0);
      }
    }
  };
  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, 1>;
#pragma unroll
  for (int t = 0; t < H; ++t) load_a(t, 0, k_of(0));
#pragma unroll
  for (int t = 0; t < RL; ++t) load_w(t, 1, k_of(0));
  if (steps > 1) {
#pragma unroll
    for (int t = 0; t < H; ++t) load_a(t, 2, k_of(1));
#pragma unroll
    for (int t = 0; t < RL; ++t) load_w(t, 3, k_of(1));
    vm_wait<H + RL>();
  } else {
    vm_wait<0>();
  }
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    if (t < H) read_a(0, t, abase + off[0]);
    read_w(0, t, wbase + SLOT + off[0]);
  }
  int sa = 0, sw = 1;   // this k-step's slots
  auto behind = [](int slot, int by) { return slot + by >= RING_SLOTS ? slot + by - RING_SLOTS : slot + by; };
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    const bool more = s + 2 < steps;
    const int na = behind(sa, 2), nw = behind(sw, 2), k2 = k_of(s + 2);
    lds_wait<0>(fa[0], fw[0]);
    if (dead == 0 && s + 1 == steps) {
#pragma unroll
      for (int t = 0; t < RT; ++t) fa[0][min(t, H - 1)] = fw[0][t] = zero8();
    }
    block(First{}, abase + sa * SLOT + off[1], wbase + sw * SLOT + off[1], more, behind(sa, 4), k2);
    lds_wait<0>(fa[1], fw[1]);
    if constexpr (GROUPED) {
      if (dead == 1) {   // (the only k-step)
#pragma unroll
        for (int t = 0; t < RT; ++t) fa[1][min(t, H - 1)] = fw[1][t] = zero8();
      }
    }
    if (more) vm_wait<H>();   // (A of k-step s + 2 may still be on its way)
    else vm_wait<0>();
    __builtin_amdgcn_s_barrier();
    block(Second{}, abase + na * SLOT + off[0], wbase + nw * SLOT + off[0], more, sa, k2);   // (behind the last: read, not used)
    sa = na, sw = nw;
  }
  lds_wait<0>(fa[0], fw[0]);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs' results, which the compiler does not know to wait for
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int j = 0; j < RT; ++j) asm volatile("" : "+a"(acc[i][j]));

  // A lane holds row lane % 16 of a tile and its columns 4 (lane / 16) .. + 3.
  constexpr int OUT = EPI == EPI_SILU_MUL ? RT / 2 : RT;   // column tiles of the wave's results
  const int cols = EPI == EPI_SILU_MUL ? half : N;
  const int gm0 = m0 + wm * H * 16, gn0 = bx * (RGN * OUT * 16) + wn * (OUT * 16);
  auto result = [&](int i, int j, float factor) -> f32x4 {   // of row tile i, column tile j of the results
    if constexpr (EPI == EPI_SILU_MUL) {
      f32x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = gated_unit(acc[i][2 * j][r] * factor, acc[i][2 * j + 1][r] * factor, glu);
      return v;
    } else {
      return acc[i][j];
    }
  };
  const bool scaled = GROUPED && EPI == EPI_SILU_MUL && grp.in_scale;
  const bool words = (size_t)ldc * sizeof(CT) % 16 == 0 && (uintptr_t)c % 16 == 0;   // rows of C are whole words
  if (gn0 + OUT * 16 <= cols && words) {   // the same for the whole wave
    if constexpr (sizeof(CT) == 2) {
      // As they lie, a store of the wave would write 32 bytes of 16 rows; so bfloat16 results go through LDS (32 KB of the
      // wave's own: every wave has read its last operands) and out in runs of 128 or 256 bytes (8,192 x 16,384 x 128, a
      // product that is mostly epilogue: 109 -> 83 us).
      constexpr int ROW = OUT * 32, PIECES = ROW / 16;   // bytes and 16-byte pieces of a row
      static_assert(RT * 16 * ROW * RGM * RGN <= (int)sizeof(ring), "the waves' rows fit the ring");
      char* own = reinterpret_cast<char*>(&ring[0][0]) + wave * (RT * 16 * ROW);
#pragma unroll
      for (int i = 0; i < H; ++i) {
        const int row = i * 16 + lane % 16;
        const float factor = scaled ? grp.in_scale[min(gm0 + row, M - 1)] : 1.f;
#pragma unroll
        for (int j = 0; j < OUT; ++j)   // half a piece; piece p of a row lies at position p ^ (row % PIECES)
          store_c4<CT>(reinterpret_cast<CT*>(own + row * ROW + ((2 * j + lane / 32) ^ (row % PIECES)) * 16 + lane / 16 % 2 * 8), result(i, j, factor));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      constexpr int RUN = 64 / PIECES, STORES = H * 16 / RUN;   // rows a store of the wave covers
      constexpr int AT_ONCE = STORES % 8 == 0 ? 8 : STORES % 7 == 0 ? 7 : STORES % 6 == 0 ? 6 : STORES % 5 == 0 ? 5 : 4;
      static_assert(STORES % AT_ONCE == 0, "whole turns");
#pragma unroll
      for (int it = 0; it < STORES; it += AT_ONCE) {
        f32x4 v[AT_ONCE];
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
          const int row = (it + u) * RUN + lane / PIECES;
          v[u] = *reinterpret_cast<const f32x4*>(own + row * ROW + ((lane % PIECES) ^ (row % PIECES)) * 16);
        }
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
          const int row = (it + u) * RUN + lane / PIECES;
          if (gm0 + row < M) *reinterpret_cast<f32x4*>(c + (size_t)(gm0 + row) * ldc + gn0 + lane % PIECES * 8) = v[u];
        }
      }
    } else {
      // 64 bytes of 16 rows a store: through LDS and out in runs of 256 they were no faster.  What is added to: the old values
      // of two row tiles are on their way while a third's are added to (8,192 x 4,096 x 4,096: 233 -> 228 us).
      constexpr int DEEP = EPI == EPI_ACCUMULATE ? 3 : 1;
      f32x4 old[DEEP][OUT];
      auto to_of = [&](int i) { return c + (size_t)min(gm0 + i * 16 + lane % 16, M - 1) * ldc + gn0 + 4 * (lane / 16); };
      auto ask = [&](int i) {
#pragma unroll
        for (int j = 0; j < OUT; ++j) old[i % DEEP][j] = *reinterpret_cast<const f32x4*>(to_of(i) + j * 16);
      };
      if constexpr (EPI == EPI_ACCUMULATE) {
        ask(0);
        ask(1);
      }
      // (what is stored goes by one place that moves on: eight of them at once were more than the registers hold: 1,157 x 11,280 x 128
      // in 32-bit 18.9 / 17.1 us)
      CT* at = c + (size_t)(gm0 + lane % 16) * ldc + gn0 + 4 * (lane / 16);
#pragma unroll
      for (int i = 0; i < H; ++i) {
        const int gm = gm0 + i * 16 + lane % 16;
        if constexpr (EPI == EPI_ACCUMULATE) {
          if (i + 2 < H) ask(i + 2);
        } else {
          asm volatile("" : "+v"(at));
        }
        if (gm < M) {
          CT* to = EPI == EPI_ACCUMULATE ? to_of(i) : at;
          const float factor = scaled ? grp.in_scale[gm] : 1.f;
#pragma unroll
          for (int j = 0; j < OUT; ++j) {
            f32x4 v = result(i, j, factor);
            if constexpr (EPI == EPI_ACCUMULATE) v = old[i % DEEP][j] + v;
            store_c4<CT>(to + j * 16, v);
          }
        }
        at += (size_t)16 * ldc;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    return;
  }
  // The last columns of C: four of them a lane, where none of a lane's lies beyond.  (One after the other, a column's old value was
  // waited for before the next one's was asked for, 256 of them, and the launch waited for those tiles.  us, so / now: added to, 8,192 x
  // 5,344 x 512 139 / 96, 7,161 x 3,552 x 960 113 / 71; stored in 32-bit 83 / 73, 65 / 60.)
  if (words && cols % 4 == 0) {
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const int gm = gm0 + i * 16 + lane % 16, gn = gn0 + 4 * (lane / 16);
      if (gm >= M) continue;
      CT* to = c + (size_t)gm * ldc + gn;
      const float factor = scaled ? grp.in_scale[gm] : 1.f;
      f32x4 old[OUT];
      if constexpr (EPI == EPI_ACCUMULATE)
#pragma unroll
        for (int j = 0; j < OUT; ++j)
          if (gn + j * 16 < cols) old[j] = *reinterpret_cast<const f32x4*>(to + j * 16);
#pragma unroll
      for (int j = 0; j < OUT; ++j) {
        f32x4 v = result(i, j, factor);
        if (gn + j * 16 >= cols) continue;
        if constexpr (EPI == EPI_ACCUMULATE) v = old[j] + v;
        store_c4<CT>(to + j * 16, v);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  // rows of C that are no 16-byte words
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const int gm = gm0 + i * 16 + lane % 16;
    if (gm >= M) continue;
    const float factor = scaled ? grp.in_scale[gm] : 1.f;
#pragma unroll
    for (int j = 0; j < OUT; ++j) {
      const f32x4 v = result(i, j, factor);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gn = gn0 + j * 16 + 4 * (lane / 16) + r;
        if (gn < cols) store_c<CT>(c + (size_t)gm * ldc + gn, v[r], EPI == EPI_ACCUMULATE);
      }
    }
  }
}

// GROUPED: as the tiled kernel's (row tiles of 256 rows); a product that divides k writes grp.slice_rows rows a slice.
template <int EPI, typename CT, bool GROUPED = false, int H = RT, int SHORT = RT>
__global__ __launch_bounds__(RGM * RGN * 64, 1) void gemm_ring_kernel(const bf16* __restrict__ a, int lda, const bf16* __restrict__ w, int ldw,
                                                           CT* __restrict__ c, int ldc, int M, int N, int K, int k_slice, int tall,
                                                           Groups grp, Glu glu) {
  int bx = blockIdx.x, by = blockIdx.y;
  bool head = false;   // GROUPED: the slice begins the row (other products' slices are of 64 and more: it is all one to them)
  if (k_slice > 0) {  // split k: workgroup z of a tile sums its own slice of k into its own copy of C
    int z = blockIdx.z;
    if (GROUPED) {  // the tiles in the map's order, all slices of a tile before the next one's
      const int gx = gridDim.x, gz = gridDim.z, id = bx + gx * (by + (int)gridDim.y * z);
      bx = id % gx;
      z = id / gx % gz;
      by = id / gx / gz;
      head = z == 0;
    }
    // The chip deals workgroups round its 8 dies by their number, and each die has a second-level cache of its
    // own.  With the grid as it stands a die would hold one column tile over all row tiles and all slices (8 + 32
    // different operand pieces a k-step among its 32 workgroups); numbered anew, it holds an eighth of the grid in
    // a row: one slice, some row tiles, all column tiles (4 + 8 pieces), which its cache then serves.
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy * gridDim.z;
    if (!GROUPED && total % 8 == 0) {
      const int id = bx + gx * (by + gy * z), anew = (id % 8) * (total / 8) + id / 8;
      bx = anew % gx;
      by = (anew / gx) % gy;
      z = anew / (gx * gy);
    }
    a += (size_t)z * k_slice;
    w += (size_t)z * k_slice;
    c += (size_t)z * (GROUPED ? grp.slice_rows : M) * ldc;
    K = min(k_slice, K - z * k_slice);
  }
  __shared__ __attribute__((aligned(16))) bf16 ring[RING_SLOTS][RBM * RBK];
  if constexpr (GROUPED) {
    const int32_t* tile = grp.map + 3 * by;
    const int group = tile[0];
    if (group < 0) return;   // (the whole workgroup)
    ring_tile<EPI, CT, true, H>(ring, a, lda, w + (size_t)group * grp.w_stride, ldw, c, ldc, tile[2], N, K, head, bx, tile[1], grp.up_off, grp, glu);
  } else if (SHORT == H || by < tall) {
    ring_tile<EPI, CT, false, H>(ring, a, lda, w, ldw, c, ldc, M, N, K, head, bx, by * (32 * H), N / 2, grp, glu);
  } else {
    ring_tile<EPI, CT, false, SHORT>(ring, a, lda, w, ldw, c, ldc, M, N, K, head, bx, tall * (32 * (H - SHORT)) + by * (32 * SHORT), N / 2, grp, glu);
  }
}

constexpr int RING_MIN_ROWS = 257;
// With slices of k: a thousand rows, or enough rows times k that a slice's sums, which go through memory, are the smaller
// part (611 x 2,048 x 8,192 47.5 / 44.9, but 512 rows 34.8 / 43.2; 320 x 4,096 x 14,336 78 / 69, 1,000 rows 177 / 118; 611 x
// 6,144 x 4,096 51 / 55).
inline bool ring_slices_pay(int M, int K) { return M >= 1024 || (M >= RING_MIN_ROWS && (long long)M * K >= 4500000); }
inline bool ring_takes(const void* a, int lda, const void* w, int ldw, int K) {
  return K % RING_K == 0 && K >= RING_MIN_K && lda % 8 == 0 && ldw % 8 == 0 && (uintptr_t)a % 16 == 0 &&
         (uintptr_t)w % 16 == 0;
}
inline int ring_columns(int epi, int N) { return epi == EPI_SILU_MUL ? (N / 2 + RBN / 2 - 1) / (RBN / 2) : (N + RBN - 1) / RBN; }

template <int EPI, typename CT>
int launch_ring(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, int k_slice, int slices,
                hipStream_t stream, Glu glu = Glu{}) {
  const int columns = ring_columns(EPI, N);
  const RingRows rows = ring_rows(M, columns * slices, k_slice ? k_slice : K);
  const dim3 grid(columns, rows.tiles, slices), block(RGM * RGN * 64);
  GB_REQUIRE(grid.y <= 65535, "gemm_bf16: M=%d needs more than 65535 row tiles", M);
  GB_REQUIRE(ring_has(rows.height), "gemm_bf16: no ring kernel for tiles of %d rows (M=%d)", 32 * rows.height, M);
  // as few tiles as there can be, and one round of them: all of 256 rows, the last one as it comes (some of 224 among them end no
  // sooner, and two heights are two loops to fetch: 2,473 x 2,576 x 13,312 in two slices 188 / 198 us; but eleven rounds, 6,151 x 28,672 x
  // 4,096 with SiLU-multiply, 1,157 / 1,122)
  const bool least = rows.height == 8 && rows.tiles == (M + RBM - 1) / RBM && (long long)rows.tiles * columns * slices <= 256;
  const int tall = least ? rows.tiles : rows.tall;
#define GB_H(H, SHORT)                                                                                                 \
  if (rows.height == H && (SHORT == H) == (H == 8 && tall == rows.tiles))                                              \
    hipLaunchKernelGGL((gemm_ring_kernel<EPI, CT, false, H, SHORT>), grid, block, 0, stream, a, lda, w, ldw, c, ldc, M, \
                       N, K, k_slice, tall, Groups{}, glu);
  GB_H(8, 8) GB_H(8, 7) GB_H(7, 6) GB_H(6, 5) GB_H(5, 4)
#undef GB_H
  return launched("gemm_bf16 (ring)");
}

// ------------------------------------------------------------------------ block
// Products of some hundred rows (short prompts, a new turn behind a history, mixed steps; the narrow products of a longer prompt): too
// few 256 x 256 tiles for the ring kernel.  A workgroup of 2 x 2 waves takes a tile of 32 RM rows by 32 CN rows of W, a wave RM x CN
// tiles of 16 x 16 (W as the first operand: a lane holds four neighbouring columns of a row of C).  Both operands of a k-step of 64 go
// from memory straight into a slot of LDS (a load of the wave brings eight whole lines; piece p of row r lies at p ^ ((r >> 1) & 7)), and
// S slots are all on their way but the one that is multiplied: what bounds the tiled kernel here is a round trip to memory a k-step, with
// one or two of them in registers ahead.  The height of a tile is chosen by the rows there are, in steps of 32: 131 rows are one tile of
// 160 and not two of 128.
//
// As in the ring kernel the operand reads and MFMAs are inline assembly in the order written, the barrier of a k-step stands between its
// two halves, and the waits are written by hand.  Before the barrier a wave has waited for its last operand reads of the k-step, so behind
// it the k-step's slot is free for the loads of k-step + S; and for its own loads of the next k-step, whose first operands are read
// under the second half's MFMAs.
// us, the tiled kernel (or one of 128-row tiles with W asked for by a wave of its own, up to 128 rows) / this one, the product alone: gate/up
// 16,384 x 2,048, 70 / 131 / 300 / 512 rows 22.4 / 28.6 / 39.4 / 46.2 -> 18.2 / 21.8 / 29.4 / 39.4 (744 -> 872 TFLOP/s at the last); 5,120 x 960, 131 /
// 420 / 1,000 rows 10.5 / 13.4 / 25.5 -> 7.3 / 10.9 / 16.3; 28,672 x 4,096, 131 rows 78 -> 55 (4.2 TB/s of W); QKV 6,144 x 2,048, 131 rows 19.5 (in
// slices) -> 13.2, 512 rows 23.9 -> 21.6; first passes in slices: 2,048 x 8,192, 131 rows 19.1 -> 13.9, 960 x 2,560, 611 rows 10.7 -> 9.9.
// In a step of short kernels, whose caches the kernels between have used, the shortest of these gain less or nothing: the 960 x 2,560
// and 5,120 x 960 products of a prompt of 611 rows take 11.2 to 12.5 and 13.9 to 15.4 there.
template <int RM, int CN, int S, int EPI, typename CT>
__global__ __launch_bounds__(256, 1) void gemm_block_kernel(const bf16* __restrict__ a, int lda, const bf16* __restrict__ w, int ldw,
                                                            CT* __restrict__ c, int ldc, int M, int N, int K, int k_slice) {
  constexpr int BM = 32 * RM, BN = 32 * CN, ROWS = BM + BN, L = ROWS / 32;   // L: loads of a wave that bring its share of a slot
  static_assert((S - 1) * L < 64, "a wave counts at most 63 loads on their way");
  if (k_slice > 0) {  // split k: workgroup z of a tile sums its own slice of k into its own copy of C
    const int z = blockIdx.z;
    a += (size_t)z * k_slice;
    w += (size_t)z * k_slice;
    c += (size_t)z * M * ldc;
    K = min(k_slice, K - z * k_slice);
  }
  __shared__ __attribute__((aligned(16))) bf16 slots[S][ROWS * RBK];   // the tile's rows of A, then those of W
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2, bx = blockIdx.x, m0 = blockIdx.y * BM;
  const int half = N / 2;  // EPI_SILU_MUL: number of gate rows; a wave's even column tiles hold gate rows, the odd ones their up rows
  auto w_row = [&](int r) -> int {   // row of W behind row r of the tile's; rows beyond M or N are read from a row that exists
    if (EPI == EPI_SILU_MUL) {
      const int j = r % (CN * 16) / 16, n = min(bx * (BN / 2) + r / (CN * 16) * (CN / 2 * 16) + j / 2 * 16 + r % 16, half - 1);
      return j % 2 ? half + n : n;
    }
    return min(bx * BN + r, N - 1);
  };
  const bf16* src[L];
#pragma unroll
  for (int t = 0; t < L; ++t) {
    const int row = (wave * L + t) * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
    src[t] = (row < BM ? a + (size_t)min(m0 + row, M - 1) * lda : w + (size_t)w_row(row - BM) * ldw) + piece * 8;
  }
  auto load = [&](int t, int slot, int k0) {
    __builtin_amdgcn_global_load_lds((glb_void*)(src[t] + k0), (lds_void*)&slots[slot][(wave * L + t) * 8 * RBK], 16, 0, 0);
  };
  // until k-step s has landed: of the k-steps up to `last` asked for, those behind s may be on their way
  auto landed = [&](int s, int last) {
    const int behind = last - s;
    if (behind >= S - 1) vm_wait<(S - 1) * L>();
    else if (S > 2 && behind == S - 2) vm_wait<(S > 2 ? S - 2 : 0) * L>();
    else if (S > 3 && behind == S - 3) vm_wait<(S > 3 ? S - 3 : 0) * L>();
    else if (S > 4 && behind == S - 4) vm_wait<(S > 4 ? S - 4 : 0) * L>();
    else vm_wait<0>();
  };
  f32x4 acc[RM][CN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < CN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t off[2];   // operand of half kh: row lane % 16 of a 16-row tile, piece 4 kh + lane / 16
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) off[kh] = 2 * ((lane % 16) * RBK + (((4 * kh + lane / 16) ^ ((lane >> 1) & 7)) * 8));
  constexpr uint32_t SLOT = 2 * ROWS * RBK, TILE = 2 * 16 * RBK;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)&slots[0][0];
  const uint32_t abase = base + wm * RM * TILE, wbase = base + (BM / 16 + wn * CN) * TILE;
  bf16x8 fa[2][RM], fw[2][CN];
  auto read = [&](int set, int t, uint32_t at) {   // operand t of RM + CN of a half
    if (t < RM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][t < RM ? t : 0]) : "v"(abase + at), "n"(t < RM ? t * TILE : 0) : "memory");
    else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fw[set][t < RM ? 0 : t - RM]) : "v"(wbase + at), "n"(t < RM ? 0 : (t - RM) * TILE) : "memory");
  };
  const int steps = K / RBK;
  // the MFMAs of operand set `set`; among them the reads of the other set from `at`, and (with `more`) a slot's loads
  auto block = [&](auto which, uint32_t at, bool more, int slot, int k0) {
    constexpr int set = decltype(which)::value, COUNT = RM * CN, EACH = (RM + CN + L + COUNT - 1) / COUNT;
    int next = 0;
#pragma unroll
    for (int n = 0; n < COUNT; ++n) {
      const int i = n / CN, j = (i & 1) ? CN - 1 - n % CN : n % CN;
      if constexpr (COUNT > 24) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fw[set][j]), "v"(fa[set][i]));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(fw[set][j]), "v"(fa[set][i]));
#pragma unroll
      for (int u = 0; u < EACH; ++u) {
        if (next < RM + CN) read(set ^ 1, next, at);
        else if (set == 1 && next < RM + CN + L && more) load(next - RM - CN, slot, k0);
        ++next;
      }
    }
  };
  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, 1>;
  const int first = min(S, steps);
#pragma unroll 1
  for (int s = 0; s < first; ++s)
#pragma unroll
    for (int t = 0; t < L; ++t) load(t, s, s * RBK);
  landed(0, first - 1);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int t = 0; t < RM + CN; ++t) read(0, t, off[0]);
  int slot = 0;
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    const int next = slot + 1 == S ? 0 : slot + 1;
    lds_wait<0>(fa[0], fw[0]);
    block(First{}, slot * SLOT + off[1], false, 0, 0);
    lds_wait<0>(fa[1], fw[1]);
    if (s + 1 < steps) landed(s + 1, min(steps, s + S) - 1);
    __builtin_amdgcn_s_barrier();
    block(Second{}, next * SLOT + off[0], s + S < steps, slot, (s + S) * RBK);   // (behind the last: read, not used)
    slot = next;
  }
  lds_wait<0>(fa[0], fw[0]);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs' results, which the compiler does not know to wait for
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < CN; ++j) {
      if constexpr (RM * CN > 24) asm volatile("" : "+a"(acc[i][j]));
      else asm volatile("" : "+v"(acc[i][j]));
    }

  // a lane holds row lane % 16 of a tile and its columns 4 (lane / 16) .. + 3
  constexpr int OUT = EPI == EPI_SILU_MUL ? CN / 2 : CN;   // column tiles of the wave's results
  const int cols = EPI == EPI_SILU_MUL ? half : N;
  const int gn0 = bx * (2 * OUT * 16) + wn * (OUT * 16) + 4 * (lane / 16);
  const bool words = ldc % 4 == 0 && (uintptr_t)c % (4 * sizeof(CT)) == 0;
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int gm = m0 + (wm * RM + i) * 16 + lane % 16;
    if (gm >= M) continue;
    CT* to = c + (size_t)gm * ldc + gn0;
    f32x4 v[OUT];
#pragma unroll
    for (int j = 0; j < OUT; ++j) {
      if constexpr (EPI == EPI_SILU_MUL) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = gated_unit(acc[i][2 * j][r], acc[i][2 * j + 1][r], Glu{});
      } else {
        v[j] = acc[i][j];
      }
    }
    if (words && gn0 + (OUT - 1) * 16 + 4 <= cols) {
      if constexpr (EPI == EPI_ACCUMULATE) {
        f32x4 old[OUT];   // a row's old values are all asked for before any is added to
#pragma unroll
        for (int j = 0; j < OUT; ++j) old[j] = *reinterpret_cast<const f32x4*>(to + j * 16);
#pragma unroll
        for (int j = 0; j < OUT; ++j) v[j] = old[j] + v[j];
      }
#pragma unroll
      for (int j = 0; j < OUT; ++j) store_c4<CT>(to + j * 16, v[j]);
    } else {
#pragma unroll
      for (int j = 0; j < OUT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (gn0 + j * 16 + r < cols) store_c<CT>(to + j * 16 + r, v[j][r], EPI == EPI_ACCUMULATE);
    }
  }
}

// Which tile, and into how many slices k is divided: what the launch takes is the rows (of 128 bytes) that its workgroups bring into LDS,
// at some 13 TB/s over the whole chip, and a compute unit at most 65 GB/s, or 50 of tiles of 224 rows and more, whose operand reads
// weigh more; and 3.5 us.  (Over tiles of 64 x 64 to 256 x 128, one to eight slices and the products of four models at 70 to 1,000
// rows that is within a fifth of what was measured.)  Slices are written and read again.  So the tiles are those that fill the chip
// once with the fewest bytes.
struct BlockPlan {
  int rm, cn, slices, k_slice;
  float us;
};
inline BlockPlan block_plan(int M, int N, int K, bool silu, int least_slices, int most_slices) {
  static const struct { int rm, cn; } tiles[] = {{2, 2}, {3, 2}, {4, 2}, {5, 2}, {6, 2}, {4, 3}, {5, 3},
                                                 {2, 4}, {3, 4}, {4, 4}, {5, 4}, {6, 4}, {8, 4}};
  static const int slices[] = {1, 2, 3, 4, 5, 6, 8};
  BlockPlan best{0, 0, 1, 0, 1e30f};
  const int steps = K / RBK;
  for (const auto& t : tiles) {
    if (silu && t.cn == 3) continue;
    const long long all = (long long)((M + 32 * t.rm - 1) / (32 * t.rm)) * ((N + 32 * t.cn - 1) / (32 * t.cn));
    for (int z : slices) {
      if (z < least_slices) continue;
      if (z > most_slices || (z > 1 && steps < 8 * z)) break;
      const int each = (steps + z - 1) / z;
      if ((steps + each - 1) / each != z) continue;
      const float bytes = (float)each * (t.rm + t.cn) * (32 * 128);
      const float chip = (float)(all * z) * bytes / 13e6f, unit = (float)((all * z + 255) / 256) * bytes / (t.rm + t.cn >= 7 ? 50e3f : 65e3f);
      const float us = 3.5f + (chip > unit ? chip : unit) + (z > 1 ? 3.5f + z * (float)M * N * 8.f / 4.5e6f : 0.f);
      if (us < best.us) best = BlockPlan{t.rm, t.cn, z, each * RBK, us};
    }
  }
  return best;
}
inline bool block_takes(const void* a, int lda, const void* w, int ldw, int K) {
  return K % RBK == 0 && lda % 8 == 0 && ldw % 8 == 0 && (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0;
}
// Sizes that the block kernel can take, if the operands allow; where it does, see block_pays.  Up to 64 rows: what the held kernel does not
// take.  A product that is not formed into a gated unit stays with the tiled kernel, whose fewer k-steps ahead start sooner, below a k of
// 1,024 (3,840 x 960, 65 to 128 rows: 6.3 to 6.6 us; 1,600 x 960, 131 rows 6.3, 7.0 here).
inline bool block_sizes(int M, int N, int K, bool silu) { return M > 32 && K % RBK == 0 && N % 8 == 0 && (silu ? N % 16 == 0 : K >= 1024); }
// What the ring kernel takes beside that, for the lines below and the slices of k, which were measured with tiles of 256 x 256 alone:
// a k-step of a round of them 1.75 us.  (The launch deals rows by ring_rows, whose estimate of a full round is 1.60; where the two
// kernels are compared by time, that one decides: ring_ahead.)
inline float ring_us(int M, int N, int K, int slices) {
  const long long tiles = (long long)((M + RBM - 1) / RBM) * ((N + RBN - 1) / RBN) * slices;
  return 3.5f + (float)((tiles + 255) / 256) * ((K / slices + RBK - 1) / RBK) * 1.75f + (slices > 1 ? 3.5f + slices * (float)M * N * 8.f / 4.5e6f : 0.f);
}

// Where the block kernel takes a product whole, with the tile of `p`; else the ring kernel where it can, the tiled one, or (up to 64 rows) the
// skinny one.  block_plan's estimate says little about those, whose smaller workgroups share a compute unit, so the lines are measured
// ones (9,000 products of 65 to 1,000 rows, 512 to 16,384 rows of W, k 256 to 8,192, of which 1 % are more than 4 % slower here than the
// other kernel, 2 % the other way round; us, the other kernel / this one).
//  * Beside the ring kernel: a storing product whose 256 x 256 tiles are one round stays there (300 x 32,768 x 4,096: 107 / 126), and
//    so does one for which the plan is tiles of 256 rows (512 x 49,152 x 3,072: 112 / 134); a gated unit goes by the estimates.
//  * Beside the tiled kernel it is ahead from where that has more than 256 workgroups (400 x 8,192 x 1,792: 24.4 / 20.8).  Below that a
//    compute unit has one workgroup either way and the tiled one starts sooner: 64-row tiles 256 x 4,096 x 1,280 7.8 / 9.6, ahead
//    here only with a long k and enough of them (256 x 3,072 x 8,192: 41.9 / 39.4); 128-row tiles 192 x 8,192 x 2,560 25.7 / 30.4, but
//    not where the plan is narrow tiles and the rows are no whole 128s (added into C, 1,000 x 1,600 x 1,280 17.4 / 13.9, but 640 x 2,560 x
//    1,280 10.3 / 11.9); up to 128 rows from 128 workgroups on (65 x 6,144 x 1,536 11.4 / 9.9).
//    Large tiles that leave compute units without one: 512 x 12,288 x 1,280 25.8 / 29.2 (192 tiles of 256 x 128), 640 x 5,120 x 1,024
//    15.4 / 21.7 (216 of 160 x 96); or that are a second round: 640 x 12,288 x 1,024 24.2 / 28.1.
//  * A gated unit: ahead of the tiled kernel everywhere but with those, and with tiles as tall as the tiled kernel's and a short k
//    (512 x 8,192 x 256: 6.9 / 7.5).  Beside the skinny kernel (up to 64 rows) with more than 2,048 gates, or a k of 1,024 and more, or
//    a very short one (33 x 4,096 x 960: 5.6 / 6.9; 33 x 8,208 x 960: 9.2 / 8.6).
//  * A vocabulary at up to 64 rows: from 65,536 rows of W on (48 x 49,152 x 4,096: 92 / 97, 128,256: 246 / 234).
// The ring kernel pays where its tiles of 256 occupy at least three quarters of the compute units, from two row tiles on, and the
// loads are whole 16-byte pieces; and wherever its estimate with the heights of ring_rows is below the block kernel's, which is
// also a bound below the tiled kernel's time.  (That estimate is some 10 % low for several rounds of tiles, and this one by what a
// tile's old values take.)  Not for one round of them where the tiled kernel's workgroups are resident at once (640 x 12,288 x 1,024
// 23.0 / 22.4; 930 x 8,192 x 3,072 53 / 58; 420 x 12,288 x 1,280 25.5 / 28.7).  Of 1,800 random
// products of 260 to 8,192 rows and a k of 128 to 2,048 six are more than 4 % slower than with the first line and tiles of 256 alone
// (456 x 23,440 x 320 with SiLU-multiply 18.0 / 21.0, 789 x 16,928 x 192 20.9 / 24.3, 1,439 x 10,880 x 2,048 with SiLU-multiply 72 / 79);
// their geometric mean is 0.93.  us, the block or tiled kernel / this one: 1,350 x 6,144 x 4,096 104 / 69,
// 2,200 x 4,096 x 14,336 372 / 237, 4,500 x 2,048 x 8,192 207 / 146, 700 x 16,384 x 2,048 with SiLU-multiply 60 / 48, 350 x 28,672 x
// 4,096 115 / 87, 4,096 x 5,120 x 960 58 / 47, 2,900 x 3,072 x 576 23.0 / 18.3.
inline bool ring_fills(int epi, int M, int N) { return M >= RING_MIN_ROWS && (long long)((M + RBM - 1) / RBM) * ring_columns(epi, N) >= 192; }
inline bool ring_ahead(int epi, int M, int N, int K) {
  const bool silu = epi == EPI_SILU_MUL;
  if (M < RING_MIN_ROWS || K % RBK != 0 || N % (silu ? 16 : 8) != 0) return false;
  const int columns = ring_columns(epi, N);
  const RingRows r = ring_rows(M, columns, K);
  const bool one_round = (long long)r.tiles * columns <= 256;
  if (one_round && tiled_grid(epi, M, N).groups() <= 512) return false;
  const float added = epi == EPI_ACCUMULATE ? 1.25f * (float)r.height : 0.f;
  return r.us + added <= (one_round ? 1.f : 1.1f) * block_plan(M, N, K, silu, 1, 1).us;
}
inline bool ring_pays(int epi, const void* a, int lda, const void* w, int ldw, int M, int N, int K) {
  return ring_takes(a, lda, w, ldw, K) && (ring_fills(epi, M, N) || ring_ahead(epi, M, N, K));
}
inline bool block_pays(int epi, int M, int N, int K, const BlockPlan& p, bool rings) {
  const bool silu = epi == EPI_SILU_MUL;
  if (rings && ring_ahead(epi, M, N, K)) return false;
  const long long tiles = (long long)((M + 32 * p.rm - 1) / (32 * p.rm)) * ((N + 32 * p.cn - 1) / (32 * p.cn));
  if (rings) {
    const long long ring = (long long)((M + RBM - 1) / RBM) * ((N + RBN - 1) / RBN);
    return p.us < ring_us(M, N, K, 1) && (silu || (ring > 256 && p.rm < 8));
  }
  if (M <= 64) return silu ? N > 4096 || K >= 1024 || K < 192 : N < 32768 || N >= 65536;
  if (tiles > 256 && tiles <= 512 && N < 32768) return false;
  const TiledGrid g = tiled_grid(epi, M, N);
  if (M <= 128 && !silu) return g.groups() >= 128;
  if ((p.rm == 8 && tiles < 224) || (p.cn == 3 && tiles < 240)) return false;
  if (silu) return !(p.cn == 4 && (p.rm == 4 || p.rm == 8) && K < 640);
  if (g.bm == 64) return g.groups() > 256 || (g.groups() > 128 && K >= 2560 && N > 2048);
  return g.groups() > 256 || (p.cn == 2 && M % 128 != 0);
}

// Slots of a tile: what fits LDS, once (one workgroup a compute unit) or, of the small tiles, twice.
constexpr int block_slots(int rm, int cn) { return rm + cn <= 5 ? 80 / (4 * (rm + cn)) : 160 / (4 * (rm + cn)) > 5 ? 5 : 160 / (4 * (rm + cn)); }

template <int EPI, typename CT>
int launch_block(int rm, int cn, const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, int k_slice,
                 int slices, hipStream_t stream) {
  const int cols = EPI == EPI_SILU_MUL ? N / 2 : N, bn = EPI == EPI_SILU_MUL ? 16 * cn : 32 * cn;
  const dim3 grid((cols + bn - 1) / bn, (M + 32 * rm - 1) / (32 * rm), slices), block(256);
  GB_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "gemm_bf16: M=%d needs more than 65535 row tiles", M);
#define GB_B(RM, CN)                                                                                                              \
  if (rm == (RM) && cn == (CN)) {                                                                                                 \
    hipLaunchKernelGGL((gemm_block_kernel<(RM), (CN), block_slots((RM), (CN)), EPI, CT>), grid, block, 0, stream, a, lda, w, ldw, c, \
                       ldc, M, N, K, slices > 1 ? k_slice : 0);                                                                   \
    return launched("gemm_bf16 (block)");                                                                                         \
  }
  GB_B(2, 2) GB_B(3, 2) GB_B(4, 2) GB_B(5, 2) GB_B(6, 2) GB_B(2, 4) GB_B(3, 4) GB_B(4, 4) GB_B(5, 4) GB_B(6, 4) GB_B(8, 4)
  if constexpr (EPI != EPI_SILU_MUL) { GB_B(4, 3) GB_B(5, 3) }
#undef GB_B
  return fail("gemm_bf16 (block): no tile of %d x %d", 32 * rm, 32 * cn);
}

// ------------------------------------------------------------------------- held
// Products of 17 to 64 rows that read a large W (decode steps of a busy server: gate/up, QKV, the vocabulary).  W is what
// they cost; but the skinny kernel reads all of A again in every workgroup, in front of the stream of W, and asks for W
// in half lines.  Here a workgroup for every compute unit holds the rows of A in registers (a wave the k-blocks that are
// its own: block b of 64 belongs to wave b % 8, MT x NB x 8 registers) and walks over several tiles of 16 rows of W.  A
// wave brings its blocks of W from memory straight into a ring of its own in LDS (whole lines of 128 bytes, nontemporal,
// five or six blocks of 2 KB: 80 or 96 KB on their way a compute unit) and takes them as MFMA operands from there: no barrier stands
// between a load and its use, and the ring runs on over the ends of tiles.  The eight waves' sums of a tile meet in LDS
// (two buffers, one barrier a tile); one wave adds them in the waves' order and finishes, the waves taking turns.
//
// MFMA row 4 q + e of a tile is such that a lane holds what the epilogue joins: with EPI_SILU_MUL e = 0, 1 are gate rows
// and e = 2, 3 the up rows that belong to them, with EPI_ROPE the two halves of two pairs.
//
// The memory counter: loads and stores retire in the order of issue, so waiting for all but the youngest 2 (HS - 1)
// means that a block has landed once HS - 1 blocks were asked for behind it, whatever else was issued in between.
// The sums go through LDS by inline assembly: the compiler would wait for every load into LDS before an access of its own.
constexpr int HWAVES = 8, HBLOCK = 16 * 64;   // waves, elements of a block
__device__ __forceinline__ f32x4 lds_read_f4(uint32_t addr) {
  f32x4 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr) : "memory");
  return v;
}

template <int MT, int NB, int EPI, typename CT>
__global__ __launch_bounds__(HWAVES * 64, 1) void gemm_held_kernel(const bf16* __restrict__ a, int lda, const bf16* __restrict__ w,
                                                                   int ldw, CT* __restrict__ c, int ldc, int M, int N, int K,
                                                                   int k_slice, int tiles, float eps, const float* __restrict__ parts,
                                                                   int n_parts, RopeExtras rope) {
  constexpr int HS = MT == 4 ? 5 : 6;   // blocks of a wave's ring
  constexpr int TURNS = MT == 3 ? 4 : MT, EVERY = HWAVES / TURNS;   // a wave finishes column block wave % TURNS of every EVERY-th tile
  __shared__ __attribute__((aligned(16))) bf16 ring[HWAVES][HS][HBLOCK];
  __shared__ __attribute__((aligned(16))) float part[2][HWAVES][MT][64][4];
  __shared__ float squares[HWAVES][64];   // of each row, a wave's share of the partial sums
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r = lane % 16, q = lane / 16;
  const int full_k = K;
  if (k_slice > 0) {   // workgroups (.., z) sum slice z of k into their own copy of C
    const int z = blockIdx.y;
    a += (size_t)z * k_slice;
    w += (size_t)z * k_slice;
    c += (size_t)z * M * ldc;
    K = min(k_slice, K - z * k_slice);
  }
  const int stride = gridDim.x, mine = (tiles - (int)blockIdx.x + stride - 1) / stride;   // tiles of the workgroup
  const int nb = (K / 64 - wave + HWAVES - 1) / HWAVES;   // k-blocks of the wave

  // ---- the stream of W: a load of the wave brings 8 rows of a block, 128 bytes each; piece p of row i lies at p ^ (i & 7)
  auto w_row = [&](int tile, int i) -> int {   // row of W behind MFMA row i of a tile
    const int j = 2 * (i / 4) + (i & 1);
    if (EPI == EPI_SILU_MUL) return min(tile * 8 + j, N / 2 - 1) + ((i & 2) ? N / 2 : 0);
    if (EPI == EPI_ROPE) {
      const int per_head = rope.hd / 16, head = tile / per_head, d0 = tile % per_head * 8;
      return head * rope.hd + d0 + j + ((i & 2) ? rope.hd / 2 : 0);
    }
    return min(tile * 16 + i, N - 1);
  };
  // (Through the ring come first the wave's blocks of A, a column block's after the other's, then those of W.)
  const bf16* src[2];
  int at_cols = 0, at_tile = blockIdx.x, at_block = 0, slot_in = 0, asked = 0;
  const int a_blocks = nb * MT, total = a_blocks + mine * nb;
  auto aim = [&](bool of_a) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = u * 8 + lane / 8, k = wave * 64 + ((lane % 8) ^ (i & 7)) * 8;
      if (of_a) src[u] = a + (size_t)min(at_cols * 16 + i, M - 1) * lda + k;
      else src[u] = w + (size_t)w_row(at_tile, i) * ldw + k;
    }
  };
  auto bring = [&](bool of_a) {
    const int col = at_block * (HWAVES * 64);
    if (of_a) {
      __builtin_amdgcn_global_load_lds((glb_void*)(src[0] + col), (lds_void*)&ring[wave][slot_in][0], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((glb_void*)(src[1] + col), (lds_void*)&ring[wave][slot_in][512], 16, 0, 0);
    } else {   // nontemporal: W is read once, in whole lines
      __builtin_amdgcn_global_load_lds((glb_void*)(src[0] + col), (lds_void*)&ring[wave][slot_in][0], 16, 0, 2);
      __builtin_amdgcn_global_load_lds((glb_void*)(src[1] + col), (lds_void*)&ring[wave][slot_in][512], 16, 0, 2);
    }
    slot_in = slot_in + 1 == HS ? 0 : slot_in + 1;
    ++asked;
    if (++at_block == nb) {
      at_block = 0;
      if (of_a) ++at_cols;
      else at_tile += stride;
    }
  };
  auto ask = [&]() {
    const bool of_a = asked < a_blocks;
    if (at_block == 0) aim(of_a);
    bring(of_a);
  };
  auto ask_w = [&]() {   // once every block of A has been asked for
    if (at_block == 0) aim(false);
    bring(false);
  };
  // A norm before the product: its partial sums of squares, row `lane`'s, every eighth a wave; asked for ahead of the ring.
  constexpr int PARTS_AT_ONCE = 32;
  float got[PARTS_AT_ONCE];
  if (parts != nullptr) {
#pragma unroll
    for (int u = 0; u < PARTS_AT_ONCE; ++u) {
      const int p = wave + u * HWAVES;
      got[u] = lane < M && p < n_parts ? parts[(size_t)p * 64 + lane] : 0.f;
    }
  }
#pragma unroll 1
  for (int s = 0; s < HS && s < total; ++s) ask();
  if (parts != nullptr) {
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < PARTS_AT_ONCE; ++u) sum += got[u];
    for (int p = wave + PARTS_AT_ONCE * HWAVES; p < n_parts; p += HWAVES) sum += lane < M ? parts[(size_t)p * 64 + lane] : 0.f;
    // (read behind the first tile's barrier)
    asm volatile("ds_write_b32 %0, %1" ::"v"((uint32_t)(uintptr_t)(lds_void*)&squares[wave][lane]), "v"(sum) : "memory");
  }

  // ---- what the wave's turns at finishing will need
  const int t_mine = wave % TURNS, m_mine = t_mine * 16 + r;
  const bool row_mine = t_mine < MT && m_mine < M;
  float scale = 1.f;
  float cs[2] = {1.f, 1.f}, sn[2] = {0.f, 0.f};
  int slot = 0;
  if constexpr (EPI == EPI_ROPE) {   // (at most EVERY tiles a workgroup: one turn a wave)
    const int tile = blockIdx.x + wave / TURNS * stride, per_head = rope.hd / 16;
    if (row_mine && wave / TURNS < mine) {
      if (rope.slots) slot = rope.slots[m_mine];
      if (rope.cosv && tile / per_head < rope.nh + rope.nkv) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const size_t at = (size_t)m_mine * (rope.hd / 2) + tile % per_head * 8 + 2 * q + e;
          cs[e] = rope.cosv[at], sn[e] = rope.sinv[at];
        }
      }
    }
  }
  // ---- the tiles
  const uint32_t ring_base = (uint32_t)(uintptr_t)(lds_void*)&ring[wave][0][0];
  const uint32_t part_base = (uint32_t)(uintptr_t)(lds_void*)&part[0][0][0][0][0];
  uint32_t off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) off[h] = 2 * (r * 64 + ((4 * h + q) ^ (r & 7)) * 8);
  int slot_out = 0, left = total;   // blocks not yet taken
  auto take = [&](bf16x8 (&f)[2]) {   // the next block of the ring as an operand: its place is free then
    if (left >= HS) vm_wait<2 * (HS - 1)>();
    else vm_wait<0>();
#pragma unroll
    for (int h = 0; h < 2; ++h) f[h] = lds_read16(ring_base + slot_out * (2 * HBLOCK) + off[h]);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1])::"memory");
    slot_out = slot_out + 1 == HS ? 0 : slot_out + 1;
    --left;
  };
  bf16x8 fa[MT][NB][2];   // (rows behind M are a row that exists: what comes of them is not stored)
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i < nb) {
        take(fa[t][i]);
        if (asked < total) ask();
      }
#pragma unroll 1
  for (int ti = 0; ti < mine; ++ti) {
    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (i < nb) {
        bf16x8 fw[2];
        take(fw);
        if (asked < total) ask_w();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[h], fa[t][i][h], acc[t], 0, 0, 0);
      }
    }
    const uint32_t buf = part_base + (uint32_t)((ti & 1) * (HWAVES * MT * 1024) + lane * 16);
    // (the MFMAs' results: the compiler does not know the assembly below to read them out of the registers at once)
    static_assert(MT >= 2 && MT <= 4, "the wait names every column block's sums");
    if constexpr (MT == 2) asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]));
    else if constexpr (MT == 3) asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]));
    else asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
#pragma unroll
    for (int t = 0; t < MT; ++t) asm volatile("ds_write_b128 %0, %1" ::"v"(buf + (uint32_t)((wave * MT + t) * 1024)), "v"(acc[t]) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t_mine >= MT || ti % EVERY != wave / TURNS) continue;
    // D[n, m]: the lane holds column m = r and rows 4 q + e
    f32x4 p[HWAVES];
#pragma unroll
    for (int wv = 0; wv < HWAVES; ++wv) p[wv] = lds_read_f4(buf + (uint32_t)((wv * MT + t_mine) * 1024));
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]), "+v"(p[4]), "+v"(p[5]), "+v"(p[6]), "+v"(p[7])::"memory");
    static_assert(HWAVES == 8, "the wait names the eight waves' sums");
    f32x4 v = p[0];
#pragma unroll
    for (int wv = 1; wv < HWAVES; ++wv) v += p[wv];
    if (parts != nullptr) {
      if (ti < EVERY) {   // the wave's first turn
        float sq[HWAVES];
#pragma unroll
        for (int wv = 0; wv < HWAVES; ++wv)
          asm volatile("ds_read_b32 %0, %1" : "=v"(sq[wv]) : "v"((uint32_t)(uintptr_t)(lds_void*)&squares[wv][t_mine * 16 + r]) : "memory");
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(sq[0]), "+v"(sq[1]), "+v"(sq[2]), "+v"(sq[3]), "+v"(sq[4]), "+v"(sq[5]), "+v"(sq[6]), "+v"(sq[7])::"memory");
        float sum = sq[0];
#pragma unroll
        for (int wv = 1; wv < HWAVES; ++wv) sum += sq[wv];
        scale = 1.0f / sqrtf(sum / (float)full_k + eps);
      }
      v *= scale;
    }
    if (row_mine) {
      const int tile = blockIdx.x + ti * stride;
      if constexpr (EPI == EPI_SILU_MUL) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int j = tile * 8 + 2 * q + e;
          if (j < N / 2) c[(size_t)m_mine * ldc + j] = (CT)gated_unit(v[e], v[2 + e], Glu{});
        }
      } else if constexpr (EPI == EPI_ROPE) {
        const int per_head = rope.hd / 16, head = tile / per_head, dim0 = tile % per_head * 8 + 2 * q, half = rope.hd / 2;
        const bool is_value = head >= rope.nh + rope.nkv;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          // (a product of its own each, as the skinny kernel's)
          const float lo = is_value || !rope.cosv ? v[e] : v[e] * cs[e] - v[2 + e] * sn[e];
          const float hi = is_value || !rope.cosv ? v[2 + e] : v[2 + e] * cs[e] + v[e] * sn[e];
#pragma unroll
          for (int up = 0; up < 2; ++up) {
            const bf16 y = (bf16)(up ? hi : lo);
            const int dim = dim0 + e + up * half;
            c[(size_t)m_mine * ldc + head * rope.hd + dim] = (CT)y;
            if (rope.slots != nullptr && head >= rope.nh) {
              const int page = slot / rope.page_size, at = slot % rope.page_size;
              if (!is_value)
                rope.k_pages[((size_t)page * rope.nkv + (head - rope.nh)) * rope.page_size * rope.hd + key_offset(at, dim, rope.page_size, 8)] = y;
              else
                rope.v_pages[(((size_t)page * rope.nkv + (head - rope.nh - rope.nkv)) * rope.hd + dim) * rope.page_size + at] = y;
            }
          }
        }
      } else {
        CT* to = c + (size_t)m_mine * ldc + tile * 16 + 4 * q;
        if (tile * 16 + 16 <= N && ldc % 4 == 0 && (uintptr_t)c % (4 * sizeof(CT)) == 0) {
          store_c4<CT>(to, v);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (tile * 16 + 4 * q + e < N) to[e] = (CT)v[e];
        }
      }
    }
  }
}

// Column blocks of 16 rows of A times k-blocks a wave: what fits the registers (MT x NB x 8 of them for A).
inline int held_blocks(int K) { return (K / 64 + HWAVES - 1) / HWAVES; }
inline bool held_takes(const void* a, int lda, const void* w, int ldw, int M, int K) {
  return M > 16 && M <= 64 && K % 64 == 0 && held_blocks(K) <= (M <= 32 ? 8 : 4) && lda % 8 == 0 && ldw % 8 == 0 &&
         (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0;
}
// Workgroups: as many as share the tiles evenly, at most one a compute unit (times the slices of k).
inline int held_groups(int tiles, int slices) {
  const int room = 256 / slices, each = (tiles + room - 1) / room;
  return (tiles + each - 1) / each;
}
// Where it pays (us, the skinny kernel, the wide tiles or narrow ones before / this one, each product alone, weights cold):
//   gate/up 28,672 x 4,096, 17 / 24 / 32 rows: 53 / 57 / 62 -> 42 / 45 / 45 (5.2 to 5.5 TB/s); vocabulary 128,256 x 4,096,
//   24 rows: 242 -> 176 (6 TB/s); gate/up 16,384 x 2,048, 20 / 33 / 64 rows: 19 / 21.6 / 20.8 -> 15.7 / 17 / 18; gate/up 5,120 x 960
//   behind partial sums of a norm, 53 rows: 12.5 -> 8.8; QKV 6,144 x 4,096, 24 rows 17.2 -> 15.3; 6,144 x 2,048, 20 / 64 rows
//   11.2 / 16.7 -> 10.3 / 13.3.
// What it saves is A, read once a workgroup and not once a tile or two: as many bytes as k and rows are large.  What it costs is the
// same for any k: the ring's start and, a tile, eight waves' sums that meet.  So it is ahead from a k on that is the smaller the
// more rows there are, the more the other kernel spends on a row (a norm's scale, the rotation) and the more tiles a workgroup has; where
// other kernels take the rows another way too (the block kernel a gated unit of 33 rows and more, the tiled one a vocabulary),
// from a larger one.  held_from gives that k; it was read off times of both at 64 <= k <= 4,096, 17 to 64 rows and 60 to 2,048 tiles (of
// 9,600 products it takes 1 % that are more than 4 % slower here, and leaves 7 % that would be more than 4 % faster).  us, the other
// kernel / this one, at the sides of a line: 256 tiles of a storing product, 24 rows, k 1,280 / 1,536: 5.4 / 5.7, 6.6 / 6.1; 300 tiles of a
// gated unit behind a norm, 24 rows, k 960 / 1,280: 7.5 / 7.9, 10.3 / 8.8; 64 rows, k 320 / 576: 8.3 / 8.2, 9.8 / 8.6.
// A k of 128: 2.9 / 4.4 at 257 tiles.  Few tiles (up to 256, one a workgroup): a workgroup's rows of A are then more than its rows of
// W, and the skinny kernel's sixteen waves (a k of 768 and more) bring both as fast until a k is several round trips there; its four (a
// shorter k) are behind from 576 on (960 x 576, 53 rows: 7.1 -> 6.2), and so are its half tiles of storing products from 160 tiles on.
inline int held_tiles(int epi, int N) { return epi == EPI_SILU_MUL ? (N / 2 + 7) / 8 : (N + 15) / 16; }
inline int held_from(int epi, int M, int tiles, int K, bool parts) {
  const int mt = (M + 15) / 16;
  const bool heads = epi == EPI_ROPE || (epi == EPI_STORE && parts);
  if (tiles <= 256) {
    if (K < 768) {
      if (mt == 2 || !(parts || (epi == EPI_STORE && tiles >= 160 && tiles < 256))) return 576;
      return mt == 4 && parts ? 64 : 320;
    }
    if (epi == EPI_STORE && !parts && tiles == 256) return mt == 2 ? 1536 : 1024;
    return mt == 2 && tiles < 160 ? 3072 : 768;
  }
  if (mt == 2) return tiles <= 512 ? 1280 : tiles < 768 ? 768 : tiles <= 1024 || tiles > 2048 ? 576 : epi == EPI_SILU_MUL && !parts ? 448 : 640;
  if (heads) return tiles >= 384 ? 256 : mt == 3 ? 1280 : 640;
  if (parts) return mt == 3 ? 576 : 448;
  if (epi == EPI_SILU_MUL) return tiles <= 512 ? 1280 : 2048;
  if (tiles >= 2048 && tiles < 4096) return 768;
  return mt == 4 || tiles >= 768 ? 576 : tiles <= 512 ? 960 : 640;
}
inline bool held_pays(int epi, int M, int N, int K, bool parts) {
  const int tiles = held_tiles(epi, N);
  if (epi == EPI_ROPE) {   // a wave prepares one turn at finishing
    const int groups = held_groups(tiles, 1);
    if ((tiles + groups - 1) / groups > HWAVES / (M <= 32 ? 2 : 4)) return false;
  }
  return tiles >= (K < 768 ? 60 : K >= 2048 ? 128 : epi == EPI_STORE ? 160 : 257) && K >= held_from(epi, M, tiles, K, parts);
}
template <int EPI, typename CT>
int launch_held(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, int k_slice, int slices, float eps,
                const float* parts, int n_parts, hipStream_t stream, const RopeExtras& rope = RopeExtras{}) {
  const int tiles = held_tiles(EPI, N), mt = (M + 15) / 16;
  const int nb = held_blocks(slices > 1 ? k_slice : K);
  const dim3 grid(held_groups(tiles, slices), slices), block(HWAVES * 64);
#define GB_H(MT, NB, FROM)                                                                                                      \
  if (mt == (MT) && nb > (FROM) && nb <= (NB)) {                                                                                \
    hipLaunchKernelGGL((gemm_held_kernel<(MT), (NB), EPI, CT>), grid, block, 0, stream, a, lda, w, ldw, c, ldc, M, N, K,          \
                       slices > 1 ? k_slice : 0, tiles, eps, parts, n_parts, rope);                                             \
    return launched("gemm_bf16 (held)");                                                                                        \
  }
  GB_H(2, 2, 0) GB_H(2, 4, 2) GB_H(2, 8, 4) GB_H(3, 2, 0) GB_H(3, 4, 2) GB_H(4, 2, 0) GB_H(4, 4, 2)
#undef GB_H
  return fail("gemm_bf16 (held): %d rows by a k of %d do not fit the registers", M, K);
}

// ------------------------------------------------------------------------ split k
// A product with few tiles (17 to a few hundred rows, or few rows of W) leaves most compute units idle
// and, as a skinny product, makes every workgroup read all of A.  Here the tiled kernel's workgroups
// also divide k: workgroup (tile, z) sums slice z of k into copy z of a float32 C in a workspace, and a
// second kernel adds the copies in the order of z and applies the epilogue.  Tiles of 64 or 128 rows; with
// many rows and a long k (ring_slices_pay), the ring kernel's tiles of 256.
struct SplitPlan {
  int bm, slices, k_slice;
  size_t floats;  // of workspace
  bool ring;      // the ring kernel's 256 x 256 tiles, if the operands allow (else the tiled kernel's, same slices)
  bool held;      // the held kernel's tiles of 16 rows of W, if the operands allow (else the tiled kernel's, same slices)
  int rm, cn;     // the block kernel's tiles of 32 rm x 32 cn, if the operands allow (else the tiled kernel's, same slices); 0: not
  float us;       // with those, block_plan's estimate
};

// Slices of k for the held kernel where its tiles alone are few (the O and down projections of 17 to 64 rows): four tiles a workgroup and
// more, so that it reads more of W than of A; 512 of k and more; and what a wave can hold of a slice.  Fewer slices than the wide tiles
// took, so that the pass behind them reads less.  (us, with that pass and the norm, before / now: 4,096 x 14,336, 24 / 53 rows 33.0 / 35.0 ->
// 26.7 / 29.8; 4,096 x 4,096, 17.0 / 17.7 -> 13.7 / 15.5; 2,048 x 8,192, 16.1 / 17.0 -> 13.5 / 15.2; 2,048 x 2,048, 53 rows 10.5 -> 9.9; 576 x
// 1,536, 53 rows 9.1 -> 7.6.)  Products of up to 32 rows by a k below 4,096 stay whole: the skinny kernel adds into the residual and
// prepares the norm in one launch.
inline int held_slice(int K, int slices) { return (K / 64 + slices - 1) / slices * 64; }
inline int held_slices(int M, int N, int K) {
  const int tiles = (N + 15) / 16, most = 64 * HWAVES * (M <= 32 ? 8 : 4), least = (K + most - 1) / most;
  if (tiles > 256 || least > 16 || (M <= 32 && K < 4096)) return 1;
  int want = (4 * 256 + tiles - 1) / tiles;
  want = want > 16 ? 16 : want;
  if (want > K / 512) want = K / 512;
  return want < least ? least : want;
}
inline SplitPlan split_plan(int M, int N, int K, bool silu = false) {
  SplitPlan p{M <= 64 ? 64 : 128, 1, 0, 0, false, false, 0, 0, 0.f};
  if (M > 16 && M <= 64 && K % 64 == 0 && N % 8 == 0 && !silu && held_slices(M, N, K) > 1) {
    p.k_slice = held_slice(K, held_slices(M, N, K));
    p.slices = (K + p.k_slice - 1) / p.k_slice;
    p.floats = (size_t)p.slices * M * N;
    p.held = true;
    return p;
  }
  // the block kernel's tiles, and as many slices as suit them, for a product that is divided; others keep what is in p
  auto in_blocks = [&](const SplitPlan& p) {
    if (!block_sizes(M, N, K, silu)) return p;
    // (few columns, many rows and a long k: 64-row tiles that are one to a compute unit keep theirs; 512 x 960 x 4,096 15.4 us, 17.4 in blocks)
    if (M > 64 && N <= 1024 && K >= 4096 && p.bm == 64 && !p.ring && (N + 127) / 128 * ((M + 63) / 64) * p.slices >= 224) return p;
    const BlockPlan b = block_plan(M, N, K, false, 2, 8);
    if (!b.rm || (p.ring && (M >= 1024 || ring_us(M, N, K, p.slices) <= b.us))) return p;
    return SplitPlan{p.bm, b.slices, b.k_slice, (size_t)b.slices * M * N, false, false, b.rm, b.cn, b.us};
  };
  // many rows, a long k and few 256 x 256 tiles (the down projection of a prompt): slices of k fill the
  // chip with the ring kernel's tiles once; a slice keeps 1,024 of k or more
  if (ring_slices_pay(M, K) && K >= 4096 && K % TBK == 0 && N % 8 == 0) {
    const int tiles = ((M + RBM - 1) / RBM) * ((N + RBN - 1) / RBN);
    int want = tiles < 192 ? 256 / tiles : 1;
    if (want > K / 1024) want = K / 1024;
    if (want >= 2) {
      p.k_slice = ((K + want - 1) / want + TBK - 1) / TBK * TBK;
      p.slices = (K + p.k_slice - 1) / p.k_slice;
      if (p.slices >= 2 && K - (p.slices - 1) * p.k_slice >= RING_MIN_K) {
        p.floats = (size_t)p.slices * M * N;
        p.ring = true;
        return in_blocks(p);
      }
      p.slices = 1, p.k_slice = 0;
    }
  }
  // 65 to 128 rows by many rows of W: the block kernel's tiles fill the chip by themselves, and what slices save is less than their second
  // pass costs until k is long (the time whole over the time in slices, 65 to 128 rows by 6,144 to 16,384 added into C, median and ends: k 2,048
  // 0.83, 0.64 to 1.01; 4,096 0.96, 0.77 to 1.20; 8,192 1.05, 0.87 to 1.40; 14,336 1.32, 1.15 to 1.65: 96 x 8,192 x 14,336 94 and 57 us)
  if (M > 64 && M <= 128 && K <= 8192 && K % RBK == 0 && N % 8 == 0 && N > 6112) return p;
  const int tiles = ((N + 127) / 128) * ((M + p.bm - 1) / p.bm);
  if (tiles >= 192 || N % 8 != 0) return p;
  // measured on SmolLM2-1.7B shapes: a long k (the down projection) always gains; a short one where the skinny kernel is at its weakest (33
  // to 64 rows: every workgroup reads all of A), up to 128 rows, and where the tiles are very few (the O projection of a portion of some
  // hundred rows: 16 to 64 tiles)
  if (K < 4096 && !(M > 32 && M <= 128 && K >= 1024) && !(M > 64 && K >= 2048 && tiles <= 128)) return p;
  // the tiled kernel's slices keep at least 8 k-steps (shorter ones cost more in partial sums than they gain), and of a long k, beyond
  // 64 rows, 16
  int want = (512 + tiles - 1) / tiles;
  want = want > 16 ? 16 : want;
  if (M > 64 && K >= 4096 && want > K / (16 * TBK)) want = K / (16 * TBK);
  if (want > K / (8 * TBK)) want = K / (8 * TBK);
  if (want < 2) return p;
  p.k_slice = ((K + want - 1) / want + TBK - 1) / TBK * TBK;
  p.slices = (K + p.k_slice - 1) / p.k_slice;
  if (p.slices < 2) return SplitPlan{p.bm, 1, 0, 0, false, false, 0, 0, 0.f};
  p.floats = (size_t)p.slices * M * N;
  // tiles of 64 rows where even with the slices a third of the compute units would have no workgroup
  if (tiles * p.slices < 168) p.bm = 64;
  return in_blocks(p);
}

// ws: [slices][M][N] float32.  Four columns a thread; EPI_SILU_MUL pairs column j with column N/2 + j.
template <int EPI, typename CT>
__global__ void splitk_reduce_kernel(const float* __restrict__ ws, int slices, CT* __restrict__ c, int ldc, int M, int N) {
  const int cols = EPI == EPI_SILU_MUL ? N / 2 : N, groups = cols / 4;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)M * groups) return;
  const int m = (int)(idx / groups), j = (int)(idx % groups) * 4;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f}, up = {0.f, 0.f, 0.f, 0.f};
  const size_t copy = (size_t)M * N;  // floats between one slice's copy of C and the next
  const float* row = ws + (size_t)m * N;
  int z = 0;
  for (; z + 4 <= slices; z += 4) {  // four slices' loads are on their way together; the sums keep the order of z
    f32x4 v[4], u[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      v[t] = *reinterpret_cast<const f32x4*>(row + (z + t) * copy + j);
      if (EPI == EPI_SILU_MUL) u[t] = *reinterpret_cast<const f32x4*>(row + (z + t) * copy + N / 2 + j);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sum += v[t];
      if (EPI == EPI_SILU_MUL) up += u[t];
    }
  }
  for (; z < slices; ++z) {
    sum += *reinterpret_cast<const f32x4*>(row + z * copy + j);
    if (EPI == EPI_SILU_MUL) up += *reinterpret_cast<const f32x4*>(row + z * copy + N / 2 + j);
  }
  CT* out = c + (size_t)m * ldc + j;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = sum[e];
    if (EPI == EPI_SILU_MUL) v = v / (1.0f + __expf(-v)) * up[e];
    store_c<CT>(out + e, v, EPI == EPI_ACCUMULATE);
  }
}

// The same pass for a product that accumulates into the float32 residual, one workgroup a row; with the new row
// in hand it also does the RMS norm that reads the residual next: h[m, n] = gamma[n] * (r[m, n] * s),
// s = 1 / sqrt(mean(r[m]^2) + eps), the formula of the norm's own kernel.  Rows of up to SPLIT_NORM_MAX columns.
constexpr int SPLIT_NORM_MAX = 256 * 4 * 8;
template <typename G>
__global__ __launch_bounds__(256) void splitk_reduce_norm_kernel(const float* __restrict__ ws, int slices, float* __restrict__ c,
                                                                 int ldc, int M, int N, const G* __restrict__ gamma, float eps,
                                                                 bf16* __restrict__ h, int ldh) {
  __shared__ float partial[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  f32x4 r[8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = (tid + 256 * i) * 4;
    if (j >= N) break;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};  // the slices in their order, then the residual: as the plain second pass does
    const size_t copy = (size_t)M * N;
    const float* row = ws + (size_t)m * N + j;
    const f32x4 old = *reinterpret_cast<const f32x4*>(c + (size_t)m * ldc + j);
    int z = 0;
    for (; z + 4 <= slices; z += 4) {  // four slices' loads on their way together
      f32x4 v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = *reinterpret_cast<const f32x4*>(row + (z + t) * copy);
#pragma unroll
      for (int t = 0; t < 4; ++t) sum += v[t];
    }
    for (; z < slices; ++z) sum += *reinterpret_cast<const f32x4*>(row + z * copy);
    sum = old + sum;
    *reinterpret_cast<f32x4*>(c + (size_t)m * ldc + j) = sum;
    r[i] = sum;
    ss += sum[0] * sum[0] + sum[1] * sum[1] + sum[2] * sum[2] + sum[3] * sum[3];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if (tid % 64 == 0) partial[tid / 64] = ss;
  __syncthreads();
  const float total = partial[0] + partial[1] + partial[2] + partial[3];
  const float scale = 1.0f / sqrtf(total / (float)N + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = (tid + 256 * i) * 4;
    if (j >= N) break;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (bf16)((float)gamma[j + e] * (r[i][e] * scale));
    *reinterpret_cast<bf16x4*>(h + (size_t)m * ldh + j) = o;
  }
}

// The same for the few rows of a decode step, which are as few workgroups: what bounds it are the round trips a thread makes one after
// the other, so as many threads as the row has words of four columns (at most 1,024), and a word's old value, gamma and up to AT_ONCE
// slices asked for together.  Same bits but for the order in which a row's squares are added.  (With
// 256 threads and four slices at a time, of 24 rows of 4,096: sixteen slices 33.3 -> 30.2 us with their product, eight 16.8 -> 15.4.)
constexpr int SPLIT_NORM_FEW = 64;
inline int split_norm_threads(int N) { return N >= 4096 ? 1024 : (N / 4 + 63) / 64 * 64; }
template <int AT_ONCE, typename G>
__global__ __launch_bounds__(1024) void splitk_reduce_norm_few_kernel(const float* __restrict__ ws, int slices, float* __restrict__ c,
                                                                      int ldc, int M, int N, const G* __restrict__ gamma, float eps,
                                                                      bf16* __restrict__ h, int ldh) {
  constexpr int WORDS = SPLIT_NORM_MAX / 4096;
  __shared__ float partial[16];
  const int m = blockIdx.x, tid = threadIdx.x, threads = blockDim.x;
  const size_t copy = (size_t)M * N;
  f32x4 r[WORDS];
  float g[WORDS][4], ss = 0.f;
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    const int j = (tid + threads * i) * 4;
    if (j >= N) break;
    const float* row = ws + (size_t)m * N + j;
    const f32x4 old = *reinterpret_cast<const f32x4*>(c + (size_t)m * ldc + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) g[i][e] = (float)gamma[j + e];
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int z = 0; z < slices; z += AT_ONCE) {
      f32x4 v[AT_ONCE];   // (behind the last slice: the last again, not added)
#pragma unroll
      for (int t = 0; t < AT_ONCE; ++t) v[t] = *reinterpret_cast<const f32x4*>(row + min(z + t, slices - 1) * copy);
#pragma unroll
      for (int t = 0; t < AT_ONCE; ++t)
        if (z + t < slices) sum += v[t];
    }
    sum = old + sum;
    *reinterpret_cast<f32x4*>(c + (size_t)m * ldc + j) = sum;
    r[i] = sum;
    ss += sum[0] * sum[0] + sum[1] * sum[1] + sum[2] * sum[2] + sum[3] * sum[3];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if (tid % 64 == 0) partial[tid / 64] = ss;
  __syncthreads();
  float total = partial[0];
  for (int w = 1; w < threads / 64; ++w) total += partial[w];
  const float scale = 1.0f / sqrtf(total / (float)N + eps);
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    const int j = (tid + threads * i) * 4;
    if (j >= N) break;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (bf16)(g[i][e] * (r[i][e] * scale));
    *reinterpret_cast<bf16x4*>(h + (size_t)m * ldh + j) = o;
  }
}

// Rows that are normed on the way: the folded kernel pays when there are at most 8 of them and whole tiles of 16 rows of W
// would leave compute units without a workgroup (measured: with 384 such tiles it no longer does).
inline bool fold_pays(int M, int N) { return M <= 8 && (N + 15) / 16 < 256; }

// What an accumulating product of these sizes can do for the RMS norm that reads the residual after it:
// 0 nothing; 1 (gemm_few_kernel for at most 16 rows, the skinny kernel up to 64) the operand bf16(gamma * r) and
// partial sums, see NormExtras;
// 2 (a product that divides k, given its workspace) the whole norm, in the pass that adds the slices.
inline int emit_mode(int M, int N, int K) {
  if (M > 16 && N % 4 == 0 && N <= SPLIT_NORM_MAX && split_plan(M, N, K).slices > 1) return 2;
  if (M <= 64 && !(M > 16 && N >= 32768)) return 1;
  return 0;
}
// Tiles of columns for which an emitting product of these sizes writes partial sums.
inline int emit_parts(int M, int N) {
  if (M > 64) return 0;
  return (N + 15) / 16 < 256 ? (N + 7) / 8 : (N + 15) / 16;  // half tiles while the tiles are few
}

template <int EPI, typename CT>
int launch_split(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, float* ws,
                 const SplitPlan& plan, hipStream_t stream, const NormExtras* norm = nullptr, float eps = 0.f,
                 bool second_pass = true) {
  const dim3 grid((N + 127) / 128, (M + plan.bm - 1) / plan.bm, plan.slices), block(256);
  const bool kfull = K % TBK == 0;
  const bool ring = plan.ring && ring_takes(a, lda, w, ldw, K);
  const bool blocks = plan.rm && block_takes(a, lda, w, ldw, K);
  if (blocks) {
    if (int rc = launch_block<EPI_STORE, float>(plan.rm, plan.cn, a, lda, w, ldw, ws, N, M, N, K, plan.k_slice, plan.slices, stream)) return rc;
  }
  const bool held = plan.held && held_takes(a, lda, w, ldw, M, plan.k_slice);
  if (held) {
    if (int rc = launch_held<EPI_STORE, float>(a, lda, w, ldw, ws, N, M, N, K, plan.k_slice, plan.slices, 0.f, nullptr, 0, stream)) return rc;
  }
  if (ring) {
    if (int rc = launch_ring<EPI_STORE, float>(a, lda, w, ldw, ws, N, M, N, K, plan.k_slice, plan.slices, stream)) return rc;
  }
#define GB_S(WM, FULL)                                                                                                   \
  if (!ring && !blocks && !held && (plan.bm == 64 * WM) && kfull == FULL)                                                                   \
    hipLaunchKernelGGL((gemm_tiled_kernel<WM, 2, 1, EPI_STORE, FULL, float>), grid, block, 0, stream, a, lda, w, ldw, ws, \
                       N, M, N, K, plan.k_slice, Groups{}, Glu{});
  GB_S(1, true) GB_S(1, false) GB_S(2, true) GB_S(2, false)
#undef GB_S
  if (int rc = launched("gemm_bf16 (split k)")) return rc;
  if (!second_pass) return 0;   // the caller adds the slices
  if constexpr (EPI == EPI_ACCUMULATE && std::is_same<CT, float>::value) {
    if (norm && norm->emit_h) {
#define GB_RN(KERNEL, THREADS, G)                                                                                          \
  hipLaunchKernelGGL(KERNEL, dim3(M), dim3(THREADS), 0, stream, ws, plan.slices, c, ldc, M, N, (const G*)norm->emit_gamma, eps, \
                     norm->emit_h, norm->emit_ldh)
#define GB_RNS(G)                                                                                                      \
  if (M > SPLIT_NORM_FEW) GB_RN((splitk_reduce_norm_kernel<G>), 256, G);                                               \
  else if (plan.slices > 8) GB_RN((splitk_reduce_norm_few_kernel<16, G>), split_norm_threads(N), G);                   \
  else if (plan.slices > 4) GB_RN((splitk_reduce_norm_few_kernel<8, G>), split_norm_threads(N), G);                    \
  else GB_RN((splitk_reduce_norm_few_kernel<4, G>), split_norm_threads(N), G);
      if (norm->emit_gamma_f32) { GB_RNS(float) } else { GB_RNS(bf16) }
#undef GB_RNS
#undef GB_RN
      return launched("gemm_bf16 (split k, second pass with the norm)");
    }
  }
  const int cols = EPI == EPI_SILU_MUL ? N / 2 : N;
  const size_t threads = (size_t)M * (cols / 4);
  hipLaunchKernelGGL((splitk_reduce_kernel<EPI, CT>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, ws,
                     plan.slices, c, ldc, M, N);
  return launched("gemm_bf16 (split k, second pass)");
}

// ------------------------------------------------------------------------ skinny
// grid (row tiles of W).  A workgroup of WAVES waves owns 16 rows of W and walks all of k in slices
// of ITERS*WAVES*64: wave w takes the 64-wide k blocks w, w+WAVES, ... of a slice; inside a block
// lane group q holds k = 8q..8q+7 of each half of 32 (the same split for W and for A, so the
// products pair up).  All loads of a slice are issued before its first MFMA.  The waves combine
// through LDS in wave order.  Few rows of W (a small N) are given many waves each, so that the
// launch still keeps enough loads in flight to use the memory system; no partial result ever
// leaves the workgroup, so no pass over memory is needed to combine them.
//
// EPI_STORE / EPI_ACCUMULATE: C[m, n] = or += the product.  EPI_SILU_MUL: W holds gate rows
// [0, N/2) and up rows [N/2, N); a tile takes 8 gate rows and the 8 up rows that belong to them
// and writes act[m, j] = gate / (1 + exp(-gate)) * up (crates/glassbox-core/src/model.rs:336-340)
// to C[M, N/2].

// 16 bytes of a lane that has something to read, else zeros: without a branch (SHORT) or with one, and the address behind it (before
// it, it costs the kernels that norm their rows the registers with which two workgroups fit on a unit).
template <bool SHORT>
__device__ __forceinline__ bf16x8 load_word(bool ok, const bf16* row, int k) {
  if constexpr (SHORT) return *or_zeros(ok, row + k);
  else return ok ? load8(row + k) : zero8();
}

// The A operand of one lane: 8 consecutive k of row m.  Plain: bfloat16 rows as they are.  RMS: the
// rows are the float32 residual; the operand is bf16(gamma[k] * x[k]) and sum(x^2) is gathered on
// the way, so that the caller can scale the finished product by 1/sqrt(mean(x^2) + eps): the RMS
// norm (crates/glassbox-core/src/model.rs:94-100) without a pass of its own.
// The 16 bytes that lane `lane` of the wave holds in v.
__device__ __forceinline__ bf16x8 from_lane(bf16x8 v, int lane) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  i32x4 w = __builtin_bit_cast(i32x4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_ds_bpermute(lane * 4, w[i]);
  return __builtin_bit_cast(bf16x8, w);
}

template <bool RMS, bool SHORT = false>
__device__ __forceinline__ bf16x8 load_a(const void* a, int lda, int m, int k, bool ok, const void* gamma, int gamma_f32,
                                         float& ss) {
  if (!RMS) return load_word<SHORT>(ok, (const bf16*)a + (size_t)m * lda, k);
  if (!ok) return zero8();
  const float* x = (const float*)a + (size_t)m * lda + k;
  const f32x4 x0 = *reinterpret_cast<const f32x4*>(x), x1 = *reinterpret_cast<const f32x4*>(x + 4);
  float g[8];
  if (gamma_f32) {
    const f32x4 g0 = *reinterpret_cast<const f32x4*>((const float*)gamma + k);
    const f32x4 g1 = *reinterpret_cast<const f32x4*>((const float*)gamma + k + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      g[e] = g0[e];
      g[4 + e] = g1[e];
    }
  } else {
    const bf16x8 gb = load8((const bf16*)gamma + k);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = (float)gb[e];
  }
  bf16x8 out;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float xe = e < 4 ? x0[e] : x1[e - 4];
    ss += xe * xe;
    out[e] = (bf16)(g[e] * xe);
  }
  return out;
}

// SHORT (rows that are normed already, where skinny_short() says so): the partial sums of the norm are asked for before W and added up
// behind its requests, and loads are without branches, so that all of a turn are asked for at once.  Otherwise the sums come first and
// loads are masked: many turns, and the traffic of many rows, are slower with an address chosen for every load and zeros fetched.
// (MT = 1, up to 16 rows: only with RMS.  Rows of so few that are normed already are gemm_few_kernel's.)
template <int MT, int WAVES, int ITERS, int RT, int EPI, bool RMS, bool SHORT, typename CT, bool HALF = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(const void* __restrict__ a, int lda,
                                                                 const bf16* __restrict__ w, int ldw, CT* __restrict__ c,
                                                                 int ldc, int M, int N, int K, const void* __restrict__ gamma,
                                                                 int gamma_f32, float eps, NormExtras extra, RopeExtras rope) {
  __shared__ float part[WAVES][RT][MT][64][4];
  __shared__ float sspart[RMS ? WAVES : 1][MT][64];
  constexpr int LR = MT == 2 ? 32 : 64;                 // lanes of a wave that stand for different rows in the sums below
  __shared__ float red[RMS ? 1 : WAVES][MT * 16];       // (with RMS the rows bring no partial sums)
  __shared__ float emit_sq[4][RT][MT][16];
  const float* __restrict__ parts = extra.parts;
  const int n_parts = extra.n_parts;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, q = lane / 16;
  const bf16* wrow[RT];
  bool row_ok[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int tile = blockIdx.x * RT + rt, pair_lo = 0, pair_hi = 8;
    if (EPI == EPI_ROPE && RT == 2 && rope.three_halves) tile = three_halves_tile(blockIdx.x, rt, &pair_lo, &pair_hi);
    int row;
    if (EPI == EPI_SILU_MUL) {
      row = r < 8 ? tile * 8 + r : N / 2 + tile * 8 + (r - 8);
    } else if (EPI == EPI_ROPE) {
      // a tile is 8 pairs of one head: its dims d0..d0+7 and those hd/2 further on
      const int per_head = rope.hd / 16, head = tile / per_head, d0 = (tile % per_head) * 8;
      row = head * rope.hd + (r < 8 ? d0 + r : rope.hd / 2 + d0 + (r - 8));
    } else if (HALF) {
      row = tile * 8 + (r & 7);  // a workgroup owns 8 rows of W: the tile's lower half stays empty
    } else {
      row = tile * 16 + r;
    }
    row_ok[rt] = EPI == EPI_SILU_MUL ? (tile * 8 + (r & 7) < N / 2) : HALF ? (r < 8 && row < N) : row < N;
    if (EPI == EPI_ROPE) row_ok[rt] = row_ok[rt] && (r & 7) >= pair_lo && (r & 7) < pair_hi;
    wrow[rt] = w + (size_t)(row_ok[rt] ? row : 0) * ldw;
  }

  f32x4 acc[RT][MT];
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    ss[t] = 0.f;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[rt][t][e] = 0.f;
  }

  // Partial sums of squares of the rows, one per tile of the product that made them (64 floats a tile): a lane a row, four loads
  // at once and then eight (one behind the other the rest of 384 tiles' sums cost 48 rows by 16,384 x 3,072 7 of 45 us).
  float got[4] = {0.f, 0.f, 0.f, 0.f};
  if (!RMS && parts != nullptr && lane % LR < M) {
    const float* mine = parts + lane % LR;
    constexpr int STEP = WAVES * 64 / LR;
    const int p0 = wave * (64 / LR) + lane / LR;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p0 + u * STEP < n_parts) got[u] = mine[(p0 + u * STEP) * 64];
    constexpr int AT_ONCE = SHORT ? 4 : 8;
    for (int p = p0 + 4 * STEP; p < n_parts; p += AT_ONCE * STEP) {
      float more[AT_ONCE];
#pragma unroll
      for (int u = 0; u < AT_ONCE; ++u) more[u] = p + u * STEP < n_parts ? mine[(p + u * STEP) * 64] : 0.f;
#pragma unroll
      for (int u = 0; u < AT_ONCE; ++u) got[u % 4] += more[u];
    }
  }
  auto add_up = [&] {
    if (RMS || parts == nullptr) return;
    float sum = ((got[0] + got[1]) + got[2]) + got[3];
#pragma unroll
    for (int o = LR; o < 64; o <<= 1) sum += __shfl_xor(sum, o, kWave);
    if (lane < LR && lane < MT * 16) red[wave][lane] = sum;
  };
  // a 64-wide k block is two MFMA steps of 32: lane group q holds k = 8q..8q+7 of each
  bf16x8 wf[RT][ITERS][2];
  auto ask = [&](int kbeg) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + (wave + WAVES * it) * 64 + q * 8;
        wf[rt][it][0] = load_word<SHORT>(row_ok[rt] && k < K, wrow[rt], k);
        wf[rt][it][1] = load_word<SHORT>(row_ok[rt] && k + 32 < K, wrow[rt], k + 32);
      }
  };
  if (SHORT) ask(0);
  add_up();
  for (int kbeg = 0; kbeg < K; kbeg += ITERS * WAVES * 64) {
    if (!SHORT || kbeg > 0) ask(kbeg);
    if (MT == 1) {
      bf16x8 xf[ITERS][2];
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + (wave + WAVES * it) * 64 + q * 8;
        xf[it][0] = load_a<RMS>(a, lda, r, k, r < M && k < K, gamma, gamma_f32, ss[0]);
        xf[it][1] = load_a<RMS>(a, lda, r, k + 32, r < M && k + 32 < K, gamma, gamma_f32, ss[0]);
      }
#pragma unroll
      for (int it = 0; it < ITERS; ++it)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][0], xf[it][0], acc[rt][0], 0, 0, 0);
          acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][1], xf[it][1], acc[rt][0], 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + (wave + WAVES * it) * 64 + q * 8;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          bf16x8 x0, x1;
          if (RMS) {
            const int m = t * 16 + r;
            x0 = load_a<RMS>(a, lda, m, k, m < M && k < K, gamma, gamma_f32, ss[t]);
            x1 = load_a<RMS>(a, lda, m, k + 32, m < M && k + 32 < K, gamma, gamma_f32, ss[t]);
          } else {
            // With several column blocks the rows of A are as much traffic from the cache as W is from memory, and the
            // cache serves a wave's load faster when neighbouring lanes share a piece of 64 bytes than when each asks
            // for 16 bytes of another row: lane 4R + Q loads piece Q of row R, and the operand's lane (row lane%16,
            // piece lane/16) takes it from there through the LDS crossbar.
            const int m = t * 16 + (lane >> 2), ka = k - q * 8 + (lane & 3) * 8;
            const bf16x8 y0 = load_a<false, SHORT>(a, lda, m, ka, m < M && ka < K, gamma, gamma_f32, ss[t]);
            const bf16x8 y1 = load_a<false, SHORT>(a, lda, m, ka + 32, m < M && ka + 32 < K, gamma, gamma_f32, ss[t]);
            x0 = from_lane(y0, 4 * r + q);
            x1 = from_lane(y1, 4 * r + q);
          }
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][0], x0, acc[rt][t], 0, 0, 0);
            acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][1], x1, acc[rt][t], 0, 0, 0);
          }
        }
      }
    }
  }
  // D[n, m]: lane l holds column m = l%16 and rows n = 4*(l/16) + e.  The first 256 threads own the
  // cells of the tiles: thread tid owns cell (l = tid/4, e = tid%4) of every row tile and column block.
  const int l = (tid % 256) / 4, e = tid % 4;
  const int nrow = 4 * (l / 16) + e;  // row of the tile, 0..15
  // What the owners will need from memory at the end (a cell's old value and the gamma of a norm to prepare; a
  // row's cosine, sine and cache slot) is asked for here, before the waves meet, so that it arrives while they do.
  constexpr int ROWS = HALF ? 8 : 16;  // rows of W a tile owns
  const bool emits = EPI == EPI_ACCUMULATE && extra.emit_h != nullptr;
  const bool empty = HALF && nrow >= 8;  // the lower half of a half tile
  float old[RT][MT], emit_g[RT], cs[RT][MT], sn[RT][MT];
  int slot[MT];
  if (EPI == EPI_ACCUMULATE && tid < 256) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int n = (blockIdx.x * RT + rt) * ROWS + nrow;
      emit_g[rt] = 0.f;
      if (emits && !empty && n < N)
        emit_g[rt] = extra.emit_gamma_f32 ? ((const float*)extra.emit_gamma)[n] : (float)((const bf16*)extra.emit_gamma)[n];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + l % 16;
        old[rt][t] = (!empty && m < M && n < N) ? (float)c[(size_t)m * ldc + n] : 0.f;
      }
    }
  }
  constexpr bool ROPE_EARLY = MT * RT <= 4;  // beyond that the registers would not hold what is asked for early
  if (EPI == EPI_ROPE && ROPE_EARLY && tid < 256) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = t * 16 + l % 16;
      slot[t] = (rope.slots != nullptr && m < M) ? rope.slots[m] : 0;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        int tile = blockIdx.x * RT + rt, pair_lo = 0, pair_hi = 8;
        if (RT == 2 && rope.three_halves) tile = three_halves_tile(blockIdx.x, rt, &pair_lo, &pair_hi);
        const int pair = (tile % (rope.hd / 16)) * 8 + (nrow & 7);
        const bool rotated = rope.cosv != nullptr && m < M && tile / (rope.hd / 16) < rope.nh + rope.nkv;
        cs[rt][t] = rotated ? rope.cosv[(size_t)m * (rope.hd / 2) + pair] : 1.f;
        sn[rt][t] = rotated ? rope.sinv[(size_t)m * (rope.hd / 2) + pair] : 0.f;
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][rt][t][lane][e] = acc[rt][t][e];
  if (RMS) {
#pragma unroll
    for (int t = 0; t < MT; ++t) sspart[wave][t][lane] = ss[t];
  }
  __syncthreads();
  if (tid >= 256) return;

  float v[RT][MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    float scale = 1.f;
    if (RMS) {
      // sum(x^2) of row m = t*16 + l%16: its k were spread over the waves and over the four lane groups
      float tot = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv)
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) tot += sspart[wv][t][l % 16 + 16 * qq];
      scale = 1.0f / sqrtf(tot / (float)K + eps);
    } else if (parts != nullptr) {
      float tot = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) tot += red[wv][t * 16 + l % 16];
      scale = 1.0f / sqrtf(tot / (float)K + eps);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float s = part[0][rt][t][l][e];
#pragma unroll
      for (int wv = 1; wv < WAVES; ++wv) s += part[wv][rt][t][l][e];
      v[rt][t] = s * scale;
    }
  }
  if (EPI == EPI_SILU_MUL) {
    // rows 0..7 are gate, 8..15 the matching up rows: the up values travel through LDS.  Only the
    // first four waves are here; the slice of the last wave is free once every sum above is done.
    float* up = &part[WAVES - 1][0][0][0][0];
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int t = 0; t < MT; ++t) up[(rt * MT + t) * 256 + tid] = v[rt][t];
    __syncthreads();
    if (nrow < 8) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int j = (blockIdx.x * RT + rt) * 8 + nrow;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const int m = t * 16 + l % 16;
          const float g = v[rt][t], u = up[(rt * MT + t) * 256 + tid + 128];
          if (m < M && j < N / 2) c[(size_t)m * ldc + j] = (CT)gated_unit(g, u, extra.glu);
        }
      }
    }
  } else if (EPI == EPI_ROPE) {
    // rows 0..7 and 8..15 of a tile are each other's partners: they meet through LDS as gate and up do
    float* other = &part[WAVES - 1][0][0][0][0];
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int t = 0; t < MT; ++t) other[(rt * MT + t) * 256 + tid] = v[rt][t];
    __syncthreads();
    const int half = rope.hd / 2, per_head = rope.hd / 16;
    const bool upper = nrow >= 8;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      int tile = blockIdx.x * RT + rt, pair_lo = 0, pair_hi = 8;
      if (RT == 2 && rope.three_halves) tile = three_halves_tile(blockIdx.x, rt, &pair_lo, &pair_hi);
      if ((nrow & 7) < pair_lo || (nrow & 7) >= pair_hi) continue;
      const int head = tile / per_head, pair = (tile % per_head) * 8 + (nrow & 7);
      const int dim = upper ? half + pair : pair;
      if (head * rope.hd + dim >= N) continue;
      const bool is_value = head >= rope.nh + rope.nkv, is_key = head >= rope.nh && !is_value;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + l % 16;
        if (m >= M) continue;
        float y = v[rt][t];
        if (!is_value && rope.cosv != nullptr) {
          const float p = other[(rt * MT + t) * 256 + (tid ^ 128)];
          const float co = ROPE_EARLY ? cs[rt][t] : rope.cosv[(size_t)m * half + pair];
          const float si = ROPE_EARLY ? sn[rt][t] : rope.sinv[(size_t)m * half + pair];
          y = upper ? y * co + p * si : y * co - p * si;
        }
        const bf16 yb = (bf16)y;
        c[(size_t)m * ldc + head * rope.hd + dim] = (CT)yb;
        if (rope.slots != nullptr && head >= rope.nh) {
          const int sl = ROPE_EARLY ? slot[t] : rope.slots[m], page = sl / rope.page_size, off = sl % rope.page_size;
          if (is_key)
            rope.k_pages[((size_t)page * rope.nkv + (head - rope.nh)) * rope.page_size * rope.hd +
                         key_offset(off, dim, rope.page_size, 8)] = yb;  // hd is a multiple of 16: pieces of 8
          else
            rope.v_pages[(((size_t)page * rope.nkv + (head - rope.nh - rope.nkv)) * rope.hd + dim) * rope.page_size + off] = yb;
        }
      }
    }
  } else {
    // accumulating onto the old values asked for above
    if (empty && !emits) return;
    float sq[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int n = (blockIdx.x * RT + rt) * ROWS + nrow;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + l % 16;
        sq[rt][t] = 0.f;
        if (!empty && m < M && n < N) {
          const float now = EPI == EPI_ACCUMULATE ? old[rt][t] + v[rt][t] : v[rt][t];
          c[(size_t)m * ldc + n] = (CT)now;
          if (emits) {
            extra.emit_h[(size_t)m * extra.emit_ldh + n] = (bf16)(emit_g[rt] * now);
            sq[rt][t] = now * now;
          }
        }
      }
    }
    if (emits) {
      // sum of squares over a tile's columns, per row: a row's 16 cells lie in four neighbouring lanes of each of
      // the four waves that are still here; added in a fixed order
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          float x = sq[rt][t];
          x += __shfl_xor(x, 1, kWave);
          x += __shfl_xor(x, 2, kWave);
          if (e == 0) emit_sq[wave][rt][t][l % 16] = x;
        }
      __syncthreads();  // the four waves that are still here
      const int stride = parts_stride(M);
      for (int i = tid; i < RT * MT * 16; i += 256) {
        const int rt = i / (MT * 16), t = i / 16 % MT, mm = i % 16, m = t * 16 + mm;
        const float tot = emit_sq[0][rt][t][mm] + emit_sq[1][rt][t][mm] + emit_sq[2][rt][t][mm] + emit_sq[3][rt][t][mm];
        if (m < M) extra.emit_ss[(size_t)(blockIdx.x * RT + rt) * stride + m] = tot;
      }
    }
  }
}

// ------------------------------------------------------------------------ folded (M <= 8, with the norm)
// At most 8 rows of A that are still to be normed by few rows of W (a first layer's product): the tiles of gemm_few_kernel below,
// 8 rows of W over two k ranges (k 0..31 and 64..95 of a 128-wide block, and 32..63 and 96..127), in waves that gather the sum of
// squares on the way (load_a).  The loads are nontemporal: W is read once.
template <int WAVES, int ITERS, int RT>
__global__ __launch_bounds__(WAVES * 64) void gemm_fold_kernel(const void* __restrict__ a, int lda, const bf16* __restrict__ w, int ldw,
                                                               bf16* __restrict__ c, int ldc, int M, int N, int K,
                                                               const void* __restrict__ gamma, int gamma_f32, float eps) {
  static_assert(WAVES >= 4, "the first four waves finish");
  __shared__ float part[WAVES][RT][64][4];
  __shared__ float sspart[WAVES][64];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, q = lane / 16;
  const int r8 = r & 7, khalf = (r >> 3) * 32;  // row of W and of A; which quarter of a k block: a load of the wave reads whole 128-byte lines
  const bf16* wrow[RT];
  bool row_ok[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int row = (blockIdx.x * RT + rt) * 8 + r8;
    row_ok[rt] = row < N;
    wrow[rt] = w + (size_t)(row_ok[rt] ? row : 0) * ldw;
  }
  f32x4 acc[RT];
  float ss = 0.f;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[rt][e] = 0.f;
  for (int kbeg = 0; kbeg < K; kbeg += ITERS * WAVES * 128) {
    bf16x8 wf[RT][ITERS][2], xf[ITERS][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + (wave + WAVES * it) * 128 + khalf + q * 8;
        wf[rt][it][0] = (row_ok[rt] && k < K) ? load8_once(wrow[rt] + k) : zero8();
        wf[rt][it][1] = (row_ok[rt] && k + 64 < K) ? load8_once(wrow[rt] + k + 64) : zero8();
      }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int k = kbeg + (wave + WAVES * it) * 128 + khalf + q * 8;
      xf[it][0] = load_a<true>(a, lda, r8, k, r8 < M && k < K, gamma, gamma_f32, ss);
      xf[it][1] = load_a<true>(a, lda, r8, k + 64, r8 < M && k + 64 < K, gamma, gamma_f32, ss);
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][0], xf[it][0], acc[rt], 0, 0, 0);
        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it][1], xf[it][1], acc[rt], 0, 0, 0);
      }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][rt][lane][e] = acc[rt][e];
  sspart[wave][lane] = ss;
  __syncthreads();
  // D[n, m]: lane l holds column m = l%16 and rows n = 4*(l/16) + e; thread tid of the first four waves owns cell
  // (l = tid/4, e = tid%4)
  const int l = (tid % 256) / 4, e = tid % 4;
  const int nrow = 4 * (l / 16) + e, m = l % 16;
  if (tid >= 256 || nrow >= 8 || m >= M) return;
  // sum(x^2) of row m: its k were spread over the waves, the four lane groups and the two halves
  float tot = 0.f;
#pragma unroll
  for (int wv = 0; wv < WAVES; ++wv)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) tot += sspart[wv][m + 16 * qq] + sspart[wv][m + 8 + 16 * qq];
  const float scale = 1.0f / sqrtf(tot / (float)K + eps);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int n = (blockIdx.x * RT + rt) * 8 + nrow;
    if (n >= N) continue;
    float sum = 0.f;
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv) sum += part[wv][rt][l][e] + part[wv][rt][l + 40][e];  // cell (n + 8, m + 8)
    c[(size_t)m * ldc + n] = (bf16)(sum * scale);
  }
}

inline int launch_fold(const void* a, int lda, const bf16* w, int ldw, bf16* c, int ldc, int M, int N, int K, const void* gamma,
                       int gamma_f32, float eps, hipStream_t stream) {
  const int tiles = (N + 7) / 8, blocks = (K + 127) / 128;  // 128-wide k blocks
  const int waves = blocks >= 16 ? 16 : 4;  // (eight blocks on sixteen waves were measured no faster than on four)
  const int rt = tiles >= 512 ? 2 : 1;
  const int iters = (blocks + waves - 1) / waves >= 2 ? 2 : 1;  // four loads in flight a wave were measured no faster
#define GB_CFG(WV, IT, RT)                                                                                                \
  if (waves == WV && iters == IT && rt == RT)                                                                             \
    hipLaunchKernelGGL((gemm_fold_kernel<WV, IT, RT>), dim3((tiles + RT - 1) / RT), dim3(WV * 64), 0, stream, a, lda, w, ldw, c, \
                       ldc, M, N, K, gamma, gamma_f32, eps);
  GB_CFG(4, 1, 1) GB_CFG(4, 1, 2) GB_CFG(4, 2, 1) GB_CFG(4, 2, 2)
  GB_CFG(16, 1, 1) GB_CFG(16, 1, 2) GB_CFG(16, 2, 1) GB_CFG(16, 2, 2)
#undef GB_CFG
  return launched("gemm_bf16 (folded)");
}

// -------------------------------------------------------------------------- few (M <= 16)
// Decode steps of up to sixteen requests.  A tile is 8 rows of W whose two ranges of 32 of a 64-wide k block stand side by side
// in a 16 x 16 MFMA tile (rows n and n + 8 the same row of W, columns m and m + 8 the same row of A, each over its own range; the
// cells (n, m) and (n + 8, m + 8) are the halves of a sum, the other two quarters are dropped), so that a load instruction of a
// wave reads whole 128-byte lines of 8 rows (bare reads of 16,384 x 2,048 in half lines of 16 rows 13.0 us, in whole lines,
// nontemporal, 11.4).  MB blocks of 8 rows of A share W's words.
// Such a kernel lasts a few microseconds and is made of trips to memory one behind the other, so everything that it reads is asked
// for before the first of it is waited for: the partial sums of the norm before it (a word of four rows a thread), what the
// epilogue needs, W and the rows of A, as much of k at once as the registers hold (few_plan).  Rows of W that the rotation or the
// gated unit pairs lie in one tile, four pairs, the partners mirrored (row n and 7 - n), and a cell's partner and a row's squares
// come by lane moves: one barrier in all.   parts / emit / rotation: as NormExtras and RopeExtras say.
// In steps of one row (of eight), the kernels before (16 rows of W a tile in half lines, partial sums one behind the other before
// W; 8 rows for the products by few rows of W) and now: SmolLM2-1.7B gate/up 13.9 -> 12.6 us (15.6 -> 13.3), QKV 9.5 -> 7.1
// (10.1 -> 7.7), down 9.2 -> 8.0 (11.0 -> 9.8), vocabulary 35.7 -> 31.0 (40.4 -> 33.8); SmolLM2-135M a layer 17.3 -> 13.6.  (Slower is a
// gate/up of 9 rows and more, a k of up to 400 and very many rows of W: 9 rows by 98,304 x 264 13.8 -> 15.6, in no number of tiles less.)
__device__ __forceinline__ float lane_mirror8(float v) {   // the value of lane 7 - n of the eight neighbouring lanes
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ float lane_quad(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// lanes (g, i) with g < 2 and i < 8 of a 16 x 16 result: v + the cell eight rows and eight columns further on
__device__ __forceinline__ float plus_folded(float v) {
  const unsigned t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, true);   // lane i + 8 of the row of 16
  const auto halves = __builtin_amdgcn_permlane32_swap(t, t, false, false);
  const unsigned upper = halves[1];                                                                      // of the upper half of the wave
  return v + __builtin_bit_cast(float, upper);
}

template <int MB, int WAVES, int ITERS, int RT, int EPI, typename CT>
__global__ __launch_bounds__(WAVES * 64, WAVES >= 8 ? 4 : 1) void gemm_few_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w, const float* __restrict__ parts, int lda, int ldw, int M, int N, int K, int n_parts,
    CT* __restrict__ c, int ldc, float eps, NormExtras extra, RopeExtras rope) {
  static_assert(EPI != EPI_ACCUMULATE || RT != 3, "partial sums of two tiles meet");
  constexpr int CELLS = RT * MB, OWN = (CELLS + WAVES - 1) / WAVES;   // blocks of 8 x 8 cells; those that a wave finishes
  constexpr bool PAIRS = EPI == EPI_ACCUMULATE && RT > 1;             // partial sums of 16 columns
  __shared__ __attribute__((aligned(16))) float part[WAVES][CELLS][64];   // [row of A][row of the tile]
  __shared__ __attribute__((aligned(16))) float red[WAVES][8 * MB];
  __shared__ float squares[PAIRS ? CELLS : 1][8];
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r8 = lane & 7, kpos = ((lane >> 3) & 1) * 32 + (lane >> 4) * 8;
  // words of four rows' partial sums: of up to 8 rows 8 floats a tile, beyond 64 of which 16 are wanted
  // (the sums are floats of a caller's: words of them need not begin at 16 bytes)
  typedef float floats4 __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 got = {0.f, 0.f, 0.f, 0.f};
  if (parts != nullptr) {
    auto word = [&](int i) -> f32x4 { return *reinterpret_cast<const floats4*>(parts + (MB == 1 ? 4 * i : 64 * (i >> 2) + 4 * (i & 3))); };
    if (tid < 2 * MB * n_parts) got = word(tid);
    for (int i = tid + WAVES * 64; i < 2 * MB * n_parts; i += WAVES * 64) got += word(i);
  }
  // the pair of row n of a tile whose rows are four pairs
  auto pair_of = [](int n) { return n < 4 ? n : 7 - n; };
  auto head_of = [&](int tile) { return (int)(((float)tile + 0.5f) * rope.per_tile); };   // tile / (hd / 8), exact below 2^21 tiles
  // the cells of this lane in the epilogue: row n of tile cell / MB, row m of A in block cell % MB
  const int n = lane & 7;
  float old[OWN], gamma[OWN], cs[OWN], sn[OWN];
  int slot[OWN], head[OWN], pair[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int cell = wave + WAVES * i, own = blockIdx.x * RT + cell / MB, m = cell % MB * 8 + (lane >> 3);
    old[i] = gamma[i] = sn[i] = 0.f;
    cs[i] = 1.f;
    slot[i] = head[i] = pair[i] = 0;
    if (cell >= CELLS) continue;
    if (EPI == EPI_ACCUMULATE && m < M && own * 8 + n < N) {
      old[i] = (float)c[(size_t)m * ldc + own * 8 + n];
      if (extra.emit_h != nullptr)
        gamma[i] = extra.emit_gamma_f32 ? ((const float*)extra.emit_gamma)[own * 8 + n] : (float)((const bf16*)extra.emit_gamma)[own * 8 + n];
    }
    if (EPI == EPI_ROPE) {
      head[i] = head_of(own);
      pair[i] = (own - head[i] * (rope.hd / 8)) * 4 + pair_of(n);
      if (m < M && own * 8 < N) {
        if (rope.slots != nullptr) slot[i] = rope.slots[m];
        if (rope.cosv != nullptr && head[i] < rope.nh + rope.nkv) {
          cs[i] = rope.cosv[(size_t)m * (rope.hd / 2) + pair[i]];
          sn[i] = rope.sinv[(size_t)m * (rope.hd / 2) + pair[i]];
        }
      }
    }
  }
  // (rows beyond N or M are read from one that exists: what comes of them is not stored)
  const bf16* wrow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int tile = blockIdx.x * RT + rt;
    int row;
    if (EPI == EPI_SILU_MUL) {
      const int j = min(tile * 4 + pair_of(r8), N / 2 - 1);
      row = r8 < 4 ? j : N / 2 + j;
    } else if (EPI == EPI_ROPE) {
      const int h = head_of(tile);
      row = min(h * rope.hd + (tile - h * (rope.hd / 8)) * 4 + pair_of(r8) + (r8 < 4 ? 0 : rope.hd / 2), N - 1);
    } else {
      row = min(tile * 8 + r8, N - 1);
    }
    wrow[rt] = w + (size_t)row * ldw + kpos;
  }
  const bf16* xrow[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) xrow[mb] = a + (size_t)min(mb * 8 + r8, M - 1) * lda + kpos;
  f32x4 acc[RT][MB];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[rt][mb][e] = 0.f;

  // A wave's 64-wide blocks of a turn: every WAVES-th, so that the waves read side by side (one row by 16,384 x 2,048 12.3 us, in runs
  // 13.3); of a short k, where that makes no difference, a run of neighbouring ones
  auto block_of = [&](int it) { return WAVES == 4 ? wave * ITERS + it : wave + WAVES * it; };
  constexpr int TURN = ITERS * WAVES * 64;
  for (int kbeg = 0; kbeg < K; kbeg += TURN) {
    bf16x8 wf[RT][ITERS], xf[MB][ITERS];
    if (kbeg + TURN <= K) {
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + block_of(it) * 64;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) wf[rt][it] = load8_once(wrow[rt] + k);
      }
#pragma unroll
      for (int it = 0; it < ITERS; ++it)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xf[mb][it] = load8(xrow[mb] + kbeg + block_of(it) * 64);
    } else {  // the last turn of a k that is not of whole turns: zeros beyond it
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int k = kbeg + block_of(it) * 64;
        const bool ok = k + kpos < K;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) wf[rt][it] = __builtin_nontemporal_load(or_zeros(ok, wrow[rt] + k));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xf[mb][it] = *or_zeros(ok, xrow[mb] + k);
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // all loads of a turn are asked for before the first is waited for
    if (kbeg == 0 && parts != nullptr) {
#pragma unroll
      for (int o = 2 * MB; o < 64; o <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) got[e] += __shfl_xor(got[e], o, kWave);
      if (lane < 2 * MB) *reinterpret_cast<f32x4*>(&red[wave][4 * lane]) = got;
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[rt][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[rt][it], xf[mb][it], acc[rt][mb], 0, 0, 0);
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = plus_folded(acc[rt][mb][e]);
      if (lane < 32 && (lane & 15) < 8) *reinterpret_cast<f32x4*>(&part[wave][rt * MB + mb][(lane & 7) * 8 + 4 * (lane >> 4)]) = v;
    }
  __syncthreads();
  if (wave >= CELLS) return;
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int cell = wave + WAVES * i, own = blockIdx.x * RT + cell / MB, m = cell % MB * 8 + (lane >> 3);
    if (cell >= CELLS) continue;
    float v = part[0][cell][lane];
#pragma unroll
    for (int wv = 1; wv < WAVES; ++wv) v += part[wv][cell][lane];
    if (parts != nullptr) {
      float tot = red[0][m];
#pragma unroll
      for (int wv = 1; wv < WAVES; ++wv) tot += red[wv][m];
      v *= 1.0f / sqrtf(tot / (float)K + eps);
    }
    if (EPI == EPI_SILU_MUL) {
      const float u = lane_mirror8(v);
      if (m < M && n < 4 && own * 4 + n < N / 2) c[(size_t)m * ldc + own * 4 + n] = (CT)gated_unit(v, u, extra.glu);
    } else if (EPI == EPI_ROPE) {
      const float p = lane_mirror8(v);
      if (m >= M || own * 8 >= N) continue;
      const int half = rope.hd / 2, dim = n < 4 ? pair[i] : half + pair[i];
      // (a value, and any head without angles, is no sum with its partner: of a partner that is not finite 0 would make a NaN)
      const bool turns = rope.cosv != nullptr && head[i] < rope.nh + rope.nkv;
      const bf16 yb = (bf16)(!turns ? v : n < 4 ? v * cs[i] - p * sn[i] : v * cs[i] + p * sn[i]);
      c[(size_t)m * ldc + head[i] * rope.hd + dim] = (CT)yb;
      if (rope.slots != nullptr && head[i] >= rope.nh) {
        const int page = rope.page_shift >= 0 ? slot[i] >> rope.page_shift : slot[i] / rope.page_size, off = slot[i] - page * rope.page_size;
        if (head[i] < rope.nh + rope.nkv)
          rope.k_pages[((size_t)page * rope.nkv + (head[i] - rope.nh)) * rope.page_size * rope.hd + key_offset(off, dim, rope.page_size, 8)] = yb;
        else
          rope.v_pages[(((size_t)page * rope.nkv + (head[i] - rope.nh - rope.nkv)) * rope.hd + dim) * rope.page_size + off] = yb;
      }
    } else {
      const int col = own * 8 + n;
      const bool mine = m < M && col < N;
      const float now = EPI == EPI_ACCUMULATE ? old[i] + v : v;
      if (mine) c[(size_t)m * ldc + col] = (CT)now;
      if (EPI == EPI_ACCUMULATE && extra.emit_h != nullptr) {
        if (mine) extra.emit_h[(size_t)m * extra.emit_ldh + col] = (bf16)(gamma[i] * now);
        float sq = mine ? now * now : 0.f;   // the squares of a row over the tile's columns, in a fixed order
        sq += lane_mirror8(sq);
        sq += lane_quad<0xB1>(sq);
        sq += lane_quad<0x4E>(sq);
        if (PAIRS) {
          if (n == 0) squares[cell][lane >> 3] = sq;
        } else if (n == 0 && m < M && own * 8 < N) {
          extra.emit_ss[(size_t)own * (MB == 1 ? 8 : 64) + m] = sq;
        }
      }
    }
  }
  if (PAIRS && extra.emit_h != nullptr) {
    __syncthreads();  // the waves that are still here
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int cell = wave + WAVES * i, own = blockIdx.x * RT + cell / MB, m = cell % MB * 8 + (lane >> 3);
      if (cell < CELLS && cell / MB % 2 == 0 && n == 0 && m < M && own * 8 < N)
        extra.emit_ss[(size_t)(own / 2) * (MB == 1 ? 8 : 64) + m] = squares[cell][lane >> 3] + squares[cell + MB][lane >> 3];
    }
  }
}

// How a product of up to 16 rows is cut: tiles a workgroup, its waves, and the 64-wide k blocks a wave asks for at once.
struct FewPlan {
  int rt, waves, iters;
};
inline FewPlan few_plan(int epi, int M, int N, int K) {
  const int tiles = epi == EPI_SILU_MUL ? (N / 2 + 3) / 4 : (N + 7) / 8, blocks = (K + 63) / 64;
  const bool many = M > 8;
  FewPlan p{1, 4, 2};
  // The compute unit with the most tiles ends last, so as many tiles a workgroup as leave it the fewest (8 rows by 5,120 x 960, 640 tiles,
  // in threes 4.56 us, in twos, 320 workgroups, 5.18; 9 rows by 8,000 x 1,040, 1,000 tiles, in fours 6.0, in threes, 334 workgroups,
  // 8.5).  Beyond that more tiles share the rows of A, which beyond 8 rows are as much traffic as W and weigh more; of a k of up to 512 more
  // than two only leave fewer waves (9 rows by 8,064 x 384 in fours 4.25, in twos 3.96).  Accumulating: two or four where emit_parts()
  // has sums of 16 columns, else one.
  if (epi != EPI_ACCUMULATE || (N + 15) / 16 >= 256) {
    const int step = epi == EPI_ACCUMULATE ? 2 : 1;
    int least = 0;
    for (int rt = step; rt <= (blocks <= 8 ? 2 : 4); rt += step) {
      const int cost = ((tiles + rt - 1) / rt + 255) / 256 * (many ? 5 * rt + 6 : 10 * rt + 3);
      if (rt == step || cost < least) least = cost, p.rt = rt;
    }
  }
  // All of k at once where it is short; of a longer one turns of eight waves, whose two, three or four blocks a wave leave the least of the
  // last turn empty, the most that do (one row by 28,672 x 4,096 38.3 us in turns of 32 blocks of four tiles, of two tiles 35.7).  Beyond 8 rows
  // four only of up to two tiles a workgroup and a k of up to 4,096, and of four tiles not three: the registers of two such workgroups a unit
  // end there.  In which order a cell is summed depends on the waves, not on the turns.  Few tiles by a k beyond 2,048 (O and down projections)
  // have sixteen waves: eight would be 2 to 6 % faster (one row by 4,096 x 14,336 19.7 us, 21.0), but sum in another order, and a model of 32 such
  // layers in 16 bits ends further from the results it had (0.011 of the logits' norm) than those may move.
  if (blocks <= 8) return p;
  if (blocks <= 12) {
    p.iters = 3;
    return p;
  }
  p.waves = 8;
  if (!many && p.rt == 1 && blocks > 32 && blocks <= 40) {
    p.iters = 5;   // (one row by 960 x 2,560 in one turn 3.8 us, in two of 24 blocks 4.1)
    return p;
  }
  if (blocks > 32 && p.rt <= 2 && tiles < 768) {
    p.waves = 16, p.iters = blocks <= 64 || p.rt == 2 || many ? 4 : 8;
    return p;
  }
  auto asked = [&](int it) { return (blocks + 8 * it - 1) / (8 * it) * (10 * it + 1); };
  const int most = !many || (p.rt <= 2 && blocks <= 64) ? 4 : p.rt == 4 ? 2 : 3;
  for (int it = 3; it <= most; ++it)
    if (asked(it) < asked(p.iters)) p.iters = it;
  return p;
}

template <int MB, int EPI, typename CT>
int launch_few_mb(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, float eps, const NormExtras& extra,
                  hipStream_t stream, const RopeExtras& rope) {
  const int tiles = EPI == EPI_SILU_MUL ? (N / 2 + 3) / 4 : (N + 7) / 8;
  const FewPlan p = few_plan(EPI, M, N, K);
  bool found = false;
#define GB_FEW(WV, IT, R)                                                                                                     \
  if constexpr (!(EPI == EPI_ACCUMULATE && R == 3))                                                                           \
    if (p.waves == WV && p.iters == IT && p.rt == R) {                                                                        \
      found = true;                                                                                                           \
      hipLaunchKernelGGL((gemm_few_kernel<MB, WV, IT, R, EPI, CT>), dim3((tiles + R - 1) / R), dim3(WV * 64), 0, stream, a, w, \
                         extra.parts, lda, ldw, M, N, K, extra.n_parts, c, ldc, eps, extra, rope);                            \
    }
#define GB_FEWS(WV, IT) GB_FEW(WV, IT, 1) GB_FEW(WV, IT, 2) GB_FEW(WV, IT, 3) GB_FEW(WV, IT, 4)
  // (what few_plan can ask for)
  GB_FEW(4, 2, 1) GB_FEW(4, 2, 2) GB_FEWS(4, 3) GB_FEWS(8, 2) GB_FEW(8, 3, 1) GB_FEW(8, 3, 2) GB_FEW(8, 3, 3)
  GB_FEW(8, 4, 1) GB_FEW(8, 4, 2) GB_FEW(16, 4, 1) GB_FEW(16, 4, 2)
  if constexpr (MB == 1) { GB_FEW(8, 3, 4) GB_FEW(8, 4, 3) GB_FEW(8, 4, 4) GB_FEW(8, 5, 1) GB_FEW(16, 8, 1) }
#undef GB_FEWS
#undef GB_FEW
  GB_REQUIRE(found, "gemm_bf16: no kernel of %d tiles, %d waves and %d blocks for up to 16 rows", p.rt, p.waves, p.iters);
  return launched("gemm_bf16 (few rows)");
}

template <int EPI, typename CT>
int launch_few(const bf16* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, float eps, const NormExtras& extra,
               hipStream_t stream, const RopeExtras& rope = RopeExtras{}) {
  RopeExtras rp = rope;
  if (EPI == EPI_ROPE) {
    rp.per_tile = 8.0f / (float)rope.hd;
    rp.page_shift = rope.page_size > 0 && (rope.page_size & (rope.page_size - 1)) == 0 ? __builtin_ctz(rope.page_size) : -1;
  }
  if (M <= 8) return launch_few_mb<1, EPI, CT>(a, lda, w, ldw, c, ldc, M, N, K, eps, extra, stream, rp);
  return launch_few_mb<2, EPI, CT>(a, lda, w, ldw, c, ldc, M, N, K, eps, extra, stream, rp);
}

// Waves per workgroup, k blocks in flight per wave and row tiles per workgroup.
inline void skinny_plan(int tiles, int K, int mt, int* waves, int* iters, int* rt) {
  // two row tiles a workgroup halve the re-reading of A once that still leaves workgroups for
  // three quarters of the compute units (384 tiles: better with two; 256 tiles: better with one)
  const int blocks = (K + 63) / 64;               // 64-wide k blocks
  *rt = tiles >= 384 ? 2 : 1;
  // A wave's k blocks come one after the other, each a round trip to memory: from twelve blocks on sixteen waves take
  // one or two each (a k of 960, fifteen blocks: a decode step of SmolLM2-360M 4 to 8 % faster than with four waves)
  *waves = blocks >= 12 ? 16 : 4;
  const int per_wave = (blocks + *waves - 1) / *waves;
  *iters = (mt == 1 && per_wave >= 2) ? 2 : 1;
}

// Whether rows that are normed already take the form for a short k (SHORT): up to 2,048, two turns of sixteen waves (us, without /
// with: 17 rows by 1,600 x 960 5.6 / 5.2, by 2,048 x 2,048 7.2 / 5.9, 40 rows by 1,600 x 960 6.9 / 6.7; 64 rows by 49,152 x 2,048 43.6 /
// 43.5; beyond, 40 rows by 16,384 x 3,072 36.4 / 38.9, 32 by 28,672 x 8,192 120 / 140), and up to 32 rows with one tile a workgroup of any
// k (17 rows by 4,096 x 5,120 17.4 / 15.0, 32 rows 17.5 / 16.1), but of half a tile only up to 24 (by 960 x 2,560 17 rows 7.6 / 6.8, 24
// rows 7.7 / 7.6, 32 rows 7.7 / 8.1).
inline bool skinny_short(int M, int K, int rt, bool half) { return K <= 2048 || (M <= 32 && rt == 1 && (!half || M <= 24)); }

template <int MT, int EPI, bool RMS, typename CT>
int launch_skinny_mt(int tiles, const void* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K,
                     const void* gamma, int gamma_f32, float eps, const NormExtras& extra, const RopeExtras& rope,
                     hipStream_t stream) {
  int waves, iters, rt;
  skinny_plan(tiles, K, MT, &waves, &iters, &rt);
  if constexpr ((EPI == EPI_STORE || EPI == EPI_ACCUMULATE) && !RMS) {
    // Few rows of W (a narrow model's O and down projections of more than 16 rows):
    // workgroups of 8 rows of W, half of each tile left empty, so that twice as many compute units draw on memory.
    if (tiles < 256 && extra.parts == nullptr) {
      const int halves = (N + 7) / 8;
      const bool brief = skinny_short(M, K, 1, true);
#define GB_HALF(WV, SHORT)                                                                                                 \
  if (waves == WV && brief == SHORT)                                                                                       \
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, WV, 1, 1, EPI, RMS, SHORT, CT, true>), dim3(halves), dim3(WV * 64), 0, stream, a, \
                       lda, w, ldw, c, ldc, M, N, K, gamma, gamma_f32, eps, extra, rope);
      GB_HALF(4, true) GB_HALF(16, true) GB_HALF(16, false)
#undef GB_HALF
      return launched("gemm_bf16 (skinny, half tiles)");
    }
  }
  // the rotating product with two tiles a workgroup: a tile and a half each where that divides evenly (three_halves_tile)
  RopeExtras rp = rope;
  rp.three_halves = (EPI == EPI_ROPE && rt == 2 && tiles % 3 == 0) ? 1 : 0;
  const int groups = rp.three_halves ? 2 * tiles / 3 : (tiles + rt - 1) / rt;
  const bool brief = !RMS && skinny_short(M, K, rt, false);
#define GB_CFG(WV, IT, RT, SHORT)                                                                                          \
  if (waves == WV && iters == IT && rt == RT && brief == SHORT)                                                            \
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, WV, IT, RT, EPI, RMS, SHORT, CT>), dim3(groups), dim3(WV * 64), 0, stream, a, lda, \
                       w, ldw, c, ldc, M, N, K, gamma, gamma_f32, eps, extra, rp);
  // the configurations skinny_plan and skinny_short can ask for
  GB_CFG(4, 1, 1, !RMS) GB_CFG(4, 1, 2, !RMS) GB_CFG(16, 1, 1, !RMS) GB_CFG(16, 1, 2, !RMS)
  if constexpr (!RMS) { GB_CFG(16, 1, 2, false) }
  if constexpr (!RMS && MT > 2) { GB_CFG(16, 1, 1, false) }
  if constexpr (RMS && MT == 1) { GB_CFG(4, 2, 1, false) GB_CFG(4, 2, 2, false) GB_CFG(16, 2, 1, false) GB_CFG(16, 2, 2, false) }
#undef GB_CFG
  return launched("gemm_bf16 (skinny)");
}

template <int EPI, bool RMS, typename CT>
int launch_skinny(const void* a, int lda, const bf16* w, int ldw, CT* c, int ldc, int M, int N, int K, const void* gamma,
                  int gamma_f32, float eps, const NormExtras& extra, hipStream_t stream, const RopeExtras& rope = RopeExtras{}) {
  const int tiles = EPI == EPI_SILU_MUL ? (N / 2 + 7) / 8 : (N + 15) / 16;  // EPI_ROPE: N is a multiple of 16
  const int mt = (M + 15) / 16;
#define GB_MT(T) \
  if (mt == T) return launch_skinny_mt<T, EPI, RMS, CT>(tiles, a, lda, w, ldw, c, ldc, M, N, K, gamma, gamma_f32, eps, extra, rope, stream);
  if constexpr (RMS) { GB_MT(1) }   // (up to 16 rows that are normed already: gemm_few_kernel)
  GB_REQUIRE(mt > 1, "gemm_bf16: the skinny kernel takes up to 16 rows with the norm alone");
  GB_MT(2) GB_MT(3)
#undef GB_MT
  return launch_skinny_mt<4, EPI, RMS, CT>(tiles, a, lda, w, ldw, c, ldc, M, N, K, gamma, gamma_f32, eps, extra, rope, stream);
}

// Which kernel takes a product, and how.  `emits`: emit_mode if the next norm is to be prepared, else 0; `workspace`: one is there.
enum : int { kTiled = 0, kRing = 1, kFew = 2 /* few, skinny or folded */, kHeld = 3, kBlock = 4, kSlices = 5 };
struct Route {
  int kernel;
  BlockPlan block;   // the block kernel's tile for the whole product, where it may take it
  SplitPlan split;   // the slices that were on offer (kSlices: taken)
};
inline Route route(int epi, const void* a, int lda, const void* w, int ldw, int M, int N, int K, bool gamma, bool parts, int emits, bool workspace) {
  Route r{kTiled, BlockPlan{}, SplitPlan{}};
  const bool silu = epi == EPI_SILU_MUL;
  const bool held = !gamma && !emits && epi != EPI_ACCUMULATE && held_pays(epi, M, N, K, parts) && held_takes(a, lda, w, ldw, M, K);
  const bool blocks = !held && !gamma && !parts && block_sizes(M, N, K, silu) && block_takes(a, lda, w, ldw, K);
  const bool rings = ring_pays(epi, a, lda, w, ldw, M, N, K);
  if (blocks) r.block = block_plan(M, N, K, silu, 1, 1);
  bool whole = false;
  if (workspace && M > 16 && !gamma && emits != 1 && !parts) {  // (gemm_few_kernel's rows are never divided)
    r.split = split_plan(M, N, K, silu);
    if (r.split.slices <= 1 || (silu && N % 16 != 0)) r.split = SplitPlan{};
    // a product that only stores needs no second pass: not divided where that takes less (QKV, 131 x 6,144 x 2,048: 16 us in slices, 13 whole)
    whole = blocks && epi != EPI_ACCUMULATE && r.split.rm && r.block.us < r.split.us;
    if (r.split.slices > 1 && !held && !whole) return r.kernel = kSlices, r;
  }
  if (held) return r.kernel = kHeld, r;
  if (blocks && (M > 64 || epi != EPI_ACCUMULATE) && !emits && (whole || block_pays(epi, M, N, K, r.block, rings))) return r.kernel = kBlock, r;
  // 17 to 64 rows by very many rows of W that the held kernel does not take (a long k): measured twice as fast
  // through the tiles as through the skinny kernel with four column blocks (49,152 x 2,048: 102 -> about 50 us),
  // and with two column blocks as fast or faster (49,152 x 960 at 17 to 32 rows: 30 -> 25 us)
  const bool wide_head = M > 16 && N >= 32768 && !gamma && !parts;
  if (M <= 64 && !wide_head) return r.kernel = kFew, r;
  if (rings) r.kernel = kRing;
  return r;
}

}  // namespace

// epilogue: 0 store, 1 accumulate (float32 C), 2 SiLU-multiply of stacked gate/up rows (C is [M, N/2]).
// gamma != nullptr (at most 64 rows, bfloat16 C, epilogue 0 or 2): a is the float32 residual and the
// product is that of its RMS-normed rows: bf16(gamma * x) as the operand, 1/sqrt(mean(x^2) + eps) on
// the result.
// split_ws != nullptr: a workspace of split_ws_floats floats that the product may use to divide k over
// workgroups (gb_gemm_bf16_split_floats says how many it needs; fewer than that is an error).
// emit_h != nullptr (accumulating product that gb_gemm_bf16_emit_parts accepts): the next norm's operand and
// partial sums are written beside the residual, see NormExtras.  parts != nullptr (at most 64 rows, no
// gamma): the rows of a are such an operand and the product is scaled by the norm's factor from n_parts
// partial sums; eps is that norm's.
extern "C" int gb_gemm_bf16_emit_parts(int M, int N) { return emit_parts(M, N); }
// 0, 1 or 2: see emit_mode.  With 2, gb_gemm_bf16 takes emit_gamma, emit_h and eps (no emit_ss) together with the
// workspace and writes the normed rows to emit_h.
extern "C" int gb_gemm_bf16_emit_mode(int M, int N, int K) { return emit_mode(M, N, K); }

// Floats of workspace with which gb_gemm_bf16 would split k for this product (0: it would not).
extern "C" long long gb_gemm_bf16_split_floats(int M, int N, int K) {
  if (M <= 16) return 0;
  const size_t plain = split_plan(M, N, K).floats, unit = split_plan(M, N, K, true).floats;   // (either may be asked for)
  return (long long)(plain > unit ? plain : unit);
}

// Slices into which gb_gemm_bf16_partial divides k for a product of these sizes (1: it would not divide it).
extern "C" int gb_gemm_bf16_slices(int M, int N, int K) {
  if (M <= 16) return 1;
  const SplitPlan plan = split_plan(M, N, K);
  return plan.slices > 1 ? plan.slices : 1;
}

// The first pass alone of a product that divides k: ws receives [slices][M][N] float32, slice z the product over the
// z-th run of k, for a reader that adds them in their order (as the second pass of gb_gemm_bf16 would).
extern "C" int gb_gemm_bf16_partial(const void* a, int lda, const void* w, int ldw, float* ws, long long ws_floats, int M,
                                    int N, int K, hipStream_t stream) {
  GB_REQUIRE(M > 16 && N > 0 && K > 0 && K % 8 == 0, "gemm_bf16_partial: bad sizes M=%d N=%d K=%d", M, N, K);
  GB_REQUIRE(ldw % 8 == 0 && lda % 8 == 0 && lda >= K && ldw >= K, "gemm_bf16_partial: row strides (%d, %d)", lda, ldw);
  GB_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0) && ws && ((uintptr_t)ws % 16 == 0),
             "gemm_bf16_partial: operands and workspace must be 16-byte aligned");
  const SplitPlan plan = split_plan(M, N, K);
  GB_REQUIRE(plan.slices > 1, "gemm_bf16_partial: a product of M=%d N=%d K=%d does not divide k", M, N, K);
  GB_REQUIRE((long long)plan.floats <= ws_floats, "gemm_bf16_partial: the workspace holds %lld floats, %zu are needed", ws_floats,
             plan.floats);
  return launch_split<EPI_STORE, float>((const bf16*)a, lda, (const bf16*)w, ldw, (float*)nullptr, N, M, N, K, ws, plan, stream,
                                        nullptr, 0.f, false);
}

// The kernel that gb_gemm_bf16 (epilogues 0 to 2, no gamma, no norm to prepare; with a workspace or without) or gb_gemm_bf16_rope
// (epilogue 3, no gamma) launches for these sizes: 0 tiled, 1 ring, 2 few or skinny, 3 held, 4 block, 5 slices of k.
extern "C" int gb_gemm_bf16_route(int M, int N, int K, int epilogue, int parts, int workspace) {
  if (epilogue == EPI_ROPE) return held_pays(epilogue, M, N, K, parts != 0) && held_takes(nullptr, K, nullptr, K, M, K) ? kHeld : kFew;
  return route(epilogue, nullptr, K, nullptr, K, M, N, K, false, parts != 0, 0, workspace != 0).kernel;
}

extern "C" int gb_gemm_bf16(const void* a, int lda, const void* w, int ldw, void* c, int ldc, int c_dtype, int M, int N,
                            int K, int epilogue, const void* gamma, int gamma_dtype, float eps, const void* emit_gamma,
                            int emit_gamma_dtype, void* emit_h, int emit_ldh, float* emit_ss, const float* parts, int n_parts,
                            float* split_ws, long long split_ws_floats, hipStream_t stream) {
  GB_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16: bad sizes M=%d N=%d K=%d", M, N, K);
  GB_REQUIRE(K % 8 == 0, "gemm_bf16: the inner size K=%d must be a multiple of 8 (16-byte operand loads)", K);
  GB_REQUIRE(ldw % 8 == 0 && lda % (gamma ? 4 : 8) == 0, "gemm_bf16: row strides (%d, %d) must keep rows 16-byte aligned", lda, ldw);
  GB_REQUIRE(epilogue >= 0 && epilogue <= 2, "gemm_bf16: unknown epilogue %d", epilogue);
  const int ncols = epilogue == EPI_SILU_MUL ? N / 2 : N;
  GB_REQUIRE(epilogue != EPI_SILU_MUL || N % 2 == 0, "gemm_bf16: stacked gate/up rows need an even N, got %d", N);
  GB_REQUIRE(lda >= K && ldw >= K && ldc >= ncols, "gemm_bf16: a leading dimension is shorter than its row");
  GB_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_bf16: operands must be 16-byte aligned");
  GB_REQUIRE(epilogue != EPI_ACCUMULATE || c_dtype == kF32, "gemm_bf16: accumulation is into a float32 result");
  GB_REQUIRE(c_dtype == kF32 || c_dtype == kBF16, "gemm_bf16: unknown result dtype %d", c_dtype);
  GB_REQUIRE(!gamma || (M <= 64 && c_dtype == kBF16 && epilogue != EPI_ACCUMULATE && ((uintptr_t)gamma % 16 == 0) &&
                        (gamma_dtype == kF32 || gamma_dtype == kBF16)),
             "gemm_bf16: the fused RMS norm serves up to 64 rows with a bfloat16 result");
  const int emits = emit_h ? emit_mode(M, N, K) : 0;
  GB_REQUIRE(!emit_h || (epilogue == EPI_ACCUMULATE && emit_gamma && emit_ldh >= N && ((uintptr_t)emit_gamma % 16 == 0) &&
                         (emit_gamma_dtype == kF32 || emit_gamma_dtype == kBF16) &&
                         ((emits == 1 && emit_ss) || (emits == 2 && split_ws && emit_ldh % 4 == 0 && ((uintptr_t)emit_h % 8 == 0)))),
             "gemm_bf16: only an accumulating product that gb_gemm_bf16_emit_mode accepts can prepare the next norm");
  GB_REQUIRE(!parts || (M <= 64 && !gamma && n_parts > 0 && epilogue != EPI_ACCUMULATE),
             "gemm_bf16: partial sums of a norm go with at most 64 rows, no gamma, and a storing epilogue");
  const NormExtras extra{emit_gamma, emit_gamma_dtype == kF32, (bf16*)emit_h, emit_ldh, emit_ss, parts, n_parts};
  if (M == 0) return 0;
  const bf16* W = (const bf16*)w;
  const Route r = route(epilogue, a, lda, w, ldw, M, N, K, gamma != nullptr, parts != nullptr, emits, split_ws != nullptr && (uintptr_t)split_ws % 16 == 0);
  GB_REQUIRE((long long)r.split.floats <= split_ws_floats, "gemm_bf16: the split-k workspace holds %lld floats, %zu are needed",
             split_ws_floats, r.split.floats);
  const bf16* A = (const bf16*)a;
// (the launch, once for each epilogue and type of C that there is)
#define GB_EACH(LAUNCH)                                                              \
  if (epilogue == EPI_ACCUMULATE) return LAUNCH(EPI_ACCUMULATE, float);              \
  if (epilogue == EPI_SILU_MUL && c_dtype == kBF16) return LAUNCH(EPI_SILU_MUL, bf16); \
  if (epilogue == EPI_SILU_MUL) return LAUNCH(EPI_SILU_MUL, float);                  \
  if (c_dtype == kF32) return LAUNCH(EPI_STORE, float);                              \
  return LAUNCH(EPI_STORE, bf16);
#define GB_SP(EPI, CT) launch_split<EPI, CT>(A, lda, W, ldw, (CT*)c, ldc, M, N, K, split_ws, r.split, stream, &extra, eps)
#define GB_HD(EPI, CT) launch_held<EPI, CT>(A, lda, W, ldw, (CT*)c, ldc, M, N, K, 0, 1, eps, parts, n_parts, stream)
#define GB_BK(EPI, CT) launch_block<EPI, CT>(r.block.rm, r.block.cn, A, lda, W, ldw, (CT*)c, ldc, M, N, K, 0, 1, stream)
#define GB_RG(EPI, CT) launch_ring<EPI, CT>(A, lda, W, ldw, (CT*)c, ldc, M, N, K, 0, 1, stream)
#define GB_TL(EPI, CT) launch_tiled<EPI, CT>(A, lda, W, ldw, (CT*)c, ldc, M, N, K, stream)
  switch (r.kernel) {
    case kSlices: GB_EACH(GB_SP)
    case kHeld:
      if (epilogue == EPI_SILU_MUL && c_dtype == kBF16) return GB_HD(EPI_SILU_MUL, bf16);
      if (epilogue == EPI_SILU_MUL) return GB_HD(EPI_SILU_MUL, float);
      if (c_dtype == kF32) return GB_HD(EPI_STORE, float);
      return GB_HD(EPI_STORE, bf16);
    case kBlock: GB_EACH(GB_BK)
    case kRing: GB_EACH(GB_RG)
    case kTiled: GB_EACH(GB_TL)
  }
#undef GB_TL
#undef GB_RG
#undef GB_BK
#undef GB_HD
#undef GB_SP
#undef GB_EACH
  const int gf = gamma_dtype == kF32;
  if (gamma && fold_pays(M, N) && epilogue != EPI_SILU_MUL)
    return launch_fold(a, lda, W, ldw, (bf16*)c, ldc, M, N, K, gamma, gf, eps, stream);
  if (!gamma && M <= 16) {
    if (epilogue == EPI_ACCUMULATE) return launch_few<EPI_ACCUMULATE, float>(A, lda, W, ldw, (float*)c, ldc, M, N, K, eps, extra, stream);
    if (epilogue == EPI_SILU_MUL && c_dtype == kBF16) return launch_few<EPI_SILU_MUL, bf16>(A, lda, W, ldw, (bf16*)c, ldc, M, N, K, eps, extra, stream);
    if (epilogue == EPI_SILU_MUL) return launch_few<EPI_SILU_MUL, float>(A, lda, W, ldw, (float*)c, ldc, M, N, K, eps, extra, stream);
    if (c_dtype == kF32) return launch_few<EPI_STORE, float>(A, lda, W, ldw, (float*)c, ldc, M, N, K, eps, extra, stream);
    return launch_few<EPI_STORE, bf16>(A, lda, W, ldw, (bf16*)c, ldc, M, N, K, eps, extra, stream);
  }
  if (gamma) {
    if (epilogue == EPI_STORE) return launch_skinny<EPI_STORE, true, bf16>(a, lda, W, ldw, (bf16*)c, ldc, M, N, K, gamma, gf, eps, extra, stream);
    return launch_skinny<EPI_SILU_MUL, true, bf16>(a, lda, W, ldw, (bf16*)c, ldc, M, N, K, gamma, gf, eps, extra, stream);
  }
#define GB_SK(EPI, CT) return launch_skinny<EPI, false, CT>(a, lda, W, ldw, (CT*)c, ldc, M, N, K, nullptr, 0, eps, extra, stream)
  if (epilogue == EPI_STORE && c_dtype == kF32) GB_SK(EPI_STORE, float);
  if (epilogue == EPI_STORE && c_dtype == kBF16) GB_SK(EPI_STORE, bf16);
  if (epilogue == EPI_ACCUMULATE) GB_SK(EPI_ACCUMULATE, float);
  if (epilogue == EPI_SILU_MUL && c_dtype == kF32) GB_SK(EPI_SILU_MUL, float);
  GB_SK(EPI_SILU_MUL, bf16);
#undef GB_SK
}

// A product whose epilogue is the clamped gated unit (see Glu): W stacks gate rows over up rows as for epilogue 2, C is
// bfloat16 [M, N / 2].  Up to 16 rows gemm_few_kernel, up to 64 the skinny kernel, beyond them the ring or the tiled kernel.
extern "C" int gb_gemm_bf16_glu(const void* a, int lda, const void* w, int ldw, void* c, int ldc, int M, int N, int K,
                                float limit, float alpha, float plus, hipStream_t stream) {
  GB_REQUIRE(M > 0 && N > 0 && N % 2 == 0 && K > 0 && K % 8 == 0, "gemm_bf16_glu: bad sizes M=%d N=%d K=%d", M, N, K);
  GB_REQUIRE(ldw % 8 == 0 && lda % 8 == 0 && lda >= K && ldw >= K && ldc >= N / 2, "gemm_bf16_glu: row strides (%d, %d, %d)", lda, ldw, ldc);
  GB_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_bf16_glu: operands must be 16-byte aligned");
  GB_REQUIRE(limit > 0.f, "gemm_bf16_glu: the limit must be positive");
  const Glu glu{limit, alpha, plus};
  if (M <= 64) {
    const NormExtras extra{nullptr, 0, nullptr, 0, nullptr, nullptr, 0, glu};
    if (M <= 16) return launch_few<EPI_SILU_MUL, bf16>((const bf16*)a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, 0.f, extra, stream);
    return launch_skinny<EPI_SILU_MUL, false, bf16>(a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, nullptr, 0, 0.f, extra, stream);
  }
  if (ring_pays(EPI_SILU_MUL, a, lda, w, ldw, M, N, K))
    return launch_ring<EPI_SILU_MUL, bf16>((const bf16*)a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, 0, 1, stream, glu);
  return launch_tiled<EPI_SILU_MUL, bf16>((const bf16*)a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, stream, glu);
}

// Products of groups of rows, each group with a W of its own (the tiled kernel's GROUPED form): `map` holds three
// numbers for each of `tiles` row tiles of `tile_rows` (64 or 128) rows, as a kernel on the device laid them out; a
// group's W starts w_stride elements behind the one before.  Epilogue 0 stores (bfloat16 or float32), 2 forms
// silu(gate) * up, or the clamped unit (limit, alpha, plus: see Glu), from the N / 2 gate rows of a group and the up rows
// up_off rows behind them.  Tiles of 256 rows go through the ring kernel, which may divide k into `slices` (float32 results
// without an epilogue): slice z's sums lie z * slice_rows rows further on in C.  in_scale (with epilogue 2, or nullptr): one
// number a row of the product, which the row of A counts times.
extern "C" int gb_gemm_bf16_grouped(const void* a, int lda, const int32_t* rows, const void* w, int ldw, long long w_stride,
                                    int up_off, void* c, int ldc, int c_dtype, const int32_t* map, int tiles, int tile_rows,
                                    int N, int K, int epilogue, float limit, float alpha, float plus, int slices, int slice_rows,
                                    const float* in_scale, hipStream_t stream) {
  GB_REQUIRE(limit > 0.f, "gemm_bf16_grouped: the unit's limit must be positive");
  GB_REQUIRE(tiles >= 0 && N > 0 && K > 0 && (tile_rows == 64 || tile_rows == 128 || tile_rows == 256), "gemm_bf16_grouped: bad sizes tiles=%d of %d rows, N=%d K=%d",
             tiles, tile_rows, N, K);
  GB_REQUIRE(K % 8 == 0 && ldw % 8 == 0 && lda % 8 == 0 && w_stride % 8 == 0 && lda >= K && ldw >= K,
             "gemm_bf16_grouped: the inner size, the row strides and the distance between groups (%d, %d, %d, %lld) must keep rows 16-byte aligned",
             K, lda, ldw, w_stride);
  GB_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0) && map, "gemm_bf16_grouped: operands must be 16-byte aligned");
  GB_REQUIRE(epilogue == EPI_STORE || (epilogue == EPI_SILU_MUL && N % 2 == 0 && c_dtype == kBF16),
             "gemm_bf16_grouped: the epilogue is a store or silu(gate) * up into bfloat16, got %d", epilogue);
  GB_REQUIRE(c_dtype == kF32 || c_dtype == kBF16, "gemm_bf16_grouped: unknown result dtype %d", c_dtype);
  const int cols = epilogue == EPI_SILU_MUL ? N / 2 : N, bn = epilogue == EPI_SILU_MUL ? 64 : 128;
  GB_REQUIRE(ldc >= cols && tiles <= 65535, "gemm_bf16_grouped: rows of C are shorter than the product's, or more than 65535 row tiles");
  if (tiles == 0) return 0;
  GB_REQUIRE(slices >= 1 && (slices == 1 || (tile_rows == 256 && epilogue == EPI_STORE && c_dtype == kF32 && slice_rows > 0)),
             "gemm_bf16_grouped: %d slices of k go with tiles of 256 rows and float32 results", slices);
  const Groups grp{map, rows, w_stride, up_off, slice_rows, in_scale};
  const bf16* A = (const bf16*)a;
  const bf16* W = (const bf16*)w;
  if (tile_rows == 256) {
    GB_REQUIRE(ring_takes(a, lda, w, ldw, K), "gemm_bf16_grouped: tiles of 256 rows need an inner size of whole 32s, %d and more, not %d", RING_MIN_K, K);
    const int k_slice = slices == 1 ? 0 : (K / RING_K + slices - 1) / slices * RING_K;
    GB_REQUIRE(slices == 1 || (slices - 1) * (long long)k_slice < K, "gemm_bf16_grouped: %d slices of k=%d leave some without a step", slices, K);
    const int rbn = epilogue == EPI_SILU_MUL ? RBN / 2 : RBN;
    const dim3 rgrid((cols + rbn - 1) / rbn, tiles, slices), rblock(RGM * RGN * 64);
    if (epilogue == EPI_SILU_MUL)
      hipLaunchKernelGGL((gemm_ring_kernel<EPI_SILU_MUL, bf16, true>), rgrid, rblock, 0, stream, A, lda, W, ldw, (bf16*)c, ldc, 0, N, K, 0, 0, grp, Glu{limit, alpha, plus});
    else if (c_dtype == kF32)
      hipLaunchKernelGGL((gemm_ring_kernel<EPI_STORE, float, true>), rgrid, rblock, 0, stream, A, lda, W, ldw, (float*)c, ldc, 0, N, K, k_slice, 0, grp, Glu{});
    else
      hipLaunchKernelGGL((gemm_ring_kernel<EPI_STORE, bf16, true>), rgrid, rblock, 0, stream, A, lda, W, ldw, (bf16*)c, ldc, 0, N, K, 0, 0, grp, Glu{});
    return launched("gemm_bf16 (grouped ring)");
  }
  const dim3 grid((cols + bn - 1) / bn, tiles), block(256);
  const bool kfull = K % TBK == 0;
#define GB_G(WM, EPI, CT, FULL)                                                                                              \
  if (tile_rows == 64 * WM && epilogue == EPI && kfull == FULL && (EPI == EPI_SILU_MUL || (c_dtype == kF32) == std::is_same_v<CT, float>)) \
    hipLaunchKernelGGL((gemm_tiled_kernel<WM, 2, 1, EPI, FULL, CT, true>), grid, block, 0, stream, A, lda, W, ldw, (CT*)c, ldc, 0, N, K, 0, grp, Glu{limit, alpha, plus});
#define GB_GG(WM, FULL) GB_G(WM, EPI_SILU_MUL, bf16, FULL) GB_G(WM, EPI_STORE, float, FULL) GB_G(WM, EPI_STORE, bf16, FULL)
  GB_GG(1, true) GB_GG(1, false) GB_GG(2, true) GB_GG(2, false)
#undef GB_GG
#undef GB_G
  return launched("gemm_bf16 (grouped)");
}

// The QKV product of a step of at most 64 rows with EPI_ROPE (see RopeExtras): c is the stacked rows
// [M][(nh + 2 nkv) hd] (or [M][nh hd] with nkv == 0: queries only), bfloat16.  gamma / parts as in
// gb_gemm_bf16 (the norm before the product).
extern "C" int gb_gemm_bf16_rope(const void* a, int lda, const void* w, int ldw, void* c, int ldc, int M, int N, int K,
                                 const void* gamma, int gamma_dtype, float eps, const float* parts, int n_parts,
                                 const float* cosv, const float* sinv, const int32_t* slots, void* k_pages, void* v_pages,
                                 int nh, int nkv, int hd, int page_size, hipStream_t stream) {
  GB_REQUIRE(M > 0 && M <= 64 && N > 0 && K > 0 && K % 8 == 0, "gemm_bf16_rope: bad sizes M=%d N=%d K=%d (at most 64 rows)", M, N, K);
  GB_REQUIRE(hd >= 16 && hd % 16 == 0 && nh > 0 && nkv >= 0 && N == (nh + 2 * nkv) * hd,
             "gemm_bf16_rope: N=%d is not (nh + 2 nkv) hd with nh=%d nkv=%d hd=%d (a multiple of 16)", N, nh, nkv, hd);
  GB_REQUIRE(ldw % 8 == 0 && lda % (gamma ? 4 : 8) == 0 && lda >= K && ldw >= K && ldc >= N && ((uintptr_t)a % 16 == 0) &&
                 ((uintptr_t)w % 16 == 0),
             "gemm_bf16_rope: operands must be 16-byte aligned rows");
  GB_REQUIRE((cosv == nullptr) == (sinv == nullptr), "gemm_bf16_rope: cos and sin come together");
  GB_REQUIRE(!slots || (k_pages && v_pages && page_size > 0 && nkv > 0), "gemm_bf16_rope: slots given without pages");
  GB_REQUIRE(!gamma || (((uintptr_t)gamma % 16 == 0) && (gamma_dtype == kF32 || gamma_dtype == kBF16) && !parts),
             "gemm_bf16_rope: gamma must be aligned float32 or bfloat16, and not given together with parts");
  GB_REQUIRE(!parts || n_parts > 0, "gemm_bf16_rope: partial sums of a norm without a count");
  const NormExtras extra{nullptr, 0, nullptr, 0, nullptr, parts, n_parts};
  const RopeExtras rope{cosv, sinv, slots, (bf16*)k_pages, (bf16*)v_pages, nh, nkv, hd, page_size, 0, 0.f, -1};
  if (!gamma && held_pays(EPI_ROPE, M, N, K, parts != nullptr) && held_takes(a, lda, w, ldw, M, K))
    return launch_held<EPI_ROPE, bf16>((const bf16*)a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, 0, 1, eps, parts, n_parts, stream, rope);
  if (gamma)
    return launch_skinny<EPI_ROPE, true, bf16>(a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, gamma, gamma_dtype == kF32,
                                               eps, extra, stream, rope);
  if (M <= 16) return launch_few<EPI_ROPE, bf16>((const bf16*)a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, eps, extra, stream, rope);
  return launch_skinny<EPI_ROPE, false, bf16>(a, lda, (const bf16*)w, ldw, (bf16*)c, ldc, M, N, K, nullptr, 0, eps, extra,
                                              stream, rope);
}

// the launches of a layer can be recorded and made again for the layers like it (common.h)
GB_TAPED(gb_gemm_bf16)
GB_TAPED(gb_gemm_bf16_partial)
GB_TAPED(gb_gemm_bf16_grouped)
GB_TAPED(gb_gemm_bf16_glu)
GB_TAPED(gb_gemm_bf16_rope)
