// Tall-skinny QR (BVOrthogonalize with block method TSQR / TSQRCHOL) for
// gfx950 (MI355X).  Reference: bvorthog.c:615-659 and bvlapack.c:347-480,
// 510-560 (geqrf + orgqr on each process, a binary tree of QR factorizations
// of stacked R factors across processes).
//
// On one GPU the tree runs over tiles of rows instead of processes: a tile is
// factored by one workgroup, its rows in registers (4 waves of 2 or 4 rows per
// lane up to 32 columns, 8 waves of one row per lane up to 64: 512 or 1024 rows):
//   level 0: every tile's Householder QR of its rows
//            of V(:, l:k) (held in registers) is computed; the kernel writes the
//            Householder vectors over the tile and its k x k R into the
//            stacked matrix of level 1;
//   level i: the same kernel on the stacked R factors, until one tile is left,
//            whose R is the R of the whole block.
// Q is then formed top-down: each tile applies its reflectors to the k x k
// block of the level above that belongs to it (padded with zero rows), in
// place; the top tile forms its explicit factor (the orgqr of the tile).
//
// The R of a tree differs from the R of one flat Householder QR (what geqrf
// computes on one process) only in the signs of its rows.  Those signs follow
// from the first k rows of Q: Householder QR of A and of Q D (D the signs of
// diag(R), so that R D has a positive diagonal) use the same reflectors, and
// the sign LAPACK picks for column j is minus the sign of the pivot of an LU
// factorization of those k rows that subtracts each chosen sign from its
// pivot (Ballard, Demmel, Grigori, Jacquelin, Nguyen, Solomonik, "Reconstructing
// Householder vectors from tall-skinny QR", IPDPS 2014).  The host computes
// these k signs from a one-tile run of the level-0 kernel and the full level-0
// pass applies them as it stores Q, so Q and R equal geqrf/orgqr's up to
// rounding at no extra pass over V.
//
// The vector ALU bounds the tiles: a step of 32 columns is about 190 FP64
// operations and 330 others per wave (the wave reduction by lane swaps, the
// sums broadcast through scalar registers).  Two choices keep it there: one
// reduction per Householder step (it gives the norm of the column and its
// products with the others together), and a register window that moves one
// column to the left with each update, so no step selects registers by the
// column number.  Four waves per tile make the tree three levels shallower than
// one wave (128 rows) for one LDS exchange per step; with 1, 4, 8 waves 32
// columns of 2.1M rows take 1.94, 1.47, 1.67 ms.  Measured against one wave per
// tile with two shuffle reductions per step (up to 32 columns) and one thread per
// row (beyond), 2.1M rows FP64: 8 columns 314 -> 238 us, 16: 721 -> 523, 24: 2.04 ->
// 0.95 ms, 32: 2.75 -> 1.47, 48: 13.0 -> 4.9, 64: 16.9 -> 7.2 (floor of 32 columns at
// the copy rate: 0.45 ms, V read and written twice).  Forming Q by matrix products
// (tsqr_form_kernel) then took 32 columns to 1.30 ms.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <vector>

#include "sa_device.h"
#include "sa_internal.h"

namespace sa {

constexpr int TS_MAXK = 64;    // most columns per call

// A tile is W waves of 64 RPL rows: wave w, lane l, r hold row 64 (w RPL + r) + l
// of it, K columns each in registers.  Rows 0..K-1, whose entries become R,
// are the first row slot of wave 0.
template <typename T, int K, int W>
struct TsShared {
  T part[2][W][K];        // per-wave partial products (two buffers: steps alternate)
  T row[2][K];            // row j of the window
};

// A value that is uniform across the wave, read from lane l (l uniform).
template <typename T>
__device__ __forceinline__ T ts_readlane(T v, int l) {
  if constexpr (sizeof(T) == 8) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
  }
}

__host__ __device__ constexpr int ts_pow2(int k) { return k <= 8 ? 8 : (k <= 16 ? 16 : (k <= 32 ? 32 : 64)); }

// The LDS exchange of a step between the waves of a tile; the global loads and
// stores stay in flight.
__device__ __forceinline__ void ts_exchange() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Orders a wave's LDS stores before the loads of its other lanes that follow,
// and its loads before stores that follow.  The hardware keeps a wave's LDS
// operations in order; without this the compiler need not, as no lane reads
// what it wrote itself.
__device__ __forceinline__ void ts_wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The wave's sums of u x[.][c] over its rows for the columns c < KS: lane l
// returns the one of column l / (64 / SP), SP = ts_pow2(KS).  The first step of
// the reduce-scatter takes the products as they are formed.
template <typename T, int K, int RPL, int KS>
__device__ __forceinline__ T ts_wave_dots(const T (&x)[RPL][K], const T (&u)[RPL], int lane) {
  constexpr int SP = ts_pow2(KS), H = SP / 2;
  auto dot = [&](int c) {
    T d = u[0] * x[0][c];
#pragma unroll
    for (int r = 1; r < RPL; r++) d += u[r] * x[r][c];
    return d;
  };
  T p[H];
#pragma unroll
  for (int i = 0; i < H; i++)
    p[i] = scatter_add<32>(i < KS ? dot(i < KS ? i : 0) : (T)0, i + H < KS ? dot(i + H < KS ? i + H : 0) : (T)0, lane);
  return wave_scatter<H, 16>(p, lane);
}

// The tile's sums in the same layout, on every wave (waves added in order).
template <typename T, int K, int W, int SP>
__device__ __forceinline__ T ts_tile_sum(int lane, int par, const TsShared<T, K, W> &sh) {
  constexpr int LPC = 64 / SP;
  const int c = min(lane / LPC, K - 1);
  T s = sh.part[par][0][c];
#pragma unroll
  for (int q = 1; q < W; q++) s += sh.part[par][q][c];
  return s;
}

// Householder steps j0 <= j < j1 (dgeqr2 / dlarfg order).  The window x[.][0..KS)
// starts at column j: each step stores its finished column and the update
// writes the others one place to the left, so that every register index is
// fixed.  One reduction per step: with u the column below row j, the products
// u^T x_c give sigma = u^T u and, for v = (1, u / (alpha - beta)), v^T x_c = x_c(j) +
// u^T x_c / (alpha - beta).
template <typename T, int K, int RPL, int W, int KS>
__device__ __forceinline__ void ts_factor_phase(T (&x)[RPL][K], int j0, int j1, int k, int lane, int wv, int nb,
                                                T *ytile, int64_t ldy, T *tau_b, T *R_b, int64_t ldr,
                                                TsShared<T, K, W> &sh) {
  constexpr int SP = ts_pow2(KS), LPC = 64 / SP;
  // one copy of the step body: an unrolled step loop outgrows the instruction cache
#pragma nounroll
  for (int j = j0; j < j1; j++) {
    const int par = j & 1;
    T u[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) u[r] = 64 * (wv * RPL + r) + lane > j ? x[r][0] : (T)0;
    if (wv == 0 && lane == j) {
#pragma unroll
      for (int c = 0; c < KS; c++) sh.row[par][c] = x[0][c];
    }
    T d = ts_wave_dots<T, K, RPL, KS>(x, u, lane);
    const int cl = lane / LPC;
    if (lane % LPC == 0 && cl < KS) sh.part[par][wv][cl] = d;
    ts_exchange();
    d = ts_tile_sum<T, K, W, SP>(lane, par, sh);
    const T xc = sh.row[par][min(cl, KS - 1)];
    const T sigma = ts_readlane(d, 0), alpha = ts_readlane(xc, 0);
    T tau = 0, beta = alpha, scal = 0;
    if (sigma != (T)0) {               // else H = I, as dlarfg does for a zero column
      const T nrm = sqrt(alpha * alpha + sigma);
      beta = alpha >= (T)0 ? -nrm : nrm;
      tau = (beta - alpha) / beta;
      scal = (T)1 / (alpha - beta);
    }
    const T w = tau * (xc + scal * d);
    T v[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) {
      const int row = 64 * (wv * RPL + r) + lane;
      const T q = u[r] * scal;         // u / (alpha - beta): the product, corrected once
      v[r] = row > j ? q + (u[r] - q * (alpha - beta)) * scal : (row == j ? (T)1 : (T)0);
      const T nj = row > j ? v[r] : (row == j ? beta : x[r][0]);
      if (ytile && row < nb) ytile[row + (int64_t)j * ldy] = nj;
      if (r == 0 && wv == 0 && lane < k) R_b[lane + (int64_t)j * ldr] = lane <= j ? nj : (T)0;
    }
    if (wv == 0 && lane == 0) tau_b[j] = tau;
#pragma unroll
    for (int c = 1; c < KS; c++) {
      const T wc = ts_readlane(w, c * LPC);
#pragma unroll
      for (int r = 0; r < RPL; r++) x[r][c - 1] = x[r][c] - v[r] * wc;
    }
  }
}

// Eight steps with a window of KS columns, then the next eight with KS - 8.
template <typename T, int K, int RPL, int W, int KS>
__device__ __forceinline__ void ts_factor_all(T (&x)[RPL][K], int k, int lane, int wv, int nb, T *ytile, int64_t ldy,
                                              T *tau_b, T *R_b, int64_t ldr, TsShared<T, K, W> &sh) {
  constexpr int J = K - KS;
  ts_factor_phase<T, K, RPL, W, KS>(x, J, min(k, J + 8), k, lane, wv, nb, ytile, ldy, tau_b, R_b, ldr, sh);
  if constexpr (KS > 8) ts_factor_all<T, K, RPL, W, KS - 8>(x, k, lane, wv, nb, ytile, ldy, tau_b, R_b, ldr, sh);
}

// One tree level: tile b covers rows [TR b, TR b + nb), TR = 64 RPL W, of the
// rows x k matrix A (column-major, lda).  Y (may equal A; nullptr: not kept)
// receives the Householder vectors and R in geqrf layout, tau[b k + j] the
// scalars and rows b k .. b k + k - 1 of R (ldr) the tile's k x k R (rows at
// or beyond nb zero).
template <typename T, int K, int RPL, int W>
__global__ __launch_bounds__(64 * W) void tsqr_factor_kernel(const T *A, int64_t lda, int64_t rows, int k,
                                                                          T *Y, int64_t ldy, T *__restrict__ tau,
                                                                          T *__restrict__ R, int64_t ldr) {
  constexpr int TR = 64 * RPL * W;
  __shared__ TsShared<T, K, W> sh;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * TR;
  const int nb = (int)min((int64_t)TR, rows - r0);
  T x[RPL][K];
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int row = 64 * (wv * RPL + r) + lane;
#pragma unroll
    for (int c = 0; c < K; c++) x[r][c] = (c < k && row < nb) ? A[r0 + row + (int64_t)c * lda] : (T)0;
  }
  ts_factor_all<T, K, RPL, W, K>(x, k, lane, wv, nb, Y ? Y + r0 : nullptr, ldy, tau + b * k, R + b * k, ldr,
                                 sh);
}

// Q of one tree level, reflector by reflector (up to 8 columns; what it computes
// is said at tsqr_form_kernel).  Each lane reads only its own rows of Y, those of
// step j - 1 one step ahead, so out may equal Y.
template <typename T, int K, int RPL, int W>
__global__ __launch_bounds__(64 * W) void tsqr_form_steps_kernel(const T *Y, int64_t ldy, int64_t rows, int k,
                                                                 const T *__restrict__ tau, const T *__restrict__ C,
                                                                 int64_t ldc, T *out, int64_t ldo,
                                                                 const T *__restrict__ sgn) {
  constexpr int TR = 64 * RPL * W, SP = ts_pow2(K), LPC = 64 / SP;
  __shared__ TsShared<T, K, W> sh;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * TR;
  const int nb = (int)min((int64_t)TR, rows - r0);
  const int kk = min(k, nb);                    // rows of C_b beyond the tile's rows meet zero rows of its R
  const T *ytile = Y + r0, *tau_b = tau + b * k;
  T q[RPL][K];
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int row = 64 * (wv * RPL + r) + lane;
#pragma unroll
    for (int c = 0; c < K; c++) {
      if (C) q[r][c] = (row < kk && c < k) ? C[b * k + row + (int64_t)c * ldc] : (T)0;
      else q[r][c] = row == c ? (T)1 : (T)0;
    }
  }
  T yn[RPL];
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int row = 64 * (wv * RPL + r) + lane;
    yn[r] = row < nb ? ytile[row + (int64_t)(kk - 1) * ldy] : (T)0;
  }
#pragma nounroll
  for (int j = kk - 1; j >= 0; j--) {
    const int par = j & 1;
    T v[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) {
      const int row = 64 * (wv * RPL + r) + lane;
      v[r] = row > j ? yn[r] : (row == j ? (T)1 : (T)0);
    }
    if (j > 0) {
#pragma unroll
      for (int r = 0; r < RPL; r++) {
        const int row = 64 * (wv * RPL + r) + lane;
        yn[r] = row < nb ? ytile[row + (int64_t)(j - 1) * ldy] : (T)0;
      }
    }
    const T tj = tau_b[j];
    T d = ts_wave_dots<T, K, RPL, K>(q, v, lane);
    if (lane % LPC == 0 && lane / LPC < K) sh.part[par][wv][lane / LPC] = d;
    ts_exchange();
    d = ts_tile_sum<T, K, W, SP>(lane, par, sh);
    const T w = tj * d;
#pragma unroll
    for (int c = 0; c < K; c++) {
      const T wc = ts_readlane(w, c * LPC);
#pragma unroll
      for (int r = 0; r < RPL; r++) q[r][c] -= v[r] * wc;
    }
  }
#pragma unroll
  for (int r = 0; r < RPL; r++) {
    const int row = 64 * (wv * RPL + r) + lane;
    if (row < nb) {
#pragma unroll
      for (int c = 0; c < K; c++)
        if (c < k) out[r0 + row + (int64_t)c * ldo] = sgn ? q[r][c] * sgn[c] : q[r][c];
    }
  }
}

// Shared memory of tsqr_form_kernel: the tile's Gram matrix beside what its
// phases use in turn.
template <typename T, int K, int W>
struct TsForm {
  static constexpr int NB = (K + 15) / 16, KP = 16 * NB, LD = KP + 1, NBLK = NB * (NB + 1) / 2;
  T G[KP * LD];                        // (Y^T Y)(j, i) at G[j LD + i], j < i
  T tau[KP];
  union {
    T tr[W][KP * 17];                  // 16 rows of a wave, transposed
    T sum[(W + 1) / 2][NBLK * 256];    // Gram blocks on their way to wave 0
    struct {
      T X[KP * LD], Y1[KP * LD], C[KP * LD];   // row by row
    } s;
  };
};

// Q of one tree level: tile b applies its reflectors (rows x k Y in geqrf
// layout, scalars tau[b k ..]) in descending order to [C_b; 0], C_b = rows b k
// .. b k + k - 1 of the Q of the level above (ldc), which gives its rows of Q;
// with C == nullptr (the top tile) to [I; 0], the explicit Householder factor
// (dorg2r).  The result, times sgn[c] per column when sgn is given, goes to
// out (may equal Y: a workgroup reads its whole tile before it writes).
//
// The reflectors are applied together (compact WY form; Schreiber and Van Loan,
// SIAM J. Sci. Stat. Comput. 10, 1989): Q = [C; 0] - Y X, where row j of X is
// what reflector j would subtract, x_j = tau_j (y_j^T [C; 0] - sum_{i > j}
// (y_j^T y_i) x_i).  The tile's rows are read once into registers, lane l holding
// row l % 16 and column l / 16 of each 16 x 4 block; Y^T Y (through a transpose
// in LDS) and Y X are matrix products on the MFMA units and what is left, k x k
// per tile, is a triangular solve.  Memory bounds it (the level over V of 2.1M
// rows and 32 columns FP64 takes 386 us, 226 at the copy rate), then the solve,
// which only the two tiles a CU holds overlap (64 columns FP64 spill 104 bytes per
// lane beside that).  Against applying the
// reflectors one by one, each a reduction and an update of all columns (the
// whole factorization, 2.1M rows FP64): 16 columns 523 -> 481 us, 24 950 -> 874,
// 32 1471 -> 1301, 48 4.9 -> 3.4 ms, 64 7.2 -> 5.0; 8 columns, which the matrix units
// pad to 16, 238 -> 260, so they keep the steps.  Eight waves per tile have the
// shorter phases; with 32 columns FP64 they lose to four (1375 us).
template <typename T, int K, int RPL, int W>
__global__ __launch_bounds__(64 * W) void tsqr_form_kernel(const T *Y, int64_t ldy, int64_t rows, int k,
                                                           const T *__restrict__ tau, const T *__restrict__ C,
                                                           int64_t ldc, T *out, int64_t ldo,
                                                           const T *__restrict__ sgn) {
  using F = TsForm<T, K, W>;
  using V4 = typename Vec4<T>::type;
  constexpr int TR = 64 * RPL * W, NB = F::NB, KP = F::KP, LD = F::LD, NBLK = F::NBLK;
  constexpr int RB = 4 * RPL, NU = (K + 3) / 4, NT = 64 * W;   // 16-row blocks per wave, 4-column steps
  extern __shared__ __align__(16) unsigned char ts_raw[];
  F &sh = *reinterpret_cast<F *>(ts_raw);
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * TR;
  const int nb = (int)min((int64_t)TR, rows - r0);
  const int kk = min(k, nb);                    // rows of C_b beyond the tile's rows meet zero rows of its R
  T y[RB][NU];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
    const int row = 16 * (wv * RB + rb) + c16;
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int c = 4 * u + g;
      y[rb][u] = (c < kk && row < nb) ? Y[r0 + row + (int64_t)c * ldy] : (T)0;
    }
  }
  constexpr int NC = (KP * KP + NT - 1) / NT;
  T cv[NC];                                     // C_b, on its way to LDS
#pragma unroll
  for (int i = 0; i < NC; i++) {
    const int r = (t + i * NT) % KP, c = (t + i * NT) / KP;
    if (C) cv[i] = (r < kk && c < k) ? C[b * k + r + (int64_t)c * ldc] : (T)0;
    else cv[i] = (r == c && r < kk) ? (T)1 : (T)0;
  }
  for (int i = t; i < KP; i += NT) sh.tau[i] = i < kk ? tau[b * k + i] : (T)0;
  if (wv == 0) {                                // unit lower trapezoidal: R is above
#pragma unroll
    for (int rb = 0; rb < NB; rb++)
#pragma unroll
      for (int u = 0; u < NU; u++) {
        const int row = 16 * rb + c16, c = 4 * u + g;
        y[rb][u] = row > c ? y[rb][u] : ((row == c && c < kk) ? (T)1 : (T)0);
      }
  }
  // ---- G = Y^T Y, the blocks on and above the diagonal -----------------------
  V4 acc[NBLK];
#pragma unroll
  for (int q = 0; q < NBLK; q++) acc[q] = (V4){0, 0, 0, 0};
  T *tr = sh.tr[wv];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
#pragma unroll
    for (int u = 0; u < NU; u++) tr[(4 * u + g) * 17 + c16] = y[rb][u];
    ts_wave_order();
#pragma unroll
    for (int h = 0; h < 4; h++) {
      T a[NB];
#pragma unroll
      for (int q = 0; q < NB; q++) a[q] = 16 * q + c16 < 4 * NU ? tr[(16 * q + c16) * 17 + 4 * h + g] : (T)0;
      int at = 0;
#pragma unroll
      for (int q = 0; q < NB; q++)
#pragma unroll
        for (int p = q; p < NB; p++, at++) acc[at] = mfma16x16x4(a[q], a[p], acc[at]);
    }
    ts_wave_order();                            // the next 16 rows overwrite these
  }
  // waves in pairs, the same order every time
#pragma unroll
  for (int half = W / 2; half >= 1; half /= 2) {
    __syncthreads();
    if (wv >= half && wv < 2 * half) {
#pragma unroll
      for (int q = 0; q < NBLK; q++)
#pragma unroll
        for (int v = 0; v < 4; v++) sh.sum[wv - half][q * 256 + v * 64 + lane] = acc[q][v];
    }
    __syncthreads();
    if (wv < half) {
#pragma unroll
      for (int q = 0; q < NBLK; q++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[q][v] += sh.sum[wv][q * 256 + v * 64 + lane];
    }
  }
  __syncthreads();
  if (wv == 0) {
    int at = 0;
#pragma unroll
    for (int q = 0; q < NB; q++)
#pragma unroll
      for (int p = q; p < NB; p++, at++)
#pragma unroll
        for (int v = 0; v < 4; v++) sh.G[(16 * q + mfma_row<T>(g, v)) * LD + 16 * p + c16] = acc[at][v];
#pragma unroll
    for (int rb = 0; rb < NB; rb++)
#pragma unroll
      for (int u = 0; u < NU; u++) sh.s.Y1[(16 * rb + c16) * LD + 4 * u + g] = y[rb][u];
  }
#pragma unroll
  for (int i = 0; i < NC; i++) {
    const int r = (t + i * NT) % KP, c = (t + i * NT) / KP;
    if (c < KP) sh.s.C[r * LD + c] = cv[i];
  }
  __syncthreads();
  // ---- X, 16 rows at a time from the last -------------------------------------
#pragma unroll
  for (int q = NB - 1; q >= 0; q--) {
    for (int e = t; e < 16 * KP; e += NT) {
      const int j = 16 * q + e / KP, c = e % KP;
      T s = (T)0;
      if (j < 4 * NU) {
#pragma unroll 8
        for (int r = 16 * q; r < KP; r++) s += sh.s.Y1[r * LD + j] * sh.s.C[r * LD + c];
#pragma unroll 8
        for (int i = 16 * (q + 1); i < KP; i++) s -= sh.G[j * LD + i] * sh.s.X[i * LD + c];
      }
      sh.s.X[j * LD + c] = s;
    }
    __syncthreads();
    if (t < KP) {
      T x[16];
#pragma unroll
      for (int j = 15; j >= 0; j--) {
        T s = sh.s.X[(16 * q + j) * LD + t];
#pragma unroll
        for (int i = 15; i > j; i--) s -= sh.G[(16 * q + j) * LD + 16 * q + i] * x[i];
        x[j] = sh.tau[16 * q + j] * s;
        sh.s.X[(16 * q + j) * LD + t] = x[j];
      }
    }
    __syncthreads();
  }
  // ---- Q = [C; 0] - Y X ---------------------------------------------------------
#pragma unroll
  for (int q = 0; q < NB; q++) {
    T xa[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) xa[u] = sh.s.X[(4 * u + g) * LD + 16 * q + c16];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      V4 d = (V4){0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < NU; u++) d = mfma16x16x4(xa[u], y[rb][u], d);
      const int row = 16 * (wv * RB + rb) + c16;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int c = 16 * q + mfma_row<T>(g, v);
        if (row < nb && c < k) {
          T o = row < KP ? sh.s.C[row * LD + c] - d[v] : -d[v];
          out[r0 + row + (int64_t)c * ldo] = sgn ? o * sgn[c] : o;
        }
      }
    }
  }
}

// ---- host side ----------------------------------------------------------------

void tsqr_signs(const double *Qtop, const double *R, int64_t n, int k, double *f) {
  std::vector<double> U(Qtop, Qtop + (size_t)k * k), D(k);
  for (int j = 0; j < k; j++) {
    D[j] = R[j + (size_t)j * k] < 0.0 ? -1.0 : 1.0;
    for (int i = 0; i < k; i++) U[i + (size_t)j * k] *= D[j];
  }
  for (int j = 0; j < k; j++) {
    const double piv = U[j + (size_t)j * k];
    // dlarfg: beta = -sign(alpha) ||x||; a column with no rows below the
    // diagonal (the last of a square block) is left as it is (tau = 0)
    const double sj = (j == n - 1) ? (piv < 0.0 ? -1.0 : 1.0) : (piv < 0.0 ? 1.0 : -1.0);
    f[j] = D[j] * sj;
    const double d = piv - sj;
    U[j + (size_t)j * k] = d;
    for (int i = j + 1; i < k; i++) U[i + (size_t)j * k] /= d;
    for (int c = j + 1; c < k; c++)
      for (int i = j + 1; i < k; i++) U[i + (size_t)c * k] -= U[i + (size_t)j * k] * U[j + (size_t)c * k];
  }
}

namespace {

// Tree workspace, one per host thread (each has its own stream): kept between
// calls, grown when a call needs more, released with the process.
struct TsWork {
  void *buf = nullptr;
  size_t bytes = 0;
};

template <typename T>
struct TsLevel {
  T *M;
  int64_t ld, rows;
  int G;
  T *tau;
};

template <typename T, int K>
int tsqr_t(BV &V, int l, int k, bool formq, double *R_host, double *f, hipStream_t s) {
  constexpr int RPL = K <= 16 ? 4 : (K <= 32 ? 2 : 1), WV = K <= 32 ? 4 : 8, TR = 64 * RPL * WV;
  constexpr int WF = K == 32 && sizeof(T) == 8 ? 4 : 8;   // waves of a tile whose Q is formed
  auto factor = [&](const T *A, int64_t lda, int64_t rows, int G, T *Y, int64_t ldy, T *tau, T *R, int64_t ldr) {
    tsqr_factor_kernel<T, K, RPL, WV><<<G, 64 * WV, 0, s>>>(A, lda, rows, k - l, Y, ldy, tau, R, ldr);
  };
  auto form = [&](const T *Y, int64_t ldy, int64_t rows, int G, const T *tau, const T *C, int64_t ldc, T *out,
                  int64_t ldo, const T *sg) {
    if constexpr (K <= 8)
      tsqr_form_steps_kernel<T, K, RPL, WV><<<G, 64 * WV, 0, s>>>(Y, ldy, rows, k - l, tau, C, ldc, out, ldo, sg);
    else
      tsqr_form_kernel<T, K, TR / (64 * WF), WF><<<G, 64 * WF, sizeof(TsForm<T, K, WF>), s>>>(Y, ldy, rows, k - l, tau,
                                                                                           C, ldc, out, ldo, sg);
  };
  if constexpr (K > 8) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
      err = hipFuncSetAttribute((const void *)tsqr_form_kernel<T, K, TR / (64 * WF), WF>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(TsForm<T, K, WF>));
    });
    SA_HIP(err);
  }
  const int nk = k - l;
  const int64_t n = V.n;
  // level sizes: rows_{i+1} = tiles_i * nk until one tile is left
  std::vector<TsLevel<T>> L;
  size_t need = 0;
  auto al = [](size_t e) { return (e + 63) / 64 * 64; };
  for (int64_t rows = n;;) {
    const int64_t G = (rows + TR - 1) / TR;
    SA_CHECK(G <= (int64_t)1 << 30, "TSQR: too many tiles");
    L.push_back({nullptr, 0, rows, (int)G, nullptr});
    need += al((size_t)G * nk);                             // tau
    if (G == 1) break;
    rows = G * nk;
    need += al((size_t)rows * nk);                          // next level's matrix
  }
  need += al((size_t)nk * nk) + al((size_t)TR * nk) + al(nk);   // R, probe tile, signs
  thread_local TsWork W;
  if (W.bytes < need * sizeof(T)) {
    if (W.buf) (void)hipFree(W.buf);
    W.buf = nullptr;
    W.bytes = 0;
    SA_HIP(hipMalloc(&W.buf, need * sizeof(T)));
    W.bytes = need * sizeof(T);
  }
  T *p = (T *)W.buf;
  L[0].M = (T *)V.data + (int64_t)l * V.ld;
  L[0].ld = V.ld;
  for (size_t i = 0; i < L.size(); i++) {
    L[i].tau = p;
    p += al((size_t)L[i].G * nk);
    if (i + 1 < L.size()) {
      L[i + 1].M = p;
      L[i + 1].ld = L[i + 1].rows;
      p += al((size_t)L[i + 1].rows * nk);
    }
  }
  T *Rtop = p;
  p += al((size_t)nk * nk);
  T *probe = p;
  p += al((size_t)TR * nk);
  T *sgn = p;
  const int top = (int)L.size() - 1;
  for (int i = 0; i <= top; i++) {
    T *Rout = i == top ? Rtop : L[i + 1].M;
    const int64_t ldr = i == top ? nk : L[i + 1].ld;
    factor(L[i].M, L[i].ld, L[i].rows, L[i].G, formq ? L[i].M : nullptr, L[i].ld, L[i].tau, Rout, ldr);
  }
  SA_HIP(hipGetLastError());
  std::vector<T> buf((size_t)nk * nk);
  SA_HIP(hipMemcpyAsync(buf.data(), Rtop, sizeof(T) * buf.size(), hipMemcpyDeviceToHost, s));
  SA_HIP(hipStreamSynchronize(s));
  for (size_t e = 0; e < buf.size(); e++) R_host[e] = (double)buf[e];
  if (!formq) return 0;
  for (int i = top; i >= 1; i--)
    form(L[i].M, L[i].ld, L[i].rows, L[i].G, L[i].tau, i == top ? nullptr : L[i + 1].M, i == top ? 0 : L[i + 1].ld,
         L[i].M, L[i].ld, nullptr);
  const T *C0 = top == 0 ? nullptr : L[1].M;
  const int64_t ldc0 = top == 0 ? 0 : L[1].ld;
  // the first nk rows of Q (tile 0 holds them: n >= nk) for the signs
  form(L[0].M, L[0].ld, L[0].rows, 1, L[0].tau, C0, ldc0, probe, TR, nullptr);
  SA_HIP(hipGetLastError());
  SA_HIP(hipMemcpy2DAsync(buf.data(), sizeof(T) * nk, probe, sizeof(T) * TR, sizeof(T) * nk, nk,
                          hipMemcpyDeviceToHost, s));
  SA_HIP(hipStreamSynchronize(s));
  std::vector<double> Qtop(buf.begin(), buf.end());
  tsqr_signs(Qtop.data(), R_host, n, nk, f);
  for (int j = 0; j < nk; j++) buf[j] = (T)f[j];
  SA_HIP(hipMemcpyAsync(sgn, buf.data(), sizeof(T) * nk, hipMemcpyHostToDevice, s));
  form(L[0].M, L[0].ld, L[0].rows, L[0].G, L[0].tau, C0, ldc0, L[0].M, L[0].ld, sgn);
  SA_HIP(hipGetLastError());
  SA_HIP(hipStreamSynchronize(s));
  return 0;
}

template <typename T>
int tsqr_k(BV &V, int l, int k, bool formq, double *R_host, double *f, hipStream_t s) {
  const int nk = k - l;
  if (nk <= 8) return tsqr_t<T, 8>(V, l, k, formq, R_host, f, s);
  if (nk <= 16) return tsqr_t<T, 16>(V, l, k, formq, R_host, f, s);
  if (nk <= 24) return tsqr_t<T, 24>(V, l, k, formq, R_host, f, s);
  if (nk <= 32) return tsqr_t<T, 32>(V, l, k, formq, R_host, f, s);
  if (nk <= 48) return tsqr_t<T, 48>(V, l, k, formq, R_host, f, s);
  return tsqr_t<T, 64>(V, l, k, formq, R_host, f, s);
}

}  // namespace

int launch_tsqr(BV &V, int l, int k, bool formq, double *R_host, double *f, hipStream_t s) {
  const int nk = k - l;
  SA_CHECK(nk >= 1 && nk <= TS_MAXK, "TSQR: at most 64 active columns per call");
  SA_CHECK(V.n >= nk, "TSQR: fewer rows than active columns");
  return V.prec == SA_FP64 ? tsqr_k<double>(V, l, k, formq, R_host, f, s)
                           : tsqr_k<float>(V, l, k, formq, R_host, f, s);
}

int bv_top_block(const BV &V, int l, int k, double *out) {
  const int nk = k - l;
  const size_t es = V.prec == SA_FP64 ? sizeof(double) : sizeof(float);
  std::vector<char> buf(es * nk * nk);
  SA_HIP(hipMemcpy2D(buf.data(), es * nk, (const char *)V.data + es * (size_t)l * V.ld, es * V.ld, es * nk, nk,
                     hipMemcpyDeviceToHost));
  for (size_t e = 0; e < (size_t)nk * nk; e++)
    out[e] = V.prec == SA_FP64 ? ((const double *)buf.data())[e] : (double)((const float *)buf.data())[e];
  return 0;
}

}  // namespace sa
