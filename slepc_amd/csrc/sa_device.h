// Device-side constants and helpers shared by the HIP sources (gfx950,
// wave size 64, 256-thread workgroups).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sa {

constexpr int BLK = 256;
constexpr int CH = 64;          // rows per chunk (one row per lane of a wave)
constexpr int LDP = CH + 1;     // padded LDS column stride
constexpr int RBLK = 1024;      // threads of the one-workgroup reductions

__device__ __forceinline__ double safe_sqrt(double a) { return a < 0.0 ? 0.0 : sqrt(a); }

// A load that is non-temporal when NT (data read once, larger than the
// caches: streaming it past the last-level cache keeps the caches for reused
// data and reads faster) and ordinary otherwise.
template <bool NT, typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// The dispatcher hands workgroups to the 8 XCDs round-robin by index, so
// consecutive blocks land on different L2s.  xcd_block maps the dispatch
// index b of a G-block grid to a logical block such that each XCD takes one
// contiguous range of about G/8 blocks (a bijection for any G): row-blocked
// kernels whose rows share neighbours (stencil planes) then find them in
// their own XCD's L2.
constexpr int N_XCD = 8;
__device__ __forceinline__ int xcd_block(int b, int G) {
  const int q = G / N_XCD, r = G % N_XCD, x = b % N_XCD, i = b / N_XCD;
  return x * q + min(x, r) + i;
}

// Cross-lane sums of a wave in the vector ALU (DPP within rows of 16 lanes,
// the gfx950 row and half swaps beyond them): a few cycles per step, where
// a shuffle through the LDS unit costs over a hundred.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;             // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;  // lane ^ 7 in 8 lanes, lane ^ 15 in 16
constexpr int DPP_ROR8 = 0x128;                             // lane ^ 8 in 16 lanes

// Lanes below M of each 2M lanes return x + (x of lane + M), the others
// y + (y of lane - M), M = 32 or 16: one step of a reduce-scatter, and with
// y = x the sum over the pair.
template <int M>
__device__ __forceinline__ uint32_t swap_lanes(uint32_t x, uint32_t y, uint32_t *other) {
  static_assert(M == 32 || M == 16, "rows of 16 lanes or halves of the wave");
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    *other = r[1];
    return r[0];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    *other = r[1];
    return r[0];
  }
}
template <int M>
__device__ __forceinline__ double swap_add(double x, double y) {
  const uint64_t a = __builtin_bit_cast(uint64_t, x), b = __builtin_bit_cast(uint64_t, y);
  uint32_t lo1, hi1;
  const uint32_t lo0 = swap_lanes<M>((uint32_t)a, (uint32_t)b, &lo1);
  const uint32_t hi0 = swap_lanes<M>((uint32_t)(a >> 32), (uint32_t)(b >> 32), &hi1);
  return __builtin_bit_cast(double, ((uint64_t)hi0 << 32) | lo0) +
         __builtin_bit_cast(double, ((uint64_t)hi1 << 32) | lo1);
}
template <int M>
__device__ __forceinline__ float swap_add(float x, float y) {
  uint32_t o;
  const uint32_t k = swap_lanes<M>(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), &o);
  return __builtin_bit_cast(float, k) + __builtin_bit_cast(float, o);
}
// The sum over N consecutive lanes (a power of two), in each of them.
template <int N, typename T>
__device__ __forceinline__ T lanes_sum(T v) {
  if constexpr (N >= 2) v += dpp_mov<DPP_XOR1>(v);
  if constexpr (N >= 4) v += dpp_mov<DPP_XOR2>(v);
  if constexpr (N >= 8) v += dpp_mov<DPP_HALF_MIRROR>(v);
  if constexpr (N >= 16) v += dpp_mov<DPP_MIRROR>(v);
  if constexpr (N >= 32) v = swap_add<16>(v, v);
  if constexpr (N >= 64) v = swap_add<32>(v, v);
  return v;
}
// One step of a reduce-scatter at lane bit M: lanes with the bit clear keep x,
// the others y, and add their partner's copy of it.
template <int M, typename T>
__device__ __forceinline__ T scatter_add(T x, T y, int lane) {
  if constexpr (M >= 16) {
    return swap_add<M>(x, y);
  } else {
    constexpr int CTRL = M == 8 ? DPP_ROR8 : (M == 4 ? DPP_HALF_MIRROR : (M == 2 ? DPP_XOR2 : DPP_XOR1));
    const bool hi = (lane & M) != 0;
    asm volatile("" : "+v"(x), "+v"(y));   // keeps the choice a select, not an indexed read
    return (hi ? y : x) + dpp_mov<CTRL>(hi ? x : y);
  }
}
// Reduce-scatter of p[0..N) over the wave (N a power of two up to 64): lane l
// returns the sum over the lanes of p[l / (64 / N)].  With M below 32 the steps
// above it have been taken: N values are left for the 2M lanes of a group.
template <int N, int M = 32, int CAP, typename T>
__device__ __forceinline__ T wave_scatter(T (&p)[CAP], int lane) {
  if constexpr (N > 1) {
#pragma unroll
    for (int i = 0; i < N / 2; i++) p[i] = scatter_add<M>(p[i], p[i + N / 2], lane);
    return wave_scatter<N / 2, M / 2>(p, lane);
  } else {
    return lanes_sum<2 * M>(p[0]);
  }
}

// out[col] = sum_b part[col * G + b] for col < ncol.  Each wave reduces four
// columns at a time (columns w, w+nw, w+2nw, w+3nw) with four loads per column
// in flight, then a shuffle reduction; the order of the additions is fixed, so
// every caller reducing the same partials obtains the same bits.
__device__ inline void sum_partials_block(const double *part, int G, int ncol, double *out) {
  constexpr int NB = 4;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, nw = blockDim.x >> 6;
  for (int c0 = w; c0 < ncol; c0 += NB * nw) {
    double s[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) s[k] = 0.0;
    int b = lane;
    for (; b + 192 < G; b += 256) {
#pragma unroll
      for (int k = 0; k < NB; k++) {
        const int col = c0 + k * nw;
        if (col < ncol) {
          const double *p = part + (size_t)col * G;
          s[k] += (p[b] + p[b + 64]) + (p[b + 128] + p[b + 192]);
        }
      }
    }
    for (; b < G; b += 64) {
#pragma unroll
      for (int k = 0; k < NB; k++) {
        const int col = c0 + k * nw;
        if (col < ncol) s[k] += part[(size_t)col * G + b];
      }
    }
#pragma unroll
    for (int k = 0; k < NB; k++) {
      double v = s[k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      const int col = c0 + k * nw;
      if (lane == 0 && col < ncol) out[col] = v;
    }
  }
}

// MFMA 16x16x4 in FP64 and FP32: C(16x16) += A(16x4) B(4x16).  Lane l
// supplies A(l%16, l/16) and B(l/16, l%16); element v of its result is
// C(g+4v, l%16) in FP64 and C(4g+v, l%16) in FP32, g = l/16.
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dbl4 mfma16x16x4(double a, double b, dbl4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ flt4 mfma16x16x4(float a, float b, flt4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename T> struct Vec4;
template <> struct Vec4<double> { typedef dbl4 type; };
template <> struct Vec4<float> { typedef flt4 type; };

// Row of the MFMA 16x16x4 result held in element v by lane group g.
template <typename T>
__device__ __forceinline__ int mfma_row(int g, int v) {
  return sizeof(T) == 8 ? g + 4 * v : 4 * g + v;
}

}  // namespace sa
