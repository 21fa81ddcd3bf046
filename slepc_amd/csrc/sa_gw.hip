// The Gram-Schmidt slots of one basis (sa_gs_device.h has the rule and the state
// machine), streaming the basis through registers.
//
// A workgroup of 8 waves walks chunks of 128 rows (two per lane; one per lane
// above 96 columns) in grid-stride order, so that the workgroups in flight
// read one contiguous stretch of every column.  Wave w holds the columns w,
// w + 8, ...: a chunk is up to NC loads per lane, those of the next chunk in
// flight while the current one is used.  The update v - V h needs one sum over
// the waves per chunk (LDS, one barrier that leaves the loads in flight); the
// dot products accumulate in FP64 registers and meet in one wave reduction at
// the end.
//
// HBM bounds it: the basis is read three times per two-pass step, and a slot
// reads 6.2 TB/s at 57 columns of 2.1M FP64 rows (949 MB in 152 us).  The
// kernel before it staged 64-row chunks in LDS, with three barriers per chunk
// and nothing in flight across them, and reached 4.9 TB/s.  Sweeps at 128^3:
// convection-diffusion FP64, columns 33-64, 17.5 -> 14.1 ms; 27-point FP64,
// columns 49-96, 44.9 -> 34.9 ms; columns 97-124, 42.8 -> 30.0 ms; 27-point FP32,
// 1.3M rows, columns 49-96, 16.3 -> 11.8 ms, 97-126, 15.5 -> 12.4.  Bases of FP64 in
// the last-level cache gain least: 5-point, columns 33-64, 240,000 rows 2.32 ->
// 2.08 ms, 300,000 2.71 -> 2.50, 399,000 3.41 -> 3.09; 300,000 rows, columns 1-30
// 1.56 -> 1.31, 49-96 6.98 -> 5.06.
#include <algorithm>

#include "sa_gs_device.h"

namespace sa {

namespace {

constexpr int GW_W = 8, GW_T = 64 * GW_W;      // waves and threads per workgroup

template <typename T, int VL> struct GwVec { typedef T type __attribute__((ext_vector_type(VL))); };

// VL rows of a column from row r (a multiple of VL), rows at or beyond n as zeros.
template <bool NT, int VL, typename T>
__device__ __forceinline__ typename GwVec<T, VL>::type gw_load(const T *p, int64_t r, int64_t n) {
  typedef typename GwVec<T, VL>::type VT;
  if (r + VL <= n) return ld_stream<NT>(reinterpret_cast<const VT *>(p + r));
  VT x = (VT)(T)0;
#pragma unroll
  for (int e = 0; e < VL; e++)
    if (r + e < n) x[e] = p[r + e];
  return x;
}

// Barrier for data exchanged through LDS: the LDS operations are complete, the
// global loads of the next chunk stay in flight.
__device__ __forceinline__ void gw_lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Chunks first, first + step, ... of the basis: v = (v - V cf) * scl when UPD
// (cf only when MULT), the dot products with the new v into acc and self when
// DOTS.  cf: this wave's coefficients.  All threads of the workgroup call it.
template <typename T, int NC, int VL, bool NT, bool MULT, bool UPD, bool DOTS>
__device__ __forceinline__ void gw_rows(const GsArgs<T> &a, int64_t first, int64_t step, T scl, const T (&cf)[NC],
                                        T (*red)[GW_W][64 * VL], double (&acc)[NC], double &self) {
  typedef typename GwVec<T, VL>::type VT;
  constexpr int CR = 64 * VL;
  // FP32 products against up to 16 columns are added in FP64 one by one: pairs of
  // a lane's two rows leave 5.3e-11 in the norm of 354,000 rows where the shorter
  // sums of a 64-row tile left 3.5e-11.  Beyond, those sums had 5 rows and more,
  // and pairs save 1.5% of a sweep (27-point, 1.3M rows, columns 49-96).
  constexpr bool ONE = sizeof(T) == 4 && NC <= 2;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = a.c;
  const int64_t nch = (a.n + CR - 1) / CR;
  T *vc = a.V + (int64_t)c * a.ld;
  VT x[NC], y[NC], v, vy;
  auto fetch = [&](int64_t ch) {
    const int64_t r = ch * CR + lane * VL;
    if constexpr (MULT || DOTS) {
#pragma unroll
      for (int i = 0; i < NC; i++) {
        const int col = i * GW_W + w;
        if (col < c) y[i] = gw_load<NT, VL>(a.V + (int64_t)col * a.ld, r, a.n);
      }
    }
    vy = gw_load<false, VL>(vc, r, a.n);
  };
#pragma unroll
  for (int i = 0; i < NC; i++) y[i] = (VT)(T)0;
  if (first < nch) fetch(first);
  int it = 0;
  for (int64_t ch = first; ch < nch; ch += step, it++) {
#pragma unroll
    for (int i = 0; i < NC; i++) x[i] = y[i];
    v = vy;
    if (ch + step < nch) fetch(ch + step);
    if constexpr (UPD) {
      VT tot = (VT)(T)0;
      if constexpr (MULT) {
        VT p = (VT)(T)0;
#pragma unroll
        for (int i = 0; i < NC; i++)
          if (i * GW_W + w < c) p += x[i] * cf[i];
        // two buffers: a wave may start the next chunk while others still read this one
        *reinterpret_cast<VT *>(&red[it & 1][w][lane * VL]) = p;
        gw_lds_barrier();
        VT q[GW_W];
#pragma unroll
        for (int u = 0; u < GW_W; u++) q[u] = *reinterpret_cast<const VT *>(&red[it & 1][u][lane * VL]);
        tot = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
      }
      v = (v - tot) * scl;
      if ((it & (GW_W - 1)) == w) {              // the waves store in turn
        const int64_t r = ch * CR + lane * VL;
        if (r + VL <= a.n) {
          *reinterpret_cast<VT *>(vc + r) = v;
        } else {
#pragma unroll
          for (int e = 0; e < VL; e++)
            if (r + e < a.n) vc[r + e] = v[e];
        }
      }
    }
    if constexpr (DOTS) {
      T s = (T)0;
#pragma unroll
      for (int e = 0; e < VL; e++) {
        if constexpr (ONE) self += (double)v[e] * (double)v[e];
        else s += v[e] * v[e];
      }
      if constexpr (!ONE) self += (double)s;
#pragma unroll
      for (int i = 0; i < NC; i++)
        if (i * GW_W + w < c) {
          T d = (T)0;
#pragma unroll
          for (int e = 0; e < VL; e++) {
            if constexpr (ONE) acc[i] += (double)x[i][e] * (double)v[e];
            else d += x[i][e] * v[e];
          }
          if constexpr (!ONE) acc[i] += (double)d;
        }
    }
  }
}

// The sums over the wave of acc and self: into out[col] (LDS) or part[col * G + b].
template <int NC>
__device__ __forceinline__ void gw_combine(double (&acc)[NC], double self, int c, double *out, double *part, int G,
                                           int b) {
  constexpr int SP = NC <= 2 ? 2 : (NC <= 4 ? 4 : (NC <= 8 ? 8 : 16)), LPC = 64 / SP;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double p[SP];
#pragma unroll
  for (int i = 0; i < SP; i++) p[i] = i < NC ? acc[i < NC ? i : 0] : 0.0;
  const double d = wave_scatter<SP>(p, lane);
  const int sl = lane / LPC, col = sl * GW_W + w;
  if (lane % LPC == 0 && sl < NC && col < c) {
    if (out) out[col] = d;
    else part[(size_t)col * G + b] = d;
  }
  if (w == c % GW_W) {
    const double s = lanes_sum<64>(self);
    if (lane == 0) {
      if (out) out[c] = s;
      else part[(size_t)c * G + b] = s;
    }
  }
}

template <typename T, int NC>
__device__ __forceinline__ void gw_coef(T (&cf)[NC], const double *s_dots, int c) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < NC; i++) cf[i] = i * GW_W + w < c ? (T)s_dots[i * GW_W + w] : (T)0;
}

// One slot of column a.c (gs_slot of sa_gs_device.h, the same states).
template <typename T, int NC, int VL, bool NT>
__global__ __launch_bounds__(GW_T) void gw_kernel(GsArgs<T> a) {
  __shared__ __align__(16) T red[2][GW_W][64 * VL];
  __shared__ double s_dots[GS_MAXC + 1];
  __shared__ GsState s_st;
  __shared__ int s_act, s_rec;
  __shared__ double s_scale;
  const int t = threadIdx.x, b = blockIdx.x, c = a.c;
  const bool lead = b == 0;
  if (t == 0) s_st = a.st[(a.slot + 1) % GS_NSTATE];
  if (a.slot > 1)
    for (int i = t; i <= c; i += GW_T) s_dots[i] = a.dots_in[i];
  __syncthreads();
  double acc[NC], self = 0.0;
  T cf[NC];
#pragma unroll
  for (int i = 0; i < NC; i++) {
    acc[i] = 0.0;
    cf[i] = (T)0;
  }
  if (a.slot == 1) {
    const bool stopped = s_st.stop != 0;
    if (lead && t == 0) {
      GsState S = s_st;
      if (stopped) {
        S.done = 1;
        S.dots_ready = 0;
      } else {
        S.pass = 0; S.pending = 0; S.lindep = 0; S.done = 0; S.dots_ready = 1;
      }
      a.st[0] = S;
    }
    if (stopped) return;
    gw_rows<T, NC, VL, NT, false, false, true>(a, b, a.G, (T)1, cf, red, acc, self);
    gw_combine(acc, self, c, nullptr, a.part_out, a.G, b);
    return;
  }
  if (s_st.done || !s_st.dots_ready) {        // nothing left for this column
    if (lead && t == 0) {
      GsState S = s_st;
      S.dots_ready = 0;
      a.st[a.slot - 1] = S;
    }
    return;
  }
  gs_decide_block<T, GW_T>(a, s_dots, &s_st, &s_act, &s_rec, &s_scale, lead);
  int act = s_act;
  int64_t first = b, step = a.G;
  if (act == ACT_MULT_DOTS && a.slot == 3) {
    // Third pass or failed estimate: the lead workgroup finishes the column
    // over all rows (the others took the same decision and leave v alone).
    if (!lead) return;
    first = 0;
    step = 1;
    if (t == 0) s_st.slow_total++;
    while (act == ACT_MULT_DOTS) {             // ends: S.pass < 3 bounds the passes
      gw_coef(cf, s_dots, c);
#pragma unroll
      for (int i = 0; i < NC; i++) acc[i] = 0.0;
      self = 0.0;
      __syncthreads();
      gw_rows<T, NC, VL, NT, true, true, true>(a, first, step, (T)1, cf, red, acc, self);
      gw_combine(acc, self, c, s_dots, nullptr, 0, 0);
      __syncthreads();                         // the sums, and every store of v before it is read again
      gs_decide_block<T, GW_T>(a, s_dots, &s_st, &s_act, &s_rec, &s_scale, true);
      act = s_act;
    }
  }
  const T scl = (T)s_scale;
  if (act == ACT_MULT_DOTS) {
    gw_coef(cf, s_dots, c);
    gw_rows<T, NC, VL, NT, true, true, true>(a, first, step, scl, cf, red, acc, self);
    gw_combine(acc, self, c, nullptr, a.part_out, a.G, b);
  } else if (act == ACT_MULT_SCALE) {
    gw_coef(cf, s_dots, c);
    gw_rows<T, NC, VL, NT, true, true, false>(a, first, step, scl, cf, red, acc, self);
  } else {
    gw_rows<T, NC, VL, NT, false, true, false>(a, first, step, scl, cf, red, acc, self);
  }
}

template <typename T, int NC>
void gw_nt(const GsArgs<T> &a, bool nt, hipStream_t s) {
  constexpr int VL = NC > 12 ? 1 : 2;     // two rows of 16 columns spill: FP32 columns 97-126 of 1.3M rows 26.0 ms, one row 12.3
  if (nt) hipLaunchKernelGGL((gw_kernel<T, NC, VL, true>), dim3(a.G), dim3(GW_T), 0, s, a);
  else hipLaunchKernelGGL((gw_kernel<T, NC, VL, false>), dim3(a.G), dim3(GW_T), 0, s, a);
}

template <typename T>
int gw_slot(const GsArgs<T> &a, bool nt, hipStream_t s) {
  const int c = a.c;
  if (c <= 2 * GW_W) gw_nt<T, 2>(a, nt, s);
  else if (c <= 4 * GW_W) gw_nt<T, 4>(a, nt, s);
  else if (c <= 6 * GW_W) gw_nt<T, 6>(a, nt, s);
  else if (c <= 8 * GW_W) gw_nt<T, 8>(a, nt, s);
  else if (c <= 12 * GW_W) gw_nt<T, 12>(a, nt, s);
  else gw_nt<T, 16>(a, nt, s);
  SA_HIP(hipGetLastError());
  return 0;
}

}  // namespace

// Two workgroups per CU where their registers allow it (FP64 up to 32 columns,
// FP32 up to 96), else one; more only adds partial sums (FP64 convection-
// diffusion sweep at 128^3 with 1, 2, 4 per CU: 14.14, 14.36, 14.66 ms; FP32
// 27-point sweep of 1.3M rows: 13.1, 11.8, 12.5 ms).
int gw_blocks(int64_t n, int prec, int c) {
  const int per_cu = c <= (prec == SA_FP64 ? 32 : 96) ? 2 : 1;
  return (int)std::min<int64_t>(std::max<int64_t>(1, (n + 127) / 128), per_cu * (int64_t)num_cus());
}

int launch_gw_slot(const GsArgs<double> &a, bool nt, hipStream_t s) { return gw_slot(a, nt, s); }
int launch_gw_slot(const GsArgs<float> &a, bool nt, hipStream_t s) { return gw_slot(a, nt, s); }

}  // namespace sa
