// The Arnoldi/Lanczos sweep as one resident kernel, for bases that fit the
// register files of the GPU (gfx950: 256 CUs with 512 KB of vector registers).
//
// The launch-per-slot sweep (sa_gs.hip) pays five dependent launches per Krylov
// step and reads the basis three times from the caches; at n = 65,536 that is
// 28 us per step, most of it launch latency.  Here one launch runs the whole
// sweep.  Workgroup b owns R = 64 Q rows for its duration and keeps their part
// of every basis column in registers: wave w of W holds the columns w, w + W,
// w + 2W, ... (S slots), lane l the rows l, l + 64, ... of the block.  A dot
// product is then Q fused multiply-adds per column and one wave reduction, an
// update Q S of them and a sum over the waves in LDS; the basis is read from
// memory once and each new column written once.
//
// What the workgroups exchange (the new vector for the next SpMV, the partial
// dot products, their totals) goes through tagged words: a 64-bit word carries
// 32 bits of data and the 32-bit number of the exchange, stored and loaded as
// one relaxed agent-scope atomic.  A reader polls the word itself until the
// number is the one it waits for, so the data arrives with its own flag: no
// fence (an agent-scope release writes back an L2), no barrier, and no order
// between different words is relied upon.  A word is only overwritten once
// every reader has consumed it: the words of a reduction depend on all
// workgroups having read the totals of the one before, and a column of the
// basis is published after the reductions that followed the last SpMV.
//
// One reduction is two exchanges: every workgroup publishes its partial sums,
// one wave per column adds them in a fixed order (results do not depend on
// timing) and publishes the total, which every workgroup reads and takes the
// same decision from (gs_rule).  Letting every workgroup read all partial sums
// itself saves the second exchange but measured slower from 32 workgroups on
// (3.5 against 2.9 us per reduction).
//
// The operator's rows and the list of the remote entries they refer to are
// kept in LDS, so a step fetches each remote entry once, all in one round
// trip (27-point operator, 256 rows per workgroup: 6.2 us per step when every
// nonzero fetches its own, 3.2 with the list).
//
// What bounds it is the latency of the five exchanges of a step, about 1.3 us
// each (a store to memory and a load that misses the L2): of 10-11 us per step
// at n = 10,000 and 65,536 they take 7, the decision and the update 2, the dot
// products 0.7.  Measured against the slots of 64-row tiles: 64 steps at n =
// 65,536 770 us (1,880), 16 steps from column 16 at n = 10,000 200 us (374), FP32
// 32 steps from column 32 at n = 354,000 628 us (2,479).
//
// All workgroups must be on the GPU together.  The grid has at most one
// workgroup per CU, and the process admits only sweeps whose workgroups fit
// the CUs together (PsAdmit); kernels of other streams only delay them.  If
// others hold the CUs all the same (another process), every wait ends after a
// bounded number of polls, the kernel exits and reports it, and the host runs
// the sweep slot by slot instead, and after repeated failures those that follow
// without a try (Backoff).
#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "sa_budget.h"
#include "sa_gs_device.h"

namespace sa {

namespace {

constexpr int PS_W = 8;                 // waves per workgroup
constexpr int PS_T = 64 * PS_W;         // threads per workgroup
constexpr int PS_READ0 = PS_T - GS_MAXC;   // first of the threads that read the totals (the last two waves)
constexpr int PS_OWN = PS_READ0 / 64;   // waves that add partial sums
constexpr int PS_COPIES = 8;            // copies of the totals

template <typename T>
struct PsArgs {
  int64_t n0, n1;             // the rows it computes: n0 .. n1 - 1 (operator columns and words count from 0)
  int64_t xn, ld;             // words of a vector's low halves, stride of the basis
  T *V;
  const int32_t *rp, *ci;     // operator, or null: column c0 itself is orthonormalised
  const T *val;
  int c0, c1;                 // columns to compute: c0 .. c1
  int G;                      // workgroups
  int nzcap, hcap, wcap;      // LDS for the block's operator: nonzeros, remote columns, their span
  uint64_t *xw, *pw, *tw;     // exchanged words: vector, partial sums, totals
  unsigned int *abort_word;   // set to `base` by a workgroup that gave up
  T *backup;                  // without operator: the vector as it was
  uint32_t base;              // number of the first exchange of this sweep
  GsState *st;                // device state
  GsMirror *host;             // pinned host mirror
  double *dbuf;
  int dm;
  double eta;
  int refine;
  int polls;                  // polls after which a wait gives up
};

__device__ __forceinline__ uint64_t ps_load(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ps_store(uint64_t *p, uint32_t data, uint32_t tag) {
  __hip_atomic_store(p, (uint64_t)data | ((uint64_t)tag << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A double as two tagged words at lo and hi, a float as one.
__device__ __forceinline__ void ps_put(uint64_t *lo, uint64_t *hi, double v, uint32_t tag) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  ps_store(lo, (uint32_t)u, tag);
  ps_store(hi, (uint32_t)(u >> 32), tag);
}
__device__ __forceinline__ double ps_join(uint64_t lo, uint64_t hi) {
  return __builtin_bit_cast(double, (lo & 0xffffffffull) | (hi << 32));
}
__device__ __forceinline__ bool ps_is(uint64_t w, uint32_t tag) { return (uint32_t)(w >> 32) == tag; }

// One poll without success: whether to go on.
template <typename T>
__device__ __forceinline__ bool ps_again(const PsArgs<T> &a, int &spin) {
  if (++spin > a.polls) return false;
  return (spin & 1023) != 0 ||
         __hip_atomic_load(a.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != a.base;
}

// x[c[u]] of the columns in `need` (a bit each), published under tag.
template <typename T, int U>
__device__ __forceinline__ bool ps_gather(const PsArgs<T> &a, const int32_t (&c)[U], unsigned need, uint32_t tag,
                                          T (&xv)[U]) {
  int spin = 0;
  for (;;) {
    uint64_t lo[U], hi[U];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (need & (1u << u)) {
        lo[u] = ps_load(a.xw + c[u]);
        if constexpr (sizeof(T) == 8) hi[u] = ps_load(a.xw + a.xn + c[u]);
      }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (need & (1u << u)) {
        if constexpr (sizeof(T) == 8) {
          if (ps_is(lo[u], tag) && ps_is(hi[u], tag)) {
            xv[u] = ps_join(lo[u], hi[u]);
            need &= ~(1u << u);
          }
        } else if (ps_is(lo[u], tag)) {
          xv[u] = __builtin_bit_cast(float, (uint32_t)lo[u]);
          need &= ~(1u << u);
        }
      }
    if (!need) return true;
    if (!ps_again(a, spin)) return false;
  }
}

constexpr int PS_D = 4;                 // partial sums per lane and column: up to 256 workgroups

// Sum of the G partial sums of one column over the wave, each awaited under
// tag; lo/hi: the column's words.
template <typename T>
__device__ __forceinline__ double ps_collect(const PsArgs<T> &a, const uint64_t *lo, const uint64_t *hi, int lane,
                                             uint32_t tag, bool *ok) {
  double v[PS_D];
  unsigned need = 0;
#pragma unroll
  for (int u = 0; u < PS_D; u++) {
    v[u] = 0.0;
    if (lane + 64 * u < a.G) need |= 1u << u;
  }
  int spin = 0;
  while (need) {
    uint64_t l[PS_D], h[PS_D];
#pragma unroll
    for (int u = 0; u < PS_D; u++)
      if (need & (1u << u)) {
        l[u] = ps_load(lo + lane + 64 * u);
        h[u] = ps_load(hi + lane + 64 * u);
      }
#pragma unroll
    for (int u = 0; u < PS_D; u++)
      if ((need & (1u << u)) && ps_is(l[u], tag) && ps_is(h[u], tag)) {
        v[u] = ps_join(l[u], h[u]);
        need &= ~(1u << u);
      }
    if (need && !ps_again(a, spin)) {
      *ok = false;
      break;
    }
  }
  return lanes_sum<64>((v[0] + v[1]) + (v[2] + v[3]));
}

// The remote columns that the block's operator rows (nz column indices ci)
// refer to, each once: lists them in hcol and writes to scol the position of
// every nonzero's column in [own rows | list].  Returns their number, or -1
// when the columns span more than wcap or number more than hcap.  bits, pre:
// wcap / 32 words each; called by all threads.
__device__ int ps_list_halo(const int32_t *__restrict__ ci, int nz, int64_t r0, int rows, int R, uint32_t *bits,
                            uint32_t *pre, int wcap, int32_t *hcol, int hcap, uint16_t *scol, int *s_tmp) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int mn = 0x7fffffff, mx = -1;
  for (int i = t; i < nz; i += PS_T) {
    mn = min(mn, ci[i]);
    mx = max(mx, ci[i]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mn = min(mn, __shfl_xor(mn, o, 64));
    mx = max(mx, __shfl_xor(mx, o, 64));
  }
  if (lane == 0) {
    s_tmp[w] = mn;
    s_tmp[PS_W + w] = mx;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PS_W; q++) {
    mn = min(mn, s_tmp[q]);
    mx = max(mx, s_tmp[PS_W + q]);
  }
  __syncthreads();
  if (mx < mn || mx - mn >= wcap) return -1;
  const int nw = ((mx - mn) >> 5) + 1;
  for (int i = t; i < nw; i += PS_T) bits[i] = 0;
  __syncthreads();
  for (int i = t; i < nz; i += PS_T) {
    const int64_t lc = ci[i] - r0;
    const int d = ci[i] - mn;
    if (lc < 0 || lc >= rows) atomicOr(&bits[d >> 5], 1u << (d & 31));
  }
  __syncthreads();
  // exclusive prefix of the words' populations: a run of words per thread
  const int run = (nw + PS_T - 1) / PS_T, i0 = min(nw, t * run), i1 = min(nw, i0 + run);
  int mine = 0;
  for (int i = i0; i < i1; i++) mine += __popc(bits[i]);
  int inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  if (lane == 63) s_tmp[w] = inc;
  __syncthreads();
  int before = 0, total = 0;
  for (int q = 0; q < PS_W; q++) {
    before += q < w ? s_tmp[q] : 0;
    total += s_tmp[q];
  }
  if (total > hcap) return -1;             // uniform: every thread has the same total
  int at = before + inc - mine;
  for (int i = i0; i < i1; i++) {
    pre[i] = at;
    for (uint32_t m = bits[i]; m; m &= m - 1) hcol[at++] = mn + 32 * i + __builtin_ctz(m);
  }
  __syncthreads();
  for (int i = t; i < nz; i += PS_T) {
    const int64_t lc = ci[i] - r0;
    const int d = ci[i] - mn;
    scol[i] = (uint16_t)((lc >= 0 && lc < rows) ? (int)lc
                                                : R + (int)pre[d >> 5] + __popc(bits[d >> 5] & ((1u << (d & 31)) - 1u)));
  }
  __syncthreads();
  return total;
}

// The lane's products of v with the first N column slots, and of v with itself,
// added to acc and self: sums of RUN rows in T, those in FP64.  Long FP32 sums
// would be the larger part of a coefficient's error: with all 22 rows of a lane
// in one, coefficients against 10 columns of 354,000 rows were 4.5e-10 of the
// vector's norm off and the norm 3.1e-10; sums as short as those of 256 threads
// on a 64-row tile (3 rows for 10 columns, 10 for 32, 11 for 40, 22 for 64) leave
// 1.8e-10 and 5.5e-11.  So FP32 products against up to 32 or 40 columns are added in
// FP64 one by one, beyond in runs of 8, with more than 64 columns of 11 at most.
template <int N, int RUN, typename T, int S, int Q>
__device__ __forceinline__ void ps_dots(T (&x)[S][Q], const T *vn, int lane, double (&acc)[S], double &self) {
#pragma unroll
  for (int q0 = 0; q0 < Q; q0 += RUN) {
    T part[N], sq = (T)0;
#pragma unroll
    for (int s = 0; s < N; s++) part[s] = (T)0;
#pragma unroll
    for (int q = q0; q < Q && q < q0 + RUN; q++) {
      const T v = vn[q * 64 + lane];
      if constexpr (RUN == 1) {
        self += (double)v * (double)v;
#pragma unroll
        for (int s = 0; s < N; s++) {
          asm volatile("" : "+v"(x[s][q]));      // converted here, not kept as doubles
          acc[s] += (double)x[s][q] * (double)v;
        }
      } else {
        sq += v * v;
#pragma unroll
        for (int s = 0; s < N; s++) part[s] += x[s][q] * v;
      }
    }
    if constexpr (RUN > 1) {
      self += (double)sq;
#pragma unroll
      for (int s = 0; s < N; s++) acc[s] += (double)part[s];
    }
  }
}

// Workgroup b of the sweep.
template <typename T, int S, int Q>
__device__ __forceinline__ void ps_block(const PsArgs<T> &a, int b) {
  constexpr int R = 64 * Q, W = PS_W;
  constexpr int SP = S <= 4 ? 4 : (S <= 8 ? 8 : 16), LPC = 64 / SP;   // lanes that end with one column's sum
  constexpr int TPR = R > PS_T / 2 ? 1 : (R > PS_T / 4 ? 2 : (R > PS_T / 8 ? 4 : 8));
  constexpr int U = 4;                       // nonzeros in flight per thread
  constexpr int NS = S > 8 ? 5 : 4;          // FP32: column slots up to which products are added in FP64
  __shared__ T va[R], vb[R];                 // the last column and the one being computed
  __shared__ T red[W * R];
  __shared__ double s_dots[GS_MAXC];
  __shared__ int32_t srp[R + 1];
  __shared__ int s_tmp[2 * W];
  __shared__ int s_fail;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *sval = reinterpret_cast<T *>(smem_raw);              // [nzcap] operator rows of the block
  T *vh = sval + a.nzcap;                                 // [hcap] remote entries of the last column
  int32_t *hcol = reinterpret_cast<int32_t *>(vh + a.hcap);   // [hcap] their columns
  uint16_t *scol = reinterpret_cast<uint16_t *>(hcol + a.hcap);   // [nzcap] columns as positions in [own rows | remote]
  uint32_t *bits = reinterpret_cast<uint32_t *>(smem_raw);   // set-up only, before sval and vh are filled
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t r0 = a.n0 + (int64_t)b * R;
  const int rows = (int)min((int64_t)R, a.n1 - r0);
  uint32_t tag = a.base;
  T *vp = va, *vn = vb;

  // the block's part of columns 0 .. c0-1, the operator's rows, the last column
  T x[S][Q];
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int col = s * W + w, row = q * 64 + lane;
      x[s][q] = (col < a.c0 && row < rows) ? a.V[(int64_t)col * a.ld + r0 + row] : (T)0;
    }
  int32_t p0 = 0;
  int nh = -1;                               // remote columns, or -1: the operator is read from memory
  if (t == 0) s_fail = 0;
  if (a.rp) {
    for (int i = t; i <= rows; i += PS_T) srp[i] = a.rp[r0 + i];
    p0 = a.rp[r0];
    const int nz = a.rp[r0 + rows] - p0;
    for (int i = t; i < R; i += PS_T) vp[i] = i < rows ? a.V[(int64_t)(a.c0 - 1) * a.ld + r0 + i] : (T)0;
    if (nz <= a.nzcap) {
      nh = ps_list_halo(a.ci + p0, nz, r0, rows, R, bits, bits + a.wcap / 32, a.wcap, hcol, a.hcap, scol, s_tmp);
      if (nh >= 0)
        for (int i = t; i < nz; i += PS_T) sval[i] = a.val[p0 + i];
    }
  } else {
    for (int i = t; i < R; i += PS_T) {
      const T v = i < rows ? a.V[(int64_t)a.c0 * a.ld + r0 + i] : (T)0;
      vn[i] = v;
      if (i < rows) a.backup[r0 + i] = v;
    }
  }
  GsState st = a.st[2];
  st.stop = 0; st.stop_col = 0; st.lindep = 0; st.beta = 0.0;
  double hreg = 0.0;                         // coefficient t of the current column (workgroup 0)
  __syncthreads();

  for (int c = a.c0; c <= a.c1; c++) {
    // ---- vn = A vp ----------------------------------------------------------
    if (a.rp) {
      const T *first = c == a.c0 ? a.V + (int64_t)(c - 1) * a.ld : nullptr;   // the sweep's first vector: in memory
      bool ok = true;
      if (nh >= 0) {
        for (int h0 = 0; h0 < nh; h0 += 2 * PS_T) {
          int32_t cc[2];
          T xv[2];
          unsigned need = 0;
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int h = h0 + u * PS_T + t;
            cc[u] = 0;
            if (h < nh) {
              cc[u] = hcol[h];
              need |= 1u << u;
            }
          }
          if (first) {
#pragma unroll
            for (int u = 0; u < 2; u++)
              if (need & (1u << u)) xv[u] = first[cc[u]];
          } else if (need) {
            ok = ps_gather(a, cc, need, tag, xv) && ok;
          }
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int h = h0 + u * PS_T + t;
            if (h < nh) vh[h] = xv[u];
          }
        }
        __syncthreads();
      }
      const int lg = t % TPR;
      for (int r = t / TPR; r < R; r += PS_T / TPR) {
        T s = (T)0;
        if (r < rows) {
          const int pb = srp[r] - p0, pe = srp[r + 1] - p0;
          for (int p = pb + lg; p < pe; p += U * TPR) {
            T av[U], xv[U];
            if (nh >= 0) {
#pragma unroll
              for (int u = 0; u < U; u++) {
                const int pk = min(p + u * TPR, pe - 1), cc = scol[pk];
                av[u] = sval[pk];
                xv[u] = *(cc < R ? vp + cc : vh + (cc - R));
              }
            } else {
              int32_t cc[U];
              unsigned need = 0;
#pragma unroll
              for (int u = 0; u < U; u++) {
                const int pk = min(p + u * TPR, pe - 1);
                av[u] = a.val[p0 + pk];
                cc[u] = a.ci[p0 + pk];
              }
#pragma unroll
              for (int u = 0; u < U; u++) {
                const int64_t lc = cc[u] - r0;
                xv[u] = (T)0;
                if (lc >= 0 && lc < rows) xv[u] = vp[lc];
                else if (p + u * TPR < pe) need |= 1u << u;
              }
              if (first) {
#pragma unroll
                for (int u = 0; u < U; u++)
                  if (need & (1u << u)) xv[u] = first[cc[u]];
              } else if (need) {
                ok = ps_gather(a, cc, need, tag, xv) && ok;
              }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
              if (p + u * TPR < pe) s += av[u] * xv[u];
          }
        }
        s = lanes_sum<TPR>(s);
        if (lg == 0) vn[r] = s;              // rows beyond the block: 0
      }
      if (!ok) s_fail = 1;
      __syncthreads();
    }
    st.pass = 0; st.pending = 0; st.lindep = 0; st.done = 0; st.dots_ready = 1;

    // ---- passes of classical Gram-Schmidt --------------------------------------
    while (true) {
      tag++;
      // partial dot products of the block, and its sum of squares in the place
      // of column c (held by no wave yet)
      {
        double p[SP], acc[S], self = 0.0;
#pragma unroll
        for (int s = 0; s < S; s++) acc[s] = 0.0;
        if constexpr (sizeof(T) == 8) ps_dots<S, Q>(x, vn, lane, acc, self);
        else if (c < NS * W) ps_dots<NS, 1>(x, vn, lane, acc, self);
        else ps_dots<S, (S > 8 ? Q : 8)>(x, vn, lane, acc, self);
#pragma unroll
        for (int s = 0; s < SP; s++) p[s] = s < S ? (s * W + w == c ? self : acc[s < S ? s : 0]) : 0.0;
        const double d = wave_scatter<SP>(p, lane);
        const int sl = lane / LPC, col = sl * W + w;
        if (lane % LPC == 0 && sl < S && col <= c) {
          if (a.G == 1) s_dots[col] = d;     // nobody to exchange with
          else ps_put(a.pw + (size_t)(2 * col) * a.G + b, a.pw + (size_t)(2 * col + 1) * a.G + b, d, tag);
        }
        if (c >= S * W && w == W - 1) {      // no place for column c: the last one of a full basis
          const double sd = lanes_sum<64>(self);
          if (lane == 0 && a.G == 1) s_dots[c] = sd;
          else if (lane == 0) ps_put(a.pw + (size_t)(2 * c) * a.G + b, a.pw + (size_t)(2 * c + 1) * a.G + b, sd, tag);
        }
      }
      bool ok = true;
      if (a.G == 1) {
      } else if (w < PS_OWN) {
        // totals of the columns this workgroup adds: column b, b + G, ...; a
        // copy for each of 8 groups of workgroups, so that fewer poll one word
        for (int col = b + w * a.G; col <= c; col += PS_OWN * a.G) {
          const uint64_t *lo = a.pw + (size_t)(2 * col) * a.G;
          const double s = ps_collect(a, lo, lo + a.G, lane, tag, &ok);
          if (!__all(ok)) break;
          if (lane < PS_COPIES) ps_put(a.tw + (2 * lane) * GS_MAXC + col, a.tw + (2 * lane + 1) * GS_MAXC + col, s, tag);
        }
      } else {
        const int i = t - PS_READ0;
        if (i <= c) {
          const uint64_t *lo = a.tw + (2 * (b % PS_COPIES)) * GS_MAXC + i, *hi = lo + GS_MAXC;
          int spin = 0;
          uint64_t l, h;
          while (true) {
            l = ps_load(lo);
            h = ps_load(hi);
            if (ps_is(l, tag) && ps_is(h, tag)) break;
            if (!ps_again(a, spin)) {
              ok = false;
              break;
            }
          }
          s_dots[i] = ps_join(l, h);
        }
      }
      if (!ok) s_fail = 1;
      __syncthreads();
      if (s_fail) {                          // a wait gave up: leave, the host starts over
        if (t == 0) {
          __hip_atomic_store(a.abort_word, a.base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          a.host->fail = 1;
        }
        return;
      }
      // V h of the block, per wave (unused when only a scaling is left, rare)
      {
        T cf[S];
#pragma unroll
        for (int s = 0; s < S; s++) cf[s] = s * W + w < c ? (T)s_dots[s * W + w] : (T)0;
#pragma unroll
        for (int q = 0; q < Q; q++) {
          T p = (T)0;
#pragma unroll
          for (int s = 0; s < S; s++) p += x[s][q] * cf[s];
          red[w * R + q * 64 + lane] = p;
        }
      }
      // the same decision in every thread of every workgroup
      double sq = 0.0, scale;
      if (lane < c) sq = s_dots[lane] * s_dots[lane];
      if (lane + 64 < c) sq += s_dots[lane + 64] * s_dots[lane + 64];
      sq = lanes_sum<64>(sq);
      int rec;
      const int act = gs_rule(st, s_dots, sq, c, a.eta, a.refine, &scale, &rec);
      if (rec && t < c) hreg = (st.pass == 1 ? 0.0 : hreg) + s_dots[t];
      // v = (v - V h) * scale
      __syncthreads();
      const T scl = (T)scale;
      for (int r = t; r < R; r += PS_T) {
        T tot = (T)0;
        if (act != ACT_SCALE_ONLY) {
          T e[W];
#pragma unroll
          for (int q = 0; q < W; q++) e[q] = red[q * R + r];
          tot = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
        }
        const T v = (vn[r] - tot) * scl;
        vn[r] = v;
        if (st.done && r < rows) {
          if (c < a.c1 && !st.stop) {
            if constexpr (sizeof(T) == 8) ps_put(a.xw + r0 + r, a.xw + a.xn + r0 + r, v, tag);
            else ps_store(a.xw + r0 + r, __builtin_bit_cast(uint32_t, v), tag);
          }
          a.V[(int64_t)c * a.ld + r0 + r] = v;
        }
      }
      __syncthreads();
      if (st.done) break;
    }
    if (b == 0) {
      double *h = a.dbuf + (size_t)c * a.dm;
      if (t < c) h[t] = hreg;
      if (t == 0) h[c] = st.lindep ? 0.0 : st.nrm;
    }
    if (st.stop || c == a.c1) break;
    // column c joins the basis
#pragma unroll
    for (int s = 0; s < S; s++)
      if (s * W + w == c)
#pragma unroll
        for (int q = 0; q < Q; q++) x[s][q] = vn[q * 64 + lane];
    T *tmp = vp;
    vp = vn;
    vn = tmp;
  }
  if (b == 0 && t == 0) {
    st.dots_ready = 0;
    a.st[2] = st;
    a.host->st = st;
    a.host->ok = 1;
  }
}

template <typename T, int S, int Q>
__global__ __launch_bounds__(PS_T) void ps_sweep_kernel(PsArgs<T> a) {
  ps_block<T, S, Q>(a, blockIdx.x);
}

// Sweeps of several problems side by side, stacked row by row in one basis:
// problem i has the workgroups b0 .. b0 + G - 1, its own columns, state,
// coefficients and exchange words.
template <typename T, int S, int Q>
__global__ __launch_bounds__(PS_T) void ps_batch_kernel(PsArgs<T> a, const PsProb *__restrict__ probs,
                                                        const int *__restrict__ of_block) {
  const int i = of_block[blockIdx.x];
  const PsProb p = probs[i];
  a.n0 = p.n0; a.n1 = p.n1;
  a.c0 = p.c0; a.c1 = p.c1; a.G = p.G;
  a.pw += (size_t)2 * GS_MAXC * p.b0;
  a.tw += (size_t)2 * PS_COPIES * GS_MAXC * i;
  a.st += (size_t)GS_NSTATE * p.id;
  a.dbuf += (size_t)a.dm * a.dm * p.id;
  ps_block<T, S, Q>(a, blockIdx.x - p.b0);
}

// ---- admission: the sweeps in flight together must fit the CUs --------------
// Workgroups go to the 8 XCDs in turn, so a sweep of G workgroups takes
// ceil(G / 8) CUs of each; the budget is one XCD's CUs, and no sweep takes more
// workgroups than ps_most().
int ps_most() { return std::min(num_cus() / N_XCD * N_XCD, 64 * PS_D); }

struct PsAdmit {
  static Budget &budget() {
    static Budget b(num_cus() / N_XCD);
    return b;
  }
  const int units;
  const bool in;
  explicit PsAdmit(int G) : units((G + N_XCD - 1) / N_XCD), in(budget().take(units)) {}
  ~PsAdmit() {
    if (in) budget().give(units);
  }
};

// LDS of a workgroup's operator rows: its capacities in a, its bytes returned.
// The rows' nonzeros with a quarter to spare (more than the room allows is
// caught in the kernel), up to 4 remote entries per row in what they leave, a
// quarter at least, and in the same memory at set-up two bits per column of
// their span.
template <typename T, int Q>
size_t ps_lds(PsArgs<T> &a, size_t room, double nz_per_row, int64_t n) {
  constexpr int R = 64 * Q;
  const size_t nz = (size_t)(1.25 * nz_per_row * R) + 64;
  const size_t left = room - std::min(nz * (sizeof(T) + 2), room - room / 4);
  a.hcap = (int)std::min({(size_t)4 * R, (size_t)4096, left / (sizeof(T) + 4)}) & ~1;
  const size_t rest = room - (size_t)a.hcap * (sizeof(T) + 4);
  a.nzcap = (int)(std::min(nz, rest / (sizeof(T) + 2)) & ~(size_t)1);
  const size_t span = ((size_t)n + 31) / 32 * 32;
  a.wcap = (int)(std::min(span, (size_t)(a.nzcap + a.hcap) * sizeof(T) * 4) / 32 * 32);
  return (size_t)a.nzcap * (sizeof(T) + 2) + (size_t)a.hcap * (sizeof(T) + 4);
}

// What the LDS leaves beside a kernel's static arrays, made available to it.
template <typename T, int Q, typename K>
int ps_room(K *kern, std::once_flag &once, hipError_t &err, size_t *room) {
  constexpr int R = 64 * Q;
  constexpr size_t fixed = sizeof(T) * (2 + PS_W) * R + 8 * GS_MAXC + 4 * (R + 1) + 1024;   // static LDS and slack
  *room = (size_t)lds_max_bytes() - fixed;
  std::call_once(once, [&] {
    err = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)*room);
  });
  SA_HIP(err);
  return 0;
}

template <typename T, int S, int Q>
int ps_go(BV &V, const Mat *A, PsArgs<T> &a, hipStream_t s) {
  constexpr int R = 64 * Q;
  auto *kern = ps_sweep_kernel<T, S, Q>;
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  size_t room, shm = 0;
  SA_TRY((ps_room<T, Q>(kern, once, err, &room)));
  if (A) shm = ps_lds<T, Q>(a, room, (double)A->nnz / (double)std::max(1, A->n), V.n);
  a.G = (int)((V.n + R - 1) / R);
  a.host->ok = a.host->fail = 0;
  PsAdmit admit(a.G);
  if (!admit.in) return 0;
  hipLaunchKernelGGL(kern, dim3(a.G), dim3(PS_T), shm, s, a);
  SA_HIP(hipGetLastError());
  SA_HIP(hipStreamSynchronize(s));
  return 0;
}

template <typename T, int S>
int ps_rows(BV &V, const Mat *A, PsArgs<T> &a, int q, hipStream_t s) {
  constexpr int M = sizeof(T) == 8 ? 88 : 176;     // as in ps_pick
  if constexpr (S * 22 <= M) if (q == 22) return ps_go<T, S, 22>(V, A, a, s);
  if constexpr (S * 16 <= M) if (q == 16) return ps_go<T, S, 16>(V, A, a, s);
  if constexpr (S * 11 <= M) if (q == 11) return ps_go<T, S, 11>(V, A, a, s);
  if constexpr (S * 8 <= M) if (q == 8) return ps_go<T, S, 8>(V, A, a, s);
  if constexpr (S * 6 <= M) if (q == 6) return ps_go<T, S, 6>(V, A, a, s);
  if (q == 4) return ps_go<T, S, 4>(V, A, a, s);
  if (q == 2) return ps_go<T, S, 2>(V, A, a, s);
  return ps_go<T, S, 1>(V, A, a, s);
}

// 64-row chunks per workgroup for n rows and S column slots, 0 when the basis
// does not fit.  A thread keeps S * Q values: at most 88 doubles or 176 floats
// (the largest spill up to 136 B per lane and still take 0.4 of the slots'
// time).  Up to 64 workgroups, or 4 chunks each, more rows per workgroup cost
// nothing (n = 10,000: 198, 200, 198 us with 1, 2, 4 chunks) and leave CUs to
// the sweeps of other threads; beyond that as few rows as the CUs allow.  When
// the application runs several solves at once (share), half the CUs if they
// hold the basis: two sweeps then run side by side, each 6% longer (eight
// 256x256 family solves on 8 threads: 110 eigenpairs/s on all CUs, 166 on half
// of them, 121 on a quarter; on 4 threads 117, 191, 147).
template <typename T>
int ps_pick(int64_t n, int S, int share) {
  constexpr int M = sizeof(T) == 8 ? 88 : 176;
  const int most = ps_most();
  for (int want : {share >= 2 ? std::max(64, most / 2) : most, most})
    for (int q : {1, 2, 4, 6, 8, 11, 16, 22}) {
      const int64_t G = (n + 64 * q - 1) / (64 * q);
      if (S * q <= M && G <= want && (G <= 64 || q >= 4)) return q;
    }
  return 0;
}

// Polls before a wait gives up: about half a second, or SLEPC_AMD_SWEEP_POLLS
// (0: at the first poll without success, so that sweeps of more than one
// workgroup run by slots).
int ps_polls() {
  static const int v = [] {
    const char *e = std::getenv("SLEPC_AMD_SWEEP_POLLS");
    const int k = e ? std::atoi(e) : -1;
    return k < 0 ? 1 << 19 : std::min(k, 1 << 19);
  }();
  return v;
}

template <typename T>
int ps_run(BV &V, const Mat *A, int c0, int c1, double eta, hipStream_t s, bool *done) {
  const int S = c1 <= 32 ? 4 : (c1 <= 64 ? 8 : (c1 <= 96 ? 12 : 16));
  const int q = ps_pick<T>(V.n, S, V.ps.share);
  if (!q || !V.ps.backoff.due()) return 0;
  PsArgs<T> a{};
  a.n0 = 0; a.n1 = a.xn = V.n; a.ld = V.ld; a.V = static_cast<T *>(V.data);
  if (A) { a.rp = A->rowptr; a.ci = A->col; a.val = static_cast<const T *>(A->val); }
  a.c0 = c0; a.c1 = c1;
  a.xw = V.ps.words;
  a.pw = a.xw + (sizeof(T) / 4) * V.n;
  a.tw = a.pw + (size_t)2 * GS_MAXC * num_cus();
  a.abort_word = reinterpret_cast<unsigned int *>(a.tw + 2 * PS_COPIES * GS_MAXC);
  a.backup = reinterpret_cast<T *>(a.tw + 2 * PS_COPIES * GS_MAXC + 1);
  // at most 4 reductions per column (three passes and a measured norm); 0 is
  // the number that fresh words carry
  const uint32_t most = 4u * (uint32_t)(c1 - c0 + 1) + 2u;
  if (V.ps.tag > 0xffffffffu - most) {
    SA_HIP(hipMemsetAsync(V.ps.words, 0, V.ps.bytes, s));
    V.ps.tag = 1;
  }
  a.base = V.ps.tag;
  V.ps.tag += most;
  a.st = V.st; a.host = reinterpret_cast<GsMirror *>(V.st_host); a.dbuf = V.dbuf; a.dm = V.m; a.eta = eta; a.refine = V.refine;
  a.polls = ps_polls();
  const int64_t passes = a.host->st.passes_total;   // the mirror is the state after every column or sweep
  int rc;
  switch (S) {
    case 4: rc = ps_rows<T, 4>(V, A, a, q, s); break;
    case 8: rc = ps_rows<T, 8>(V, A, a, q, s); break;
    case 12: rc = ps_rows<T, 12>(V, A, a, q, s); break;
    default: rc = ps_rows<T, 16>(V, A, a, q, s); break;
  }
  SA_TRY(rc);
  *done = a.host->ok && !a.host->fail;
  if (*done) {
    V.ps.tally.resident++;
    V.ps.backoff.succeeded();
  } else if (a.host->fail) {
    V.ps.tally.gave_up++;
    V.ps.backoff.failed();
    if (a.host->ok) {   // the lead finished, another did not: the slots count these passes again
      a.host->st.passes_total = passes;
      SA_HIP(hipMemcpyAsync(V.st + 2, &a.host->st, sizeof(GsState), hipMemcpyHostToDevice, s));
    }
  }
  if (a.host->fail && !A)   // the vector as it was, for the slots
    SA_HIP(hipMemcpyAsync(a.V + (size_t)c0 * a.ld, a.backup, sizeof(T) * V.n, hipMemcpyDeviceToDevice, s));
  return 0;
}

// ---- several problems at once -------------------------------------------------
template <typename T, int S, int Q>
int psb_go(const PsBatch &w, PsArgs<T> &a, int blocks, double nz_per_row, hipStream_t s) {
  auto *kern = ps_batch_kernel<T, S, Q>;
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  size_t room;
  SA_TRY((ps_room<T, Q>(kern, once, err, &room)));
  const size_t shm = ps_lds<T, Q>(a, room, nz_per_row, a.xn);
  PsAdmit admit(blocks);
  if (!admit.in) {
    w.fail->fail = 1;
    return 0;
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(PS_T), shm, s, a, (const PsProb *)w.probs, (const int *)w.of_block);
  SA_HIP(hipGetLastError());
  SA_HIP(hipStreamSynchronize(s));
  return 0;
}

template <typename T, int S>
int psb_rows(const PsBatch &w, PsArgs<T> &a, int q, int blocks, double nz, hipStream_t s) {
  constexpr int M = sizeof(T) == 8 ? 88 : 176;
  if constexpr (S * 22 <= M) if (q == 22) return psb_go<T, S, 22>(w, a, blocks, nz, s);
  if constexpr (S * 16 <= M) if (q == 16) return psb_go<T, S, 16>(w, a, blocks, nz, s);
  if constexpr (S * 11 <= M) if (q == 11) return psb_go<T, S, 11>(w, a, blocks, nz, s);
  if (q == 8) return psb_go<T, S, 8>(w, a, blocks, nz, s);
  return psb_go<T, S, 4>(w, a, blocks, nz, s);
}

template <typename T>
int psb_run(PsBatch &w, PsArgs<T> &a, std::vector<PsProb> &pr, double nz_per_row, hipStream_t s, bool *done) {
  constexpr int M = sizeof(T) == 8 ? 88 : 176;
  const int most = ps_most();
  int c1 = 0, len = 0;
  int64_t nmax = 0;
  for (const PsProb &p : pr) {
    if (p.n1 <= p.n0 || p.c1 < p.c0) return 0;
    c1 = std::max(c1, p.c1);
    len = std::max(len, p.c1 - p.c0 + 1);
    nmax = std::max(nmax, p.n1 - p.n0);
  }
  if (c1 > 64) return 0;
  const int S = c1 <= 32 ? 4 : 8;
  // as few rows per workgroup as lets all problems run in one launch; when
  // none does, the most, and as many launches as that takes
  int q = 0;
  for (int t : {4, 8, 11, 16, 22}) {
    if (S * t > M) break;
    q = t;
    int64_t total = 0;
    for (const PsProb &p : pr) total += (p.n1 - p.n0 + 64 * q - 1) / (64 * q);
    if (total <= most) break;
  }
  if ((nmax + 64 * q - 1) / (64 * q) > most || !w.backoff.due()) return 0;
  const uint32_t tags = 4u * (uint32_t)len + 2u;
  *w.fail = GsMirror{};
  for (size_t i0 = 0; i0 < pr.size();) {
    int blocks = 0;
    size_t i1 = i0;
    std::vector<int> of_block;
    for (; i1 < pr.size(); i1++) {
      PsProb &p = pr[i1];
      p.G = (int)((p.n1 - p.n0 + 64 * q - 1) / (64 * q));
      if (blocks + p.G > most) break;
      p.b0 = blocks;
      blocks += p.G;
      of_block.insert(of_block.end(), p.G, (int)(i1 - i0));
    }
    if (w.tag > 0xffffffffu - tags) {
      SA_HIP(hipMemsetAsync(w.words, 0, w.bytes, s));
      w.tag = 1;
    }
    a.base = w.tag;
    w.tag += tags;
    // the copies have read their source when the launch below has been awaited
    SA_HIP(hipMemcpyAsync(w.probs, pr.data() + i0, sizeof(PsProb) * (i1 - i0), hipMemcpyHostToDevice, s));
    SA_HIP(hipMemcpyAsync(w.of_block, of_block.data(), sizeof(int) * blocks, hipMemcpyHostToDevice, s));
    SA_TRY((S == 4 ? psb_rows<T, 4>(w, a, q, blocks, nz_per_row, s) : psb_rows<T, 8>(w, a, q, blocks, nz_per_row, s)));
    if (w.fail->fail) {
      w.tally.gave_up++;
      w.backoff.failed();
      return 0;
    }
    i0 = i1;
  }
  *done = true;
  w.tally.resident++;
  w.backoff.succeeded();
  return 0;
}

}  // namespace

size_t ps_bytes(int64_t n, int prec) {
  const size_t es = prec_size(prec);
  if (n == 0 || n > (int64_t)num_cus() * 64 * (prec == SA_FP64 ? 16 : 22)) return 0;
  return 8 * ((es / 4) * (size_t)n + (size_t)2 * GS_MAXC * num_cus() + 2 * PS_COPIES * GS_MAXC + 1) + es * (size_t)n;
}

int ps_sweep(BV &V, const Mat *A, int c0, int c1, double eta, hipStream_t s, bool *done) {
  *done = false;
  const int64_t gave_up = V.ps.tally.gave_up;
  if (V.ps.words && c1 < GS_MAXC)
    SA_TRY((V.prec == SA_FP64 ? ps_run<double>(V, A, c0, c1, eta, s, done) : ps_run<float>(V, A, c0, c1, eta, s, done)));
  V.ps.tally.slots += !*done && V.ps.tally.gave_up == gave_up;
  return 0;
}

void ps_batch_free(PsBatch &w) {
  if (w.words) (void)hipFree(w.words);
  if (w.probs) (void)hipFree(w.probs);
  if (w.of_block) (void)hipFree(w.of_block);
  if (w.fail) (void)hipHostFree(w.fail);
  const SweepTally t = w.tally;
  w = PsBatch();
  w.tally = t;
}

bool ps_batch_alloc(PsBatch &w, int64_t nrows, int prec, int P, hipStream_t s) {
  if (w.words) return true;
  // a launch has at most num_cus() workgroups, so no more problems
  const int most = std::min(P, num_cus());
  w.pw = (prec_size(prec) / 4) * (size_t)nrows;
  w.tw = w.pw + (size_t)2 * GS_MAXC * num_cus();
  w.abort_word = w.tw + (size_t)2 * PS_COPIES * GS_MAXC * most;
  w.bytes = 8 * (w.abort_word + 1);
  if (hipMalloc((void **)&w.words, w.bytes) != hipSuccess ||
      hipMalloc((void **)&w.probs, sizeof(PsProb) * most) != hipSuccess ||
      hipMalloc((void **)&w.of_block, sizeof(int) * num_cus()) != hipSuccess ||
      hipHostMalloc((void **)&w.fail, sizeof(GsMirror)) != hipSuccess ||
      hipMemsetAsync(w.words, 0, w.bytes, s) != hipSuccess) {
    (void)hipGetLastError();
    ps_batch_free(w);
    return false;
  }
  w.tag = 1;
  return true;
}

int ps_batch_sweep(PsBatch &w, int prec, void *V, int64_t ld, int64_t nrows, const int32_t *rp, const int32_t *ci,
                   const void *val, int64_t nnz, std::vector<PsProb> &pr, GsState *st, double *dbuf, int m, double eta,
                   hipStream_t s, bool *done) {
  *done = false;
  const double nz = nrows ? (double)nnz / (double)nrows : 0.0;
  auto run = [&](auto zero) {
    using T = decltype(zero);
    PsArgs<T> a{};
    a.xn = nrows; a.ld = ld; a.V = static_cast<T *>(V);
    a.rp = rp; a.ci = ci; a.val = static_cast<const T *>(val);
    a.xw = w.words; a.pw = w.words + w.pw; a.tw = w.words + w.tw;
    a.abort_word = reinterpret_cast<unsigned int *>(w.words + w.abort_word);
    a.st = st; a.host = w.fail; a.dbuf = dbuf; a.dm = m; a.eta = eta; a.refine = GS_REFINE_IFNEEDED;
    a.polls = ps_polls();
    return psb_run<T>(w, a, pr, nz, s, done);
  };
  return prec == SA_FP64 ? run(0.0) : run(0.0f);
}

}  // namespace sa
