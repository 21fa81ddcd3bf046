// Gram-Schmidt step of the Arnoldi/Lanczos sweep on one basis, for gfx950
// (MI355X): the host launch sequence of the three slot kernels (sa_gw.hip) and
// the per-column reductions between them.  Bases that fit the GPU's registers
// take the resident sweep (sa_sweep.hip) instead.  Every decision of the reference's rules
// (bvorthog.c:91-217, 380-427) is taken on the device.
#include <algorithm>

#include "sa_gs_device.h"

namespace sa {

// Reduction of a slot's partial sums before the next slot: one workgroup per
// column.  It runs even when the slot produced no dot products (the next slot
// then ignores them), which saves the round trip of reading the state first.
__global__ __launch_bounds__(BLK) void gs_sum_kernel(const double *part, int G, double *dots) {
  gs_sum_column(part, G, (int)blockIdx.x, dots);
}

__global__ void gs_reset_kernel(GsState *st) {
  if (threadIdx.x == 0) {
    GsState S = st[2];
    S.stop = 0; S.stop_col = 0; S.pending = 0; S.lindep = 0; S.pass = 0;
    S.done = 0; S.dots_ready = 0; S.beta = 0.0;
    st[2] = S;
  }
}

// The three slots of column c and the reductions between them.  The SpMV is a
// kernel of its own ahead of slot 1: fused into a slot it gathers row by row
// with every workgroup of the slot waiting for it.  After a breakdown neither
// it nor the slots write a column.
template <typename T>
static int gs_launch(BV &V, const Mat *A, int c, double eta, hipStream_t s) {
  GsArgs<T> a{};
  a.n = V.n; a.ld = V.ld; a.V = static_cast<T *>(V.data); a.c = c;
  a.st = V.st; a.dbuf = V.dbuf; a.m = V.m; a.eta = eta;
  a.refine = V.refine;
  a.G = std::min(V.ws.maxG, gw_blocks(V.n, V.prec, c));
  const bool nt = (int64_t)V.ld * V.m * (int64_t)sizeof(T) > GS_NT_BYTES;
  double *pa = V.ws.part, *pb = V.ws.part + (size_t)V.ws.maxG * (GS_MAXC + 1);
  double *da = V.ws.dots, *db = V.ws.dots + (GS_MAXC + 1);
  if (A) SA_TRY(launch_spmv(*A, a.V + (size_t)(c - 1) * a.ld, a.V + (size_t)c * a.ld, s, &V.st[2].stop));
  for (int slot = 1; slot <= 3; slot++) {
    a.slot = slot;
    a.part_out = slot == 1 ? pa : pb;
    a.dots_in = slot == 2 ? da : db;
    SA_TRY(launch_gw_slot(a, nt, s));
    if (slot < 3)
      hipLaunchKernelGGL(gs_sum_kernel, dim3(c + 1), dim3(BLK), 0, s, (const double *)a.part_out, a.G,
                         slot == 1 ? da : db);
  }
  SA_HIP(hipGetLastError());
  return 0;
}

int launch_gs_column(BV &V, const Mat *A, int c, double eta, hipStream_t s) {
  SA_CHECK(c >= 0 && c < GS_MAXC && c < V.m, "column index out of range for the Gram-Schmidt kernel");
  SA_CHECK(!A || (A->prec == V.prec && A->n == V.n), "matrix and basis sizes or precisions differ");
  SA_CHECK(!A || c > 0, "SpMV step needs a previous column");
  if (V.prec == SA_FP64) return gs_launch<double>(V, A, c, eta, s);
  return gs_launch<float>(V, A, c, eta, s);
}

int launch_gs_reset(BV &V, hipStream_t s) {
  hipLaunchKernelGGL(gs_reset_kernel, dim3(1), dim3(64), 0, s, V.st);
  SA_HIP(hipGetLastError());
  return 0;
}

}  // namespace sa
