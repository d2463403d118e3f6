// Kernels of the adjoint (transposed) evaluate pass, FP64 (its near field and the
// field pass: kernels_near64.hip).  In the adjoint every block is the forward kernel block K(target - source;
// source normal) contracted over the target DOF instead of the source DOF, so
// the pass is the exact transpose of the forward operator whatever the
// kernel's symmetry.  No rounding-order contract applies (FMA contraction on).
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace kifmm {

// ---------------------------------------------------------------------------
// Equivalent surface <- targets (adjoint of M2T into UE and of L2T into DE):
// out(node)[q] += sum_t K_mm(t - y_q)^T w(t); one workgroup per task, each lane
// owns up to two surface samples.
// ---------------------------------------------------------------------------
constexpr int kSurfT = 256;

template <int KM>
__global__ __launch_bounds__(kSurfT) void k_surf_t(SurfTArgs a, KParams<double> pm) {
  constexpr int sd = src_dof(KM), td = trg_dof(KM);
  __shared__ double sp[kSurfT * 3];
  __shared__ double sv[kSurfT * td];
  const SurfTask tk = a.tasks[blockIdx.x];
  const double4 g = a.geom[tk.node];
  const int lane = threadIdx.x;
  double yp[2][3];
  double acc[2][sd];
  bool act[2];
  for (int u = 0; u < 2; u++) {
    const int q = lane + u * kSurfT;
    act[u] = q < a.n_sam;
    const int qq = act[u] ? q : 0;
    yp[u][0] = g.x + g.w * a.sam[3 * qq];
    yp[u][1] = g.y + g.w * a.sam[3 * qq + 1];
    yp[u][2] = g.z + g.w * a.sam[3 * qq + 2];
    for (int s = 0; s < sd; s++) acc[u][s] = 0.0;
  }
  for (int it = tk.ibeg; it < tk.iend; it++) {
    const int leaf = a.items[it];
    const int b = a.trg_beg[leaf], nt = a.trg_num[leaf];
    for (int base = 0; base < nt; base += kSurfT) {
      const int m = min(kSurfT, nt - base);
      __syncthreads();
      if (lane < m) {
        const int64_t q = int64_t(b + base + lane);
        for (int d = 0; d < 3; d++) sp[3 * lane + d] = a.tpos[3 * q + d];
        for (int t = 0; t < td; t++) sv[lane * td + t] = a.tw[q * td + t];
      }
      __syncthreads();
      for (int j = 0; j < m; j++) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
          if (!act[u]) continue;
          double blk[sd * td];
          kblock<KM, double>(pm, sp[3 * j] - yp[u][0], sp[3 * j + 1] - yp[u][1], sp[3 * j + 2] - yp[u][2], 0.0,
                             0.0, 0.0, blk);
#pragma unroll
          for (int t = 0; t < td; t++)
#pragma unroll
            for (int s = 0; s < sd; s++) acc[u][s] += blk[t * sd + s] * sv[j * td + t];
        }
      }
    }
  }
  double* o = a.out + int64_t(tk.node) * a.sz_out;
  for (int u = 0; u < 2; u++) {
    if (!act[u]) continue;
    const int q = lane + u * kSurfT;
    for (int s = 0; s < sd; s++) o[q * sd + s] += acc[u][s];
  }
}

hipError_t launch_surface_adjoint(int km, const SurfTArgs& a, const KParams<double>& pm, hipStream_t s) {
  if (a.ntasks <= 0) return hipSuccess;
  if (a.n_sam > 2 * kSurfT) return hipErrorInvalidValue;
  switch (km) {
    case 111: k_surf_t<111><<<dim3(unsigned(a.ntasks)), dim3(kSurfT), 0, s>>>(a, pm); break;
    case 301: k_surf_t<301><<<dim3(unsigned(a.ntasks)), dim3(kSurfT), 0, s>>>(a, pm); break;
    case 511: k_surf_t<511><<<dim3(unsigned(a.ntasks)), dim3(kSurfT), 0, s>>>(a, pm); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace kifmm
