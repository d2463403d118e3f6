// HIP kernels of the FP64 evaluate pass for gfx950 (CDNA4, wave64).
//
// Phase -> kernel:
//   load densities (fmm3d_eval_mpi.cpp:443-461)           k_gather
//   S2M (:577) / X-list S2L (:1253)                       k_surface
//   M2M, UC->UE, L2L, DC->DE (:583-592, :1371-1382)       k_gemm (level-batched, indexed columns)
//   V-list (:1007-1059)                                   k_fft_fwd, k_had_scalar, k_had_vec, k_fft_inv
//   U-list S2T, W-list S2T/M2T, X-list S2T, L2T
//     (:773-785, :1146-1165, :1249, :1383-1435)            kernels_near64.hip
//   write back (:1490-1510)                               k_scatter
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "device.hpp"
#include "gemm.hpp"
#include "hadamard.hpp"
#include "pair64.hpp"

namespace kifmm {

// ---------------------------------------------------------------------------
__global__ void k_gather(const double* __restrict__ in, const int* __restrict__ perm,
                         double* __restrict__ out, int64_t n, int dof) {
  int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= n) return;
  int64_t o = perm[k];
  for (int d = 0; d < dof; d++) out[k * dof + d] = in[o * dof + d];
}

__global__ void k_scatter(const double* __restrict__ in, const int* __restrict__ perm,
                          double* __restrict__ out, int64_t n, int dof) {
  int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= n) return;
  int64_t o = perm[k];
  for (int d = 0; d < dof; d++) out[o * dof + d] = in[k * dof + d];
}

// Densities of nrhs right-hand sides, caller's layout [r][k][dof] -> leaf order
// [sinv[k]][r][dof] (the right-hand sides of a source side by side).
__global__ void k_load_rhs(const double* __restrict__ in, const int* __restrict__ sinv, double* __restrict__ out,
                           int64_t n, int dof, int nrhs) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n * nrhs) return;
  const int64_t r = i / n, k = i % n, o = sinv[k];
  for (int d = 0; d < dof; d++) out[(o * nrhs + r) * dof + d] = in[i * dof + d];
}

// Values of nrhs right-hand sides, leaf order [r][k][dof] -> caller's [r][perm[k]][dof].
__global__ void k_store_rhs(const double* __restrict__ in, const int* __restrict__ perm, double* __restrict__ out,
                            int64_t n, int dof, int nrhs) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n * nrhs) return;
  const int64_t r = i / n, k = i % n, o = r * n + perm[k];
  for (int d = 0; d < dof; d++) out[o * dof + d] = in[i * dof + d];
}

// Up to kZeroRanges buffers in one launch (four launches of about 2.3 us each, and
// their gaps, in front of every pass before: 9 of a 4,000-point pass's 132 us).
__global__ void k_zero_ranges(ZeroRanges z) {
  double* p = z.p[blockIdx.y];
  const int64_t n = z.n[blockIdx.y];
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
    p[i] = 0.0;
}

hipError_t launch_gather(const double* in, const int* perm, double* out, int64_t n, int dof, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_gather<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(in, perm, out, n, dof);
  return hipGetLastError();
}
hipError_t launch_scatter(const double* in, const int* perm, double* out, int64_t n, int dof, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_scatter<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(in, perm, out, n, dof);
  return hipGetLastError();
}
hipError_t launch_load_rhs(const double* in, const int* sinv, double* out, int64_t n, int dof, int nrhs,
                           hipStream_t s) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  k_load_rhs<<<dim3(unsigned((n * nrhs + 255) / 256)), dim3(256), 0, s>>>(in, sinv, out, n, dof, nrhs);
  return hipGetLastError();
}
hipError_t launch_store_rhs(const double* in, const int* perm, double* out, int64_t n, int dof, int nrhs,
                            hipStream_t s) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  k_store_rhs<<<dim3(unsigned((n * nrhs + 255) / 256)), dim3(256), 0, s>>>(in, perm, out, n, dof, nrhs);
  return hipGetLastError();
}
// One thread per (row, right-hand side, column); 16-byte stores when the row
// length is even (rows of 8-byte-aligned length: 152, 296, ...).
__global__ void k_zero_rows(double* base, const int* rows, int nrows, int len, int nrhs, int64_t nstride) {
  const int half = len / 2;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(nrows) * nrhs * half) return;
  const int col = int(i % half);
  const int64_t kr = i / half;
  const int k = int(kr % nrows), r = int(kr / nrows);
  double* row = base + (int64_t(rows[k]) + r * nstride) * len;
  reinterpret_cast<double2*>(row)[col] = make_double2(0.0, 0.0);
}
__global__ void k_zero_rows_odd(double* base, const int* rows, int nrows, int len, int nrhs, int64_t nstride) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(nrows) * nrhs * len) return;
  const int col = int(i % len);
  const int64_t kr = i / len;
  const int k = int(kr % nrows), r = int(kr / nrows);
  base[(int64_t(rows[k]) + r * nstride) * len + col] = 0.0;
}
hipError_t launch_zero_rows(double* base, const int* rows, int nrows, int len, int nrhs, int64_t nstride,
                            hipStream_t s) {
  if (nrows <= 0 || nrhs <= 0 || len <= 0) return hipSuccess;
  if (len % 2 == 0) {
    const int64_t n = int64_t(nrows) * nrhs * (len / 2);
    k_zero_rows<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(base, rows, nrows, len, nrhs, nstride);
  } else {
    const int64_t n = int64_t(nrows) * nrhs * len;
    k_zero_rows_odd<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(base, rows, nrows, len, nrhs, nstride);
  }
  return hipGetLastError();
}

hipError_t launch_zero_ranges(const ZeroRanges& z, hipStream_t s) {
  int64_t n = 0;
  for (int k = 0; k < kZeroRanges; k++) n = std::max(n, z.n[k]);
  if (n <= 0) return hipSuccess;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 16384);
  k_zero_ranges<<<dim3(unsigned(blocks), kZeroRanges), dim3(256), 0, s>>>(z);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Exact sources -> check surface of a node (S2M into UC, S2L into DC).
// One workgroup per task; each lane owns up to two surface points.
// ---------------------------------------------------------------------------
constexpr int kSurfThreads = 256;

template <int KT, int NR>
__global__ __launch_bounds__(kSurfThreads) void k_surface(SurfArgs a, KParams<double> pu) {
  constexpr int SD = src_dof(KT), TD = trg_dof(KT);
  __shared__ double sp[kSurfThreads * 3];
  __shared__ double sn[kSurfThreads * 3];
  __shared__ double sv[kSurfThreads * SD * NR];
  const SurfTask tk = a.tasks[blockIdx.x];
  const double4 g = a.geom[tk.node];
  const int lane = threadIdx.x;
  const int64_t rstep = a.nstride * a.sz_out;
  double tp[2][3];
  double acc[2][NR][TD];
  bool act[2];
  for (int u = 0; u < 2; u++) {
    const int q = lane + u * kSurfThreads;
    act[u] = q < a.n_sam;
    const int qq = act[u] ? q : 0;
    tp[u][0] = g.x + g.w * a.sam[3 * qq];
    tp[u][1] = g.y + g.w * a.sam[3 * qq + 1];
    tp[u][2] = g.z + g.w * a.sam[3 * qq + 2];
    // start from the current check value and add term by term (dgemv order)
#pragma unroll
    for (int r = 0; r < NR; r++)
      for (int t = 0; t < TD; t++)
        acc[u][r][t] = act[u] && r < a.nr
                           ? a.out[(a.r0 + r) * rstep + int64_t(tk.node) * a.sz_out + q * TD + t] : 0.0;
  }
  for (int it = tk.ibeg; it < tk.iend; it++) {
    const int node = a.items[it];
    const int b = a.src_beg[node], ns = a.src_num[node];
    for (int base = 0; base < ns; base += kSurfThreads) {
      const int m = min(kSurfThreads, ns - base);
      __syncthreads();
      if (lane < m) {
        const int64_t gg = int64_t(b + base + lane);
        for (int d = 0; d < 3; d++) { sp[3 * lane + d] = a.spos[3 * gg + d]; sn[3 * lane + d] = a.snor[3 * gg + d]; }
#pragma unroll
        for (int r = 0; r < NR; r++)
          for (int s = 0; s < SD; s++)
            sv[(lane * NR + r) * SD + s] = r < a.nr ? a.sden[(gg * a.nrhs + a.r0 + r) * SD + s] : 0.0;
      }
      __syncthreads();
      for (int j = 0; j < m; j++) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
          if (!act[u]) continue;
          double blk[SD * TD];
          kblock<KT, double>(pu, tp[u][0] - sp[3 * j], tp[u][1] - sp[3 * j + 1], tp[u][2] - sp[3 * j + 2],
                             sn[3 * j], sn[3 * j + 1], sn[3 * j + 2], blk);
#pragma unroll
          for (int r = 0; r < NR; r++)
#pragma unroll
            for (int t = 0; t < TD; t++)
#pragma unroll
              for (int s = 0; s < SD; s++) acc[u][r][t] += blk[t * SD + s] * sv[(j * NR + r) * SD + s];
        }
      }
    }
  }
  for (int u = 0; u < 2; u++) {
    if (!act[u]) continue;
    const int q = lane + u * kSurfThreads;
#pragma unroll
    for (int r = 0; r < NR; r++) {
      if (r >= a.nr) continue;
      double* o = a.out + (a.r0 + r) * rstep + int64_t(tk.node) * a.sz_out;
      for (int t = 0; t < TD; t++) o[q * TD + t] = acc[u][r][t];
    }
  }
}

// ---------------------------------------------------------------------------
// Level-batched translations and pseudo-inverse applies: see gemm.hpp.
hipError_t launch_gemm(const GemmArgs& g, hipStream_t s) { return launch_gemm_seq(g, s); }

// ---------------------------------------------------------------------------
// V list.  Forward: UE samples (scaled 2^(l*deg)) scattered onto the (2np)^3
// grid and transformed (r2c, FFTW layout).  Only the np^3 block at offset np/2
// is non-zero, so the three DFT passes run over that block.  One wave per
// node; each lane transforms whole lines, and since the twiddle exponent of
// input x and output k is ((x + np/2) k) mod n with x and k unrolled at compile
// time (NP is a template parameter), the n twiddles sit in registers.  Every
// output is summed over its inputs in ascending order, as the separable DFT of
// the reference layout does.
// ---------------------------------------------------------------------------
constexpr int kMaxNp = 8;

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// 3- and 6-point DFTs, X[k] = sum_n x[n] exp(SGN 2 pi i n k / N) (SGN = -1:
// forward, +1: inverse).  Three points: t1 = b + c, t2 = a - t1/2,
// r = SGN i (sqrt(3)/2)(b - c); X = (a + t1, t2 + r, t2 - r).  Six points: radix 2
// over two 3-point transforms of the even and odd samples with twiddles
// w6^k = exp(SGN 2 pi i k / 6), X[k] = E[k] + w6^k D[k], X[k+3] = E[k] - w6^k D[k].
template <int SGN>
__device__ inline void dft3(double2 a, double2 b, double2 c, double2& X0, double2& X1, double2& X2) {
  constexpr double kS = 0.86602540378443864676;
  const double2 t1 = cadd(b, c);
  const double2 t2 = make_double2(a.x - 0.5 * t1.x, a.y - 0.5 * t1.y);
  const double2 d = csub(b, c);
  const double2 r = make_double2(-SGN * kS * d.y, SGN * kS * d.x);
  X0 = cadd(a, t1);
  X1 = cadd(t2, r);
  X2 = csub(t2, r);
}
template <int SGN>
__device__ inline void dft6(const double2 (&x)[6], double2 (&X)[6]) {
  constexpr double kS = 0.86602540378443864676;
  double2 E[3], D[3];
  dft3<SGN>(x[0], x[2], x[4], E[0], E[1], E[2]);
  dft3<SGN>(x[1], x[3], x[5], D[0], D[1], D[2]);
  const double2 t1 = cmul(make_double2(0.5, SGN * kS), D[1]);
  const double2 t2 = cmul(make_double2(-0.5, SGN * kS), D[2]);
  X[0] = cadd(E[0], D[0]); X[3] = csub(E[0], D[0]);
  X[1] = cadd(E[1], t1);   X[4] = csub(E[1], t1);
  X[2] = cadd(E[2], t2);   X[5] = csub(E[2], t2);
}
// Mixed path, np = 6.  Forward line transform from the 6 block samples at grid
// positions b + 3 to the 12 frequencies: out[k] = sum_b in[b] w^((b+3) k); the
// even outputs are the 6-point DFT of the samples placed at (b + 3) mod 6, the
// odd outputs the same of in[b] w^(b+3).  w: the 12 forward twiddles.
__device__ inline void pad12_fwd(const double2 (&in)[6], const double2 (&w)[12], double2 (&out)[12]) {
  double2 e[6], o[6], E[6], D[6];
#pragma unroll
  for (int b = 0; b < 6; b++) {
    const int p = (b + 3) % 6;
    e[p] = in[b];
    o[p] = cmul(in[b], w[(b + 3) % 12]);
  }
  dft6<-1>(e, E);
  dft6<-1>(o, D);
#pragma unroll
  for (int m = 0; m < 6; m++) { out[2 * m] = E[m]; out[2 * m + 1] = D[m]; }
}
// Inverse line transform from 12 frequencies to the 6 block positions a + 3:
// out[a] = sum_k in[k] wi^((a+3) k) = E[j] + wi^(a+3) D[j], j = (a + 3) mod 6,
// with E, D the 6-point inverse DFTs of the even and odd frequencies.
__device__ inline void pad12_inv(const double2 (&in)[12], const double2 (&wi)[12], double2 (&out)[6]) {
  double2 e[6], o[6], E[6], D[6];
#pragma unroll
  for (int m = 0; m < 6; m++) { e[m] = in[2 * m]; o[m] = in[2 * m + 1]; }
  dft6<1>(e, E);
  dft6<1>(o, D);
#pragma unroll
  for (int a = 0; a < 6; a++) out[a] = cadd(E[(a + 3) % 6], cmul(wi[(a + 3) % 12], D[(a + 3) % 6]));
}

__device__ inline void store_c(double2* p, double2 v) { *p = v; }
__device__ inline void store_c(float2* p, double2 v) { *p = make_float2(float(v.x), float(v.y)); }
__device__ inline double2 load_c(const double2* p) { return *p; }
__device__ inline double2 load_c(const float2* p) { const float2 v = *p; return make_double2(v.x, v.y); }

// C2 = storage type of the spectra (double2, or float2 for the mixed path).
template <int NP, typename C2>
__global__ __launch_bounds__(64) void k_fft_fwd(VlistArgs v, C2* dspec) {
  constexpr int N = 2 * NP, HH = NP + 1, O = NP / 2;
  // mixed path at np = 6: the y and z line transforms by two 6-point DFTs
  // (the FP64 path keeps the ascending-order sums of the reference layout)
  constexpr bool kFast = NP == 6 && std::is_same<C2, float2>::value;
  // mixed path: packed half spectrum (spec_pack), the FP64 path the full r2c
  // layout (ka n + kb) h + kc
  constexpr bool kPack = std::is_same<C2, float2>::value;
  constexpr int HS = kPack ? spec_packed_len(NP) : N * N * HH;
  constexpr int NSAM = NP * NP * NP - (NP - 2) * (NP - 2) * (NP - 2);
  // mixed path: the line results between passes are kept in LDS as FP32 (the
  // spectra are stored in FP32 anyway), which halves the LDS of a workgroup
  using LT = typename std::conditional<std::is_same<C2, float2>::value, float2, double2>::type;
  __shared__ double xb[NP * NP * NP];
  __shared__ LT t1[NP * NP * HH];
  __shared__ LT t2[NP * N * HH];
  const int slot = blockIdx.x;  // right-hand side slot / nsrc, source slot % nsrc
  const int node = v.src_node[slot % v.nsrc];
  const int64_t urow = int64_t(node) + int64_t(slot / v.nsrc) * v.nstride;
  const int lane = threadIdx.x;
  double2 w[N];  // exp(-2 pi i m / n)
#pragma unroll
  for (int m = 0; m < N; m++) w[m] = v.twiddle[m];
  const int l = v.depth[node] + v.root_level;
  constexpr int R = (NSAM + 63) / 64;  // lane rounds over the surface samples
  bool big = false;  // a sample is not finite, or so large that its spectrum may not be
  for (int s = 0; s < v.sd; s++) {
    const double scale = ldexp(1.0, int(l * v.deg[s]));
    // all rounds' samples are loaded before the grid is cleared and filled
    double uv[R];
    int sh[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      // unconditional loads (a lane past the samples reads sample 0), so the
      // rounds' loads are issued together
      const int q = lane + 64 * r;
      const bool ok = q < NSAM;
      const int qq = ok ? q : 0;
      sh[r] = v.shell[qq];
      const double u = v.UE[urow * v.sz_ue + qq * v.sd + s];
      uv[r] = ok ? u * scale : 0.0;
      if constexpr (!kPack) big = big || !(fabs(uv[r]) < 1e290);
    }
    __syncthreads();
    for (int e = lane; e < NP * NP * NP; e += 64) xb[e] = 0.0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++)
      if (lane + 64 * r < NSAM) xb[sh[r]] = uv[r];
    __syncthreads();
    // along x (c): real -> half spectrum; line (a, b)
    for (int ab = lane; ab < NP * NP; ab += 64) {
      double xv[NP];
#pragma unroll
      for (int c = 0; c < NP; c++) xv[c] = xb[ab * NP + c];
#pragma unroll
      for (int kc = 0; kc < HH; kc++) {
        double2 acc = make_double2(0, 0);
#pragma unroll
        for (int c = 0; c < NP; c++) {
          const double2 tw = w[((c + O) * kc) % N];
          acc.x += xv[c] * tw.x; acc.y += xv[c] * tw.y;
        }
        store_c(&t1[ab * HH + kc], acc);
      }
    }
    __syncthreads();
    // along y (b); line (a, kc)
    for (int e = lane; e < NP * HH; e += 64) {
      const int a = e / HH, kc = e % HH;
      double2 in[NP];
#pragma unroll
      for (int b = 0; b < NP; b++) in[b] = load_c(&t1[(a * NP + b) * HH + kc]);
      if constexpr (kFast) {
        double2 out[N];
        pad12_fwd(in, w, out);
#pragma unroll
        for (int kb = 0; kb < N; kb++) store_c(&t2[(a * N + kb) * HH + kc], out[kb]);
      } else {
#pragma unroll
        for (int kb = 0; kb < N; kb++) {
          double2 acc = make_double2(0, 0);
#pragma unroll
          for (int b = 0; b < NP; b++) acc = cadd(acc, cmul(in[b], w[((b + O) * kb) % N]));
          store_c(&t2[(a * N + kb) * HH + kc], acc);
        }
      }
    }
    __syncthreads();
    // along z (a) -> global, frequency (ka, kb, kc); line (kb, kc)
    // (jfast: the DOFs of a frequency side by side)
    C2* out = v.jfast ? dspec + int64_t(slot) * v.sd * HS + s : dspec + (int64_t(slot) * v.sd + s) * HS;
    const int st = v.jfast ? v.sd : 1;
    auto zline = [&](int e, double2 (&o)[N]) {  // the n outputs of line e = kb h + kc
      double2 in[NP];
#pragma unroll
      for (int a = 0; a < NP; a++) in[a] = load_c(&t2[a * N * HH + e]);
      if constexpr (kFast) {
        pad12_fwd(in, w, o);
      } else {
#pragma unroll
        for (int ka = 0; ka < N; ka++) {
          double2 acc = make_double2(0, 0);
#pragma unroll
          for (int a = 0; a < NP; a++) acc = cadd(acc, cmul(in[a], w[((a + O) * ka) % N]));
          o[ka] = acc;
        }
      }
    };
    if constexpr (kPack) {
      // the lines of the planes kc in [1, np-1] first: line li = kb (np-1) +
      // kc - 1 stores frequency ka at li + ka NI; then the lines p = 2 kb +
      // (kc == np) of the planes kc = 0, np, which store ka in [0, np] without
      // the mirrors.  Every lane round is of one kind.
      constexpr int NI = N * (NP - 1);
      for (int li = lane; li < NI; li += 64) {
        double2 o[N];
        zline((li / (NP - 1)) * HH + li % (NP - 1) + 1, o);
#pragma unroll
        for (int ka = 0; ka < N; ka++) store_c(out + (li + ka * NI) * st, o[ka]);
      }
      for (int p = lane; p < 2 * N; p += 64) {
        const int e = (p >> 1) * HH + (p & 1) * NP;
        const SpecLine<NP> L(e);
        double2 o[N];
        zline(e, o);
#pragma unroll
        for (int ka = 0; ka <= NP; ka++)
          if (!L.plane_conj(ka)) store_c(out + L.plane_index(ka) * st, o[ka]);
      }
      // the row's padding (the Hadamard sweeps it with the other frequencies)
      constexpr int NC = spec_packed_count(NP);
      for (int q = NC + lane; q < HS; q += 64) store_c(out + q * st, make_double2(0, 0));
    } else {
      for (int e = lane; e < N * HH; e += 64) {
        double2 o[N];
        zline(e, o);
#pragma unroll
        for (int ka = 0; ka < N; ka++) store_c(out + (ka * N * HH + e) * st, o[ka]);
      }
    }
  }
  if constexpr (!kPack) {
    if (v.nonfin) {
      const int any = __any(big);
      if (lane == 0) v.nonfin[slot] = any;
    }
  }
}

// Scalar-kernel Hadamard (see hadamard.hpp for the scheme).  A workgroup's table:
// 16 frequencies (88 KB); lane = frequency x 4 target pairs, so a wave sweeps one
// group, its source list is uniform, and a source value (read by 16 lanes as one
// 256-byte row, the same for the 4 pairs) serves two targets a lane.  Every
// target sees its terms in V-list order with the 1/G factor applied per term
// (UpwEqu2DwnChk_dgemv + cptwvv); PRE: 1/G is a power of two and is taken into
// the table.  At 4,334 groups (np 6) 2.1-2.6 ms, 3.7 with the table in L2; at 72
// groups (np 4) 33 us, 204 before.
constexpr int kHadF = 16;

template <bool PRE>
__global__ __launch_bounds__(1024) void k_had_scalar(VlistArgs v, double nrm, int nchunk, int nsplit) {
  __shared__ double2 T[343 * kHadF];
  __shared__ int lists[16][2 * kPairStride];
  __shared__ int next;
  if (threadIdx.x == 0) next = 0;
  int chunk, split;
  if (!had_block(nchunk, nsplit, chunk, split)) return;
  const int H = v.H, f0 = chunk * kHadF;
  const int nvg = v.ngrp * v.nrhs;
  for (int e = threadIdx.x; e < 343 * kHadF; e += blockDim.x) {
    double2 t = v.m2l[int64_t(e / kHadF) * H + min(f0 + e % kHadF, H - 1)];
    if constexpr (PRE) { t.x *= nrm; t.y *= nrm; }
    T[e] = t;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, fl = lane & 15, sg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const bool fok = f0 + fl < H;
  const int f = fok ? f0 + fl : H - 1;
  // targets 2 sg and 2 sg + 1: slot = slot of the halo index - offset of the child
  const double2* tl = T + fl - ((sg >> 1) * 49 + (sg & 1) * 7) * kHadF;
  const int m0 = 1 << (2 * sg);
  int* ls = lists[wave];      // the group's source slots
  int* lw = ls + kPairStride;  // the table positions of their halo indices, membership << 16
  // lane l stages the list entries l, 64 + l, ... (the next group's are loaded
  // during this one's sums); padding: the group's first source, no member
  constexpr int NE = (kPairStride + 63) / 64;
  int es[NE], ew[NE], cnt_n = 0, bad_n = 0;
  auto fetch = [&](int vg) {
    const int g = vg / v.nrhs, rh = vg % v.nrhs;
    const int* ps = v.psrc + int64_t(g) * kPairStride;
    const int* pw = v.pslot + int64_t(g) * kPairStride;
    cnt_n = v.pcnt[g];
    const int s0 = ps[0];
#pragma unroll
    for (int e = 0; e < NE; e++) {
      const int k = lane + 64 * e < kPairStride ? lane + 64 * e : 0;
      es[e] = ps[k];
      ew[e] = ((pw[k] >> 9) & 0x3ff) * kHadF | (pw[k] >> 20) << 16;
      if (es[e] < 0) es[e] = s0;
    }
    bad_n = 0;
#pragma unroll
    for (int e = 0; e < NE; e++) bad_n |= v.nonfin[int64_t(rh) * v.nsrc + es[e]];
  };
  // an XCD's workgroups of one chunk advance through the groups side by side, so
  // that their sources' rows are shared in its L2; a workgroup's waves take its
  // groups from a counter (the lists' lengths differ several times over)
  auto take = [&]() {
    int c = 0;
    if (lane == 0) c = atomicAdd(&next, 1);
    c = __builtin_amdgcn_readfirstlane(c);
    return (c / nw * nsplit + split) * nw + c % nw;
  };
  int vg = take();
  if (vg < nvg) fetch(vg);
  for (int vn; vg < nvg; vg = vn) {
    const int g = vg / v.nrhs, rh = vg % v.nrhs;
    const int cnt = __builtin_amdgcn_readfirstlane(cnt_n);
    const bool bad = __any(bad_n);
#pragma unroll
    for (int e = 0; e < NE; e++)
      if (lane + 64 * e < kPairStride) {
        ls[lane + 64 * e] = es[e];
        lw[lane + 64 * e] = ew[e];
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    vn = take();
    if (vn < nvg) fetch(vn);
    const double2* dsp = v.dspec + int64_t(rh) * v.nsrc * H;
    double2 acc[2] = {make_double2(0, 0), make_double2(0, 0)};
    auto term = [&](int i, double2 t, double2 d) {
      const double2 p = cmul(t, d);
      if constexpr (PRE) acc[i] = cadd(acc[i], p);
      else acc[i] = make_double2(acc[i].x + nrm * p.x, acc[i].y + nrm * p.y);
    };
    auto source = [&](int k) { return (dsp + int64_t(__builtin_amdgcn_readfirstlane(ls[k])) * H)[unsigned(f)]; };
    if (!bad) {
      // Every source's values are finite, so a source adds zeros (its spectra) to
      // the targets that it is adjacent to and no membership is looked at.
      // A ring of 8 sources' values (the lists are padded to 8), each reloaded for
      // 8 sources on once it is used; the next source's spectra are read during
      // this one's sums.
      double2 d[8], tc[2], tn[2];
      auto spectra = [&](int k, double2 (&t)[2]) {
        const double2* p = tl + (lw[k] & 0xffff);
        t[0] = p[0];
        t[1] = p[-kHadF];
      };
#pragma unroll
      for (int u = 0; u < 8; u++) d[u] = source(u);
      spectra(0, tc);
      for (int k = 0; k < cnt; k += 8) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
          spectra(k + u + 1, tn);
          __builtin_amdgcn_sched_barrier(0);
          term(0, tc[0], d[u]);
          term(1, tc[1], d[u]);
          __builtin_amdgcn_sched_barrier(0);
          d[u] = source(k + 8 + u);  // (past the list: padding)
          tc[0] = tn[0];
          tc[1] = tn[1];
        }
      }
    } else {
      for (int k = 0; k < cnt; k++) {
        const int w = lw[k];
        const double2* t = tl + (w & 0xffff);
        const double2 d = source(k);
        if ((w >> 16) & m0) term(0, t[0], d);
        if ((w >> 16) & (m0 << 1)) term(1, t[-kHadF], d);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the lists are read before they are replaced
    if (!fok) continue;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int tg = v.tgt[g * 8 + 2 * sg + i];
      if (tg >= 0) v.espec[int64_t(tg + rh * v.ntrg) * H + f] = acc[i];
    }
  }
}

// Inverse: unnormalised c2r of each target spectrum, evaluated only on the
// surface samples, added into DC (effVal2PlnVal + regVal2SamVal).  Same line
// scheme as the forward transform; the first pass reads the spectrum straight
// from global memory (lines are contiguous across lanes).
template <int NP, typename C2>
__global__ __launch_bounds__(64) void k_fft_inv(VlistArgs v, const C2* espec) {
  constexpr int N = 2 * NP, HH = NP + 1, O = NP / 2;
  constexpr bool kFast = NP == 6 && std::is_same<C2, float2>::value;
  constexpr bool kPack = std::is_same<C2, float2>::value;
  constexpr int HS = kPack ? spec_packed_len(NP) : N * N * HH;
  constexpr int NSAM = NP * NP * NP - (NP - 2) * (NP - 2) * (NP - 2);
  using LT = typename std::conditional<std::is_same<C2, float2>::value, float2, double2>::type;
  __shared__ LT y1[NP * N * HH];
  __shared__ LT y2[NP * NP * HH];
  __shared__ int qof[NP * NP * NP];  // block index -> surface sample, -1 inside
  const int slot = blockIdx.x;  // right-hand side slot / ntrg, target slot % ntrg
  const int node = v.trg_node[slot % v.ntrg];
  const int64_t drow = int64_t(node) + int64_t(slot / v.ntrg) * v.nstride;
  const int lane = threadIdx.x;
  double2 w[N];  // exp(+2 pi i m / n)
#pragma unroll
  for (int m = 0; m < N; m++) { const double2 t = v.twiddle[m]; w[m] = make_double2(t.x, -t.y); }
  for (int e = lane; e < NP * NP * NP; e += 64) qof[e] = -1;
  __syncthreads();
  for (int q = lane; q < NSAM; q += 64) qof[v.shell[q]] = q;
  double* dc = v.DC + drow * v.sz_dc;
  const int lvl = v.depth[node] + v.root_level;
  for (int i = 0; i < v.td; i++) {
    const double oscale = v.deg_out ? ldexp(1.0, int(lvl * v.deg_out[i])) : 1.0;
    const C2* in = espec + (int64_t(slot) * v.td + i) * HS;
    __syncthreads();
    // along z (a), only block rows a' in [0,np); line (kb, kc)
    auto zline = [&](const double2 (&x)[N], int e) {  // line e = kb h + kc from its n inputs
      if constexpr (kFast) {
        double2 o6[NP];
        pad12_inv(x, w, o6);
#pragma unroll
        for (int a = 0; a < NP; a++) store_c(&y1[a * N * HH + e], o6[a]);
      } else {
#pragma unroll
        for (int a = 0; a < NP; a++) {
          double2 acc = make_double2(0, 0);
#pragma unroll
          for (int ka = 0; ka < N; ka++) acc = cadd(acc, cmul(x[ka], w[((a + O) * ka) % N]));
          store_c(&y1[a * N * HH + e], acc);
        }
      }
    };
    if constexpr (kPack) {
      // packed spectrum: the lines of the planes kc in [1, np-1] (li = kb (np-1)
      // + kc - 1 reads frequency ka at li + ka NI), then those of the planes
      // kc = 0, np (p = 2 kb + (kc == np), a value that is not stored is the
      // conjugate of its mirror), so each lane round is of one kind.  With one
      // round of each (np <= 6) both rounds' inputs are loaded before either is
      // transformed.
      constexpr int NI = N * (NP - 1);
      auto eline = [](int li) { return (li / (NP - 1)) * HH + li % (NP - 1) + 1; };
      auto eplane = [](int p) { return (p >> 1) * HH + (p & 1) * NP; };
      auto ldp = [&](const SpecLine<NP>& L, int ka) -> C2 {
        C2 t = in[L.plane_index(ka)];
        if (L.plane_conj(ka)) t.y = -t.y;
        return t;
      };
      if constexpr (NI <= 64 && 2 * N <= 64) {
        const int li = lane < NI ? lane : 0, p = lane < 2 * N ? lane : 0;
        const SpecLine<NP> L(eplane(p));
        C2 ri[N], rp[N];
#pragma unroll
        for (int ka = 0; ka < N; ka++) ri[ka] = in[li + ka * NI];
#pragma unroll
        for (int ka = 0; ka < N; ka++) rp[ka] = ldp(L, ka);
        double2 x[N];
        if (lane < NI) {
#pragma unroll
          for (int ka = 0; ka < N; ka++) x[ka] = load_c(&ri[ka]);
          zline(x, eline(li));
        }
        if (lane < 2 * N) {
#pragma unroll
          for (int ka = 0; ka < N; ka++) x[ka] = load_c(&rp[ka]);
          zline(x, eplane(p));
        }
      } else {
        for (int li = lane; li < NI; li += 64) {
          double2 x[N];
#pragma unroll
          for (int ka = 0; ka < N; ka++) x[ka] = load_c(in + li + ka * NI);
          zline(x, eline(li));
        }
        for (int p = lane; p < 2 * N; p += 64) {
          const SpecLine<NP> L(eplane(p));
          double2 x[N];
#pragma unroll
          for (int ka = 0; ka < N; ka++) {
            const C2 t = ldp(L, ka);
            x[ka] = load_c(&t);
          }
          zline(x, eplane(p));
        }
      }
    } else if constexpr (N * HH > 128) {
      for (int e = lane; e < N * HH; e += 64) {
        double2 x[N];
#pragma unroll
        for (int ka = 0; ka < N; ka++) x[ka] = load_c(in + ka * N * HH + e);
        zline(x, e);
      }
    } else {
      // the n h lines fit two rounds of the 64 lanes (np <= 7): both rounds'
      // inputs are loaded before either is transformed, so the load latency is
      // paid once per node
      const int e0 = lane, e1 = lane + 64;
      const bool has1 = e1 < N * HH;
      C2 r0[N], r1[N];
#pragma unroll
      for (int ka = 0; ka < N; ka++) r0[ka] = in[ka * N * HH + (e0 < N * HH ? e0 : 0)];
#pragma unroll
      for (int ka = 0; ka < N; ka++) r1[ka] = in[ka * N * HH + (has1 ? e1 : 0)];
#pragma unroll
      for (int half = 0; half < 2; half++) {
        const int e = half ? e1 : e0;
        if (e >= N * HH) continue;
        double2 x[N];
#pragma unroll
        for (int ka = 0; ka < N; ka++) x[ka] = load_c(half ? &r1[ka] : &r0[ka]);
        zline(x, e);
      }
    }
    __syncthreads();
    // along y (b), only b' in [0,np); line (a, kc)
    for (int e = lane; e < NP * HH; e += 64) {
      const int a = e / HH, kc = e % HH;
      double2 x[N];
#pragma unroll
      for (int kb = 0; kb < N; kb++) x[kb] = load_c(&y1[(a * N + kb) * HH + kc]);
      if constexpr (kFast) {
        double2 o6[NP];
        pad12_inv(x, w, o6);
#pragma unroll
        for (int b = 0; b < NP; b++) store_c(&y2[(a * NP + b) * HH + kc], o6[b]);
      } else {
#pragma unroll
        for (int b = 0; b < NP; b++) {
          double2 acc = make_double2(0, 0);
#pragma unroll
          for (int kb = 0; kb < N; kb++) acc = cadd(acc, cmul(x[kb], w[((b + O) * kb) % N]));
          store_c(&y2[(a * NP + b) * HH + kc], acc);
        }
      }
    }
    __syncthreads();
    // along x (c), c2r at the surface samples; line (a, b)
    for (int ab = lane; ab < NP * NP; ab += 64) {
      double2 yy[HH];
#pragma unroll
      for (int kc = 0; kc < HH; kc++) yy[kc] = load_c(&y2[ab * HH + kc]);
      // the line's check values are loaded together (absent samples read
      // element 0 and are not stored), so the loads are not serialised
      int qc[NP];
      double old[NP];
#pragma unroll
      for (int c = 0; c < NP; c++) qc[c] = qof[ab * NP + c];
      if (v.dc_store) {  // 0 + x: the same sums as reading the zeroed values
#pragma unroll
        for (int c = 0; c < NP; c++) old[c] = 0.0;
      } else {
#pragma unroll
        for (int c = 0; c < NP; c++) old[c] = dc[(qc[c] < 0 ? 0 : qc[c]) * v.td + i];
      }
#pragma unroll
      for (int c = 0; c < NP; c++) {
        double val = yy[0].x + yy[N / 2].x * (((c + O) & 1) ? -1.0 : 1.0);
#pragma unroll
        for (int kc = 1; kc < N / 2; kc++) {
          const double2 tw = w[((c + O) * kc) % N];
          val += 2.0 * (yy[kc].x * tw.x - yy[kc].y * tw.y);
        }
        if (qc[c] >= 0) dc[qc[c] * v.td + i] = old[c] + (v.deg_out ? oscale * val : val);
      }
    }
  }
}

template <typename C2>
static hipError_t launch_fft_fwd_any(const VlistArgs& v, C2* dspec, hipStream_t s) {
  const dim3 g(unsigned(int64_t(v.nsrc) * v.nrhs)), b(64);
  switch (v.np) {
    case 3: k_fft_fwd<3, C2><<<g, b, 0, s>>>(v, dspec); break;
    case 4: k_fft_fwd<4, C2><<<g, b, 0, s>>>(v, dspec); break;
    case 5: k_fft_fwd<5, C2><<<g, b, 0, s>>>(v, dspec); break;
    case 6: k_fft_fwd<6, C2><<<g, b, 0, s>>>(v, dspec); break;
    case 7: k_fft_fwd<7, C2><<<g, b, 0, s>>>(v, dspec); break;
    case 8: k_fft_fwd<8, C2><<<g, b, 0, s>>>(v, dspec); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename C2>
static hipError_t launch_fft_inv_any(const VlistArgs& v, const C2* espec, hipStream_t s) {
  const dim3 g(unsigned(int64_t(v.ntrg) * v.nrhs)), b(64);
  switch (v.np) {
    case 3: k_fft_inv<3, C2><<<g, b, 0, s>>>(v, espec); break;
    case 4: k_fft_inv<4, C2><<<g, b, 0, s>>>(v, espec); break;
    case 5: k_fft_inv<5, C2><<<g, b, 0, s>>>(v, espec); break;
    case 6: k_fft_inv<6, C2><<<g, b, 0, s>>>(v, espec); break;
    case 7: k_fft_inv<7, C2><<<g, b, 0, s>>>(v, espec); break;
    case 8: k_fft_inv<8, C2><<<g, b, 0, s>>>(v, espec); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_vlist(const VlistArgs& v0, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  if (v0.ngrp <= 0) return hipSuccess;
  if (v0.np > kMaxNp || v0.nrhs < 1) return hipErrorInvalidValue;
  VlistArgs v = v0;
  v.jfast = 1;  // as k_had_vec reads it (one DOF: the same layout)
  // a flag per source spectrum, behind the spectra (their buffer has one more entry a row)
  v.nonfin = reinterpret_cast<int*>(v.dspec + int64_t(v.nsrc) * v.nrhs * v.sd * v.H);
  hipError_t e = launch_fft_fwd_any<double2>(v, v.dspec, s);
  if (e != hipSuccess) return e;
  if (e0) (void)hipEventRecord(e0, s);
  const double nrm = 1.0 / double(v.n * v.n * v.n);
  const bool pre = (v.n & (v.n - 1)) == 0;  // 1/G is a power of two
  if (v.sd == 1 && v.td == 1) {
    const int nchunk = (v.H + kHadF - 1) / kHadF;
    const HadShape h = had_shape(nchunk, int64_t(v.ngrp) * v.nrhs, 1);
    const dim3 grid(had_grid(nchunk, h.S)), block(64 * h.W);
    if (pre) k_had_scalar<true><<<grid, block, 0, s>>>(v, nrm, nchunk, h.S);
    else k_had_scalar<false><<<grid, block, 0, s>>>(v, nrm, nchunk, h.S);
    e = hipGetLastError();
  } else {
    if (v.sd == 4 && v.td == 3) e = launch_had_vec<4, 3>(v, pre, nrm, s);
    else if (v.sd == 3 && v.td == 3) e = launch_had_vec<3, 3>(v, pre, nrm, s);
    else if (v.sd == 3 && v.td == 4) e = launch_had_vec<3, 4>(v, pre, nrm, s);
    else e = hipErrorInvalidValue;
  }
  if (e != hipSuccess) return e;
  if (e1) (void)hipEventRecord(e1, s);
  return launch_fft_inv_any<double2>(v, v.espec, s);
}

hipError_t launch_fft_fwd32(const VlistArgs& v, float2* dspec, hipStream_t s) {
  if (v.nsrc <= 0) return hipSuccess;
  if (v.np > kMaxNp || v.nrhs < 1) return hipErrorInvalidValue;
  return launch_fft_fwd_any<float2>(v, dspec, s);
}

hipError_t launch_fft_inv32(const VlistArgs& v, const float2* espec, hipStream_t s) {
  if (v.ntrg <= 0) return hipSuccess;
  if (v.np > kMaxNp || v.nrhs < 1) return hipErrorInvalidValue;
  return launch_fft_inv_any<float2>(v, espec, s);
}

// ---------------------------------------------------------------------------
// FP64 direct sum (Dense3d_MPI::evaluate, dense3d_mpi.cpp:75-141) at nt
// check targets over all sources.  Workgroup (x, y) takes 256 Q targets (Q per
// thread, so that an LDS read of a source serves Q pairs: one target a thread is
// bound by the LDS) and source chunk y; the chunk's sources (leaf order, density
// read through the source permutation) are staged through LDS 256 at a time and
// every thread sweeps them with the pair form of pair64.hpp (r < 1e-8 excluded).
// Each chunk writes its partial sums to part[y][target][TD]; k_direct_sum adds
// the chunks in chunk order (deterministic for a given chunk count).  4,096
// targets, 1M sources, Laplace: 2.3 ms (5.7 with one target a thread, square root
// and division).  The reciprocal square root has no value where r^2 overflows: a
// target (or a domain, src_r2 its largest squared coordinate) that far away is summed
// again with the kernel block, which gives 0 there.
template <int KT, int Q>
__global__ __launch_bounds__(256) void k_direct_part(KParams<double> p, int64_t ns, int64_t chunk,
                                                     const double* __restrict__ spos, const double* __restrict__ snor,
                                                     const int* __restrict__ sperm, const double* __restrict__ sden,
                                                     int nt, const double* __restrict__ tpos, double src_r2,
                                                     double* __restrict__ part) {
  constexpr int SD = src_dof(KT), TD = trg_dof(KT);
  constexpr bool NOR = needs_normals_ct(KT);
  constexpr int WO = NOR ? 6 : 3, REC = (WO + SD + 1) / 2 * 2;
  __shared__ __align__(16) double rec[256 * REC];
  __shared__ int infs[4];
  const int tid = threadIdx.x;
  double tx[Q], ty[Q], tz[Q], acc[Q][TD];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int i = (int(blockIdx.x) * Q + q) * 256 + tid;
    const double* t = tpos + 3 * int64_t(i < nt ? i : nt - 1);
    tx[q] = t[0]; ty[q] = t[1]; tz[q] = t[2];
#pragma unroll
    for (int d = 0; d < TD; d++) acc[q][d] = 0.0;
  }
  const double h = ratio64<KT>(p);
  const int64_t j0 = int64_t(blockIdx.y) * chunk, j1 = j0 + chunk < ns ? j0 + chunk : ns;
  for (int64_t b = j0; b < j1; b += 256) {
    const int64_t j = b + tid;
    bool inf = false;  // a density staged here is not finite (where that matters)
    __syncthreads();
    double* o = rec + tid * REC;
    if (j < j1) {
#pragma unroll
      for (int d = 0; d < 3; d++) o[d] = spos[3 * j + d];
      if constexpr (NOR)
        for (int d = 0; d < 3; d++) o[3 + d] = snor[3 * j + d];
      const int64_t k = sperm[j];
#pragma unroll
      for (int d = 0; d < SD; d++) {
        o[WO + d] = sden[k * SD + d] * weight64<KT>(p, d);
        if constexpr (both_signs64(KT, false)) inf = inf || !(fabs(sden[k * SD + d]) < INFINITY);
      }
    } else {  // padding: far away, zero density
#pragma unroll
      for (int d = 0; d < REC; d++) o[d] = d ? 0.0 : 1e18;
    }
    if constexpr (both_signs64(KT, false)) infs[tid >> 6] = __any(inf);
    __syncthreads();
    const int cnt = j1 - b < 256 ? int(j1 - b) : 256;
    if constexpr (both_signs64(KT, false)) {
      inf = infs[0] | infs[1] | infs[2] | infs[3];
#pragma unroll 1
      for (int k = 0; inf && k < cnt; k++) {
        const double* sr = rec + k * REC;
#pragma unroll
        for (int q = 0; q < Q; q++) {
          const double x = tx[q] - sr[0], y = ty[q] - sr[1], z = tz[q] - sr[2];
          const double r2 = fma(x, x, fma(y, y, z * z));
          const double inv = r2 < kMinDif * kMinDif ? 0.0 : rsqrt64(r2);
          pair64_block<KT, false>(h, x, y, z, inv, sr + 3, sr + WO, acc[q]);
        }
      }
      if (inf) continue;
    }
    for (int k = 0; k < cnt; k++) {
      const double* sr = rec + k * REC;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const double x = tx[q] - sr[0], y = ty[q] - sr[1], z = tz[q] - sr[2];
        const double r2 = fma(x, x, fma(y, y, z * z));
        const double inv = r2 < kMinDif * kMinDif ? 0.0 : rsqrt64(r2);
        pair64<KT>(h, x, y, z, inv, sr + 3, sr + WO, acc[q]);
      }
    }
  }
  unsigned far = 0;  // targets to be summed again
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int i = (int(blockIdx.x) * Q + q) * 256 + tid;
    if (i >= nt) continue;
    far |= tx[q] * tx[q] + ty[q] * ty[q] + tz[q] * tz[q] + src_r2 < 1e300 ? 0u : 1u << q;
#pragma unroll
    for (int d = 0; d < TD; d++) part[(int64_t(blockIdx.y) * nt + i) * TD + d] = acc[q][d];
  }
#pragma unroll 1
  for (int q = 0; far; q++, far >>= 1) {
    const int i = (int(blockIdx.x) * Q + q) * 256 + tid;
    if (!(far & 1)) continue;
    const double* t = tpos + 3 * int64_t(i);
    double v[TD] = {};
#pragma unroll 1
    for (int64_t j = j0; j < j1; j++) {
      double blk[SD * TD], n[3] = {0.0, 0.0, 0.0};
      if constexpr (NOR)
        for (int d = 0; d < 3; d++) n[d] = snor[3 * j + d];
      kblock<KT, double>(p, t[0] - spos[3 * j], t[1] - spos[3 * j + 1], t[2] - spos[3 * j + 2], n[0], n[1], n[2], blk);
      const double* w = sden + int64_t(sperm[j]) * SD;
#pragma unroll
      for (int d = 0; d < TD; d++)
#pragma unroll
        for (int e = 0; e < SD; e++) v[d] += blk[d * SD + e] * w[e];
    }
    for (int d = 0; d < TD; d++) part[(int64_t(blockIdx.y) * nt + i) * TD + d] = v[d];
  }
}

__global__ void k_direct_sum(const double* __restrict__ part, int nchunk, int64_t n, double* __restrict__ out) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = 0.0;
  for (int c = 0; c < nchunk; c++) v += part[int64_t(c) * n + i];
  out[i] = v;
}

// ---------------------------------------------------------------------------
#define KIFMM_USER_KERNELS(X) X(111) X(121) X(311) X(312) X(321) X(322) X(511) X(521)

hipError_t launch_surface(int kt, const SurfArgs& a0, const KParams<double>& pu, hipStream_t s) {
  if (a0.ntasks <= 0) return hipSuccess;
  if (a0.n_sam > 2 * kSurfThreads || a0.nrhs < 1) return hipErrorInvalidValue;
  for (int r0 = 0; r0 < a0.nrhs; r0 += kMaxNr) {
    SurfArgs a = a0;
    a.r0 = r0;
    a.nr = std::min(kMaxNr, a0.nrhs - r0);
    const dim3 g(unsigned(a.ntasks)), b(kSurfThreads);
    switch (kt * 16 + rhs_group(a.nr)) {
#define KIFMM_CASE_NR(K, R) case K * 16 + R: k_surface<K, R><<<g, b, 0, s>>>(a, pu); break;
#define KIFMM_CASE(K) KIFMM_CASE_NR(K, 1) KIFMM_CASE_NR(K, 2) KIFMM_CASE_NR(K, 4) KIFMM_CASE_NR(K, 8)
      KIFMM_USER_KERNELS(KIFMM_CASE)
#undef KIFMM_CASE
#undef KIFMM_CASE_NR
      default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Targets a thread of the direct sum: up to 4, as long as a workgroup's 256 Q
// targets are there.
static int direct_targets(int nt) { return nt >= 1024 ? 4 : nt >= 512 ? 2 : 1; }

DirectPlan plan_direct(int64_t ns, int nt, int td, int64_t cap_doubles) {
  DirectPlan d{};
  if (nt <= 0) return d;
  const int64_t per_chunk = int64_t(nt) * td;
  if (per_chunk > cap_doubles) return d;  // nchunk 0: the workspace cannot hold one chunk
  const int64_t tiles = (nt + 256 * direct_targets(nt) - 1) / (256 * direct_targets(nt));
  const int64_t blocks = std::max<int64_t>(1, (ns + 255) / 256);
  // about 8 workgroups per CU over 256 CUs, within the workspace
  int64_t nchunk = std::min<int64_t>({blocks, std::max<int64_t>(1, (2048 + tiles - 1) / tiles),
                                      cap_doubles / per_chunk, 65535});
  nchunk = std::max<int64_t>(1, nchunk);
  d.chunk = ((ns + nchunk - 1) / nchunk + 255) / 256 * 256;
  if (d.chunk == 0) d.chunk = 256;
  d.nchunk = int(std::max<int64_t>(1, (ns + d.chunk - 1) / d.chunk));
  d.work_doubles = int64_t(d.nchunk) * per_chunk;
  return d;
}

hipError_t launch_direct(int kt, const KParams<double>& p, int64_t ns, const double* spos, const double* snor,
                         const int* sperm, const double* sden, int nt, const double* tpos, double src_r2,
                         const DirectPlan& d, double* work, double* tval, hipStream_t s) {
  if (nt <= 0) return hipSuccess;
  if (d.nchunk <= 0 || !work || d.chunk <= 0 || int64_t(d.nchunk) * d.chunk < ns) return hipErrorInvalidValue;
  const int q = direct_targets(nt);
  const dim3 grid(unsigned((nt + 256 * q - 1) / (256 * q)), unsigned(d.nchunk));
  switch (kt) {
#define KIFMM_CASE_Q(K, Q) \
    k_direct_part<K, Q><<<grid, dim3(256), 0, s>>>(p, ns, d.chunk, spos, snor, sperm, sden, nt, tpos, src_r2, work)
#define KIFMM_CASE(K)                   \
    case K:                             \
      if (q == 4) KIFMM_CASE_Q(K, 4);   \
      else if (q == 2) KIFMM_CASE_Q(K, 2); \
      else KIFMM_CASE_Q(K, 1);          \
      break;
    KIFMM_USER_KERNELS(KIFMM_CASE)
#undef KIFMM_CASE
#undef KIFMM_CASE_Q
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t n = int64_t(nt) * trg_dof(kt);
  k_direct_sum<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(work, d.nchunk, n, tval);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Fixed scratch for callers that cannot allocate: the direct sum's partial
// sums live in this array, one copy per GPU, held until the process ends.
// Every slot a call reads is written earlier in the same call, so nothing is
// cleared; calls that overlap on one GPU share it and race.
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

hipError_t scratch_address(double** out) {
  *out = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    // the array's device address on the current GPU (the host-side name is
    // only a stand-in and must never reach a kernel)
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace kifmm
