// Indexed batched GEMM of the FP64 path in exact dgemv order: separate multiply
// and add, k ascending, accumulate steps seeded from C.
// C[:, cidx[j]] = (acc ? C : 0) + rs (.) (A_z * (ks (.) B[:, bidx[j]])).
// A_z is M x K column-major; z = blockIdx.z selects one of several matrices and
// its column range [zoff[z], zoff[z+1]) (the 8 L2L child matrices of a level run
// in one launch).
//
// The order rules out matrix cores, FMA and a split of K, so a launch is bound
// by the FP64 VALU (two instructions a term) where it has many columns and by
// the length of its K chain where it has few (the top levels, and K = 8 nUE of
// M2M).  k_gemm_seq serves the former: a lane owns one column and a wave 64
// columns x R rows; the R entries of A of a k are uniform, so they come from
// scalar loads straight into the multiplies' scalar operand, and a k costs one
// 8-byte LDS read for 2 R vector instructions.  Four waves of a workgroup take
// consecutive row sets of the same 64 columns, whose B slabs of GT_K terms are
// staged in LDS (two buffers, the next slab's loads in flight during the current
// one).  200,000 columns of M 152, K 296 take 945 us (half the rate of the
// unfused instructions); 16 rows a wave or slabs of 32 are slower.  k_gemm_row
// serves the latter.  A 64 x 64 tile a workgroup of 4 x 4 outputs a lane, used
// before both, took 277 us where M2M (M 296, K 1216) has 832 columns (79 now)
// and 102 us where it has 8 (27 now).
#pragma once
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace kifmm {

constexpr int GT_W = 4;           // waves a workgroup
constexpr int GT_R = 8;           // rows a wave
constexpr int GT_N = 64;          // columns a workgroup: one a lane
constexpr int GT_K = 16;          // k of a staged slab
constexpr int GT_T = 64 * GT_W;
constexpr int GT_B = GT_K * GT_N / GT_T;  // B elements a thread stages
constexpr int GT_S = 12;                  // period of the K scale (ksd divides it)
typedef const __attribute__((address_space(4))) double* gt_cptr;

template <int R>
__global__ __launch_bounds__(GT_T) void k_gemm_seq(GemmArgs g) {
  __shared__ double Bs[2][GT_K][GT_N + 1];
  __shared__ double sct[GT_S + GT_K];
  const int z = blockIdx.z;
  const int cbeg = g.zoff ? g.zoff[z] : 0, cend = g.zoff ? g.zoff[z + 1] : g.ncol;
  const int n0 = cbeg + int(blockIdx.y) * GT_N;
  if (n0 >= cend) return;
  const int tid = threadIdx.x, lane = tid & 63;
  // rows [mw, mw + R) of which this wave stores those from m0 on (the last
  // waves' sets are moved up to end at M; their other rows are other waves')
  const int m0 = (int(blockIdx.x) * GT_W + __builtin_amdgcn_readfirstlane(tid >> 6)) * R;
  const int mw = m0 + R <= g.M ? m0 : g.M - R;
  gt_cptr A = (gt_cptr)(g.A + int64_t(z) * g.a_zstride + mw);
  const int K = g.K, M = g.M;
  const int n = n0 + lane;
  const bool nok = n < cend;
  double* col = g.C + int64_t(nok ? g.cidx[n] : 0) * g.ldc;
  double c[R];
#pragma unroll
  for (int i = 0; i < R; i++) c[i] = g.accumulate && nok && mw + i >= m0 ? col[mw + i] : 0.0;
  if (tid < GT_S + GT_K) sct[tid] = g.kscale[tid % g.ksd];
  // staging: GT_K / GT_B threads a column, GT_B consecutive k each; a column
  // past the last reads the first one
  const int js = tid / (GT_K / GT_B), ks = (tid % (GT_K / GT_B)) * GT_B;
  const double* bcol = g.B + int64_t(g.bidx[n0 + js < cend ? n0 + js : n0]) * g.ldb + ks;
  double rb[GT_B];
  auto fetch = [&](int k0) {
    if (k0 + GT_K <= K) {
#pragma unroll
      for (int u = 0; u < GT_B; u++) rb[u] = bcol[k0 + u];
    } else {
#pragma unroll
      for (int u = 0; u < GT_B; u++) rb[u] = bcol[k0 + ks + u < K ? k0 + u : -ks];
    }
  };
  // batches of U terms: the A entries and B values of the next one are loaded
  // while this one is summed
  constexpr int U = 16 / R, NB = GT_K / U;
  double a0[U][R];
  auto load_a = [&](int k, double (&a)[U][R]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int i = 0; i < R; i++) a[u][i] = A[int64_t(k + u) * M + i];
  };
  auto sum = [&](const double (&a)[U][R], const double (&b)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int i = 0; i < R; i++) c[i] = c[i] + a[u][i] * b[u];
  };
  fetch(0);
  load_a(0, a0);
  __syncthreads();
  int buf = 0, sp = 0, k0 = 0;
  for (; k0 + GT_K <= K; k0 += GT_K, buf ^= 1) {
#pragma unroll
    for (int u = 0; u < GT_B; u++) Bs[buf][ks + u][js] = rb[u] * sct[sp + ks + u];
    sp = sp + GT_K % GT_S >= GT_S ? sp + GT_K % GT_S - GT_S : sp + GT_K % GT_S;
    __syncthreads();  // also: every wave has left the other buffer's terms
    if (k0 + GT_K < K) fetch(k0 + GT_K);
    double b0[U];
#pragma unroll
    for (int u = 0; u < U; u++) b0[u] = Bs[buf][u][lane];
#pragma unroll
    for (int j = 0; j < NB; j++) {
      double a1[U][R], b1[U];
      // (the last batch's entries, K >= U of them, are read again at the end)
      const int kn = k0 + (j + 1) * U;
      load_a(j + 1 < NB || kn + U <= K ? kn : K - U, a1);
      if (j + 1 < NB) {
#pragma unroll
        for (int u = 0; u < U; u++) b1[u] = Bs[buf][(j + 1) * U + u][lane];
      }
      __builtin_amdgcn_sched_barrier(0);  // the loads above are issued before the sums
      sum(a0, b0);
#pragma unroll
      for (int u = 0; u < U; u++) {
#pragma unroll
        for (int i = 0; i < R; i++) a0[u][i] = a1[u][i];
        if (j + 1 < NB) b0[u] = b1[u];
      }
    }
  }
  if (k0 < K) {  // the last K % GT_K terms
#pragma unroll
    for (int u = 0; u < GT_B; u++) Bs[buf][ks + u][js] = rb[u] * sct[sp + ks + u];
    __syncthreads();
    for (int kk = 0; k0 + kk < K; kk++) {
      const double b = Bs[buf][kk][lane];
#pragma unroll
      for (int i = 0; i < R; i++) c[i] = c[i] + A[int64_t(k0 + kk) * M + i] * b;
    }
  }
  if (!nok) return;
#pragma unroll
  for (int i = 0; i < R; i++)
    if (mw + i >= m0) col[mw + i] = g.accumulate ? c[i] : g.rscale[(mw + i) % g.rsd] * c[i];
}

// The same sums for launches with too few columns to fill the chip above: one
// wave a workgroup, its lanes 16 rows x 4 column sets of C columns, so that a
// narrow strip of A (one 128-byte line a term) serves a wave and the strips of a
// matrix spread over many CUs.  A is streamed from global memory D terms ahead
// into registers (independent loads that return in order; no wave waits for
// another at a barrier); the 4 C columns of B are scaled and staged GR_K terms at
// a time in LDS and read Q terms ahead of their sums.
constexpr int GR_K = 128;

template <int C, int D, int Q>
__global__ __launch_bounds__(64) void k_gemm_row(GemmArgs g) {
  static_assert(GR_K % D == 0 && D % (2 * Q) == 0, "whole rings a slab, an even number of batches a ring");
  constexpr int NC = 4 * C;  // columns a wave
  __shared__ __align__(16) double Bs[GR_K][NC];
  const int z = blockIdx.z;
  const int cbeg = g.zoff ? g.zoff[z] : 0, cend = g.zoff ? g.zoff[z + 1] : g.ncol;
  const int n0 = cbeg + int(blockIdx.y) * NC;
  if (n0 >= cend) return;
  const int lane = threadIdx.x, K = g.K, M = g.M;
  const int m = int(blockIdx.x) * 16 + (lane & 15), cg = (lane >> 4) * C;
  const unsigned mr = unsigned(m < M ? m : M - 1);
  const double* A = g.A + int64_t(z) * g.a_zstride;
  double c[C], a[D];
#pragma unroll
  for (int q = 0; q < C; q++) {
    const int n = n0 + cg + q < cend ? n0 + cg + q : n0;  // a column past the last repeats the first
    c[q] = g.accumulate ? g.C[int64_t(g.cidx[n]) * g.ldc + mr] : 0.0;
  }
  // staging: lane = term of a column, all NC columns
  const double* bcol[NC];
#pragma unroll
  for (int q = 0; q < NC; q++) bcol[q] = g.B + int64_t(g.bidx[n0 + q < cend ? n0 + q : n0]) * g.ldb;
  constexpr int SB = GR_K / 64;
  double rb[SB][NC];
  auto fetch_b = [&](int k0) {
#pragma unroll
    for (int u = 0; u < SB; u++) {
      const int k = k0 + lane + 64 * u < K ? k0 + lane + 64 * u : 0;
#pragma unroll
      for (int q = 0; q < NC; q++) rb[u][q] = bcol[q][k];
    }
  };
  // A through a buffer resource: the lane's row in the vector offset, the term in
  // the scalar offset (one scalar add and min a load; past the last term: it again)
  const unsigned M8 = unsigned(M) * 8u, last = unsigned(K - 1) * M8, mr8 = mr * 8u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, int(unsigned(K) * M8), 0x00020000);
  unsigned so = 0;
  auto load_a = [&]() {
    const double v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ra, mr8, so, 0));
    so = so + M8 < last ? so + M8 : last;
    return v;
  };
  fetch_b(0);
#pragma unroll
  for (int j = 0; j < D; j++) a[j] = load_a();
  for (int k0 = 0; k0 < K; k0 += D) {
    const int kb = k0 % GR_K;
    if (kb == 0) {
      __syncthreads();
#pragma unroll
      for (int u = 0; u < SB; u++) {
        const double sc = g.kscale[(k0 + lane + 64 * u) % g.ksd];
#pragma unroll
        for (int q = 0; q < NC; q++) Bs[lane + 64 * u][q] = rb[u][q] * sc;
      }
      __syncthreads();
      if (k0 + GR_K < K) fetch_b(k0 + GR_K);
    }
    if (k0 + D <= K) {
      double b[2][Q][C];
      auto read_b = [&](int j, double (&d)[Q][C]) {
#pragma unroll
        for (int u = 0; u < Q; u++)
#pragma unroll
          for (int q = 0; q < C; q++) d[u][q] = Bs[kb + j + u][cg + q];
      };
      read_b(0, b[0]);
#pragma unroll
      for (int j = 0; j < D; j += Q) {
        if (j + Q < D) read_b(j + Q, b[(j / Q + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // the reads are issued before the sums
#pragma unroll
        for (int u = 0; u < Q; u++)
#pragma unroll
          for (int q = 0; q < C; q++) c[q] = c[q] + a[j + u] * b[(j / Q) & 1][u][q];
        __builtin_amdgcn_sched_barrier(0);  // and the loads after them, into the same registers
#pragma unroll
        for (int u = 0; u < Q; u++) a[j + u] = load_a();
      }
    } else {
#pragma unroll
      for (int j = 0; j < D; j++)
        if (k0 + j < K) {
#pragma unroll
          for (int q = 0; q < C; q++) c[q] = c[q] + a[j] * Bs[kb + j][cg + q];
        }
    }
  }
  if (m >= M) return;
#pragma unroll
  for (int q = 0; q < C; q++) {
    if (n0 + cg + q >= cend) break;
    double* col = g.C + int64_t(g.cidx[n0 + cg + q]) * g.ldc;
    col[m] = g.accumulate ? c[q] : g.rscale[m % g.rsd] * c[q];
  }
}

inline hipError_t launch_gemm_seq(const GemmArgs& g, hipStream_t s) {
  if (g.ncol <= 0) return hipSuccess;
  if (g.M < GT_R || g.K < GT_R || g.ksd < 1 || GT_S % g.ksd) return hipErrorInvalidValue;
  const int nz = g.zoff ? g.nz : 1;
  // Column-per-lane waves from about one a SIMD on: below that a wave's chain of
  // scalar-load latencies is what counts, and the strips, whose chains are short,
  // win (M 152, K 296: 2,000 columns 42 us in strips and 59 here, 4,096 columns
  // 56 and 45; M 296, K 1216: 1,444 columns 112 and 152, 4,334 columns 310 and 197).
  const int64_t colblk = int64_t((g.max_zcol + GT_N - 1) / GT_N);
  if (colblk * nz * ((g.M + GT_R - 1) / GT_R) >= 1100) {
    k_gemm_seq<GT_R><<<dim3(unsigned((g.M + GT_W * GT_R - 1) / (GT_W * GT_R)), unsigned(colblk), unsigned(nz)),
                       dim3(GT_T), 0, s>>>(g);
    return hipGetLastError();
  }
  // Strips: 1, 2 or 4 columns a lane.  A lane's time grows by half a chain a
  // column, so few columns are spread over waves first (M 296, K 1216: 64 columns
  // 30 / 36 / 52 us with 1 / 2 / 4 a lane, 512 columns 126 / 66 / 70, 832 columns
  // 164 / 92 / 79).
  const int64_t rb = (g.M + 15) / 16;
  auto grid = [&](int C) { return dim3(unsigned(rb), unsigned((g.max_zcol + 4 * C - 1) / (4 * C)), unsigned(nz)); };
  auto waves = [&](int C) { return rb * ((g.max_zcol + 4 * C - 1) / (4 * C)) * nz; };
  if (waves(4) >= 800) k_gemm_row<4, 32, 2><<<grid(4), dim3(64), 0, s>>>(g);
  else if (waves(2) >= 320) k_gemm_row<2, 32, 8><<<grid(2), dim3(64), 0, s>>>(g);
  else k_gemm_row<1, 32, 16><<<grid(1), dim3(64), 0, s>>>(g);
  return hipGetLastError();
}

}  // namespace kifmm
