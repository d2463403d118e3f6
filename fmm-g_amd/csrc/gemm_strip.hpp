// FP64 matrix-core GEMM of small and middle launches (mixed path, transposed passes):
// C[:, cidx[j]] (+)= rs (.) (A_z * (ks (.) B[:, bidx[j]])).
#pragma once
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace kifmm {

// The products of k_gemm_mfma by single waves, for launches whose tiles would not
// fill the chip.
//
// The instruction, v_mfma_f64_4x4x4f64: four independent 4 x 4 x 4 products in 16
// clocks.  A register-only loop of it reaches 71-73 TFLOP/s from one wave a SIMD on;
// the 16 x 16 x 4 form 25-35 with one wave and 49 with eight.  Both run the same
// chain of fused multiply-adds, k ascending, so they give the same bits, whatever
// the tile.  Here the four products are the four 4-row groups of a 16-row block with
// one 4-column group (its B values are read by all four).  Operand layout: lane l
// supplies A[4 ((l / 4) % 4) + l % 4][l / 16], that is row l % 16, and
// B[l / 16][l % 4]; its result is D[4 ((l / 4) % 4) + l / 16][l % 4].  (In a 160 x 64
// tile of its own it was no faster than the 16 x 16 x 4 form inside a pass: 128 VGPRs
// for four waves a SIMD spill.)
//
// A wave takes 16 R rows x 4 Q columns, with its A operands read straight
// into registers DP steps of four terms ahead and its columns of B staged 64 terms
// at a time in LDS of its own (read and scaled a term a lane, so that no load is
// scattered).  No wave waits for another, so a step costs its MFMAs and not a
// slab's barrier and latencies (about 1,200 clocks a slab in the tile, which a launch
// of few tiles pays in full).  W waves a workgroup: neighbouring columns
// of the same rows, whose A lines they share in the L1; or, SPLIT, the K chunks of
// the same rows and columns, W at a time, whose products are summed here in chunk
// order (no workspace and no launch for the sum).  The two parts of a B are two
// sweeps; terms past a part's end are zeros.  Bound by the serial chain of its K
// when it is alone, by the A and B loads (each read M / 16 R or columns / 4 Q times)
// when there are many.
template <int R, int Q, int DP, int W, bool SPLIT>
__global__ __launch_bounds__(64 * W) void k_gemm_strip(GemmArgs g) {
  constexpr int NC = 4 * Q, KC = 64, ST = KC / 4;  // columns a wave, terms and steps a stage
  constexpr int NV = 16 * R * NC;                  // products of a wave
  static_assert(ST % DP == 0, "whole rings a stage");
  static_assert(!SPLIT || NV <= 64 * W, "a thread a sum");
  __shared__ __align__(16) double Bs_[W][KC][NC];
  __shared__ double part[SPLIT ? 2 : 1][SPLIT ? W : 1][SPLIT ? NV : 1];
  const int z = blockIdx.z;
  const int cbeg = g.zoff ? g.zoff[z] : 0, cend = g.zoff ? g.zoff[z + 1] : g.ncol;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lk = lane >> 4;
  const int n0 = cbeg + (SPLIT ? int(blockIdx.y) : int(blockIdx.y) * W + wave) * NC;
  const int m0 = int(blockIdx.x) * 16 * R;
  const int M = g.M;
  if (n0 >= cend) return;
  double (*Bs)[NC] = Bs_[wave];
  // A through a buffer resource (term in the scalar offset, lane's row and term of
  // four in the vector offset)
  const unsigned M8 = unsigned(M) * 8u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)(g.A + int64_t(z) * g.a_zstride), (short)0,
                                                                      int(unsigned(g.K) * M8), 0x00020000);
  unsigned arow[R];
#pragma unroll
  for (int r = 0; r < R; r++) arow[r] = unsigned(min(m0 + 16 * r + (lane & 15), M - 1)) * 8u;
  double acc[R][Q];
  // terms [ka, kb); term k of column n is base[idx[n] * ld + k - first]
  auto sweep = [&](int ka, int kb, int first, const double* base, const int* idx, int64_t ld,
                   bool scaled) __attribute__((always_inline)) {
    if (ka >= kb) return;
    const double* col[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) col[c] = base + int64_t(idx[n0 + c < cend ? n0 + c : n0]) * ld - first;
    double rb[NC], sc;
    auto fetch = [&](int k0) {  // a term a lane
      const int k = min(k0 + lane, kb - 1);
      sc = k0 + lane < kb ? (scaled ? g.kscale[(k - first) % g.ksd] : 1.0) : 0.0;
#pragma unroll
      for (int c = 0; c < NC; c++) rb[c] = col[c][k];
    };
    unsigned al[R], sa = unsigned(ka) * M8;
    const unsigned last = kb - ka >= 4 ? unsigned(kb - 4) * M8 : sa;
#pragma unroll
    for (int r = 0; r < R; r++) al[r] = arow[r] + unsigned(lk) * M8;
    double a[DP][R];
    auto load = [&](double (&av)[R]) {  // the next whole step (past the last: it again)
#pragma unroll
      for (int r = 0; r < R; r++) av[r] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ra, al[r], sa, 0));
      sa = min(sa + 4u * M8, last);
    };
    // position of column 4 q + j of a term: j Q + q, so a lane's columns lie together
    auto step = [&](const double (&av)[R], int t) {
      const double* b = &Bs[4 * t + lk][(lane & 3) * Q];
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const double v = b[q];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][q] = __builtin_amdgcn_mfma_f64_4x4x4f64(av[r], v, acc[r][q], 0, 0, 0);
      }
    };
    const int nf = (kb - ka) / 4;  // whole steps
    fetch(ka);
    if (nf > 0)
#pragma unroll
      for (int p = 0; p < DP; p++) load(a[p]);
    for (int t0 = 0; t0 < nf || t0 * 4 < kb - ka; t0 += ST) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int c = 0; c < NC; c++) {
        // (a term past the end may be of another part: not multiplied)
        Bs[lane][(c & 3) * Q + (c >> 2)] = sc != 0.0 ? rb[c] * sc : 0.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (ka + 4 * (t0 + ST) < kb) fetch(ka + 4 * (t0 + ST));
      if (t0 + ST <= nf) {
#pragma unroll
        for (int p = 0; p < ST; p++) {
          step(a[p % DP], p);
          load(a[p % DP]);
        }
      } else {
        const int rest = nf - t0;
#pragma unroll
        for (int p = 0; p < ST; p++)
          if (p < rest) {
            step(a[p % DP], p);
            load(a[p % DP]);
          }
        if ((kb - ka) % 4) {  // the last 1 to 3 terms: lanes past them read the last one
          const unsigned k = unsigned(min(ka + 4 * nf + lk, kb - 1));
#pragma unroll
          for (int r = 0; r < R; r++)
            a[0][r] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ra, arow[r] + k * M8, 0, 0));
          step(a[0], rest);
        }
      }
    }
  };
  auto chunk = [&](int kbeg, int kend) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int q = 0; q < Q; q++) acc[r][q] = 0.0;
    if (g.k1 > 0) sweep(kbeg, min(kend, g.k1), 0, g.B1, g.cidx, g.ldb1, false);
    sweep(max(kbeg, g.k1), kend, g.k1, g.B, g.bidx, g.ldb, true);
  };
  if constexpr (SPLIT) {
    double sum = 0.0;
    int buf = 0;
    for (int c0 = 0; c0 < g.ksplit; c0 += W, buf ^= 1) {
      const int c = c0 + wave;
      if (c < g.ksplit) {
        chunk(c * g.kchunk, min(g.K, (c + 1) * g.kchunk));
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
          for (int r = 0; r < R; r++)
            part[buf][wave][(4 * q + (lane & 3)) * 16 * R + 16 * r + (lane & 12) + lk] =
                g.rscale[min(m0 + 16 * r + (lane & 12) + lk, M - 1) % g.rsd] * acc[r][q];
      }
      // (a buffer is written again two rounds on, past the next round's barrier)
      __syncthreads();
      if (threadIdx.x < NV)
        for (int w = 0; w < min(W, g.ksplit - c0); w++) sum += part[buf][w][threadIdx.x];
    }
    const int n = n0 + int(threadIdx.x) / (16 * R), m = m0 + int(threadIdx.x) % (16 * R);
    if (threadIdx.x < NV && n < cend && m < M) {
      double* dst = g.C + int64_t(g.cidx[n]) * g.ldc + m;
      *dst = g.accumulate ? *dst + sum : sum;
    }
  } else {
    chunk(0, g.K);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int n = n0 + 4 * q + (lane & 3);
      if (n >= cend) continue;
      double* col = g.C + int64_t(g.cidx[n]) * g.ldc;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int m = m0 + 16 * r + (lane & 12) + lk;
        if (m >= M) continue;
        const double v = g.rscale[m % g.rsd] * acc[r][q];
        col[m] = g.accumulate ? col[m] + v : v;
      }
    }
  }
}

template <int R, int Q, int DP, int W, bool SPLIT>
inline void launch_gemm_strip(const GemmArgs& g, hipStream_t s) {
  const int cols = 4 * Q * (SPLIT ? 1 : W);
  const dim3 grid(unsigned((g.M + 16 * R - 1) / (16 * R)), unsigned((g.max_zcol + cols - 1) / cols),
                  unsigned(g.zoff ? g.nz : 1));
  k_gemm_strip<R, Q, DP, W, SPLIT><<<grid, dim3(64 * W), 0, s>>>(g);
}

}  // namespace kifmm
