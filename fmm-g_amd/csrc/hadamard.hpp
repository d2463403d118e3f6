// FP64 V-list Hadamard sums in V-list (node) order, with the reference's rounding,
// with the translation spectra in LDS.
//
// Every (source, target) pair of a sibling group reads its own translation
// spectrum, so with one wave a group and the spectra in L2 the sums ran at the
// L2's rate (16 bytes a complex multiply-add and lane).  Here a workgroup keeps
// the whole table (343 offset slots) of a few frequencies in LDS and sweeps many
// groups with it; its lanes are those frequencies times targets (and groups), so
// a source value loaded once serves all its targets, and what bounds the sums is
// the arithmetic (10 unfused FP64 instructions a complex multiply-add).  The
// host's lists give each source of a group as a word: halo coordinates + 1 (3 x 3
// bits), offset slot of the halo index (10 bits, from bit 9), membership of the 8
// targets (from bit 20).  A source that is adjacent to a target is left out (its
// spectrum in the table is zero, but the source's value may not be finite).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"

namespace kifmm {

constexpr int kHadSlots = 392;  // LDS slots: 7 x 7 x 8 (z padded to 8)

typedef const __attribute__((address_space(4))) int* had_ci;  // read by scalar loads
__device__ inline had_ci had_cptr(const int* p) { return (had_ci)p; }

// Workgroup -> (frequency chunk, split of the groups).  An XCD (workgroup id mod 8)
// takes consecutive chunks, all splits of a chunk next to each other.
inline unsigned had_grid(int nchunk, int nsplit) { return unsigned((nchunk + 7) / 8 * 8) * unsigned(nsplit); }
__device__ inline bool had_block(int nchunk, int nsplit, int& chunk, int& split) {
  const int per8 = (nchunk + 7) / 8, q = int(blockIdx.x) >> 3;
  chunk = (int(blockIdx.x) & 7) * per8 + q / nsplit;
  split = q % nsplit;
  return chunk < nchunk;
}

// Launch shape: W waves a workgroup, each sweeping gw groups at a time, the
// groups dealt to S workgroups a chunk, one workgroup a CU (LDS), 32 CUs an XCD.
// A workgroup's time is its table load (0.4 of a wave's sweep of a group) and its
// waves' sweeps, W / 4 of them a SIMD (a lone wave a SIMD waits on its loads half
// of the time), half a sweep of it for the last ones.  Measured, FP64 scalar:
// 4,334 groups x 63 chunks 2.08 ms with W 16, S 4 (2.12 with S 12, 2.18 with S 32,
// 2.49 with W 8, S 4); 72 groups x 20 chunks 36 us with W 8, S 8 (42 with W 16, 51
// with W 4).
struct HadShape {
  int W, S;
};
inline HadShape had_shape(int nchunk, int64_t nvg, int gw) {
  HadShape best{16, 1};
  double tb = 1e300;
  const int per_xcd = (nchunk + 7) / 8;
  for (int W = 16; W >= 4; W /= 2) {
    const int64_t pass = int64_t(W) * gw;
    const int s_max = int(std::min<int64_t>(32, (nvg + pass - 1) / pass));
    for (int S = 1; S <= s_max; S++) {
      const double t = double((per_xcd * S + 31) / 32) *
                       (0.4 + (std::max(1.0, double(nvg) / double(pass * S)) + 0.5) * std::max(W / 4, 2));
      if (t < tb * (1 - 1e-9)) { tb = t; best = {W, S}; }
    }
  }
  return best;
}

__device__ inline double2 had_mul(double2 t, double2 d) {  // the complex product, unfused
  return make_double2(t.x * d.x - t.y * d.y, t.x * d.y + t.y * d.x);
}

// Vector kernels (SD source, TD target DOFs).  Lane = frequency (2) x 8 targets x
// 4 groups; each lane keeps the TD sums of its target.  The table is laid out
// component by component, a slot's 2 frequencies side by side, its z coordinate
// permuted by the parities of x and y so that the 8 targets' slots of a source
// fall into different banks.  The source spectra are stored with the DOFs of a
// frequency side by side ([source][frequency][SD]), so a chunk reads whole cache
// lines.  PRE: 1/G is a power of two (np 4 and 8) and is taken into the table,
// which leaves every product and sum as it is.  584 groups of the Stokes kernel at
// np 6: 5.2 ms (12.9 with the table in L2).
template <int SD, int TD, bool PRE>
__global__ __launch_bounds__(1024) void k_had_vec(VlistArgs v, double nrm, int nchunk, int nsplit) {
  constexpr int FL = 2, GQ = 4;
  __shared__ double2 T[SD * TD * kHadSlots * FL];
  int chunk, split;
  if (!had_block(nchunk, nsplit, chunk, split)) return;
  const int H = v.H, f0 = chunk * FL;
  const int nvg = v.ngrp * v.nrhs;
  for (int e = threadIdx.x; e < 343 * SD * TD * FL; e += blockDim.x) {
    const int fl = e % FL, row = e / FL, slot = row / (SD * TD), c = row % (SD * TD);
    const int X = slot / 49, Y = (slot / 7) % 7, Z = slot % 7;
    double2 t = v.m2l[int64_t(row) * H + min(f0 + fl, H - 1)];
    if constexpr (PRE) { t.x *= nrm; t.y *= nrm; }
    T[(c * kHadSlots + X * 56 + Y * 8 + (Z ^ ((Y & 1) * 2 + (X & 1) * 4))) * FL + fl] = t;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, fl = lane % FL, tau = (lane / FL) & 7, gq = lane / (8 * FL);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int bx = tau >> 2, by = (tau >> 1) & 1, bz = tau & 1;
  const bool fok = f0 + fl < H;
  const int f = fok ? f0 + fl : H - 1;
  for (int gb = (split * nw + wave) * GQ; gb < nvg; gb += nsplit * nw * GQ) {
    const bool gok = gb + gq < nvg;
    const int vg = gok ? gb + gq : nvg - 1, g = vg / v.nrhs, rh = vg % v.nrhs;
    const double2* dsp = v.dspec + (int64_t(rh) * v.nsrc * H + f) * SD;
    const int4* ps = reinterpret_cast<const int4*>(v.psrc + int64_t(g) * kPairStride);
    const int4* pw = reinterpret_cast<const int4*>(v.pslot + int64_t(g) * kPairStride);
    const int own = v.pcnt[g], s0 = v.psrc[int64_t(g) * kPairStride];
    int cnt = own;
#pragma unroll
    for (int d = 8 * FL; d < 64; d <<= 1) cnt = max(cnt, __shfl_xor(cnt, d, 64));
    cnt = __builtin_amdgcn_readfirstlane(cnt);  // the longest of the wave's lists
    double2 acc[TD];
#pragma unroll
    for (int i = 0; i < TD; i++) acc[i] = make_double2(0, 0);
    // four sources a batch; beyond a list's end its first source with the
    // padding's word (no target)
    struct Batch { int s[4], w[4]; };
    auto words = [&](int k, Batch& b) {
      const bool in = k < own;
      const int4 s4 = ps[in ? k / 4 : 0], w4 = pw[in ? k / 4 : 0];
      b.s[0] = s4.x; b.s[1] = s4.y; b.s[2] = s4.z; b.s[3] = s4.w;
      b.w[0] = w4.x; b.w[1] = w4.y; b.w[2] = w4.z; b.w[3] = w4.w;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (!in) b.w[u] = kHadPadWord;
        if (!in || b.s[u] < 0) b.s[u] = s0;
      }
    };
    auto sources = [&](const Batch& b, int u, double2 (&d)[SD]) {
#pragma unroll
      for (int j = 0; j < SD; j++) d[j] = dsp[int64_t(b.s[u]) * H * SD + j];
    };
    Batch bc, bn;
    double2 d[2][SD];
    words(0, bc);
    sources(bc, 0, d[0]);
    for (int k = 0; k < cnt; k += 4) {
      words(k + 4, bn);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (u < 3) sources(bc, u + 1, d[(u + 1) & 1]);
        else sources(bn, 0, d[0]);
        const int w = bc.w[u];
        const int X = (w & 7) - bx, Y = ((w >> 3) & 7) - by, Z = ((w >> 6) & 7) - bz;
        if (!((w >> (20 + tau)) & 1)) continue;  // adjacent, or past the list's end
        const double2* t = T + (X * 56 + Y * 8 + (Z ^ ((Y & 1) * 2 + (X & 1) * 4))) * FL + fl;
#pragma unroll
        for (int i = 0; i < TD; i++)
#pragma unroll
          for (int j = 0; j < SD; j++) {
            const double2 p = had_mul(t[(j * TD + i) * kHadSlots * FL], d[u & 1][j]);
            if constexpr (PRE) acc[i] = make_double2(acc[i].x + p.x, acc[i].y + p.y);
            else acc[i] = make_double2(acc[i].x + nrm * p.x, acc[i].y + nrm * p.y);
          }
      }
      bc = bn;
    }
    const int tg = v.tgt[g * 8 + tau];
    if (!fok || !gok || tg < 0) continue;
#pragma unroll
    for (int i = 0; i < TD; i++) v.espec[(int64_t(tg + rh * v.ntrg) * TD + i) * H + f] = acc[i];
  }
}

template <int SD, int TD>
inline hipError_t launch_had_vec(const VlistArgs& v, bool pre, double nrm, hipStream_t s) {
  const int nchunk = (v.H + 1) / 2;
  const HadShape h = had_shape(nchunk, int64_t(v.ngrp) * v.nrhs, 4);
  const dim3 grid(had_grid(nchunk, h.S)), block(64 * h.W);
  if (pre) k_had_vec<SD, TD, true><<<grid, block, 0, s>>>(v, nrm, nchunk, h.S);
  else k_had_vec<SD, TD, false><<<grid, block, 0, s>>>(v, nrm, nchunk, h.S);
  return hipGetLastError();
}

}  // namespace kifmm
