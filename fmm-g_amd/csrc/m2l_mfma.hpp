// Scalar-kernel Hadamard of the mixed path (sd = td = 1) on the matrix cores.
//
// The halo sweep of k_m2l_tile<., true> (same sums, same order, same bits): target
// child t of a group receives, for every colleague offset q and source child c, the
// product T(2q + c - t) X(c), in three real chains (Gauss's form).  For one frequency
// and offset that is an 8 x 8 matrix of spectra times a column a group.
// v_mfma_f32_4x4x1f32 runs it as the vector unit does, one rounded multiply-add a
// product (compared to the bit, subnormals included), at twice the rate: 16 blocks of
// 4 x 4 = two halves of the targets x 32 groups.
//
// A wave takes one frequency of a tile of up to 32 groups; a workgroup eight
// neighbouring frequencies (64-byte pieces of the spectra rows).  The colleagues of
// the tile's groups overlap (32 groups of a full level have 144 different ones, not
// 832), so their child spectra are read once into LDS (76 KB: two workgroups a CU)
// and gathered from there: per offset four child spectra a lane, the first half of
// the wave the even children, the second the odd ones, which the instruction's
// half-wave broadcast hands to both target halves.  The 8 x 8 spectra of an offset
// are one register a chain, a lane an entry, and the broadcast of one 4-row block
// picks the source child.  Past the staging no wave waits for another.
//
// Bound by the matrix cores (busy 60% of the time) and, not hidden, by the staging
// and the LDS gathers between the products (half of the LDS cycles are bank
// conflicts).  Laplace np 6: 8 million points 5.05 -> 3.53 ms in a run of passes (5.43
// -> 4.05 in the kernel trace of a few), a million uniform points 757 -> 517 us,
// 100,000 points 164 -> 117 us.  In that trace, with the offset's spectra gathered from
// the table by every wave, or staged by the workgroup behind a barrier an offset: 4.3
// ms; child spectra staged in batches of eight loads: 4.9 ms.
#pragma once
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace kifmm {

constexpr int kMtF = 8;                    // frequencies (waves) a workgroup
constexpr int kMtP = kM2lTileParents + 1;  // colleagues, and one of zeros
constexpr int kMtS = 8 * kMtP + 4;         // spectra of a frequency; frequencies start 8 banks apart
constexpr int kMtT = 28;                   // translation spectra of a frequency and offset (27)
static_assert(kMtS % 8 == 4 && kMtS >= 8 * kMtP, "bank spread");

__global__ __launch_bounds__(64 * kMtF, 4) void k_m2l_mfma(VlistArgs v, const float2* __restrict__ dspec,
                                                           const float2* __restrict__ m2l, float2* __restrict__ espec,
                                                           float nrm, int ntile, int per_xcd) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  __shared__ __align__(16) float2 xs[kMtF * kMtS];
  __shared__ float2 ts[2][kMtF][kMtT];
  const int bx = blockIdx.x;
  // an XCD takes a run of tiles; a tile's two pieces of a 128-byte line in turn
  const int tile = (bx & 7) * per_xcd + (bx >> 4);
  if (tile >= ntile) return;
  const int H = v.H, tid = threadIdx.x, rhs = blockIdx.z;
  const int4 inf = v.mt_inf[tile];  // first group, groups, colleagues, offsets with sources
  const int f0 = (int(blockIdx.y) * 2 + ((bx >> 3) & 1)) * kMtF;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), th = lane >> 5;
  const int fl = tid % kMtF, i0 = tid / kMtF;  // staging and storing: frequency, and the first row of a round of 64
  constexpr int T = 64;
  // the wave's 27 spectra around an offset, a lane one: loaded two and three offsets
  // ahead, in LDS (of the wave's own: no wave waits for another) one ahead
  constexpr int NQ = 13;  // offsets q; 26 - q = -q runs on the conjugates
  const int td = min(lane, 26);
  const float2* tf = m2l + int64_t((td / 9) * 49 + ((td / 3) % 3) * 7 + td % 3) * H + f0 + wave;
  float2 tr[2];
  auto load_t = [&](int j) __attribute__((always_inline)) {
    tr[j & 1] = tf[int64_t(2 * (j / 9) * 49 + 2 * ((j / 3) % 3) * 7 + 2 * (j % 3)) * H];
  };
  auto store_t = [&](int j) __attribute__((always_inline)) {
    if (lane < 27) ts[j & 1][wave][lane] = tr[j & 1];
  };
  // waits for the LDS traffic only: loads stay in flight
  auto barrier = []() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  int tg[4];       // the targets this thread stores
  unsigned pk[7];  // colleague numbers of this lane's group, a byte an offset
  {
    // eight rows of one child and neighbouring colleagues a wave and round
    const int* rows = v.mt_row + int64_t(tile) * 8 * kM2lTileParents;  // [child][colleague]
    const float2* base = dspec + int64_t(rhs) * v.nsrc * H + f0 + fl;
    constexpr int U = 8 * kM2lTileParents / T;  // rounds
    static_assert(8 * kM2lTileParents % T == 0 && kM2lTileParents % 8 == 0, "whole rounds, a child a wave");
    int row[U];
    float2 x[U];
#pragma unroll
    for (int u = 0; u < U; u++) row[u] = rows[i0 + u * T];
    load_t(0);
#pragma unroll
    for (int u = 0; u < 7; u++) pk[u] = (v.mt_idx + int64_t(tile) * (7 * 32))[u * 32 + (lane & 31)];
#pragma unroll
    for (int u = 0; u < U; u++) x[u] = row[u] >= 0 ? base[int64_t(row[u]) * H] : make_float2(0.f, 0.f);
#pragma unroll
    for (int u = 0; u < 4; u++) tg[u] = v.tgt[int64_t(inf.x) * 8 + min(i0 + u * T, 8 * inf.y - 1)];
    store_t(0);
    load_t(1);
    load_t(2);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * T;
      xs[fl * kMtS + i / kM2lTileParents * kMtP + i % kM2lTileParents] = x[u];
    }
    barrier();
    // colleague number inf.z: no source
    if (tid < 8 * kMtF) xs[fl * kMtS + i0 * kMtP + inf.z] = make_float2(0.f, 0.f);
    barrier();
  }
  // this lane's entry of the 8 x 8 spectra: source child c, target child t
  const int tc = (lane >> 2) & 7, tt = 4 * th + (lane & 3);
  const int dl = ((tc >> 2) - (tt >> 2) + 1) * 9 + (((tc >> 1) & 1) - ((tt >> 1) & 1) + 1) * 3 + ((tc & 1) - (tt & 1) + 1);
  const float2* xw = xs + wave * kMtS + th * kMtP;
  const unsigned qmask = unsigned(inf.w);
  f4 k1 = {0.f, 0.f, 0.f, 0.f}, k2 = k1, k3 = k1;
  // offset q with the translation spectra t
  auto sweep = [&](int q, const float2 (&x)[4], float2 t) __attribute__((always_inline)) {
    const float tsum = t.x + t.y;
#define KIFMM_MT_STEP(C)                                                                                   \
  k1 = __builtin_amdgcn_mfma_f32_4x4x1f32(t.x, x[(C) / 2].x, k1, 3, C, 1 + (C) % 2);                       \
  k2 = __builtin_amdgcn_mfma_f32_4x4x1f32(t.y, x[(C) / 2].y, k2, 3, C, 1 + (C) % 2);                       \
  k3 = __builtin_amdgcn_mfma_f32_4x4x1f32(tsum, x[(C) / 2].x + x[(C) / 2].y, k3, 3, C, 1 + (C) % 2);
    if ((qmask >> q) & 1) {
      KIFMM_MT_STEP(0) KIFMM_MT_STEP(1) KIFMM_MT_STEP(2) KIFMM_MT_STEP(3)
      KIFMM_MT_STEP(4) KIFMM_MT_STEP(5) KIFMM_MT_STEP(6) KIFMM_MT_STEP(7)
    }
#undef KIFMM_MT_STEP
  };
  auto gather = [&](int q, float2 (&x)[4]) __attribute__((always_inline)) {
    const float2* xp = xw + ((pk[q / 4] >> (8 * (q % 4))) & 255u);
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = xp[2 * k * kMtP];
  };
  float2 xa[4], xb[4];
  gather(0, xa);
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    // (a wave's LDS accesses keep their order: what offset q - 1 read is read)
    if (q + 1 < NQ) store_t(q + 1);
    if (q + 3 < NQ) load_t(q + 3);
    const float2 t = ts[q & 1][wave][dl];
    float2 tm = ts[q & 1][wave][26 - dl];
    tm.y = -tm.y;
    gather(26 - q, xb);
    sweep(q, xa, t);
    if (q + 1 < NQ) gather(q + 1, xa);
    sweep(26 - q, xb, tm);
  }
  barrier();
  // through LDS, so that a row's eight frequencies are stored together
  constexpr int SO = 256 + 4;
#pragma unroll
  for (int r = 0; r < 4; r++)
    xs[wave * SO + (lane & 31) * 8 + 4 * th + r] =
        make_float2((k1[r] - k2[r]) * nrm, (k3[r] - k1[r] - k2[r]) * nrm);
  barrier();
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int i = i0 + u * T;
    if (i < 8 * inf.y && tg[u] >= 0) espec[(int64_t(rhs) * v.ntrg + tg[u]) * H + f0 + fl] = xs[fl * SO + i];
  }
}

}  // namespace kifmm
