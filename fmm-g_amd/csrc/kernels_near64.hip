// FP64 near field (U, W, X fallbacks, M2T, L2T; fmm3d_eval_mpi.cpp:773-785,
// :1146-1165, :1249, :1383-1435), its gradient (Laplace) and its transpose, one
// kernel for all: the points of a chunk meet the sources of the chunk's items.
//
// The sums feed no pseudo-inverse, so their order is free, and what bounds them
// is the FP64 VALU (12 instructions and a quarter-rate reciprocal square root a
// Laplace pair) with the LDS close behind (32 bytes a source and lane set).  A
// workgroup of two waves packs its items' sources, item after item, into full LDS
// blocks (short leaves share a staging round; an item is found by walking those
// that start inside the block), and a lane holds two of the chunk's points, so
// that one LDS read of a source serves two pairs.  Lanes form S copies of the
// point pairs; copy c sweeps the block's sources c, c + S, ..., two at a time, the
// same number of rounds for all copies (they run on into padding: zero density,
// outside the domain).  Neighbouring copies read neighbouring records, whose length
// is 32 bytes or an odd multiple of 16, so their reads fall into different banks
// (with a contiguous share a copy, 8 copies met in one bank).  Pairs closer than the
// reference's 1e-8 cut contribute nothing; the test is made only in blocks that hold
// the leaf's own sources unless the host could not keep the other items 1e-7 away
// (see NearChunk).  2.3e9 Laplace pairs (1M clustered points): 1.54 ms, 4.36 with one
// point a lane, an item a staging round, square root and division; 2.06 in leaf order
// instead of largest chunk first (the last chunks ran alone).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "pair64.hpp"

namespace kifmm {

enum Near64Mode { NEAR64_VAL = 0, NEAR64_GRAD = 1, NEAR64_T = 2 };
constexpr int kN64Win = 128;
static_assert(kNearChunk <= kN64Threads, "a lane for every two points and more");
typedef const __attribute__((address_space(1))) double* n64_ptr;
// Offset of an item's source `row` among rows of `len` values.  64 bits: one leaf's
// densities over all right-hand sides may pass 2^32 values.
__host__ __device__ constexpr int64_t n64_off(unsigned row, unsigned len) { return int64_t(uint64_t(row) * len); }
static_assert(n64_off(131071, 3 * 10950) == 4305682350 && n64_off(1500000000, 3) == 4500000000, "past 32 bits");

template <int KT, int NR, int MODE>
struct Near64 {
  static constexpr int KM = mm_kernel(KT);
  static constexpr bool TR = MODE == NEAR64_T, GRAD = MODE == NEAR64_GRAD;
  static constexpr bool NOR = needs_normals_ct(KT);
  // the equivalent surfaces have a kernel of their own: a pass for each kind
  static constexpr int PASSES = TR || KM == KT ? 1 : 2;
  static constexpr int W0 = TR ? trg_dof(KT) : src_dof(KT);            // densities a source, exact items
  static constexpr int W1 = TR ? W0 : src_dof(KM);                     // and surface items
  static constexpr int WM = (W0 > W1 ? W0 : W1) * NR;
  static constexpr int OUT = GRAD ? 3 : TR ? src_dof(KT) : trg_dof(KT);  // values a point
  static constexpr bool SNOR = NOR && !TR;                             // normals staged (TR: the point's own)
  static constexpr int LEN = (3 + (SNOR ? 3 : 0) + WM + 1) / 2 * 2;
  static constexpr int REC = LEN > 4 && LEN % 4 == 0 ? LEN + 2 : LEN;  // doubles a staged source
  // sources a block: full rounds of the threads, within about 16 KB for one
  // right-hand side; the same for more, whose sums then run in the same order (up to
  // 77 KB with eight: two workgroups a CU.  2.8M points, 511: 48 ms, and 43 with the
  // kernel before, which staged 128 sources and formed a pair's block once for all)
  static constexpr int NB = 3 + (SNOR ? 3 : 0) + WM / NR <= 6 ? 256 : 128;
  static constexpr int PAD = NB + 2 * kN64Copies;
  struct Item { double cw[4]; n64_ptr pos, den, nor; };
  struct Shared {
    __align__(16) double rec[PAD * REC];
    int pre[kN64Win + 1];
    unsigned char kind[kN64Win];
    int wsum[2];
    union {
      Item item[kN64Win];
      double red[kN64Threads * 2 * OUT];
    };
    unsigned inf[2];
  };
};

template <int KT, int NR, int MODE>
__global__ __launch_bounds__(kN64Threads) void k_near64(NearArgs a, KParams<double> pu, KParams<double> pm) {
  using C = Near64<KT, NR, MODE>;
  constexpr int KM = C::KM, NB = C::NB, REC = C::REC, OUT = C::OUT, PO = C::SNOR ? 6 : 3;
  __shared__ typename C::Shared sh;
  const NearChunk ch = a.chunks[a.order ? a.order[blockIdx.x] : int(blockIdx.x)];
  const int lane = threadIdx.x;
  const int tn = max(ch.tnum, 1), tl = (tn + 1) / 2;
  const int S = near64_copies(tn);
  const int ti = lane % tl, sub = lane / tl;
  const bool active = sub < S;
  // points ti and ti + tl (absent: the first one again, not stored)
  const int64_t q0 = ch.tbeg + ti, q1 = ch.tbeg + (ti + tl < ch.tnum ? ti + tl : ti);
  double px[2], py[2], pz[2], pn[2][C::TR && C::NOR ? 3 : 1];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const double* p = a.tpos + 3 * (q ? q1 : q0);
    px[q] = p[0]; py[q] = p[1]; pz[q] = p[2];
    if constexpr (C::TR && C::NOR)
      for (int d = 0; d < 3; d++) pn[q][d] = a.tnor[3 * (q ? q1 : q0) + d];
  }
  // padding past the block
  if (lane < C::PAD - NB)
    for (int e = 0; e < REC; e++) sh.rec[(NB + lane) * REC + e] = e == 0 ? a.padx : 0.0;
  double acc[2][NR][OUT];
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
      for (int t = 0; t < OUT; t++) acc[q][r][t] = 0.0;
  const int64_t rs_ue = a.nstride * a.sz_ue, rs_de = a.nstride * a.sz_de;  // right-hand-side steps
#pragma unroll 1
  for (int pass = 0; pass < C::PASSES; pass++) {
    for (int w0 = ch.ibeg; w0 < ch.iend; w0 += kN64Win) {
      const int nw = min(ch.iend - w0, kN64Win);
      __syncthreads();
      int sz = 0;
      if (lane < nw) {
        const int code = a.items[w0 + lane], node = code >> 2, kind = code & 3;
        const bool ex = kind == ITEM_EXACT, ue = kind == ITEM_UE;
        auto& it = sh.item[lane];
        if (C::PASSES == 1 || ex == (pass == 0)) sz = ex ? a.src_num[node] : (ue ? a.n_ue : a.n_de);
        if (ex) {
          const int64_t b = a.src_beg[node];
          it.pos = (n64_ptr)(a.spos + 3 * b);
          it.nor = (n64_ptr)(a.snor + 3 * b);
          it.den = (n64_ptr)(a.sden + (b * a.nrhs + a.r0) * C::W0);
          it.cw[0] = it.cw[1] = it.cw[2] = 0.0;
          it.cw[3] = 1.0;
        } else {
          const double4 g = a.geom[node];
          it.pos = it.nor = (n64_ptr)(ue ? a.sam_ue : a.sam_de);
          it.den = (n64_ptr)(ue ? a.UE + int64_t(node) * a.sz_ue + a.r0 * rs_ue
                               : a.DE + int64_t(node) * a.sz_de + a.r0 * rs_de);
          it.cw[0] = g.x; it.cw[1] = g.y; it.cw[2] = g.z; it.cw[3] = g.w;
        }
        sh.kind[lane] = (unsigned char)kind;
      }
      int inc = sz;  // prefix of the item sizes
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(inc, d, 64);
        if ((lane & 63) >= d) inc += y;
      }
      if ((lane & 63) == 63) sh.wsum[lane >> 6] = inc;
      __syncthreads();
      if (lane >= 64) inc += sh.wsum[0];
      sh.pre[lane + 1] = inc;
      if (lane == 0) sh.pre[0] = 0;
      __syncthreads();
      const int total = sh.pre[nw];
      // slots of the leaf's own item in this window (empty if absent)
      const int ow = ch.own >= 0 ? ch.ibeg + ch.own - w0 : -1;
      const int own0 = ow >= 0 && ow < nw ? sh.pre[ow] : 0, own1 = ow >= 0 && ow < nw ? sh.pre[ow + 1] : 0;
      int icur = 0;  // (uniform) the item of slot `base`, the last j with pre[j] <= base
      for (int base = 0; base < total; base += NB) {
        const int m = min(NB, total - base);
        const bool cut = !ch.unchk || (own0 < base + m && own1 > base);
        // items of this thread's slots, walking the items that start in the block
        constexpr int NS = NB / kN64Threads;
        int lo[NS], j = icur + 1;
#pragma unroll
        for (int e = 0; e < NS; e++) lo[e] = icur;
        for (; j < nw; j++) {
          const int sj = __builtin_amdgcn_readfirstlane(sh.pre[j]);
          if (sj >= base + m) break;
#pragma unroll
          for (int e = 0; e < NS; e++)
            if (base + kN64Threads * e + lane >= sj) lo[e] = j;
        }
        int inext = j - 1;
        while (inext + 1 < nw && __builtin_amdgcn_readfirstlane(sh.pre[inext + 1]) <= base + NB) inext++;
        icur = inext;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NS; e++) {
          const int slot = kN64Threads * e + lane;
          double* rec = sh.rec + slot * REC;
          if (slot < m) {
            const unsigned off = unsigned(base + slot - sh.pre[lo[e]]);
            const int kind = sh.kind[lo[e]];
            const bool ex = kind == ITEM_EXACT;
            const auto& it = sh.item[lo[e]];
            const n64_ptr ps = it.pos + n64_off(off, 3);
            const double w = it.cw[3];
            rec[0] = fma(w, ps[0], it.cw[0]);
            rec[1] = fma(w, ps[1], it.cw[1]);
            rec[2] = fma(w, ps[2], it.cw[2]);
            if constexpr (C::SNOR) {
              if (pass == 0) {
                const n64_ptr pn_ = it.nor + n64_off(off, 3);
                rec[3] = pn_[0]; rec[4] = pn_[1]; rec[5] = pn_[2];
              }
            }
            if constexpr (C::PASSES == 1) {
              const n64_ptr pd = it.den + n64_off(off, ex && !C::TR ? a.nrhs * C::W0 : C::W0);
              const int64_t rstep = ex ? int64_t(C::W0) : kind == ITEM_UE ? rs_ue : rs_de;
#pragma unroll
              for (int r = 0; r < NR; r++)
#pragma unroll
                for (int s = 0; s < C::W0; s++)
                  rec[PO + r * C::W0 + s] =
                      r < a.nr ? pd[r * rstep + s] * (ex || C::TR ? weight64<KT>(pu, s) : weight64<KM>(pm, s)) : 0.0;
            } else if (pass == 0) {
              const n64_ptr pd = it.den + n64_off(off, a.nrhs * C::W0);
#pragma unroll
              for (int r = 0; r < NR; r++)
#pragma unroll
                for (int s = 0; s < C::W0; s++)
                  rec[PO + r * C::W0 + s] = r < a.nr ? pd[r * C::W0 + s] * weight64<KT>(pu, s) : 0.0;
            } else {
              const n64_ptr pd = it.den + n64_off(off, C::W1);
              const int64_t rstep = kind == ITEM_UE ? rs_ue : rs_de;
#pragma unroll
              for (int r = 0; r < NR; r++)
#pragma unroll
                for (int s = 0; s < C::W1; s++)
                  rec[PO + r * C::W1 + s] = r < a.nr ? pd[r * rstep + s] * weight64<KM>(pm, s) : 0.0;
            }
          } else {
            for (int e2 = 0; e2 < REC; e2++) rec[e2] = e2 == 0 ? a.padx : 0.0;
          }
        }
        if constexpr (both_signs64(KT, C::TR)) {
          // right-hand sides with a density here that is not finite
          unsigned inf = 0, any = 0;
#pragma unroll
          for (int e = 0; e < NS; e++) {
            const double* w = sh.rec + (kN64Threads * e + lane) * REC + PO;
#pragma unroll
            for (int i = 0; i < NR * C::W0; i++) inf |= fabs(w[i]) < INFINITY ? 0u : 1u << (i / C::W0);
          }
#pragma unroll
          for (int r = 0; r < NR; r++) any |= __any(inf & (1u << r)) ? 1u << r : 0u;
          sh.inf[lane >> 6] = any;
        }
        __syncthreads();
        if (!active) continue;
        const int L = ((m + S - 1) / S + 1) & ~1;
        const double* rec = sh.rec + sub * REC;
        const int step = S * REC;
        auto sweep = [&](auto K_, auto cut_, double h) {
          constexpr int K = decltype(K_)::value;
          constexpr bool CUT = decltype(cut_)::value;
          constexpr int WK = C::TR ? trg_dof(K) : src_dof(K);
          for (int i = 0; i < L; i += 2, rec += 2 * step) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
              const double* s = rec + u * step;
#pragma unroll
              for (int q = 0; q < 2; q++) {
                double x = px[q] - s[0], y = py[q] - s[1], z = pz[q] - s[2];
                const double r2 = fma(x, x, fma(y, y, z * z));
                double inv = rsqrt64(r2);
                const bool near = CUT && r2 < kMinDif * kMinDif;
                if constexpr (!C::GRAD) inv = near ? 0.0 : inv;
                if constexpr (C::TR) { x = -x; y = -y; z = -z; }  // the points are the sources
#pragma unroll
                for (int r = 0; r < NR; r++) {
                  const double* w = s + PO + r * WK;
                  if constexpr (C::GRAD) {
                    // (a cut pair's density is not looked at, finite or not)
                    const double g = -w[0] * inv * (inv * inv), c = near ? 0.0 : g;
                    acc[q][r][0] = fma(c, x, acc[q][r][0]);
                    acc[q][r][1] = fma(c, y, acc[q][r][1]);
                    acc[q][r][2] = fma(c, z, acc[q][r][2]);
                  } else if constexpr (C::TR) {
                    pair64_t<K>(h, x, y, z, inv, pn[q], w, acc[q][r]);
                  } else {
                    pair64<K>(h, x, y, z, inv, s + 3, w, acc[q][r]);
                  }
                }
              }
            }
          }
        };
        using TT = std::true_type;
        using FT = std::false_type;
        if (pass == 0) {
          const double h = ratio64<KT>(pu);
          if constexpr (both_signs64(KT, C::TR)) {
            const unsigned any = __builtin_amdgcn_readfirstlane(sh.inf[0] | sh.inf[1]);
            if (any) {  // (the other right-hand sides keep their sums' bits)
#pragma unroll 1
              for (int i = 0; i < L; i++, rec += step)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                  const double sg = C::TR ? -1.0 : 1.0;
                  const double x = sg * (px[q] - rec[0]), y = sg * (py[q] - rec[1]), z = sg * (pz[q] - rec[2]);
                  const double r2 = fma(x, x, fma(y, y, z * z));
                  const double inv = r2 < kMinDif * kMinDif ? 0.0 : rsqrt64(r2);
#pragma unroll
                  for (int r = 0; r < NR; r++) {
                    const double* n = C::TR ? pn[q] : rec + 3;
                    const double* w = rec + PO + r * C::W0;
                    if (any & (1u << r)) pair64_block<KT, C::TR>(h, x, y, z, inv, n, w, acc[q][r]);
                    else if constexpr (C::TR) pair64_t<KT>(h, x, y, z, inv, n, w, acc[q][r]);
                    else pair64<KT>(h, x, y, z, inv, n, w, acc[q][r]);
                    __builtin_amdgcn_sched_barrier(0);
                  }
                }
              continue;
            }
          }
          if (cut) sweep(std::integral_constant<int, KT>{}, TT{}, h);
          else sweep(std::integral_constant<int, KT>{}, FT{}, h);
        } else if constexpr (C::PASSES == 2) {
          const double h = ratio64<KM>(pm);
          if (cut) sweep(std::integral_constant<int, KM>{}, TT{}, h);
          else sweep(std::integral_constant<int, KM>{}, FT{}, h);
        }
      }
    }
  }
  // sum of the S copies, one right-hand side at a time
#pragma unroll
  for (int r = 0; r < NR; r++) {
    __syncthreads();
    if (active && sub > 0)
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int t = 0; t < OUT; t++) sh.red[((lane - tl) * 2 + q) * OUT + t] = acc[q][r][t];
    __syncthreads();
    if (lane >= tl || r >= a.nr) continue;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      if (ti + q * tl >= ch.tnum) continue;
      double v[OUT];
#pragma unroll
      for (int t = 0; t < OUT; t++) v[t] = acc[q][r][t];
      for (int u = 1; u < S; u++)
#pragma unroll
        for (int t = 0; t < OUT; t++) v[t] += sh.red[(((u - 1) * tl + lane) * 2 + q) * OUT + t];
      const int64_t o = q ? q1 : q0;
      double* out = a.tval + int64_t(a.r0 + r) * a.tstride + (a.tperm ? int64_t(a.tperm[o]) : o) * OUT;
#pragma unroll
      for (int t = 0; t < OUT; t++) out[t] = v[t];
    }
  }
}

#define KIFMM_NEAR64_KERNELS(X) X(111) X(121) X(311) X(312) X(321) X(322) X(511) X(521)

hipError_t launch_near(int kt, const NearArgs& a0, const KParams<double>& pu, const KParams<double>& pm,
                       hipStream_t s) {
  if (a0.nchunks <= 0) return hipSuccess;
  if (a0.nrhs < 1) return hipErrorInvalidValue;
  for (int r0 = 0; r0 < a0.nrhs; r0 += kMaxNr) {
    NearArgs a = a0;
    a.r0 = r0;
    a.nr = std::min(kMaxNr, a0.nrhs - r0);
    const dim3 g(unsigned(a.nchunks)), b(kN64Threads);
    switch (kt * 16 + rhs_group(a.nr)) {
#define KIFMM_CASE_NR(K, R) case K * 16 + R: k_near64<K, R, NEAR64_VAL><<<g, b, 0, s>>>(a, pu, pm); break;
#define KIFMM_CASE(K) KIFMM_CASE_NR(K, 1) KIFMM_CASE_NR(K, 2) KIFMM_CASE_NR(K, 4) KIFMM_CASE_NR(K, 8)
      KIFMM_NEAR64_KERNELS(KIFMM_CASE)
#undef KIFMM_CASE
#undef KIFMM_CASE_NR
      default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_near_grad(int kt, const NearArgs& a, const KParams<double>& pu, const KParams<double>& pm,
                            hipStream_t s) {
  if (kt != 111) return hipErrorInvalidValue;
  if (a.nchunks <= 0) return hipSuccess;
  k_near64<111, 1, NEAR64_GRAD><<<dim3(unsigned(a.nchunks)), dim3(kN64Threads), 0, s>>>(a, pu, pm);
  return hipGetLastError();
}

hipError_t launch_near_adjoint(int kt, const NearArgs& a, const KParams<double>& pu, hipStream_t s) {
  if (a.nchunks <= 0) return hipSuccess;
  const dim3 g(unsigned(a.nchunks)), b(kN64Threads);
  switch (kt) {
#define KIFMM_CASE(K) case K: k_near64<K, 1, NEAR64_T><<<g, b, 0, s>>>(a, pu, pu); break;
    KIFMM_NEAR64_KERNELS(KIFMM_CASE)
#undef KIFMM_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace kifmm
