// FP64 pair interactions of the kernels that feed no pseudo-inverse (near field,
// its transpose, the gradient, the direct sum): 1/r from one reciprocal square
// root instead of a square root and divisions, the kernel's constants taken into
// the density where it is staged, and the density contracted at once (the 3 x 3
// blocks have the form G delta_ij + H x_i x_j, so G w + H (x.w) x costs a third of
// forming and applying the block).  Fused multiply-adds throughout: no rounding
// order is kept here.  Closed forms: kernel3d.hpp.
#pragma once
#include <hip/hip_runtime.h>

#include "kernel3d.hpp"

namespace kifmm {

// 1 / sqrt(x) for normal x: the hardware estimate (about 2^-23) and one step of
// third order, e = 1 - x y^2, y (1 + e / 2 + 3 e^2 / 8), which leaves rounding.
__device__ __forceinline__ double rsqrt64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

__device__ __forceinline__ double dot3(double ax, double ay, double az, const double* b) {
  return fma(ax, b[0], fma(ay, b[1], az * b[2]));
}

// Factor of density component s of kernel K and of its transpose.  The Navier
// kernels' is the constant that no nu makes zero (511: H / mu, 521: C); the other
// one, zero at nu = 3/4 (G) and nu = 1/2 (A), stands as its ratio to it.
template <int K>
__device__ __forceinline__ double weight64(const KParams<double>& p, int s) {
  if constexpr (K == 121) return -p.a;
  else if constexpr (K == 301) return s == 3 ? p.b : p.a;
  else if constexpr (K == 311) return p.a * p.b;
  else if constexpr (K == 321) return -p.a;
  else if constexpr (K == 511) return p.b * p.c;
  else if constexpr (K == 521) return p.c;
  else return p.a;  // 111, 312, 322
}
// Ratio of the other constant to the one in weight64 (511: G / H, 521: A / C).
template <int K>
__device__ __forceinline__ double ratio64(const KParams<double>& p) {
  if constexpr (K == 511) return p.a / p.b;
  else if constexpr (K == 521) return p.a / p.c;
  else return 0.0;
}

// acc += K(x; n) w for one pair, x = target - source, inv = 1/|x| (0: no
// contribution), n the source normal, w the density with weight64 applied.
template <int K>
__device__ __forceinline__ void pair64(double h, double x, double y, double z, double inv, const double* n,
                                       const double* w, double* acc) {
  if constexpr (K == 111) {
    acc[0] = fma(inv, w[0], acc[0]);
  } else {
    const double inv2 = inv * inv, inv3 = inv2 * inv;
    if constexpr (K == 121) {
      acc[0] = fma(inv3 * dot3(x, y, z, n), w[0], acc[0]);
    } else if constexpr (K == 312) {
      acc[0] = fma(inv3, dot3(x, y, z, w), acc[0]);
    } else if constexpr (K == 322) {
      const double nw = dot3(n[0], n[1], n[2], w), rn = dot3(x, y, z, n);
      acc[0] = fma(inv3, fma(-3.0 * rn * inv2, dot3(x, y, z, w), nw), acc[0]);
    } else if constexpr (K == 301 || K == 311 || K == 511) {
      double f = dot3(x, y, z, w);
      if constexpr (K == 301) f += w[3];
      const double g = inv3 * f, c = K == 511 ? h * inv : inv;
      acc[0] = fma(c, w[0], fma(g, x, acc[0]));
      acc[1] = fma(c, w[1], fma(g, y, acc[1]));
      acc[2] = fma(c, w[2], fma(g, z, acc[2]));
    } else if constexpr (K == 321) {
      const double g = inv3 * inv2 * dot3(x, y, z, n) * dot3(x, y, z, w);
      acc[0] = fma(g, x, acc[0]);
      acc[1] = fma(g, y, acc[1]);
      acc[2] = fma(g, z, acc[2]);
    } else if constexpr (K == 521) {
      // A (rn w + n (x.w)) + B x (n.w) + C rn (x.w) x, B = -A
      const double rn = dot3(x, y, z, n), f = dot3(x, y, z, w), nw = dot3(n[0], n[1], n[2], w);
      const double hi = h * inv3, a = hi * rn, b = hi * f, g = fma(inv3 * inv2 * rn, f, -hi * nw);
      acc[0] = fma(a, w[0], fma(b, n[0], fma(g, x, acc[0])));
      acc[1] = fma(a, w[1], fma(b, n[1], fma(g, y, acc[1])));
      acc[2] = fma(a, w[2], fma(b, n[2], fma(g, z, acc[2])));
    }
  }
}

// Whether the sums above (TR: those of the transpose below) form terms of both signs
// from one density component: an infinite one would give NaN where the kernel block
// times it is an infinity.
__host__ __device__ constexpr bool both_signs64(int kt, bool tr) { return kt == 521 || (kt == 322 && !tr); }
// The same pair with the block formed first, for densities that are not finite.
template <int K, bool TR>
__device__ __forceinline__ void pair64_block(double h, double x, double y, double z, double inv, const double* n,
                                             const double* w, double* acc) {
  const double v[3] = {x, y, z}, rn = dot3(x, y, z, n), inv2 = inv * inv, inv3 = inv2 * inv;
  if constexpr (K == 322) {
#pragma unroll
    for (int s = 0; s < 3; s++) acc[0] += inv3 * fma(-3.0 * rn * inv2, v[s], n[s]) * w[s];
  } else {
    const double hi = h * inv3, g = inv3 * inv2 * rn;
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
      for (int s = 0; s < 3; s++) {
        const double b = g * v[t] * v[s] + hi * (n[t] * v[s] - v[t] * n[s] + (t == s ? rn : 0.0));
        acc[TR ? s : t] += b * w[TR ? t : s];
      }
  }
}

// acc += K(x; n)^T w, w per target DOF, acc per source DOF.
template <int K>
__device__ __forceinline__ void pair64_t(double h, double x, double y, double z, double inv, const double* n,
                                         const double* w, double* acc) {
  if constexpr (K == 111 || K == 121 || K == 311 || K == 321) {
    pair64<K>(h, x, y, z, inv, n, w, acc);  // symmetric blocks
  } else {
    const double inv2 = inv * inv, inv3 = inv2 * inv;
    if constexpr (K == 511) {
      // symmetric too; with one right-hand side h w, formed once for two points, is
      // less than h / r a pair
      const double u = inv2 * dot3(x, y, z, w);
      acc[0] = fma(inv, fma(u, x, h * w[0]), acc[0]);
      acc[1] = fma(inv, fma(u, y, h * w[1]), acc[1]);
      acc[2] = fma(inv, fma(u, z, h * w[2]), acc[2]);
    } else if constexpr (K == 312) {
      const double g = inv3 * w[0];
      acc[0] = fma(g, x, acc[0]);
      acc[1] = fma(g, y, acc[1]);
      acc[2] = fma(g, z, acc[2]);
    } else if constexpr (K == 322) {
      const double a = inv3 * w[0], t = -3.0 * dot3(x, y, z, n) * inv2;
      acc[0] = fma(fma(t, x, n[0]), a, acc[0]);
      acc[1] = fma(fma(t, y, n[1]), a, acc[1]);
      acc[2] = fma(fma(t, z, n[2]), a, acc[2]);
    } else if constexpr (K == 521) {
      const double rn = dot3(x, y, z, n), f = dot3(x, y, z, w), nw = dot3(n[0], n[1], n[2], w);
      const double hi = h * inv3, a = hi * rn, b = -hi * f, g = fma(inv3 * inv2 * rn, f, hi * nw);
      acc[0] = fma(a, w[0], fma(b, n[0], fma(g, x, acc[0])));
      acc[1] = fma(a, w[1], fma(b, n[1], fma(g, y, acc[1])));
      acc[2] = fma(a, w[2], fma(b, n[2], fma(g, z, acc[2])));
    }
  }
}

}  // namespace kifmm
