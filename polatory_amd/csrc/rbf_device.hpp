// Device-side RBF evaluation phi(r^2) with the constants folded per call site.
//
//   bh3  phi = -slope * sqrt(r^2 + c^2)        (rbf/polyharmonic_odd.hpp:32-43, kSign=-1)
//   th3  phi = +slope * (r^2 + c^2)^(3/2)      (rbf/polyharmonic_odd.hpp:120-136)
//   exp  phi = psill * exp(-3 r / range)       (rbf/cov_exponential.hpp:33-40)
//
// Call sites work in a local length unit h (r_phys = h * r_local); the folded
// constants (a, b) absorb h so that phi(r_local^2) = phi_phys(h r_local):
//   bh3: a = -slope*h,   b = (c/h)^2   -> a * sqrt(r2 + b)
//   th3: a =  slope*h^3, b = (c/h)^2   -> a * rho^3, rho = sqrt(r2 + b)
//   exp: a =  psill,     b = -3 h / range -> a * exp(b * sqrt(r2))
#pragma once

#include "common.hpp"

namespace pam {

struct PhiConsts {
  double a, b;
};

inline PhiConsts phi_consts(const RbfDesc& rbf, double h) {
  switch (rbf.kind) {
    case kBh3: return {-rbf.p0 * h, (rbf.p1 / h) * (rbf.p1 / h)};
    case kTh3: return {rbf.p0 * h * h * h, (rbf.p1 / h) * (rbf.p1 / h)};
    case kExp: return {rbf.p0, -3.0 * h / rbf.p1};
  }
  throw_invalid("unknown rbf kind");
}

template <int KIND>
__device__ __forceinline__ double phi_f64(double r2, double a, double b) {
  if constexpr (KIND == kBh3) {
    return a * sqrt(r2 + b);
  } else if constexpr (KIND == kTh3) {
    double rho = sqrt(r2 + b);
    return a * (rho * rho * rho);
  } else {
    return a * exp(b * sqrt(r2));
  }
}

// FP32 form: raw hardware square root (v_sqrt_f32, ~1 ulp) and exp2-based exp.
template <int KIND>
__device__ __forceinline__ float phi_f32(float r2, float a, float b) {
  if constexpr (KIND == kBh3) {
    return a * __builtin_amdgcn_sqrtf(r2 + b);
  } else if constexpr (KIND == kTh3) {
    float rho = __builtin_amdgcn_sqrtf(r2 + b);
    return a * (rho * rho * rho);
  } else {
    return a * __expf(b * __builtin_amdgcn_sqrtf(r2));
  }
}

// The constant b that phi_shape<T> expects: the FP32 exponential is 2^(b r),
// with log2 e folded in before the rounding to FP32.
template <class T>
inline double phi_shape_const(int kind, double b) {
  return sizeof(T) == 4 && kind == kExp ? b * 1.4426950408889634074 : b;
}

// Square root for the FP64 sums, x > 0 and finite: the hardware reciprocal
// square root (v_rsq_f64, accurate to about 2^-23 relative), one Goldschmidt
// step and a Newton correction of the remainder (Markstein's method), within a
// few ulp of the correctly rounded sqrt in 7 instructions instead of the
// compiler's IEEE-rounded expansion. The correction's factor h needs no step
// of its own: its 2^-23 meet a remainder below 2^-44.
__device__ __forceinline__ double sqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double s0 = x * y, h = 0.5 * y;
  const double s = fma(s0, fma(-s0, h, 0.5), s0);
  return fma(fma(-s, s, x), h, s);
}

// 1 / sqrt(x), x > 0 and finite: the hardware's reciprocal root and one
// correction of third order, within an ulp.
__device__ __forceinline__ double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y, e * fma(0.375, e, 0.5), y);
}

// sum_k c_k m_k(x, y, z) over the monomials of degree 0..2
// (polynomial/monomial_basis.hpp:198-209 order: 1, x, y, z, x^2, xy, xz, y^2, yz, z^2).
__device__ __forceinline__ double poly_value(int degree, const double* __restrict__ c, double x, double y,
                                             double z) {
  double acc = c[0];
  if (degree >= 1) acc += c[1] * x + c[2] * y + c[3] * z;
  if (degree >= 2) acc += c[4] * x * x + c[5] * x * y + c[6] * x * z + c[7] * y * y + c[8] * y * z + c[9] * z * z;
  return acc;
}

// phi without its factor a, for loops that fold a into the weights:
// r2c = r^2 + b for bh3 / th3 (the caller seeds its sum of squares with b),
// r2c = r^2 for exp.
template <class T, int KIND>
__device__ __forceinline__ T phi_shape(T r2c, T b) {
  if constexpr (sizeof(T) == 8) {
    if constexpr (KIND == kBh3) {
      return sqrt_pos(r2c);
    } else if constexpr (KIND == kTh3) {
      return r2c * sqrt_pos(r2c);
    } else {
      return exp(b * sqrt_pos(r2c));
    }
  } else {
    if constexpr (KIND == kBh3) {
      return __builtin_amdgcn_sqrtf(r2c);
    } else if constexpr (KIND == kTh3) {
      return r2c * __builtin_amdgcn_sqrtf(r2c);
    } else {
      return __builtin_amdgcn_exp2f(b * __builtin_amdgcn_sqrtf(r2c));
    }
  }
}

// Seed of the sum of squares that phi_shape expects. FP64: at least 1e-290, so
// that the root of a coincident pair needs no test (r is then 1e-145 h).
template <class T, int KIND>
__device__ __forceinline__ T phi_seed(T b) {
  const T s = KIND == kExp ? T(0) : b;
  if constexpr (sizeof(T) == 8) return fmax(s, 1e-290);
  else return s;
}

// Gradient and Hessian in physical units from differences u in a local unit h
// (rbf/polyharmonic_odd.hpp:41-72, rbf/cov_exponential.hpp:42-62):
//   grad phi = ag f u,  H a = (ag / h) f (a + t u (u . a)),
// with (ag, b) from grad_consts(rbf, h) and f, t from grad_terms at
// r2c = |u|^2 + grad_seed(b):
//   bh3: ag = -slope,           f = 1 / sqrt(r2c)                      t = -1 / r2c
//   th3: ag = 3 slope h^2,      f = sqrt(r2c)                          t = 1 / r2c
//   exp: ag = -3 psill / range, f = exp(b r) / r, r = sqrt(r2c)        t = -(1 - b r) / r2c
// At r2c = 0 the polyharmonic terms are zero; the exponential's are undefined,
// as in the reference.
inline PhiConsts grad_consts(const RbfDesc& rbf, double h) {
  const PhiConsts pc = phi_consts(rbf, h);
  switch (rbf.kind) {
    case kBh3: return {pc.a / h, pc.b};
    case kTh3: return {3.0 * pc.a / h, pc.b};
    case kExp: return {pc.a * pc.b / h, pc.b};
  }
  throw_invalid("unknown rbf kind");
}

// FP64: at least 1e-200 (polyharmonic kernels), so that 1 / sqrt is finite.
template <class T, int KIND>
__device__ __forceinline__ T grad_seed(T b) {
  if constexpr (KIND == kExp) return T(0);
  else if constexpr (sizeof(T) == 8) return fmax(b, 1e-200);
  else return b;
}

template <class T, int KIND, bool kHess>
__device__ __forceinline__ void grad_terms(T r2c, T b, T* f, T* t) {
  if constexpr (sizeof(T) == 8) {
    if constexpr (KIND == kTh3 && !kHess) {
      *f = sqrt_pos(r2c);
    } else {
      const double y = rsqrt_nr(r2c);
      if constexpr (KIND == kBh3) {
        // The Hessian's first term does not vanish with u.
        *f = kHess && !(r2c > 1e-190) ? 0.0 : y;
        *t = -(y * y);
      } else if constexpr (KIND == kTh3) {
        *f = r2c * y;
        *t = y * y;
      } else {
        const double br = b * (r2c * y);
        *f = exp(br) * y;
        *t = (br - 1.0) * (y * y);
      }
    }
  } else {
    if constexpr (KIND == kBh3) {
      *f = r2c > 0.0f ? __builtin_amdgcn_rsqf(r2c) : 0.0f;
      *t = r2c > 0.0f ? -1.0f / r2c : 0.0f;
    } else if constexpr (KIND == kTh3) {
      *f = __builtin_amdgcn_sqrtf(r2c);
      *t = r2c > 0.0f ? 1.0f / r2c : 0.0f;
    } else {
      const float rs = __builtin_amdgcn_rsqf(r2c);
      *f = __expf(b * (r2c * rs)) * rs;
      *t = -(1.0f - b * sqrtf(r2c)) / r2c;
    }
  }
}

template <class T, int KIND>
__device__ __forceinline__ T phi_t(T r2, T a, T b) {
  if constexpr (sizeof(T) == 8) {
    return phi_f64<KIND>(r2, a, b);
  } else {
    return phi_f32<KIND>(r2, a, b);
  }
}

// Value, gradient and Hessian of the isotropic kernel at a difference u that
// is already transformed by the anisotropy (rbf/polyharmonic_odd.hpp:32-72,
// rbf/cov_exponential.hpp:33-62). Polyharmonic of degree K (bh3: K = 1, sign
// -1; th3: K = 3, sign +1), rho = sqrt(|u|^2 + c^2):
//   g = sign K slope rho^(K-2) u,  H = sign K slope rho^(K-2) (I + (K-2) u u^T / rho^2),
//   both zero at rho = 0.
// Exponential, r = |u|:
//   g = -3 psill e^(-3 r / range) / (range r) u,
//   H = (same factor) (I - (1/r^2 + 3 / (range r)) u u^T)   (no guard at r = 0).
template <int KIND>
__host__ __device__ inline double rbf_value_iso(double p0, double p1, const double u[3]) {
  const double q = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  if constexpr (KIND == kBh3) {
    return -p0 * sqrt(q + p1 * p1);
  } else if constexpr (KIND == kTh3) {
    const double rho = sqrt(q + p1 * p1);
    return p0 * (rho * rho * rho);
  } else {
    return p0 * exp(-3.0 * (sqrt(q) / p1));
  }
}

template <int KIND>
__host__ __device__ inline double rbf_grad_factor(double p0, double p1, const double u[3], double* t) {
  // Returns the factor f with g = f u; t receives the coefficient of u u^T in
  // H / f - I.
  const double q = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  if constexpr (KIND == kBh3 || KIND == kTh3) {
    constexpr int K = KIND == kBh3 ? 1 : 3;
    constexpr double sign = KIND == kBh3 ? -1.0 : 1.0;
    const double rho2 = q + p1 * p1;
    const double rho = sqrt(rho2);
    if (rho == 0.0) {
      *t = 0.0;
      return 0.0;
    }
    *t = (K - 2) / rho2;
    const double rk = K == 1 ? 1.0 / rho : rho;  // rho^(K-2)
    return sign * K * p0 * rk;
  } else {
    const double r = sqrt(q);
    *t = -(1.0 / (r * r) + 3.0 / (p1 * r));
    return -3.0 * p0 * exp(-3.0 * (r / p1)) / (p1 * r);
  }
}

template <int KIND>
__host__ __device__ inline void rbf_grad_iso(double p0, double p1, const double u[3], double g[3]) {
  double t;
  const double f = rbf_grad_factor<KIND>(p0, p1, u, &t);
  for (int k = 0; k < 3; k++) g[k] = f * u[k];
}

template <int KIND>
__host__ __device__ inline void rbf_hess_iso(double p0, double p1, const double u[3], double h[9]) {
  double t;
  const double f = rbf_grad_factor<KIND>(p0, p1, u, &t);
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) h[3 * i + j] = f * ((i == j ? 1.0 : 0.0) + t * u[i] * u[j]);
}

// Dispatch a templated functor on the runtime kind.
template <class F>
inline void dispatch_kind(int kind, F&& f) {
  switch (kind) {
    case kBh3: f(std::integral_constant<int, kBh3>{}); return;
    case kTh3: f(std::integral_constant<int, kTh3>{}); return;
    case kExp: f(std::integral_constant<int, kExp>{}); return;
  }
  throw_invalid("unknown rbf kind");
}

}  // namespace pam
