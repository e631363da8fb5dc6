// FP64 direct O(N M) sums: values, gradients, Hessian columns, and the sums
// over sources with 3-vector weights (gradient data), in one kernel.
//
// Bound by FP64 VALU issue. Per pair three differences, three FMAs and a
// square root (or its reciprocal) from the hardware's reciprocal root with one
// correction of third order, instead of the compiler's rounded root (and
// division): about 22 FP64 operations for a value of a polyharmonic kernel.
// The sum of squares is seeded with the kernel's offset or 1e-290, so that a
// coincident pair needs no test; squares that overflow give NaN this way, and
// a workgroup whose sums are not numbers adds its range again with the plain
// expressions. Sources with 3-vector weights are summed in one pass over the
// pairs (three gradient passes or three Hessian columns before).
// MI355X, triharmonic, 30,011 points + 15,013 with vector weights, all pairs:
// values 0.96 to 0.68 ms, values from vector weights 1.43 to 0.39 ms,
// gradients 0.72 to 0.37 ms, gradients from vector weights 4.2 to 0.25 ms.
#include <algorithm>
#include <cstring>
#include <vector>

#include "device_api.hpp"
#include "rbf_device.hpp"

namespace pam {

namespace {

constexpr int kDt = 256;  // threads; sources staged per tile

// What a direct sum adds up per pair, u = t - s, phi' the kernel's gradient
// factor (grad phi = phi' u), H its Hessian:
//   kDirValue     w phi                      one output
//   kDirGradient  w grad phi                 three
//   kDirDipole    -(v . grad phi)            one, v the source's vector weight
//   kDirHessian   -H v                       three
enum DirectMode : int { kDirValue = 0, kDirGradient = 1, kDirDipole = 2, kDirHessian = 3 };
constexpr int out_per(int mode) { return mode == kDirValue || mode == kDirDipole ? 1 : 3; }
constexpr bool vector_weights(int mode) { return mode == kDirDipole || mode == kDirHessian; }

// Constants of a direct sum: a multiplies the weights (kernel or gradient
// factor), b as in phi_shape / grad_terms; p0, p1 for the plain expressions.
struct DirectConsts {
  double a, b, p0, p1;
};

DirectConsts direct_consts(const RbfDesc& rbf, int mode) {
  const PhiConsts c = mode == kDirValue ? phi_consts(rbf, 1.0) : grad_consts(rbf, 1.0);
  return {mode >= kDirDipole ? -c.a : c.a, c.b, rbf.p0, rbf.p1};
}

// How n_trg targets and n_src sources are shared out: workgroups of tp target
// slots (R targets each) x kDt / tp source splits, sources in nchunks chunks.
struct DirectSplit {
  int r, tp, gx, nchunks;
  int64_t chunk;
};

DirectSplit direct_split(int64_t n_trg, int64_t n_src) {
  DirectSplit d;
  // Many targets: 256 slots of two targets. Fewer: 64 slots (a wavefront),
  // four splits of the sources; below that as many slots as targets. 257
  // targets x 10,000 sources: 87 us with 256 slots and chunks of 1,024, 8 us
  // this way. One, two or four targets per thread between 16,384 and 32,768
  // targets are within 7 % of each other.
  d.r = n_trg >= 16384 ? 2 : 1;
  d.tp = n_trg >= 32768 ? kDt : 64;
  while (d.tp > 1 && d.tp / 2 >= n_trg) d.tp /= 2;
  d.gx = ceil_div(n_trg, static_cast<int64_t>(d.tp) * d.r);
  // Enough workgroups to fill 256 CUs several times, at least 64 sources per
  // thread (1,024 where a workgroup covers 512 targets).
  const int64_t want = std::max<int64_t>(1, (2048 + static_cast<int64_t>(d.gx) * d.r - 1) / (static_cast<int64_t>(d.gx) * d.r));
  const int64_t least = d.tp == kDt ? 1024 : 64 * (kDt / d.tp);
  d.chunk = std::max((n_src + want - 1) / want, least);
  d.nchunks = static_cast<int>(n_src > 0 ? (n_src + d.chunk - 1) / d.chunk : 1);
  return d;
}

// One pair's term into acc. w: the weight or the vector weight times
// DirectConsts::a; r2 is seeded (direct_seed).
template <int KIND, int MODE>
__device__ __forceinline__ void direct_pair(double dx, double dy, double dz, double r2, double b, const double (&w)[3],
                                            double (&acc)[3]) {
  if constexpr (MODE == kDirValue) {
    const double rho = sqrt_pos(r2);
    if constexpr (KIND == kBh3) acc[0] = fma(w[0], rho, acc[0]);
    else if constexpr (KIND == kTh3) acc[0] = fma(w[0], rho * r2, acc[0]);
    else acc[0] = fma(w[0], exp(b * rho), acc[0]);
  } else {
    double f, t = 0.0;  // as in grad_terms
    if constexpr (KIND == kTh3 && MODE != kDirHessian) {
      f = sqrt_pos(r2);
    } else {
      const double y = rsqrt_nr(r2);
      if constexpr (KIND == kBh3) {
        f = y;
        if constexpr (MODE == kDirHessian) {
          t = -(y * y);
          f = r2 > 1e-280 ? f : 0.0;  // zero for coincident points, where the vector's own term is left
        }
      } else if constexpr (KIND == kTh3) {
        f = r2 * y;
        t = y * y;
      } else {
        const double br = b * (r2 * y);
        f = exp(br) * y;
        t = (br - 1.0) * (y * y);
      }
    }
    if constexpr (MODE == kDirGradient) {
      f *= w[0];
      acc[0] = fma(f, dx, acc[0]);
      acc[1] = fma(f, dy, acc[1]);
      acc[2] = fma(f, dz, acc[2]);
    } else {
      const double uv = fma(dz, w[2], fma(dy, w[1], dx * w[0]));
      if constexpr (MODE == kDirDipole) {
        acc[0] = fma(f, uv, acc[0]);
      } else {
        const double tu = t * uv;
        acc[0] = fma(f, fma(tu, dx, w[0]), acc[0]);
        acc[1] = fma(f, fma(tu, dy, w[1]), acc[1]);
        acc[2] = fma(f, fma(tu, dz, w[2]), acc[2]);
      }
    }
  }
}

// The same term by the plain expressions; w without the factor DirectConsts::a
// except its sign.
template <int KIND, int MODE>
__device__ void direct_pair_plain(const double (&u)[3], const DirectConsts& c, const double (&w)[3], double (&acc)[3]) {
  if constexpr (MODE == kDirValue) {
    acc[0] += w[0] * rbf_value_iso<KIND>(c.p0, c.p1, u);
  } else {
    double t;
    const double f = rbf_grad_factor<KIND>(c.p0, c.p1, u, &t);
    if constexpr (MODE == kDirGradient) {
      for (int k = 0; k < 3; k++) acc[k] += w[0] * (f * u[k]);
    } else {
      const double uv = u[0] * w[0] + u[1] * w[1] + u[2] * w[2];
      if constexpr (MODE == kDirDipole) {
        acc[0] -= f * uv;
      } else {
        for (int k = 0; k < 3; k++) acc[k] -= f * (w[k] + t * u[k] * uv);
      }
    }
  }
}

template <int MODE>
struct DirectTile {
  double4 p[kDt];                               // position, weight
  double v[vector_weights(MODE) ? kDt : 1][3];  // vector weight
};

// Sum of a thread's R targets (t) over its share of the sources [j0, j1):
// tile slots si, si + splits, .... a3: the vector weights' map (A for data
// weights; null: the weight times the vector col). Every thread of the
// workgroup takes part.
template <int KIND, int MODE, int R, class W>
__device__ __forceinline__ void direct_range(DirectTile<MODE>& tile, const DirectConsts& c,
                                             const double* __restrict__ src, W weight, int64_t j0, int64_t j1, int si,
                                             int splits, const double (&t)[R][3], double (&acc)[R][3]) {
  constexpr bool kVec = vector_weights(MODE);
  // No seed for the exponential's gradient, which is undefined at r = 0.
  const double seed = KIND == kExp ? (MODE == kDirValue ? 1e-290 : 0.0) : fmax(c.b, 1e-290);
#pragma unroll
  for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = acc[r][2] = 0.0;
  bool plain = false;
  for (;;) {
    for (int64_t jt = j0; jt < j1; jt += kDt) {
      __syncthreads();
      const int64_t j = jt + threadIdx.x;
      if (j < j1) {
        double w[3];
        weight(j, plain ? 1.0 : c.a, w);
        tile.p[threadIdx.x] = make_double4(src[3 * j], src[3 * j + 1], src[3 * j + 2], w[0]);
        if constexpr (kVec)
          for (int k = 0; k < 3; k++) tile.v[threadIdx.x][k] = w[k];
      }
      __syncthreads();
      const int cnt = static_cast<int>(j1 - jt < kDt ? j1 - jt : kDt);
      if (!plain) {
#pragma unroll 4
        for (int k = si; k < cnt; k += splits) {
          const double4 q = tile.p[k];
          const double w[3] = {q.w, kVec ? tile.v[kVec ? k : 0][1] : 0.0, kVec ? tile.v[kVec ? k : 0][2] : 0.0};
#pragma unroll
          for (int r = 0; r < R; r++) {
            const double dx = t[r][0] - q.x, dy = t[r][1] - q.y, dz = t[r][2] - q.z;
            direct_pair<KIND, MODE>(dx, dy, dz, fma(dz, dz, fma(dy, dy, fma(dx, dx, seed))), c.b, w, acc[r]);
          }
        }
      } else {
        for (int k = si; k < cnt; k += splits) {
          const double4 q = tile.p[k];
          const double w[3] = {q.w, kVec ? tile.v[kVec ? k : 0][1] : 0.0, kVec ? tile.v[kVec ? k : 0][2] : 0.0};
          for (int r = 0; r < R; r++) {
            const double u[3] = {t[r][0] - q.x, t[r][1] - q.y, t[r][2] - q.z};
            direct_pair_plain<KIND, MODE>(u, c, w, acc[r]);
          }
        }
      }
    }
    bool bad = false;
#pragma unroll
    for (int r = 0; r < R; r++) bad |= !(fabs(acc[r][0]) + fabs(acc[r][1]) + fabs(acc[r][2]) < INFINITY);
    if (plain || !__syncthreads_or(bad)) return;
    plain = true;
    for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = acc[r][2] = 0.0;
  }
}

// Sums of the source splits, in order, for the threads of split 0.
template <int MODE, int R>
__device__ __forceinline__ void direct_fold(double (*red)[kDt], int tp, int ti, int si, double (&acc)[R][3]) {
  constexpr int kOut = out_per(MODE);
  const int splits = kDt / tp;
  if (splits == 1) return;
#pragma unroll
  for (int r = 0; r < R; r++)
    for (int k = 0; k < kOut; k++) {
      __syncthreads();
      red[0][threadIdx.x] = acc[r][k];
      __syncthreads();
      if (si == 0) {
        double s = red[0][ti];
        for (int m = 1; m < splits; m++) s += red[0][ti + m * tp];
        acc[r][k] = s;
      }
    }
}

struct DirectArgs {
  DirectConsts c;
  const double* src;
  const double* w;   // n_src, or 3 n_src data weights (mapped by a)
  int64_t n_src;
  const double* trg;
  int64_t n_trg;
  double* partial;   // [chunk][target][out_per]
  int64_t chunk;
  int tp;
  double a[9];       // row-major map of the vector weights: v = a w3
  double col[3];     // scalar weights in a Hessian sum: v = w col
  int scalar;        // the weights are scalars
};

template <int KIND, int MODE, int R>
__global__ void __launch_bounds__(kDt) direct_kernel(DirectArgs g) {
  __shared__ DirectTile<MODE> tile;
  __shared__ double red[1][kDt];
  const int tp = g.tp, splits = kDt / tp;
  const int ti = threadIdx.x & (tp - 1), si = threadIdx.x / tp;
  const int64_t j0 = static_cast<int64_t>(blockIdx.y) * g.chunk;
  const int64_t j1 = j0 + g.chunk < g.n_src ? j0 + g.chunk : g.n_src;
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * tp * R + ti;
  double t[R][3], acc[R][3];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = i0 + static_cast<int64_t>(r) * tp;
    for (int k = 0; k < 3; k++) t[r][k] = i < g.n_trg ? g.trg[3 * i + k] : 0.0;
  }
  auto weight = [&](int64_t j, double f, double (&w)[3]) {
    if constexpr (!vector_weights(MODE)) {
      w[0] = f * g.w[j];
    } else if (g.scalar) {
      const double s = f * g.w[j];
      for (int k = 0; k < 3; k++) w[k] = s * g.col[k];
    } else {
      const double x = g.w[3 * j], y = g.w[3 * j + 1], z = g.w[3 * j + 2];
      for (int k = 0; k < 3; k++) w[k] = f * (fma(g.a[3 * k + 2], z, fma(g.a[3 * k + 1], y, g.a[3 * k] * x)));
    }
  };
  direct_range<KIND, MODE, R>(tile, g.c, g.src, weight, j0, j1, si, splits, t, acc);
  direct_fold<MODE, R>(red, tp, ti, si, acc);
  if (si != 0) return;
  constexpr int kOut = out_per(MODE);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = i0 + static_cast<int64_t>(r) * tp;
    if (i >= g.n_trg) continue;
    for (int k = 0; k < kOut; k++)
      g.partial[(static_cast<int64_t>(blockIdx.y) * g.n_trg + i) * kOut + k] = acc[r][k];
  }
}

// Chunks in order; n: targets x outputs per target.
__global__ void reduce_partial_kernel(const double* __restrict__ partial, int nchunks, int64_t n,
                                      double* __restrict__ out, int accumulate) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double acc = 0.0;
#pragma unroll 8
  for (int c = 0; c < nchunks; c++) acc += partial[c * n + i];
  out[i] = accumulate ? out[i] + acc : acc;
}

struct Map3 {
  double a[9];
};

// out[i] = A^T (sum of the chunks in order)
__global__ void reduce_partial3_kernel(const double* __restrict__ partial, int nchunks, int64_t n_trg, Map3 A,
                                       double* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n_trg) return;
  double g[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
  for (int c = 0; c < nchunks; c++)
    for (int k = 0; k < 3; k++) g[k] += partial[(static_cast<int64_t>(c) * n_trg + i) * 3 + k];
  for (int k = 0; k < 3; k++) out[3 * i + k] = (A.a[k] * g[0] + A.a[3 + k] * g[1]) + A.a[6 + k] * g[2];
}

__global__ void fill_f64_kernel(double* __restrict__ out, int64_t n, double v) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = v;
}

template <int MODE>
void launch_direct(const RbfDesc& rbf, DirectArgs g, const DirectSplit& d, hipStream_t s) {
  g.c = direct_consts(rbf, MODE);
  g.chunk = d.chunk;
  g.tp = d.tp;
  const dim3 grid(d.gx, d.nchunks);
  dispatch_kind(rbf.kind, [&](auto k) {
    constexpr int K = decltype(k)::value;
    if (d.r == 2) direct_kernel<K, MODE, 2><<<grid, kDt, 0, s>>>(g);
    else direct_kernel<K, MODE, 1><<<grid, kDt, 0, s>>>(g);
  });
  PAM_LAUNCH_CHECK();
}

// A sum with three outputs per target: partials, then A^T of their sum.
template <int MODE>
void direct_sum3(const RbfDesc& rbf, DirectArgs g, double* out3, DevBuf<double>& scratch, hipStream_t s) {
  if (g.n_trg == 0) return;
  Map3 A;
  for (int k = 0; k < 9; k++) A.a[k] = rbf.aniso[k];
  int nchunks = 0;
  if (g.n_src > 0) {
    const DirectSplit d = direct_split(g.n_trg, g.n_src);
    nchunks = d.nchunks;
    scratch.resize(static_cast<size_t>(nchunks) * g.n_trg * 3);
    g.partial = scratch.get();
    launch_direct<MODE>(rbf, g, d, s);
  }
  reduce_partial3_kernel<<<ceil_div(g.n_trg, 256), 256, 0, s>>>(scratch.get(), nchunks, g.n_trg, A, out3);
  PAM_LAUNCH_CHECK();
}

// ---- batched FP64 direct sums: several query sets, each against its own
// models' sources, in one launch and one reduction ----
//
// A segment is one (query set, rbf) pair. It is split into target blocks and
// source chunks by the same rule as a single direct sum, so its partial sums,
// and hence every query set's result, do not depend on which other query sets
// share the launch.
struct DirSeg {
  const double* src;  // transformed sources, n_src x 3
  const double* w;    // weights, n_src
  int64_t n_src, chunk;
  int64_t part_off;   // its partial sums: nchunks x q_n
  int64_t q_off, q_n; // rows of the concatenated query points
  int32_t kind, gx, nchunks, work_first, tp, r;
  DirectConsts c;
  double a[9];        // anisotropy applied to the query points on load
};
static_assert(sizeof(DirSeg) % sizeof(double) == 0, "DirSeg is staged as doubles");

struct DirQuery {
  int64_t off, n;
  int32_t seg_first, n_seg, degree, pad;
  const double* coeffs;
};
static_assert(sizeof(DirQuery) % sizeof(double) == 0, "DirQuery is staged as doubles");

template <int R>
__device__ __forceinline__ void direct_segment(DirectTile<kDirValue>& tile, double (*red)[kDt], const DirSeg& g,
                                               int bx, int by, const double* __restrict__ pts,
                                               double* __restrict__ partial) {
  const int tp = g.tp, splits = kDt / tp;
  const int ti = threadIdx.x & (tp - 1), si = threadIdx.x / tp;
  const int64_t j0 = static_cast<int64_t>(by) * g.chunk;
  const int64_t j1 = j0 + g.chunk < g.n_src ? j0 + g.chunk : g.n_src;
  const int64_t i0 = static_cast<int64_t>(bx) * tp * R + ti;
  double t[R][3], acc[R][3];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = i0 + static_cast<int64_t>(r) * tp;
    t[r][0] = t[r][1] = t[r][2] = 0.0;
    if (i < g.q_n) {
      const double* p = pts + 3 * (g.q_off + i);
      const double x = p[0], y = p[1], z = p[2];
      // the rounding of transform_kernel
      for (int k = 0; k < 3; k++)
        t[r][k] = __dadd_rn(__dadd_rn(__dmul_rn(g.a[3 * k], x), __dmul_rn(g.a[3 * k + 1], y)),
                            __dmul_rn(g.a[3 * k + 2], z));
    }
  }
  auto weight = [&](int64_t j, double f, double (&w)[3]) { w[0] = f * g.w[j]; };
  switch (g.kind) {
    case kBh3: direct_range<kBh3, kDirValue, R>(tile, g.c, g.src, weight, j0, j1, si, splits, t, acc); break;
    case kTh3: direct_range<kTh3, kDirValue, R>(tile, g.c, g.src, weight, j0, j1, si, splits, t, acc); break;
    default: direct_range<kExp, kDirValue, R>(tile, g.c, g.src, weight, j0, j1, si, splits, t, acc); break;
  }
  direct_fold<kDirValue, R>(red, tp, ti, si, acc);
  if (si != 0) return;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = i0 + static_cast<int64_t>(r) * tp;
    if (i < g.q_n) partial[g.part_off + static_cast<int64_t>(by) * g.q_n + i] = acc[r][0];
  }
}

__global__ void __launch_bounds__(kDt)
direct_batch_kernel(const DirSeg* __restrict__ segs, int nseg, const double* __restrict__ pts,
                    double* __restrict__ partial) {
  __shared__ DirectTile<kDirValue> tile;
  __shared__ double red[1][kDt];
  const int b = static_cast<int>(blockIdx.x);
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (segs[mid].work_first <= b) lo = mid;
    else hi = mid - 1;
  }
  const DirSeg& g = segs[lo];
  const int local = b - g.work_first;
  if (g.r == 2) direct_segment<2>(tile, red, g, local % g.gx, local / g.gx, pts, partial);
  else direct_segment<1>(tile, red, g, local % g.gx, local / g.gx, pts, partial);
}

// One thread per query row: each segment's chunks summed in chunk order, the
// segments of a query set added in rbf order, then its polynomial.
__global__ void direct_batch_reduce_kernel(const DirQuery* __restrict__ qs, int nq,
                                           const DirSeg* __restrict__ segs, const double* __restrict__ pts,
                                           const double* __restrict__ partial, double* __restrict__ out,
                                           int64_t rows) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= rows) return;
  int lo = 0, hi = nq - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (qs[mid].off <= t) lo = mid;
    else hi = mid - 1;
  }
  const DirQuery& q = qs[lo];
  const int64_t i = t - q.off;
  double v = 0.0;
  for (int k = 0; k < q.n_seg; k++) {
    const DirSeg& g = segs[q.seg_first + k];
    double acc = 0.0;
#pragma unroll 8
    for (int c = 0; c < g.nchunks; c++) acc += partial[g.part_off + static_cast<int64_t>(c) * g.q_n + i];
    v = k == 0 ? acc : v + acc;
  }
  if (q.degree >= 0) v += poly_value(q.degree, q.coeffs, pts[3 * t], pts[3 * t + 1], pts[3 * t + 2]);
  out[t] = v;
}

}  // namespace

size_t direct_partial_size(int64_t n_trg, int64_t n_src) {
  return n_trg == 0 ? 0 : static_cast<size_t>(direct_split(n_trg, n_src).nchunks) * n_trg;
}

void direct_sum_f64_into(const RbfDesc& rbf, const double* src, const double* w, int64_t n_src,
                         const double* trg, int64_t n_trg, double* out, bool accumulate, double* partial,
                         hipStream_t s) {
  if (n_trg == 0) return;
  const DirectSplit d = direct_split(n_trg, n_src);
  if (n_src == 0) {
    fill_f64_kernel<<<ceil_div(n_trg, 256), 256, 0, s>>>(partial, n_trg, 0.0);
    PAM_LAUNCH_CHECK();
  } else {
    DirectArgs g{};
    g.src = src;
    g.w = w;
    g.n_src = n_src;
    g.trg = trg;
    g.n_trg = n_trg;
    g.partial = partial;
    launch_direct<kDirValue>(rbf, g, d, s);
  }
  reduce_partial_kernel<<<ceil_div(n_trg, 256), 256, 0, s>>>(partial, d.nchunks, n_trg, out, accumulate ? 1 : 0);
  PAM_LAUNCH_CHECK();
}

void direct_sum_f64(const RbfDesc& rbf, const double* src, const double* w, int64_t n_src,
                    const double* trg, int64_t n_trg, double* out, bool accumulate,
                    DevBuf<double>& scratch, hipStream_t s) {
  if (n_trg == 0) return;
  scratch.resize(direct_partial_size(n_trg, n_src));
  direct_sum_f64_into(rbf, src, w, n_src, trg, n_trg, out, accumulate, scratch.get(), s);
}

void direct_gradient_f64(const RbfDesc& rbf, const double* src, const double* w, int64_t n_src,
                         const double* trg, int64_t n_trg, double* out3, DevBuf<double>& scratch,
                         hipStream_t s) {
  DirectArgs g{};
  g.src = src;
  g.w = w;
  g.n_src = n_src;
  g.trg = trg;
  g.n_trg = n_trg;
  direct_sum3<kDirGradient>(rbf, g, out3, scratch, s);
}

void direct_hessian_column_f64(const RbfDesc& rbf, const double* src, const double* w, int64_t n_src,
                               const double* trg, int64_t n_trg, int kcol, double* out3, DevBuf<double>& scratch,
                               hipStream_t s) {
  if (n_trg == 0) return;
  if (kcol < 0 || kcol > 2) throw_invalid("Hessian column out of range");
  DirectArgs g{};
  g.src = src;
  g.w = w;
  g.n_src = n_src;
  g.trg = trg;
  g.n_trg = n_trg;
  g.scalar = 1;
  // the sum of H a_k w has the sign opposite to the vector-weight sum's
  for (int k = 0; k < 3; k++) g.col[k] = -rbf.aniso[3 * k + kcol];
  direct_sum3<kDirHessian>(rbf, g, out3, scratch, s);
}

void direct_dipole_f64(const RbfDesc& rbf, const double* src, const double* w3, int64_t n_src, const double* trg,
                       int64_t n_trg, double* out, DevBuf<double>& scratch, hipStream_t s) {
  if (n_trg == 0) return;
  const DirectSplit d = direct_split(n_trg, n_src);
  scratch.resize(static_cast<size_t>(d.nchunks) * n_trg);
  if (n_src > 0) {
    DirectArgs g{};
    g.src = src;
    g.w = w3;
    g.n_src = n_src;
    g.trg = trg;
    g.n_trg = n_trg;
    g.partial = scratch.get();
    for (int k = 0; k < 9; k++) g.a[k] = rbf.aniso[k];
    launch_direct<kDirDipole>(rbf, g, d, s);
  }
  reduce_partial_kernel<<<ceil_div(n_trg, 256), 256, 0, s>>>(scratch.get(), n_src > 0 ? d.nchunks : 0, n_trg, out, 0);
  PAM_LAUNCH_CHECK();
}

void direct_dipole_hessian_f64(const RbfDesc& rbf, const double* src, const double* w3, int64_t n_src,
                               const double* trg, int64_t n_trg, double* out3, DevBuf<double>& scratch,
                               hipStream_t s) {
  DirectArgs g{};
  g.src = src;
  g.w = w3;
  g.n_src = n_src;
  g.trg = trg;
  g.n_trg = n_trg;
  for (int k = 0; k < 9; k++) g.a[k] = rbf.aniso[k];
  direct_sum3<kDirHessian>(rbf, g, out3, scratch, s);
}

void DirectBatch::run(const std::vector<DirectBatchQuery>& queries,
                      const std::vector<DirectBatchTerm>& terms, hipStream_t s) {
  std::vector<DirSeg> segs;
  std::vector<DirQuery> qs;
  int64_t rows = 0, part = 0, work = 0;
  for (const DirectBatchQuery& q : queries) {
    if (q.n < 0) throw_invalid("negative query count");
    if (q.n == 0) continue;
    if (!q.pts || !q.out) throw_invalid("null query or output buffer");
    if (q.n_terms < 1 || q.first_term < 0 || q.first_term + q.n_terms > static_cast<int>(terms.size()))
      throw_invalid("query terms out of range");
    if (q.poly_degree > 2) throw_invalid("polynomial degree must be at most 2");
    if (q.poly_degree >= 0 && !q.coeffs) throw_invalid("null polynomial coefficients");
    DirQuery d{};
    d.off = rows;
    d.n = q.n;
    d.seg_first = static_cast<int32_t>(segs.size());
    d.n_seg = q.n_terms;
    d.degree = q.poly_degree;
    d.coeffs = q.coeffs;
    qs.push_back(d);
    for (int k = q.first_term; k < q.first_term + q.n_terms; k++) {
      const DirectBatchTerm& t = terms[k];
      if (t.n_src < 1 || !t.src || !t.w) throw_invalid("a batched term needs sources and weights");
      DirSeg g{};
      g.src = t.src;
      g.w = t.w;
      g.n_src = t.n_src;
      const DirectSplit sp = direct_split(q.n, t.n_src);
      g.gx = sp.gx;
      g.chunk = sp.chunk;
      g.nchunks = sp.nchunks;
      g.tp = sp.tp;
      g.r = sp.r;
      g.part_off = part;
      g.q_off = rows;
      g.q_n = q.n;
      g.kind = t.rbf.kind;
      g.work_first = static_cast<int32_t>(work);
      g.c = direct_consts(t.rbf, kDirValue);
      for (int e = 0; e < 9; e++) g.a[e] = t.rbf.aniso[e];
      segs.push_back(g);
      part += static_cast<int64_t>(g.nchunks) * q.n;
      work += static_cast<int64_t>(g.gx) * g.nchunks;
      if (work > (int64_t{1} << 30)) throw_invalid("batched direct sum too large for one launch");
    }
    rows += q.n;
  }
  if (rows == 0) return;
  // One upload: segment table, query table, then the query points.
  const size_t seg_d = segs.size() * sizeof(DirSeg) / sizeof(double);
  const size_t q_d = qs.size() * sizeof(DirQuery) / sizeof(double);
  const size_t total = seg_d + q_d + static_cast<size_t>(rows) * 3;
  double* h = up_.acquire(total);
  std::memcpy(h, segs.data(), segs.size() * sizeof(DirSeg));
  std::memcpy(h + seg_d, qs.data(), qs.size() * sizeof(DirQuery));
  double* hp = h + seg_d + q_d;
  for (const DirectBatchQuery& q : queries) {
    if (q.n == 0) continue;
    std::memcpy(hp, q.pts, sizeof(double) * 3 * static_cast<size_t>(q.n));
    hp += 3 * q.n;
  }
  up_.upload(d_in_, total, s);
  const DirSeg* d_segs = reinterpret_cast<const DirSeg*>(d_in_.get());
  const DirQuery* d_qs = reinterpret_cast<const DirQuery*>(d_in_.get() + seg_d);
  const double* d_pts = d_in_.get() + seg_d + q_d;
  d_part_.resize(static_cast<size_t>(part));
  d_out_.resize(static_cast<size_t>(rows));
  direct_batch_kernel<<<static_cast<unsigned>(work), kDt, 0, s>>>(d_segs, static_cast<int>(segs.size()),
                                                                          d_pts, d_part_.get());
  PAM_LAUNCH_CHECK();
  direct_batch_reduce_kernel<<<ceil_div(rows, 256), 256, 0, s>>>(d_qs, static_cast<int>(qs.size()), d_segs, d_pts,
                                                                d_part_.get(), d_out_.get(), rows);
  PAM_LAUNCH_CHECK();
  double* ho = down_.acquire(static_cast<size_t>(rows));
  PAM_HIP(hipMemcpyAsync(ho, d_out_.get(), sizeof(double) * rows, hipMemcpyDeviceToHost, s));
  PAM_HIP(hipStreamSynchronize(s));
  for (const DirectBatchQuery& q : queries) {
    if (q.n == 0) continue;
    std::memcpy(q.out, ho, sizeof(double) * static_cast<size_t>(q.n));
    ho += q.n;
  }
}

}  // namespace pam
