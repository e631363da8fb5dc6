// Dense FP64 kernels of the coarse grid (about 2,000 to 6,000 rows).
//
// The factorisation is right-looking with 64-wide panels, two launches per
// panel: every workgroup of the first factors the diagonal block for itself
// (one wavefront, rows in registers, pivots broadcast by lane reads) and
// multiplies its 64 rows by the block's inverse, the second updates the
// trailing tiles on FP64 MFMA. What bounds it is the chain of diagonal
// blocks. The solve is then made an operator by inverting the factor (block
// pairs of doubling size, two products each) and forming W = L^-T L^-1: about
// n^3 multiply-adds of FP64 MFMA in place of one sequential pair of
// triangular solves per row of the operator.
// 2,048 rows on MI355X: a panel step 55 us (40 + 15), the factorisation 1.8 ms
// (6.5 ms with 32-wide panels, one wavefront in LDS and three launches), the
// operator 0.46 ms (7.4 ms).
#include "coarse_dense.hpp"

namespace pam {

namespace {

constexpr int kCt = 256;   // threads
constexpr int kB = kCoarseBlk;
constexpr int kSub = 16;   // rows that one wavefront factors in registers
constexpr int kKc = 32;    // reduction chunk of the products
constexpr double kTiny = 1e-300;

using d64x4 = double __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(u)), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(u >> 32)), lane);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// 1 / sqrt(p) to about an ulp: the hardware's 2^-23 and one step of third order.
__device__ __forceinline__ double rsqrt_f64(double p) {
  const double y = __builtin_amdgcn_rsq(p);
  const double e = fma(-(p * y), y, 1.0);
  return fma(y, e * fma(0.375, e, 0.5), y);
}

// Cholesky factor and inverse of the 16 x 16 block of dg at (off, off) by one
// wavefront: lane r (and r + 16, ...) holds row r of the factor, then column r
// of the inverse. Both eliminate column by column, so that the updates of a
// step are independent and only the pivots form a chain. (A 32 x 32 block
// this way is straight-line code of some 25 KB, and fetching it took longer
// than running it: 70 us a panel step.)
__device__ __forceinline__ void wave_factor16(double (*dg)[kB + 1], double (*inv)[kB + 1], int off,
                                           int32_t* __restrict__ flag) {
  const int lane = threadIdx.x & 63, r = lane & (kSub - 1);
  double row[kSub];
#pragma unroll
  for (int c = 0; c < kSub; c++) row[c] = dg[off + r][off + c];
  bool bad = false;
  double rd = 0.0;  // lane r: 1 / L_rr
#pragma unroll
  for (int j = 0; j < kSub; j++) {
    double p = lane_value(row[j], j);
    if (!(p > 0.0)) {
      bad = true;
      p = fabs(p) + kTiny;
    }
    const double y = rsqrt_f64(p);
    if (r == j) rd = y;
    const double d = p * y;
    row[j] = r == j ? fma(fma(-d, d, p), 0.5 * y, d) : row[j] * y;
#pragma unroll
    for (int c = j + 1; c < kSub; c++) row[c] = fma(-row[j], lane_value(row[j], c), row[c]);
  }
  if (bad && lane == 0) atomicExch(flag, 1);
  double x[kSub];
#pragma unroll
  for (int i = 0; i < kSub; i++) x[i] = i == r ? 1.0 : 0.0;
#pragma unroll
  for (int i = 0; i < kSub; i++) {
    x[i] *= lane_value(rd, i);
#pragma unroll
    for (int k = i + 1; k < kSub; k++) x[k] = fma(-lane_value(row[i], k), x[i], x[k]);
  }
  if (lane < kSub) {
#pragma unroll
    for (int c = 0; c < kSub; c++) {
      dg[off + r][off + c] = c <= r ? row[c] : 0.0;
      inv[off + c][off + r] = c >= r ? x[c] : 0.0;
    }
  }
}

// acc += A B for 16 x 16 blocks by one wavefront; a(r, k), b(k, c).
template <class A, class B>
__device__ __forceinline__ void mm16(A a, B b, d64x4& acc) {
  const int lane = threadIdx.x & 63, rc = lane & 15, k0 = lane >> 4;
#pragma unroll
  for (int k = 0; k < kSub; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a(rc, k + k0), b(k + k0, rc), acc, 0, 0, 0);
}
// Register q of acc: row lane / 16 + 4 q, column lane % 16.
template <class F>
__device__ __forceinline__ void mm16_each(const d64x4& acc, F f) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 4; q++) f((lane >> 4) + 4 * q, lane & 15, acc[q]);
}

// dg (64 x 64, symmetric in its lower triangle) becomes its Cholesky factor,
// inv the factor's inverse; both with zeros above the diagonal. 16-wide steps:
// the diagonal block by one wavefront, the products of blocks on MFMA.
__device__ __forceinline__ void block_factor(double (*dg)[kB + 1], double (*inv)[kB + 1],
                                             int32_t* __restrict__ flag) {
  const int wave = threadIdx.x >> 6;
  constexpr int kN = kB / kSub;  // 4 blocks, one per wave
#pragma unroll 1
  for (int b = 0; b < kN; b++) {
    const int o = b * kSub;
    if (wave == 0) wave_factor16(dg, inv, o, flag);
    __syncthreads();
    if (b + 1 + wave < kN) {  // L_ib = A_ib inv_bb^T
      const int ro = (b + 1 + wave) * kSub;
      d64x4 acc{0.0, 0.0, 0.0, 0.0};
      mm16([&](int r, int k) { return dg[ro + r][o + k]; }, [&](int k, int c) { return inv[o + c][o + k]; }, acc);
      mm16_each(acc, [&](int r, int c, double v) { dg[ro + r][o + c] = v; });
    }
    __syncthreads();
    const int left = kN - 1 - b;
    for (int t = wave; t < left * (left + 1) / 2; t += 4) {  // A_ij - L_ib L_jb^T, i >= j
      const int i = t < 1 ? 0 : (t < 3 ? 1 : 2), j = t - i * (i + 1) / 2;
      const int ro = (b + 1 + i) * kSub, co = (b + 1 + j) * kSub;
      d64x4 acc{0.0, 0.0, 0.0, 0.0};
      mm16([&](int r, int k) { return dg[ro + r][o + k]; }, [&](int k, int c) { return dg[co + c][o + k]; }, acc);
      mm16_each(acc, [&](int r, int c, double v) { dg[ro + r][co + c] -= v; });
    }
    __syncthreads();
  }
  // inv_ij = -inv_ii sum_{j <= k < i} L_ik inv_kj, by distance from the
  // diagonal; the sum waits in the block above the diagonal, (j, i), of inv.
#pragma unroll 1
  for (int d = 1; d < kN; d++) {
    if (wave + d < kN) {
      const int jo = wave * kSub, io = (wave + d) * kSub;
      d64x4 acc{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
      for (int ko = jo; ko < io; ko += kSub)
        mm16([&](int r, int k) { return dg[io + r][ko + k]; }, [&](int k, int c) { return inv[ko + k][jo + c]; }, acc);
      mm16_each(acc, [&](int r, int c, double v) { inv[jo + r][io + c] = v; });
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      acc = d64x4{0.0, 0.0, 0.0, 0.0};
      mm16([&](int r, int k) { return inv[io + r][io + k]; }, [&](int k, int c) { return inv[jo + k][io + c]; }, acc);
      mm16_each(acc, [&](int r, int c, double v) { inv[io + r][jo + c] = -v; });
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < kB * kB; e += kCt) {
    const int r = e & 63, c = e >> 6;
    if (c / kSub > r / kSub) dg[r][c] = inv[r][c] = 0.0;
  }
  __syncthreads();
}

struct MmSmem {
  union {
    struct {
      double pa[kB][kKc + 1], pb[kB][kKc + 1];
    } p;
    double dt[kB][kB + 1];
  } u;
};

// acc += sum over k in [k0, k1) of A(r, k) B(k, c) for the calling wave's 32 x
// 32 part of a 64 x 64 tile. kAK / kBK: the operand is contiguous along k in
// memory (else along r or c), which decides how the threads load it; la(r, k)
// and lb(k, c) return 0 outside their matrices. Ends with a barrier.
template <bool kAK, bool kBK, class LA, class LB>
__device__ __forceinline__ void mm_tile(MmSmem& sm, int k0, int k1, LA la, LB lb, d64x4 (&acc)[2][2]) {
  constexpr int kPer = kB * kKc / kCt;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wi = wave >> 1, wj = wave & 1;
  double ra[kPer], rb[kPer];
  auto row_of = [&](bool along_k, int q) { return along_k ? (tid >> 5) + 8 * q : tid & 63; };
  auto k_of = [&](bool along_k, int q) { return along_k ? tid & 31 : (tid >> 6) + 4 * q; };
  auto load = [&](int k) {
#pragma unroll
    for (int q = 0; q < kPer; q++) {
      const int ka = k + k_of(kAK, q), kb = k + k_of(kBK, q);
      ra[q] = ka < k1 ? la(row_of(kAK, q), ka) : 0.0;
      rb[q] = kb < k1 ? lb(kb, row_of(kBK, q)) : 0.0;
    }
  };
  load(k0);
  for (int k = k0; k < k1; k += kKc) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; q++) {
      sm.u.p.pa[row_of(kAK, q)][k_of(kAK, q)] = ra[q];
      sm.u.p.pb[row_of(kBK, q)][k_of(kBK, q)] = rb[q];
    }
    __syncthreads();
    if (k + kKc < k1) load(k + kKc);
#pragma unroll
    for (int ks = 0; ks < kKc / 4; ks++) {
      double af[2], bf[2];
#pragma unroll
      for (int ii = 0; ii < 2; ii++) af[ii] = sm.u.p.pa[wi * 32 + ii * 16 + (lane & 15)][ks * 4 + (lane >> 4)];
#pragma unroll
      for (int jj = 0; jj < 2; jj++) bf[jj] = sm.u.p.pb[wj * 32 + jj * 16 + (lane & 15)][ks * 4 + (lane >> 4)];
#pragma unroll
      for (int ii = 0; ii < 2; ii++)
#pragma unroll
        for (int jj = 0; jj < 2; jj++)
          acc[ii][jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[ii], bf[jj], acc[ii][jj], 0, 0, 0);
    }
  }
  __syncthreads();
}

// The tile's entries as (row, column, value): MFMA register q of a lane holds
// row lane / 16 + 4 q, column lane % 16.
template <class F>
__device__ __forceinline__ void mm_each(const d64x4 (&acc)[2][2], F f) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, wi = wave >> 1, wj = wave & 1;
#pragma unroll
  for (int ii = 0; ii < 2; ii++)
#pragma unroll
    for (int jj = 0; jj < 2; jj++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        f(wi * 32 + ii * 16 + (lane >> 4) + 4 * q, wj * 32 + jj * 16 + (lane & 15), acc[ii][jj][q]);
}

// The tile through LDS, so that column-major stores are coalesced:
// store(row, column, value).
template <class F>
__device__ __forceinline__ void mm_store(MmSmem& sm, const d64x4 (&acc)[2][2], F store) {
  mm_each(acc, [&](int r, int c, double v) { sm.u.dt[r][c] = v; });
  __syncthreads();
  for (int e = threadIdx.x; e < kB * kB; e += kCt) store(e & 63, e >> 6, sm.u.dt[e & 63][e >> 6]);
}

__device__ __forceinline__ void mm_zero(d64x4 (&acc)[2][2]) {
#pragma unroll
  for (int ii = 0; ii < 2; ii++)
#pragma unroll
    for (int jj = 0; jj < 2; jj++) acc[ii][jj] = d64x4{0.0, 0.0, 0.0, 0.0};
}

// Panel step k0: workgroup 0 keeps the diagonal block's factor (in lscr: the
// other workgroups still read the block; the trailing launch moves it into a)
// and its inverse (x), workgroup b >= 1 turns rows k0 + 64 b .. + 63 of the
// panel into rows of the factor.
__global__ void __launch_bounds__(kCt)
coarse_step_kernel(double* __restrict__ a, int n, int k0, int32_t* __restrict__ flag, double* __restrict__ x,
                   double* __restrict__ lscr) {
  __shared__ double dg[kB][kB + 1];
  __shared__ double inv[kB][kB + 1];
  __shared__ MmSmem sm;
  const int tid = threadIdx.x;
  const int64_t lda = n;
  const int kb = min(kB, n - k0);
  for (int e = tid; e < kB * kB; e += kCt) {
    const int r = e & 63, c = e >> 6;
    // padded with the identity past the matrix
    dg[r][c] = (r < kb && c < kb) ? (r >= c ? a[(k0 + c) * lda + k0 + r] : 0.0) : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  block_factor(dg, inv, flag);
  if (blockIdx.x == 0) {
    const bool last = gridDim.x == 1;
    for (int e = tid; e < kB * kB; e += kCt) {
      const int r = e & 63, c = e >> 6;
      if (last) {
        if (r < kb && c <= r) a[(k0 + c) * lda + k0 + r] = dg[r][c];
      } else {
        lscr[e] = dg[r][c];
      }
      if (x && r < kb && c < kb) x[(k0 + c) * lda + k0 + r] = inv[r][c];
    }
    return;
  }
  const int r0 = k0 + kB * static_cast<int>(blockIdx.x);
  d64x4 acc[2][2];
  mm_zero(acc);
  mm_tile<false, true>(
      sm, 0, kB, [&](int r, int k) { return r0 + r < n ? a[(k0 + k) * lda + r0 + r] : 0.0; },
      [&](int k, int c) { return inv[c][k]; }, acc);
  mm_store(sm, acc, [&](int r, int c, double v) {
    if (r0 + r < n) a[(k0 + c) * lda + r0 + r] = v;
  });
}

// Trailing tile (I, J), I >= J, of panel step k0: A_IJ -= L_I L_J^T.
__global__ void __launch_bounds__(kCt)
coarse_trailing_kernel(double* __restrict__ a, int n, int k0, const double* __restrict__ lscr) {
  __shared__ MmSmem sm;
  const int64_t lda = n;
  const int t = blockIdx.x;
  int I = static_cast<int>((sqrt(8.0 * t + 1.0) - 1.0) / 2.0);
  while ((I + 1) * (I + 2) / 2 <= t) I++;
  while (I * (I + 1) / 2 > t) I--;
  const int J = t - I * (I + 1) / 2;
  if (t == 0)
    for (int e = threadIdx.x; e < kB * kB; e += kCt) {
      const int r = e & 63, c = e >> 6;
      if (c <= r) a[(k0 + c) * lda + k0 + r] = lscr[e];
    }
  const int r0 = k0 + kB + I * kB, c0 = k0 + kB + J * kB;
  d64x4 acc[2][2];
  mm_zero(acc);
  mm_tile<false, false>(
      sm, k0, k0 + kB, [&](int r, int k) { return r0 + r < n ? a[k * lda + r0 + r] : 0.0; },
      [&](int k, int c) { return c0 + c < n ? a[k * lda + c0 + c] : 0.0; }, acc);
  mm_store(sm, acc, [&](int r, int c, double v) {
    if (r0 + r < n && c0 + c <= r0 + r) a[(c0 + c) * lda + r0 + r] -= v;
  });
}

// Inverse of the factor by block pairs of size s: with [A 0; B C] the factor's
// diagonal block of rows 2 s p .. 2 s (p + 1) and A^-1, C^-1 known in x, first
// t = B A^-1, then x = -C^-1 t below the diagonal. blockIdx = (tile column,
// tile row, pair).
__global__ void __launch_bounds__(kCt)
coarse_inverse_t_kernel(const double* __restrict__ a, int n, const double* __restrict__ x, double* __restrict__ t,
                        int s) {
  __shared__ MmSmem sm;
  const int64_t lda = n;
  const int c0 = 2 * s * static_cast<int>(blockIdx.z) + kB * static_cast<int>(blockIdx.x);
  const int kend = 2 * s * static_cast<int>(blockIdx.z) + s;
  const int r0 = kend + kB * static_cast<int>(blockIdx.y);
  if (r0 >= n) return;
  d64x4 acc[2][2];
  mm_zero(acc);
  mm_tile<false, true>(
      sm, c0, kend, [&](int r, int k) { return r0 + r < n ? a[k * lda + r0 + r] : 0.0; },
      [&](int k, int c) { return x[(c0 + c) * lda + k]; }, acc);
  mm_store(sm, acc, [&](int r, int c, double v) {
    if (r0 + r < n) t[(c0 + c) * lda + r0 + r] = v;
  });
}

__global__ void __launch_bounds__(kCt)
coarse_inverse_x_kernel(int n, double* __restrict__ x, const double* __restrict__ t, int s) {
  __shared__ MmSmem sm;
  const int64_t lda = n;
  const int c0 = 2 * s * static_cast<int>(blockIdx.z) + kB * static_cast<int>(blockIdx.x);
  const int k0 = 2 * s * static_cast<int>(blockIdx.z) + s;
  const int r0 = k0 + kB * static_cast<int>(blockIdx.y);
  if (r0 >= n) return;
  d64x4 acc[2][2];
  mm_zero(acc);
  mm_tile<false, true>(
      sm, k0, min(r0 + kB, n), [&](int r, int k) { return r0 + r < n ? x[k * lda + r0 + r] : 0.0; },
      [&](int k, int c) { return t[(c0 + c) * lda + k]; }, acc);
  mm_store(sm, acc, [&](int r, int c, double v) {
    if (r0 + r < n) x[(c0 + c) * lda + r0 + r] = -v;
  });
}

// Tile (I, J) of W = x^T x into the operator's rows and columns l .. m - 1.
__global__ void __launch_bounds__(kCt)
coarse_w_kernel(const double* __restrict__ x, int n, int l, int m, double* __restrict__ op) {
  __shared__ MmSmem sm;
  const int64_t lda = n;
  const int r0 = kB * static_cast<int>(blockIdx.y), c0 = kB * static_cast<int>(blockIdx.x);
  d64x4 acc[2][2];
  mm_zero(acc);
  mm_tile<true, true>(
      sm, max(r0, c0), n, [&](int r, int k) { return r0 + r < n ? x[(r0 + r) * lda + k] : 0.0; },
      [&](int k, int c) { return c0 + c < n ? x[(c0 + c) * lda + k] : 0.0; }, acc);
  mm_each(acc, [&](int r, int c, double v) {
    if (r0 + r < n && c0 + c < n) op[static_cast<int64_t>(l + r0 + r) * m + l + c0 + c] = v;
  });
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

constexpr int kRowsPerBlock = kCt / 64;

// Q's first l rows: op[a][l + j] = op[l + j][a] = -sum_i lag[idx[l + i]][a] W_ji,
// one wavefront per row j of W.
template <int L>
__global__ void __launch_bounds__(kCt)
coarse_top_kernel(const double* __restrict__ lag, const int32_t* __restrict__ idx, int m, double* __restrict__ op) {
  const int lane = threadIdx.x & 63;
  const int j = static_cast<int>(blockIdx.x) * kRowsPerBlock + static_cast<int>(threadIdx.x >> 6);
  if (j >= m - L) return;
  const int64_t row = static_cast<int64_t>(L + j) * m;
  double acc[L];
#pragma unroll
  for (int a = 0; a < L; a++) acc[a] = 0.0;
  for (int u = L + lane; u < m; u += 64) {
    const double w = op[row + u];
    const double* q = lag + static_cast<int64_t>(idx[u]) * L;
#pragma unroll
    for (int a = 0; a < L; a++) acc[a] = fma(-q[a], w, acc[a]);
  }
#pragma unroll
  for (int a = 0; a < L; a++) {
    const double v = wave_sum(acc[a]);
    if (lane == 0) {
      op[row + a] = v;
      op[static_cast<int64_t>(a) * m + L + j] = v;
    }
  }
}

// op[a][b] = -sum_j lag[idx[l + j]][b] op[a][l + j]; one wavefront per (a, b).
template <int L>
__global__ void __launch_bounds__(64)
coarse_corner_kernel(const double* __restrict__ lag, const int32_t* __restrict__ idx, int m, double* __restrict__ op) {
  const int a = static_cast<int>(blockIdx.x) / L, b = static_cast<int>(blockIdx.x) % L;
  double acc = 0.0;
  for (int u = L + static_cast<int>(threadIdx.x); u < m; u += 64)
    acc = fma(-lag[static_cast<int64_t>(idx[u]) * L + b], op[static_cast<int64_t>(a) * m + u], acc);
  acc = wave_sum(acc);
  if (threadIdx.x == 0) op[static_cast<int64_t>(a) * m + b] = acc;
}

// The polynomial rows: op[m + a][u] = sum_b pinv[a][b] (delta_bu - sum_v
// A_top[b][v] op[v][u]); the operator's first m rows are symmetric, so column
// u is read as row u. One wavefront per u.
template <int L>
__global__ void __launch_bounds__(kCt)
coarse_poly_kernel(const double* __restrict__ atop, const double* __restrict__ pinv, int m, double* __restrict__ op) {
  const int lane = threadIdx.x & 63;
  const int u = static_cast<int>(blockIdx.x) * kRowsPerBlock + static_cast<int>(threadIdx.x >> 6);
  if (u >= m) return;
  double acc[L];
#pragma unroll
  for (int b = 0; b < L; b++) acc[b] = 0.0;
  for (int v = lane; v < m; v += 64) {
    const double w = op[static_cast<int64_t>(u) * m + v];
#pragma unroll
    for (int b = 0; b < L; b++) acc[b] = fma(-atop[static_cast<int64_t>(b) * m + v], w, acc[b]);
  }
#pragma unroll
  for (int b = 0; b < L; b++) acc[b] = wave_sum(acc[b]) + (b == u ? 1.0 : 0.0);
  if (lane == 0) {
#pragma unroll
    for (int a = 0; a < L; a++) {
      double c = 0.0;
#pragma unroll
      for (int b = 0; b < L; b++) c = fma(pinv[a * L + b], acc[b], c);
      op[static_cast<int64_t>(m + a) * m + u] = c;
    }
  }
}

template <int L>
void launch_poly_part(int m, const int32_t* idx, const double* lag, const double* atop, const double* pinv,
                      double* op, hipStream_t s) {
  if (m > L) {
    coarse_top_kernel<L><<<ceil_div(m - L, kRowsPerBlock), kCt, 0, s>>>(lag, idx, m, op);
    PAM_LAUNCH_CHECK();
  }
  coarse_corner_kernel<L><<<L * L, 64, 0, s>>>(lag, idx, m, op);
  PAM_LAUNCH_CHECK();
  coarse_poly_kernel<L><<<ceil_div(m, kRowsPerBlock), kCt, 0, s>>>(atop, pinv, m, op);
  PAM_LAUNCH_CHECK();
}

}  // namespace

void launch_coarse_factor(double* a, int n, int32_t* flag, double* x, double* lscr, hipStream_t s) {
  for (int k0 = 0; k0 < n; k0 += kB) {
    const int nt = n - k0 > kB ? ceil_div(n - k0 - kB, kB) : 0;
    coarse_step_kernel<<<1 + nt, kCt, 0, s>>>(a, n, k0, flag, x, lscr);
    PAM_LAUNCH_CHECK();
    if (nt == 0) break;
    coarse_trailing_kernel<<<nt * (nt + 1) / 2, kCt, 0, s>>>(a, n, k0, lscr);
    PAM_LAUNCH_CHECK();
  }
}

void launch_coarse_inverse(const double* a, int n, double* x, double* t, hipStream_t s) {
  for (int h = kB; h < n; h *= 2) {
    const dim3 grid(h / kB, h / kB, ceil_div(n, 2 * h));
    coarse_inverse_t_kernel<<<grid, kCt, 0, s>>>(a, n, x, t, h);
    PAM_LAUNCH_CHECK();
    coarse_inverse_x_kernel<<<grid, kCt, 0, s>>>(n, x, t, h);
    PAM_LAUNCH_CHECK();
  }
}

void launch_coarse_operator(const double* x, int m, int l, const int32_t* idx, const double* lag,
                            const double* atop, const double* pinv, double* op, hipStream_t s) {
  const int n = m - l;
  if (n > 0) {
    coarse_w_kernel<<<dim3(ceil_div(n, kB), ceil_div(n, kB)), kCt, 0, s>>>(x, n, l, m, op);
    PAM_LAUNCH_CHECK();
  }
  switch (l) {
    case 0: break;
    case 1: launch_poly_part<1>(m, idx, lag, atop, pinv, op, s); break;
    case 4: launch_poly_part<4>(m, idx, lag, atop, pinv, op, s); break;
    case 10: launch_poly_part<10>(m, idx, lag, atop, pinv, op, s); break;
    default: throw_invalid("unsupported polynomial basis size");
  }
}

}  // namespace pam
