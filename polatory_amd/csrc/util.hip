// Generic device building blocks: point transforms, bbox reduction, prefix
// sums, a stable LSD radix sort, gathers and polynomial terms.
#include <type_traits>
#include <vector>

#include "device_api.hpp"
#include "rbf_device.hpp"

namespace pam {

namespace {

struct Mat3 {
  double a[9];
};

__global__ void transform_kernel(Mat3 m, const double* __restrict__ in, int64_t n,
                                 double* __restrict__ out) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double x = in[3 * i], y = in[3 * i + 1], z = in[3 * i + 2];
  // Explicit round-to-nearest ops: no FMA contraction, so the result equals the
  // CPU evaluation of ((A0 x + A1 y) + A2 z) bit for bit.
  out[3 * i] = __dadd_rn(__dadd_rn(__dmul_rn(m.a[0], x), __dmul_rn(m.a[1], y)), __dmul_rn(m.a[2], z));
  out[3 * i + 1] = __dadd_rn(__dadd_rn(__dmul_rn(m.a[3], x), __dmul_rn(m.a[4], y)), __dmul_rn(m.a[5], z));
  out[3 * i + 2] = __dadd_rn(__dadd_rn(__dmul_rn(m.a[6], x), __dmul_rn(m.a[7], y)), __dmul_rn(m.a[8], z));
}

constexpr int kBboxThreads = 256;

__global__ void bbox_partial_kernel(const double* __restrict__ pts, int64_t n,
                                    double* __restrict__ partial) {
  __shared__ double s[6][kBboxThreads];
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    for (int k = 0; k < 3; k++) {
      double v = pts[3 * i + k];
      lo[k] = fmin(lo[k], v);
      hi[k] = fmax(hi[k], v);
    }
  }
  for (int k = 0; k < 3; k++) {
    s[k][threadIdx.x] = lo[k];
    s[3 + k][threadIdx.x] = hi[k];
  }
  __syncthreads();
  for (int off = kBboxThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      for (int k = 0; k < 3; k++) {
        s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + off]);
        s[3 + k][threadIdx.x] = fmax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + off]);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) partial[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void bbox_final_kernel(const double* __restrict__ partial, int nb, double* __restrict__ out) {
  __shared__ double s[6][kBboxThreads];
  double r[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int b = threadIdx.x; b < nb; b += kBboxThreads) {
    for (int k = 0; k < 3; k++) {
      r[k] = fmin(r[k], partial[b * 6 + k]);
      r[3 + k] = fmax(r[3 + k], partial[b * 6 + 3 + k]);
    }
  }
  for (int k = 0; k < 6; k++) s[k][threadIdx.x] = r[k];
  __syncthreads();
  for (int off = kBboxThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      for (int k = 0; k < 3; k++) {
        s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + off]);
        s[3 + k][threadIdx.x] = fmax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + off]);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[threadIdx.x] = s[threadIdx.x][0];
}

// ---- exclusive scan: 256 threads x 4 items per block ----
constexpr int kScanThreads = 256;
constexpr int kScanTile = 1024;

__global__ void scan_block_kernel(const int32_t* in, int32_t* out, int64_t n, int32_t* block_sums) {
  __shared__ int32_t s[kScanThreads];
  int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * 4;
  int32_t v[4];
  int32_t tsum = 0;
  for (int q = 0; q < 4; q++) {
    v[q] = (base + q < n) ? in[base + q] : 0;
    tsum += v[q];
  }
  s[threadIdx.x] = tsum;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    int32_t t = (static_cast<int>(threadIdx.x) >= off) ? s[threadIdx.x - off] : 0;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  int32_t run = s[threadIdx.x] - tsum;
  for (int q = 0; q < 4; q++) {
    if (base + q < n) out[base + q] = run;
    run += v[q];
  }
  if (threadIdx.x == kScanThreads - 1 && block_sums) block_sums[blockIdx.x] = s[threadIdx.x];
}

__global__ void scan_add_kernel(int32_t* out, int64_t n, const int32_t* offs) {
  int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
  int32_t o = offs[blockIdx.x];
  for (int q = 0; q < 4; q++) {
    int64_t i = base + threadIdx.x + q * kScanThreads;
    if (i < n) out[i] += o;
  }
}

// Exclusive scan of a short array in one workgroup: chunks of 4096 entries
// (4 consecutive per thread), wave scans by shuffles and a running carry.
// Every thread reads and writes only its own entries, so in may equal out.
constexpr int kScan1Threads = 1024;
constexpr int64_t kScan1Max = 65536;

__global__ void __launch_bounds__(kScan1Threads) scan_single_kernel(const int32_t* in, int32_t* out,
                                                                    int64_t n) {
  __shared__ int32_t wsum[kScan1Threads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int32_t carry = 0;
  for (int64_t base = 0; base < n; base += 4 * kScan1Threads) {
    const int64_t i0 = base + 4 * static_cast<int64_t>(tid);
    int32_t v[4];
    int32_t tsum = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      v[q] = i0 + q < n ? in[i0 + q] : 0;
      tsum += v[q];
    }
    int32_t incl = tsum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      int32_t u = __shfl_up(incl, d, 64);
      if (lane >= d) incl += u;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int32_t before = 0, total = 0;
    for (int w = 0; w < kScan1Threads / 64; w++) {
      if (w < wave) before += wsum[w];
      total += wsum[w];
    }
    int32_t run = carry + before + incl - tsum;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (i0 + q < n) out[i0 + q] = run;
      run += v[q];
    }
    carry += total;
    __syncthreads();
  }
}

void scan_rec(const int32_t* in, int32_t* out, int64_t n, int32_t* scratch, hipStream_t s) {
  if (n <= kScan1Max) {
    scan_single_kernel<<<1, kScan1Threads, 0, s>>>(in, out, n);
    PAM_LAUNCH_CHECK();
    return;
  }
  int64_t nb = (n + kScanTile - 1) / kScanTile;
  if (nb <= 1) {
    scan_block_kernel<<<1, kScanThreads, 0, s>>>(in, out, n, nullptr);
    PAM_LAUNCH_CHECK();
    return;
  }
  scan_block_kernel<<<static_cast<unsigned>(nb), kScanThreads, 0, s>>>(in, out, n, scratch);
  PAM_LAUNCH_CHECK();
  scan_rec(scratch, scratch, nb, scratch + nb, s);
  scan_add_kernel<<<static_cast<unsigned>(nb), kScanThreads, 0, s>>>(out, n, scratch);
  PAM_LAUNCH_CHECK();
}

// ---- radix sort: digits of up to 8 bits, tiles of 2,048 items ----
//
// Bound by launches up to some 100,000 items. A Morton code of 9 to 18 bits
// takes two or three passes this way (three to five with 4-bit digits, whose
// counters fitted in registers). Each wavefront of a tile ranks eight times 64
// consecutive items: lanes with the same digit find each other by one ballot
// per bit, and the digit's counter in LDS carries over to the next 64, so the
// order stays stable and reads are coalesced.
// MI355X, two trees of 1M points (18 bits, three passes instead of five and
// two copies): tree stage 0.69 to 0.65 ms; of 50k points 0.46 to 0.43 ms.
constexpr int kRsThreads = 256;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsThreads * kRsItems;
constexpr int kRsMaxBits = 8;

__global__ void __launch_bounds__(kRsThreads)
radix_hist_kernel(const uint64_t* __restrict__ keys, int64_t n, int shift, int bits, int32_t* __restrict__ hist,
                  int nblocks) {
  __shared__ int32_t cnt[1 << kRsMaxBits];
  const unsigned digits = 1u << bits;
  for (unsigned e = threadIdx.x; e < digits; e += kRsThreads) cnt[e] = 0;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kRsTile;
#pragma unroll
  for (int q = 0; q < kRsItems; q++) {
    const int64_t i = base + threadIdx.x + q * kRsThreads;
    if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & (digits - 1)], 1);
  }
  __syncthreads();
  for (unsigned e = threadIdx.x; e < digits; e += kRsThreads)
    hist[static_cast<int64_t>(e) * nblocks + blockIdx.x] = cnt[e];
}

__global__ void __launch_bounds__(kRsThreads)
radix_scatter_kernel(const uint64_t* __restrict__ kin, const int32_t* __restrict__ vin, uint64_t* __restrict__ kout,
                     int32_t* __restrict__ vout, int64_t n, int shift, int bits, const int32_t* __restrict__ offs,
                     int nblocks) {
  constexpr int kWaves = kRsThreads / 64;
  __shared__ int32_t cnt[kWaves][1 << kRsMaxBits];  // per wave: items so far, then where its first one goes
  const unsigned digits = 1u << bits;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (unsigned e = threadIdx.x; e < digits; e += kRsThreads)
    for (int w = 0; w < kWaves; w++) cnt[w][e] = 0;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kRsTile + wave * (kRsTile / kWaves) + lane;
  uint64_t key[kRsItems];
  int32_t val[kRsItems], rank[kRsItems];
#pragma unroll
  for (int q = 0; q < kRsItems; q++) {
    const int64_t i = base + 64 * q;
    key[q] = i < n ? kin[i] : 0;
    val[q] = i < n ? vin[i] : 0;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kRsItems; q++) {
    const bool valid = base + 64 * q < n;
    const unsigned d = static_cast<unsigned>(key[q] >> shift) & (digits - 1);
    uint64_t same = __ballot(valid);
    for (int b = 0; b < bits; b++) {
      const uint64_t set = __ballot((d >> b) & 1u);
      same &= ((d >> b) & 1u) ? set : ~set;
    }
    const int before = __popcll(same & ((uint64_t{1} << lane) - 1));
    const int32_t seen = cnt[wave][d];
    rank[q] = seen + before;
    // The reads of this step come before its writes, and those before the
    // next step's reads; the counters belong to this wave.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid && before == 0) cnt[wave][d] = seen + __popcll(same);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  for (unsigned e = threadIdx.x; e < digits; e += kRsThreads) {
    int32_t run = offs[static_cast<int64_t>(e) * nblocks + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const int32_t c = cnt[w][e];
      cnt[w][e] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kRsItems; q++) {
    if (base + 64 * q >= n) continue;
    const unsigned d = static_cast<unsigned>(key[q] >> shift) & (digits - 1);
    const int64_t pos = cnt[wave][d] + rank[q];
    kout[pos] = key[q];
    vout[pos] = val[q];
  }
}

__global__ void iota_kernel(int32_t* v, int64_t n) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) v[i] = static_cast<int32_t>(i);
}

__global__ void gather_f64_kernel(const double* __restrict__ in, const int32_t* __restrict__ idx,
                                  int64_t n, double* __restrict__ out) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[idx[i]];
}

__global__ void poly_eval_kernel(int degree, const double* __restrict__ pts, int64_t n,
                                 const double* __restrict__ c, double* __restrict__ out) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] += poly_value(degree, c, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]);
}

// Gradient of the polynomial part at untransformed points:
// out3[3 i + k] += d/dx_k sum_m c_m m(p_i) (monomial_basis.hpp:198-209 order).
__global__ void poly_grad_kernel(int degree, const double* __restrict__ pts, int64_t n,
                                 const double* __restrict__ c, double* __restrict__ out3) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (degree < 1) return;
  const double x = pts[3 * i], y = pts[3 * i + 1], z = pts[3 * i + 2];
  double gx = c[1], gy = c[2], gz = c[3];
  if (degree >= 2) {
    gx += 2.0 * c[4] * x + c[5] * y + c[6] * z;
    gy += c[5] * x + 2.0 * c[7] * y + c[8] * z;
    gz += c[6] * x + c[8] * y + 2.0 * c[9] * z;
  }
  out3[3 * i] += gx;
  out3[3 * i + 1] += gy;
  out3[3 * i + 2] += gz;
}

}  // namespace

void launch_transform_points(const double* aniso, const double* in, int64_t n, double* out,
                             hipStream_t s) {
  if (n == 0) return;
  Mat3 m;
  for (int i = 0; i < 9; i++) m.a[i] = aniso[i];
  transform_kernel<<<ceil_div(n, 256), 256, 0, s>>>(m, in, n, out);
  PAM_LAUNCH_CHECK();
}

void launch_bbox(const double* pts, int64_t n, double* d_out, DevBuf<double>& scratch,
                 hipStream_t s) {
  int nb = ceil_div(n, kBboxThreads);
  if (nb > 512) nb = 512;
  if (nb < 1) nb = 1;
  scratch.resize(static_cast<size_t>(nb) * 6);
  bbox_partial_kernel<<<nb, kBboxThreads, 0, s>>>(pts, n, scratch.get());
  PAM_LAUNCH_CHECK();
  bbox_final_kernel<<<1, kBboxThreads, 0, s>>>(scratch.get(), nb, d_out);
  PAM_LAUNCH_CHECK();
}

void exclusive_scan_i32(const int32_t* in, int32_t* out, int64_t n, DevBuf<int32_t>& scratch,
                        hipStream_t s) {
  if (n <= 0) return;
  int64_t need = 0;
  for (int64_t m = n; m > 1;) {
    m = (m + kScanTile - 1) / kScanTile;
    need += m;
  }
  scratch.resize(static_cast<size_t>(need + 1));
  scan_rec(in, out, n, scratch.get(), s);
}

int radix_sort_passes(int64_t n, int bits) { return n <= 1 || bits <= 0 ? 0 : (bits + kRsMaxBits - 1) / kRsMaxBits; }

void radix_sort_pairs(uint64_t* keys, int32_t* vals, int64_t n, int bits, DevBuf<uint64_t>& tk,
                      DevBuf<int32_t>& tv, DevBuf<int32_t>& hist, DevBuf<int32_t>& scratch,
                      hipStream_t s) {
  const int passes = radix_sort_passes(n, bits);
  if (passes == 0) return;
  const int nb = ceil_div(n, kRsTile);
  const int width = (bits + passes - 1) / passes;
  tk.resize(static_cast<size_t>(n));
  tv.resize(static_cast<size_t>(n));
  hist.resize((static_cast<size_t>(1) << width) * nb);
  uint64_t* ka = keys;
  int32_t* va = vals;
  uint64_t* kb = tk.get();
  int32_t* vb = tv.get();
  if (passes % 2) {  // the input is in tk, tv
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  for (int p = 0; p < passes; p++) {
    const int shift = width * p, w = std::min(width, bits - shift);
    radix_hist_kernel<<<nb, kRsThreads, 0, s>>>(ka, n, shift, w, hist.get(), nb);
    PAM_LAUNCH_CHECK();
    exclusive_scan_i32(hist.get(), hist.get(), (static_cast<int64_t>(1) << w) * nb, scratch, s);
    radix_scatter_kernel<<<nb, kRsThreads, 0, s>>>(ka, va, kb, vb, n, shift, w, hist.get(), nb);
    PAM_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
  }
}

void launch_iota(int32_t* vals, int64_t n, hipStream_t s) {
  if (n == 0) return;
  iota_kernel<<<ceil_div(n, 256), 256, 0, s>>>(vals, n);
  PAM_LAUNCH_CHECK();
}

void launch_gather_f64(const double* in, const int32_t* idx, int64_t n, double* out, hipStream_t s) {
  if (n == 0) return;
  gather_f64_kernel<<<ceil_div(n, 256), 256, 0, s>>>(in, idx, n, out);
  PAM_LAUNCH_CHECK();
}

void launch_poly_grad(int degree, const double* pts, int64_t n, const double* d_coeffs, double* out3,
                      hipStream_t s) {
  if (n == 0 || degree < 1) return;
  poly_grad_kernel<<<ceil_div(n, 256), 256, 0, s>>>(degree, pts, n, d_coeffs, out3);
  PAM_LAUNCH_CHECK();
}

void launch_poly_eval(int degree, const double* pts, int64_t n, const double* d_coeffs,
                      double* out, hipStream_t s) {
  if (n == 0 || degree < 0) return;
  poly_eval_kernel<<<ceil_div(n, 256), 256, 0, s>>>(degree, pts, n, d_coeffs, out);
  PAM_LAUNCH_CHECK();
}

}  // namespace pam
