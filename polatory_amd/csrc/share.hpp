// Near-equal shares of a range, for the kernels that deal a leaf's targets out
// to workgroups and passes and for the host.
#pragma once

#if defined(__HIPCC__)
#define PAM_HD __host__ __device__ __forceinline__
#else
#define PAM_HD inline
#endif

namespace pam {

// Shares of at most `per` items that n items need.
PAM_HD int share_count(int n, int per) { return n / per + (n % per != 0 ? 1 : 0); }

// First item of share i of k (the end of share i - 1), 0 <= i <= k: shares of
// n / k items, one more in the first n % k. With k = share_count(n, per) none
// is longer than `per`. No intermediate value exceeds n, so every n of 32 bits
// is right; n * i / k passes 2^31 at 524,288 items in shares of 128.
PAM_HD int share_begin(int n, int i, int k) {
  const int rem = n % k;
  return n / k * i + (i < rem ? i : rem);
}

}  // namespace pam
