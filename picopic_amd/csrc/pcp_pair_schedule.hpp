// The pair schedule of a collision cell (collisionsP12.cpp:356-528).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pcp {

// pairs of the n particles of one species: (0, 1), (2, 3), ... of an even n, the
// chain (0, 1), (1, 2), (2, 0) and then (3, 4), ... of an odd one
__host__ __device__ __forceinline__ uint32_t like_pairs(int n) {
  if (n % 2 == 0) return (uint32_t)(n / 2);
  return (uint32_t)((n >= 3 ? 3 : 0) + (n >= 5 ? (n - 3) / 2 : 0));
}

// The unlike pairs of a cell with N particles of the more numerous species
// and n of the other (cases 2a / 2b): each of the n meets a chain of the N,
// first particles of the reference's 1st group (c + 1 each), then of the 2nd
// (c each).  No particle of the N is in two chains, so the chains are
// independent and each runs in the reference's order.
struct UnlikeChains {
  int n, big, c;                 // chains, N, floor(N / n)
  int big1, small1, big2;        // 1st group: particles of the N, of the n; 2nd group: of the N
  __host__ __device__ __forceinline__ void set(int nel, int nion) {
    const int lo = min(nel, nion), hi = max(nel, nion);
    n = lo;
    big = hi;
    if (lo == hi || lo == 0) {
      c = 1;
      big1 = small1 = 0;
      big2 = lo;
      return;
    }
    const float ratio = (float)hi / (float)lo;
    const double ci = (double)floorf(ratio);
    const double cr = (double)ratio - ci;
    c = (int)ci;
    big1 = min((int)((ci + 1) * cr * lo), hi);
    small1 = (int)(cr * lo);
    big2 = min((int)(ci * (1 - cr) * lo), hi - big1);
  }
  // chain e: pairs of the 1st and of both groups
  __host__ __device__ __forceinline__ int first(int e) const { return min(max(big1 - e * (c + 1), 0), c + 1); }
  __host__ __device__ __forceinline__ int length(int e) const {
    return first(e) + (e >= small1 ? min(max(big2 - (e - small1) * c, 0), c) : 0);
  }
  // the N's particle (and pair ordinal) of pair j of chain e
  __host__ __device__ __forceinline__ int partner(int e, int j) const {
    const int f = first(e);
    return j < f ? e * (c + 1) + j : big1 + (e - small1) * c + (j - f);
  }
  // chains that can hold more than one pair: every one for c > 1, else the 1st group's
  __host__ __device__ __forceinline__ int long_chains() const { return c > 1 ? n : min(n, small1 + 1); }
};

}  // namespace pcp
