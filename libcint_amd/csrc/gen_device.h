// Device helpers of the kernels whose class is known at run time.
#pragma once
#include "device_common.h"
#include "gen_layout.h"

namespace mcint {

namespace ct {
#define C2S_QUAL constexpr
#include "c2s_tables.inc"
#undef C2S_QUAL
}  // namespace ct

// Nonzero Cartesian -> spherical coefficients, rows (l, m) at l*l + m.
constexpr int c2s_nnz() {
  int n = 0;
  for (int i = 0; i < 840; ++i) n += ct::c2s_coef[i] != 0.0;
  return n;
}
struct C2sSparse {
  short ptr[50];
  short k[c2s_nnz()];
  double v[c2s_nnz()];
};
constexpr C2sSparse make_c2s_sparse() {
  C2sSparse s{};
  int n = 0;
  for (int l = 0; l <= LMAX; ++l) {
    const int nc = (l + 1) * (l + 2) / 2;
    for (int m = 0; m < 2 * l + 1; ++m) {
      s.ptr[l * l + m] = (short)n;
      for (int k = 0; k < nc; ++k) {
        const double v = ct::c2s_coef[ct::c2s_offset[l] + m * nc + k];
        if (v != 0.0) {
          s.k[n] = (short)k;
          s.v[n++] = v;
        }
      }
    }
  }
  s.ptr[49] = (short)n;
  return s;
}
static __device__ const C2sSparse c2s_sparse = make_c2s_sparse();

// Mixed-radix counter of a lane's elements lane, lane + step, ... (digit 0
// fastest; the last digit is unbounded).
template <int N>
struct Odo {
  int d[N], n[N], s[N];
  __device__ __forceinline__ Odo(int lane, const int (&dims)[N], int step = GEN_LANES) {
    int a = lane, b = step;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      n[j] = dims[j];
      if (j < N - 1) {
        d[j] = (int)((unsigned)a % (unsigned)n[j]);
        a = (int)((unsigned)a / (unsigned)n[j]);
        s[j] = (int)((unsigned)b % (unsigned)n[j]);
        b = (int)((unsigned)b / (unsigned)n[j]);
      } else {
        d[j] = a;
        s[j] = b;
      }
    }
  }
  __device__ __forceinline__ void next() {
    int c = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      d[j] += s[j] + c;
      c = 0;
      if (j < N - 1 && d[j] >= n[j]) {
        d[j] -= n[j];
        c = 1;
      }
    }
  }
};

// n / 6 for n <= 4080 divisible by 6
__device__ __forceinline__ int tet_d(int l) { return (int)(((unsigned)(l * (l + 1) * (l + 2)) * 43691u) >> 18); }
// index of Cartesian exponents (x, y, z) among the components of all shells
__device__ __forceinline__ int cart_all(int x, int y, int z) {
  const int m = y + z;
  return tet_d(x + m) + ((m * (m + 1)) >> 1) + z;
}

__device__ __forceinline__ double binom_small(int n, int k) {
  double r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}

// One primitive quartet of a batch.
struct GenPrim {
  double aij, akl, a0, a1, x, fac, theta, w[3];
  double pq[3], pa[3], qc[3];
};
static_assert(sizeof(GenPrim) == GEN_PRIM_D * sizeof(double), "GEN_PRIM_D");

}  // namespace mcint
