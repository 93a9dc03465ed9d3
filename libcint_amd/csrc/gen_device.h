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

// The sets of X in LDS, three row sets and two column sets: first e (f) among
// the list | number << 16, offset | weight << 28.  Absent ones are empty.
constexpr int GEN_SETS = 5;
__device__ __forceinline__ void put_sets(const GenLayout& G, int2* sets) {
#pragma unroll
  for (int r = 0; r < 3; ++r)
    sets[r] = r < G.nbs ? make_int2(G.be[r] | (G.nes[r] << 16), G.ox[r] | (G.bw[r] << 28)) : make_int2(0, 0);
#pragma unroll
  for (int u = 0; u < 2; ++u)
    sets[3 + u] = u < G.nks ? make_int2(G.kf[u] | (G.nfs[u] << 16), G.cf[u] | (G.kw[u] << 28)) : make_int2(0, 0);
}
// Adds a component's sums (e-list position ie, f-list position jf; g0, g1, g2
// weighted 1, 2a_i, 4a_i^2, h0, h1 the first two times 2a_k) to the sets of X
// it belongs to.  The sets come from LDS: indexed by a loop variable the
// layout's arrays are read from memory one by one for every component, and
// with constant indices they take scalar registers that the rest spills.
// i-derivatives (dd|dg) of 256 primitives: 29.1 -> 25.2 ms on the generic kernel.
__device__ __forceinline__ void add_to_sets(const int2* sets, int KF, double* X, int ie, int jf, double g0, double g1,
                                            double g2, double h0, double h1) {
  const int2 c[2] = {sets[3], sets[4]};
  constexpr int OFF = (1 << 28) - 1;
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int2 q = sets[r];
    const int er = ie - (q.x & 0xffff);
    if ((unsigned)er >= ((unsigned)q.x >> 16)) continue;
    double* const row = X + (q.y & OFF) + er * KF;
    const int w = q.y >> 28;
    const double g = w == 0 ? g0 : (w == 1 ? g1 : g2), h = w ? h1 : h0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int fu = jf - (c[u].x & 0xffff);
      if ((unsigned)fu < ((unsigned)c[u].x >> 16)) row[(c[u].y & OFF) + fu] += c[u].y >> 28 ? h : g;
    }
  }
}

}  // namespace mcint
