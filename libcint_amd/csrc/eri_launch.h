// Host-side entry points of the device code (eri.hip).
#pragma once
#include "mcint_internal.h"

namespace mcint {

// Primitive-pair records of the listed shell pairs, each pair's list in
// ascending order of cce0, and pos[k] = position in pp of the k-th record in
// libcint's order; tmp is a staging buffer of the size of pp.
hipError_t launch_pairdata(const VShell* vsh, const double* env, int nv, const int* pairs,
                           int npairs, const int64_t* pair_off, double* pair_ld, PairPrim* tmp,
                           PairPrim* pp, int* pos, hipStream_t stream);

hipError_t launch_rys_batch(int n, const double* x, int64_t count, double* u, double* w,
                            hipStream_t stream);
// Short-range rule of exp(-x t^2) on [lower, 1] for count (x, lower) pairs
// (one wave each); u, w: count * n.
hipError_t launch_sr_rys_batch(int n, const double* x, const double* lower, int64_t count,
                               double* u, double* w, hipStream_t stream);

hipError_t launch_count_prims(const BasisView& B, const BucketArgs& A, unsigned long long* counter,
                              hipStream_t stream);

hipError_t launch_generic(const BasisView& B, const BucketArgs& A, hipStream_t stream);

// grad[i] += sum over the nslot accumulator copies of acc[slot * stride + i], i < n
hipError_t launch_grad_reduce(const double* acc, int nslot, int64_t stride, int n, double* grad,
                              hipStream_t stream);

// Grouped J/K digest: row pass (groups of quartets sharing (i,j), LDS of
// rows_lds bytes) and column pass (groups sharing (k,l)) into the half
// matrices J', K' (either nullable); symmetrize then forms X + X^T.
hipError_t launch_jk_grouped(const int* shls, const int64_t* off, const int* rows_q,
                             const int* rows_ptr, int nrows, size_t rows_lds, const int* cols_q,
                             const int* cols_ptr, int ncols, const double* eri, const int* ao_loc,
                             const double* D, int nao, double* Jp, double* Kp, hipStream_t stream);
// out = X + X^T of the sum of nslot copies of X, stride doubles apart
hipError_t launch_symmetrize(const double* X, double* out, int n, int nslot, int64_t stride,
                             hipStream_t stream);
// x[0..n) = 0 (a kernel, so that captured graphs hold no memset node)
hipError_t launch_zero(double* x, int64_t n, hipStream_t stream);

hipError_t launch_jk_digest(const int* shls, const int64_t* off, int64_t nq, const double* eri,
                            const int* ao_loc, const double* D, int nao, double* J, double* K,
                            hipStream_t stream);

// Register-resident kernels for the classes listed in eri_fast.h:
// mode 1 = one kernel with an in-register epilogue, 2 = chunk kernels plus
// an LDS epilogue (scratch of chunked_block_doubles() per task), 0 = none.
// Cartesian output: every kind except short range.
int fast_kernel_mode(int kind, int sph, int la, int lb, int lc, int ld, double omega);
// 1: team-of-one buckets of the chunked classes with a wave kernel run it
// instead of their chunk kernels (mcint_tune MCINT_TUNE_WAVE_KERNELS;
// read at launch, so graphs captured earlier keep their kernels)
extern int g_wave_kernels;
// per-class and team-size choice of the chunked classes' kernels
// (mcint_tune_class_wave): 0 the default rule, 1 chunk kernels, 2 wave
// kernel; indexed by class_index * 7 + log2(team lanes)
constexpr int NCLS = (LMAX + 1) * (LMAX + 1) * (LMAX + 1) * (LMAX + 1);
__host__ __device__ constexpr int class_index(int la, int lb, int lc, int ld) {
  return ((la * (LMAX + 1) + lb) * (LMAX + 1) + lc) * (LMAX + 1) + ld;
}
extern int8_t g_class_wave[NCLS * 7];
// 1 when the canonical plain class (la lb|lc ld) has a wave kernel
int wave_kernel_exists(int la, int lb, int lc, int ld);
// whether a bucket of the chunked plain class with teams of tune_team lanes
// runs its wave kernel (the rule of launch_chunks)
bool chunk_class_on_wave(int la, int lb, int lc, int ld, int tune_team, double omega, int fp32);
int chunked_block_doubles(int kind, int la, int lb, int lc, int ld);
int fast_team_lanes_max();
hipError_t launch_fast(const BasisView& B, const BucketArgs& A, hipStream_t stream);
hipError_t launch_chunked(const BasisView& B, const BucketArgs& A, hipStream_t stream);

}  // namespace mcint
