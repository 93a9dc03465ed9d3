// Device code of libmcint: pair data, root batches, primitive counts and the
// dispatch of the register kernels (the generic kernel is in generic.hip).
//
// Algorithm (the mathematics of libcint's Rys path, src/g2e.c:4425-4545,
// reorganised for the GPU):
//   per primitive quartet: Rys roots (tables), the Rys coefficients
//   b00/b10/b01/c00/c0p, the 2D vertical recurrence I(e,f) with e built on
//   centre A and f on centre C (src/g2e.c:272-421), and the products
//   [e0|f0] = sum_roots Ix*Iy*Iz accumulated over primitives;
//   per contracted quartet: the horizontal transfers (a,b| <- [e0| and
//   |c,d) <- |f0] done once on contracted data (libcint does them per
//   primitive, src/g2e.c:428-693), the Cartesian -> spherical transform
//   (src/cart2sph.c:5324-5376) and the store in libcint's Fortran order.
#include "device_common.h"

namespace mcint {

// ---------------------------------------------------------------------
// Pair data: one block per ordered virtual-shell pair, one lane per
// primitive pair.  Restates CINTset_pairdata (src/optimizer.c:288-342).
// ---------------------------------------------------------------------
// One workgroup per shell pair.  The records are staged in 'tmp' and then
// stored in ascending order of cce0 (ties by primitive index), so that the
// primitive quartets passing the screening tests of one pair against a
// fixed partner form a prefix of the list.
__global__ void pairdata_kernel(const VShell* __restrict__ vsh, const double* __restrict__ env,
                                int nv, const int* __restrict__ pairs,
                                const int64_t* __restrict__ pair_off, double* __restrict__ pair_ld,
                                PairPrim* __restrict__ tmp, PairPrim* __restrict__ pp,
                                int* __restrict__ pos) {
  const int ia = pairs[2 * blockIdx.x];
  const int ib = pairs[2 * blockIdx.x + 1];
  const VShell a = vsh[ia];
  const VShell b = vsh[ib];
  const double dx = a.r[0] - b.r[0], dy = a.r[1] - b.r[1], dz = a.r[2] - b.r[2];
  const double rr = dx * dx + dy * dy + dz * dz;
  const double* ea = env + a.pexp;
  const double* eb = env + b.pexp;
  const double log_rr0 = 1.7 - 1.5 * log(ea[a.nprim - 1] + eb[b.nprim - 1]);
  if (threadIdx.x == 0) pair_ld[(int64_t)ia * nv + ib] = log(sqrt(rr) + 1.0);
  const int64_t base = pair_off[(int64_t)ia * nv + ib];
  const int n = a.nprim * b.nprim;
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const int ip = p % a.nprim;
    const int jp = p / a.nprim;
    double mca = 0, mcb = 0;
    for (int c = 0; c < a.nctr; ++c) mca = fmax(mca, fabs(env[a.pcoef0 + c * a.nprim + ip]));
    for (int c = 0; c < b.nctr; ++c) mcb = fmax(mcb, fabs(env[b.pcoef0 + c * b.nprim + jp]));
    const double ai = ea[ip], aj = eb[jp];
    const double aij = ai + aj;
    const double inv = 1.0 / aij;
    const double e = rr * ai * aj * inv;
    PairPrim q;
    const double wj = aj * inv;
    q.px = a.r[0] + wj * (b.r[0] - a.r[0]);
    q.py = a.r[1] + wj * (b.r[1] - a.r[1]);
    q.pz = a.r[2] + wj * (b.r[2] - a.r[2]);
    q.aij = aij;
    q.kab = env[a.pcoef + ip] * env[b.pcoef + jp] * exp(-e);
    q.cce0 = e - log_rr0 - log(mca) - log(mcb);
    q.ai = ai;
    q.aj = aj;
    tmp[base + p] = q;
  }
  __syncthreads();
  // rank sort; a NaN key (never produced by finite inputs) sorts last
  auto key = [](double c) { return c == c ? c : __builtin_huge_val(); };
  for (int p = threadIdx.x; p < n; p += blockDim.x) {
    const double c = key(tmp[base + p].cce0);
    int rank = 0;
    for (int m = 0; m < n; ++m) {
      const double cm = key(tmp[base + m].cce0);
      rank += (cm < c) || (cm == c && m < p);
    }
    pp[base + rank] = tmp[base + p];
    pos[base + p] = rank;
  }
}

hipError_t launch_pairdata(const VShell* vsh, const double* env, int nv, const int* pairs,
                           int npairs, const int64_t* pair_off, double* pair_ld, PairPrim* tmp,
                           PairPrim* pp, int* pos, hipStream_t stream) {
  if (npairs <= 0) return hipSuccess;
  hipLaunchKernelGGL(pairdata_kernel, dim3(npairs), dim3(64), 0, stream, vsh, env, nv, pairs,
                     pair_off, pair_ld, tmp, pp, pos);
  return hipGetLastError();
}

__global__ void rys_batch_kernel(int n, const double* __restrict__ x, int64_t count,
                                 double* __restrict__ u, double* __restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count * n) return;
  const int64_t k = i / n;
  const int r = (int)(i - k * n);
  double uu, ww;
  rys_root_one(n, r, x[k], uu, ww);
  u[k * n + r] = uu;
  w[k * n + r] = ww;
}

hipError_t launch_rys_batch(int n, const double* x, int64_t count, double* u, double* w,
                            hipStream_t stream) {
  const int64_t tot = count * n;
  if (tot <= 0) return hipSuccess;
  hipLaunchKernelGGL(rys_batch_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, stream,
                     n, x, count, u, w);
  return hipGetLastError();
}

// Counts primitive quartets that pass libcint's screening (one lane per
// task); used by the benchmark's algorithmic FLOP model.
__global__ void count_prims_kernel(BasisView B, BucketArgs A, unsigned long long* counter) {
  const int64_t t = A.t0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= A.t1) return;
  const Task tk = A.tasks[t];
  const bool three = kind_three(A.kind);
  const bool noscreen = A.kind == KIND_2C2E;
  const VShell s0 = B.vsh[tk.sh[0]], s1 = B.vsh[tk.sh[1]], s2 = B.vsh[tk.sh[2]];
  const int nij = s0.nprim * s1.nprim;
  const int nkl = three ? s2.nprim : s2.nprim * B.vsh[tk.sh[3]].nprim;
  const PairPrim* pij = B.pp + B.pair_off[(int64_t)tk.sh[0] * B.nv + tk.sh[1]];
  const PairPrim* pkl = three ? nullptr : B.pp + B.pair_off[(int64_t)tk.sh[2] * B.nv + tk.sh[3]];
  const double ld_ij = B.pair_ld[(int64_t)tk.sh[0] * B.nv + tk.sh[1]] *
                       (A.la + A.lb + kind_bra_raise(A.kind));
  const double ld_kl = three ? 0.0
                             : B.pair_ld[(int64_t)tk.sh[2] * B.nv + tk.sh[3]] *
                                   (A.lc + A.ld + kind_ket_raise(A.kind));
  const double E = three ? B.expcutoff_3c : B.expcutoff_4c;
  if (noscreen) {
    atomicAdd(counter, (unsigned long long)nij * nkl);
    return;
  }
  int live_ij = 0, live_kl = three;
  for (int p = 0; p < nij; ++p) live_ij |= (pij[p].cce0 - ld_ij) < E;
  if (!three)
    for (int p = 0; p < nkl; ++p) live_kl |= (pkl[p].cce0 - ld_kl) < E;
  if (!(live_ij && live_kl)) return;
  unsigned long long n = 0;
  for (int kl = 0; kl < nkl; ++kl) {
    const double ckl = three ? 0.0 : pkl[kl].cce0 - ld_kl;
    if (ckl >= E) continue;
    for (int ij = 0; ij < nij; ++ij) {
      const double cij = pij[ij].cce0 - ld_ij;
      if (cij < E && cij <= (three ? E : E - ckl)) ++n;
    }
  }
  atomicAdd(counter, n);
}

hipError_t launch_count_prims(const BasisView& B, const BucketArgs& A, unsigned long long* counter,
                              hipStream_t stream) {
  const int64_t n = A.t1 - A.t0;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(count_prims_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, B,
                     A, counter);
  return hipGetLastError();
}

}  // namespace mcint

#include "eri_fast.h"

namespace mcint {
int g_wave_kernels = 1;
int8_t g_class_wave[NCLS * 7] = {};
#define MC_WAVE_HAS(a, b, c, d) \
  if (la == a && lb == b && lc == c && ld == d) return WaveCfg<a, b, c, d>::OK ? 1 : 0;
int wave_kernel_exists(int la, int lb, int lc, int ld) {
  MCINT_CHUNK_CLASSES(MC_WAVE_HAS)
  return 0;
}
#undef MC_WAVE_HAS
#define MC_WAVE_DEFAULT(a, b, c, d) \
  if (la == a && lb == b && lc == c && ld == d) return WaveCfg<a, b, c, d>::DEFAULT;
static bool wave_kernel_default(int la, int lb, int lc, int ld) {
  MCINT_CHUNK_CLASSES(MC_WAVE_DEFAULT)
  return false;
}
#undef MC_WAVE_DEFAULT
bool chunk_class_on_wave(int la, int lb, int lc, int ld, int tune_team, double omega, int fp32) {
  if (omega < 0 || fp32 || g_wave_kernels == 0 || !wave_kernel_exists(la, lb, lc, ld)) return false;
  if (g_wave_kernels == 2) return true;
  // per class and team size: the tuned choice, else the built-in rule
  // (team-of-one buckets, blocks of 480+ components)
  int tl = 0;
  while ((1 << tl) < tune_team && tl < 6) ++tl;
  const int cw = g_class_wave[class_index(la, lb, lc, ld) * 7 + tl];
  return cw ? cw == 2 : tune_team == 1 && wave_kernel_default(la, lb, lc, ld);
}
MCINT_FAST_DISPATCH
}  // namespace mcint
