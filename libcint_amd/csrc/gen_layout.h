// Work layout of the generic (any class) kernel, computed on the host and
// passed to the kernel by value.
#pragma once
#include <algorithm>

#include "mcint_internal.h"

namespace mcint {

// Bounds of what the generic kernel takes: recurrence tables of one
// primitive quartet (3 directions x roots, doubled for short range, x
// (E+1)(F+1) doubles) and Cartesian components of the e-list and f-list (all
// of l <= 14: ipip1 of (66|ss) reaches e = 14).
constexpr int GEN_VCAP = 3 * 2 * NRYS_MAX * 90;
constexpr int GEN_ECAP = 680;
constexpr int GEN_FCAP = 680;
constexpr int GEN_LANES = 64;  // lanes of a workgroup (one wave, one task at a time)

// LDS per wave, in doubles: derivative components share a pass as long as
// the whole stays below the first figure (20 KB: eight waves per CU);
// classes that need more than the second for one component (64 KB) keep
// their blocks in global scratch.
constexpr int GEN_LDS_TARGET = 2560;
constexpr int GEN_LDS_MAX = 8000;

// Cartesian components of all shells below l
__host__ __device__ constexpr int tet(int l) { return l * (l + 1) * (l + 2) / 6; }
// terms of the horizontal transfers of all Cartesian components of shell l:
// sum over (bx, by, bz) of (bx+1)(by+1)(bz+1) = C(l+5, 5)
__host__ __device__ constexpr int xfer_count(int l) {
  return (l + 5) * (l + 4) * (l + 3) * (l + 2) * (l + 1) / 120;
}

// Primitive sums are kept as row sets of the bra (shells blo..bhi on centre
// A, weighted by the bw-th power of 2 a_i) by column sets of the ket (shells
// klo..khi on C, weighted by the kw-th power of 2 a_k); derivatives are
// formed from them after contraction.  With D_p|a> = a_p|a-1_p> - 2a|a+1_p>:
//   plain    bra la..la+lb                               ket lc..lc+ld
//   ip1      bra la-1.. (1), la+1.. (2a)                 ket as plain
//   ip2 (3c) bra as plain                                ket lc-1, lc+1 (2a)
//   ipip1    bra la-2.. (1), la.. (2a), la+2.. (4a^2)    ket as plain
//   ip1ip2   bra as ip1                                  ket lc-1.. (1), lc+1.. (2a)
// X holds set r's rows by all KF ket columns; H1/H2 the bra transferred and
// transformed, H3 the ket transferred, nbg bra components at a time.
struct GenLayout {
  int nbs, blo[3], bhi[3], nes[3], bw[3], ox[3];
  int nks, klo[2], khi[2], nfs[2], kw[2], cf[2];
  int be[3], kf[2];       // first e (f) of a set among the e-list (f-list)
  int e_lo, E, f_lo, F, nE, nF, KF;
  int nbc, nkc, ncomp;  // derivative components of the bra, the ket, in all
  int nca, ncb, ncc, ncd, nAo, nBo, nCo, nDo;
  int lij, lkl, nr, nrt;
  int nX, nH1, nH2, nH3;  // doubles of X and of one bra component's passes
  // LDS doubles: block regions (nbg components per pass), then the walk's
  // tables in the same space as the passes, the transfer terms, the codes
  int PB, nbg, oH1, oH2, oV, oP, ou, ow, oTb, oTk, oI;
  int lds;          // doubles of LDS
  // matrix kernel (mm_layout): Y = (bra matrix) X in tiles of 16 rows, then
  // block = Y (ket matrix)^T; k steps of 4
  int waves;            // waves per task, 0: the class does not fit
  int nbu;              // distinct bra components (ipip1: p <= q)
  int nrow, ncol;       // rows and columns of the block
  int RT, KS, CT1;      // bra: row tiles, k steps, column tiles (of KF)
  int CT2, KS2, YS;     // ket: column tiles, k steps, row stride of Y
  int nXz;              // doubles of X with its rows padded to 4
  int spread;           // lanes share a component's primitive quartets
  int in_lds;       // blocks in LDS (else in global scratch, nblk per wave)
  int64_t nblk;     // doubles of global scratch per wave
};

// Doubles per primitive quartet of a batch besides its recurrence tables
constexpr int GEN_PRIM_D = 19;

inline GenLayout gen_layout(int kind, int sph, int la, int lb, int lc, int ld, double omega) {
  GenLayout g{};
  const bool three = kind_three(kind);
  if (three) ld = 0;
  const bool ip1 = kind_bra_der(kind) || kind == KIND_2E_IP1IP2;
  const bool ket = kind_ket_der(kind) || kind == KIND_2E_IP1IP2;
  auto bset = [&](int shift, int w) {
    if (la + shift < 0) return;
    const int r = g.nbs++;
    g.blo[r] = la + shift;
    g.bhi[r] = la + lb + shift;
    g.bw[r] = w;
    g.nes[r] = tet(g.bhi[r] + 1) - tet(g.blo[r]);
  };
  if (kind == KIND_2E_IPIP1) {
    bset(-2, 0);
    bset(0, 1);
    bset(2, 2);
  } else if (ip1) {
    bset(-1, 0);
    bset(1, 1);
  } else {
    bset(0, 0);
  }
  auto kset = [&](int shift, int w) {
    if (lc + shift < 0) return;
    const int u = g.nks++;
    g.klo[u] = lc + shift;
    g.khi[u] = lc + ld + shift;
    g.kw[u] = w;
    g.nfs[u] = tet(g.khi[u] + 1) - tet(g.klo[u]);
    g.cf[u] = g.KF;
    g.KF += g.nfs[u];
  };
  if (ket) {
    kset(-1, 0);
    kset(1, 1);
  } else {
    kset(0, 0);
  }
  g.e_lo = g.blo[0];
  g.E = g.bhi[g.nbs - 1];
  g.f_lo = g.klo[0];
  g.F = g.khi[g.nks - 1];
  g.nE = tet(g.E + 1) - tet(g.e_lo);
  g.nF = tet(g.F + 1) - tet(g.f_lo);
  for (int r = 0; r < g.nbs; ++r) {
    g.ox[r] = g.nX;
    g.be[r] = tet(g.blo[r]) - tet(g.e_lo);
    g.nX += g.nes[r] * g.KF;
  }
  for (int u = 0; u < g.nks; ++u) g.kf[u] = tet(g.klo[u]) - tet(g.f_lo);
  g.nbc = kind == KIND_2E_IPIP1 ? 9 : (ip1 ? 3 : 1);
  g.nkc = ket ? 3 : 1;
  g.ncomp = g.nbc * g.nkc;
  g.nca = ncart(la);
  g.ncb = ncart(lb);
  g.ncc = ncart(lc);
  g.ncd = ncart(ld);
  g.nAo = sph ? nsph(la) : g.nca;
  g.nBo = sph ? nsph(lb) : g.ncb;
  g.nCo = sph ? nsph(lc) : g.ncc;
  g.nDo = sph ? nsph(ld) : g.ncd;
  g.lij = la + lb + kind_bra_raise(kind);
  g.lkl = lc + ld + kind_ket_raise(kind);
  g.nr = (g.lij + g.lkl) / 2 + 1;
  g.nrt = omega < 0 ? 2 * g.nr : g.nr;
  // the bra transform is the identity for s and p and for Cartesian output;
  // the ket needs no transfer with one plain shell
  const bool bra_c2s = sph && (la > 1 || lb > 1);
  const bool ket_x = !(three && g.nkc == 1);
  g.nH1 = g.nca * g.ncb * g.KF;
  g.nH2 = bra_c2s ? g.nAo * g.nBo * g.KF : 0;
  g.nH3 = ket_x ? g.nkc * g.nAo * g.nBo * g.ncc * g.ncd : 0;
  // H3 reuses H1's region unless H2 is H1
  auto passes = [&](int n) {
    const int a = bra_c2s ? (g.nH1 > g.nH3 ? g.nH1 : g.nH3) : g.nH1;
    return n * (a + (bra_c2s ? g.nH2 : g.nH3));
  };
  const int PV = 3 * g.nrt * (g.E + 1) * (g.F + 1) + 2 * g.nrt + GEN_PRIM_D;
  const int ncode = tet((g.E > g.F ? g.E : g.F) + 1);
  // terms: weights (doubles), packed exponents (ints), starts per component
  const int ntb = xfer_count(lb), ntk = three ? 1 : xfer_count(ld);
  const int fixed = ntb + ntk + (10 + ncode + ntb + ntk + g.ncb + g.ncd + 4 + 1) / 2;
  // a batch of primitive quartets: enough (primitive, direction, root)
  // recurrences for the lanes, at most 16 KB of tables
  // (second derivatives of 20 shells, when this was chosen: 29.4 ms; 8 KB
  // 31.9 ms, 4 KB 46 ms)
  g.PB = 1;
  while (g.PB < 16 && g.PB * 3 * g.nrt < GEN_LANES && (g.PB + 1) * PV <= 2048) ++g.PB;
  const int walk = g.PB * PV;
  auto total = [&](int n) {
    const int p = passes(n);
    return g.nX + (p > walk ? p : walk) + fixed;
  };
  g.nbg = g.nbc;
  while (g.nbg > 1 && total(g.nbg) > GEN_LDS_TARGET) g.nbg = (g.nbg + 1) / 2;
  g.in_lds = total(g.nbg) <= GEN_LDS_MAX;
  const int xl = g.in_lds ? g.nX : 0, pl = g.in_lds ? passes(g.nbg) : 0;
  g.nblk = g.in_lds ? 0 : g.nX + passes(g.nbg);
  // block offsets: in LDS or in the wave's global scratch
  g.oH1 = g.nX;
  g.oH2 = g.nX + g.nbg * (bra_c2s ? (g.nH1 > g.nH3 ? g.nH1 : g.nH3) : g.nH1);
  g.oV = xl;
  g.oP = g.oV + g.PB * 3 * g.nrt * (g.E + 1) * (g.F + 1);
  g.ou = g.oP + g.PB * GEN_PRIM_D;
  g.ow = g.ou + g.PB * g.nrt;
  g.oTb = xl + (pl > walk ? pl : walk);
  g.oTk = g.oTb + ntb;
  g.oI = g.oTk + ntk;
  g.lds = g.oTb + fixed;
  return g;
}

// LDS doubles of the matrix kernel's four-wave workgroup: two of them per CU.
constexpr int MM_LDS4 = 10200;
// The matrix kernel's instances: up to this many roots, and one for more.
constexpr int MM_NRT = 6;

// Layout of the matrix kernel: X, then the walk's tables, each wave's Y and
// the partial sums of shared components in one space, then the codes.
inline GenLayout mm_layout(int kind, int sph, int la, int lb, int lc, int ld, double omega, int waves) {
  GenLayout g = gen_layout(kind, sph, la, lb, lc, ld, omega);
  const bool three = kind_three(kind);
  const int threads = 64 * waves;
  int R = 0;
  for (int r = 0; r < g.nbs; ++r) R += g.nes[r];
  g.nbu = kind == KIND_2E_IPIP1 ? 6 : g.nbc;
  g.nrow = g.nbu * g.nAo * g.nBo;
  g.ncol = g.nkc * g.nCo * (three ? 1 : g.nDo);
  g.RT = (g.nrow + 15) / 16;
  g.KS = (R + 3) / 4;
  g.CT1 = (g.KF + 15) / 16;
  g.CT2 = (g.ncol + 15) / 16;
  g.KS2 = (g.KF + 3) / 4;
  g.YS = g.CT1 * 16 + 1;
  g.nXz = g.KS * 4 * g.KF;
  g.spread = 2 * g.nE * g.nF <= threads;
  // A batch: two (primitive, direction, root) recurrences per lane, so that
  // its barriers are shared by more primitive quartets, in tables that leave
  // the LDS to several workgroups.  Second derivatives of 20 shells / three-
  // centre derivatives of 186 shells, when this was chosen: 10.9 / 4.95 ms; one recurrence per lane
  // 11.3 / 5.1; four 10.8 / 5.2; tables of 24 and 16 KB (four waves, one)
  // 11.2 / 4.9, of 32 and 16 KB 10.8 / 5.1.
  const int VT = 3 * g.nrt * (g.E + 1) * (g.F + 1);
  const int PV = VT + 2 * g.nrt + GEN_PRIM_D;
  g.PB = 1;
  while (g.PB < 16 * waves && g.PB * 3 * g.nrt < 2 * threads && (g.PB + 1) * PV <= (waves > 1 ? 3584 : 1536)) ++g.PB;
  int space = g.PB * PV;
  if (waves * 16 * g.YS > space) space = waves * 16 * g.YS;
  if (g.spread && 5 * threads > space) space = 5 * threads;
  const int ncode = tet((g.E > g.F ? g.E : g.F) + 1);
  g.oV = g.nXz;
  g.oP = g.oV + g.PB * VT;
  g.ou = g.oP + g.PB * GEN_PRIM_D;
  g.ow = g.ou + g.PB * g.nrt;
  g.oI = g.nXz + space;
  g.lds = g.oI + (10 + g.nrow + g.ncol + 2 * waves + (ncode + 1) / 2 + 1) / 2;
  g.waves = g.lds <= (waves > 1 ? MM_LDS4 : GEN_LDS_MAX) ? waves : 0;
  return g;
}

// Waves per task of a launch of n tasks with np primitive quartets in all: four
// or one on the matrix kernel, 0 on the generic one.  Work is a task's products
// (components x roots x primitive quartets).
//   Four: with 2000 products or more to share, where the list is short, tasks
//   hold many primitives (or many products of more roots than are compiled
//   in), or the LDS then leaves a CU twice the waves (i-derivatives (dd|dg) of
//   256 primitives, 3000 tasks: 44 KB for one wave, 69 for four; 52 and 11 ms).
//   None: where the bra matrix outweighs the walk and at most four columns use
//   it, of the matrix instruction's 16 (3000 Cartesian (gg|ss) of one
//   primitive: 364 us, 54 on the generic kernel), where one-wave
//   workgroups fill the LDS and tasks hold primitives for more than two to
//   four waves (int2e_ip1ip2 (fp|df) of 256: 97 and 34 ms), and for (s|s) and
//   (p|s), which are set-up alone (30 000 (s|s) of one primitive: 206 and 146 us).
// Over 2716 lists (280 classes of every kind, s to i shells, 1 to 256 primitive
// quartets, 300 to 30 000 tasks) this takes 1.04 times the fastest of the three
// on geometric average; by tasks and primitives alone 1.14.
constexpr int64_t MM_TASKS = 1024;
constexpr double MM_PRIMS = 24, MM_WORK = 2000, MM_WORK4 = 50000;
inline int mm_waves(int kind, int sph, int la, int lb, int lc, int ld, double omega, int64_t n, int64_t np) {
  const GenLayout g1 = mm_layout(kind, sph, la, lb, lc, ld, omega, 1);
  const GenLayout g4 = mm_layout(kind, sph, la, lb, lc, ld, omega, 4);
  const double prims = (double)np / (double)n, work = prims * g1.nE * g1.nF * g1.nrt;
  const bool four = g4.waves && work >= MM_WORK;
  if (four && n < MM_TASKS) return 4;
  const int bra = g1.RT * g1.KS;
  if (g1.KS2 == 1 && bra >= 240 && work < 32.0 * bra) return 0;
  if (kind == KIND_2C2E && work < 4) return 0;
  // waves of a CU (160 KB of LDS, 256 CUs): by the LDS, and with this list
  const int lds = 160 * 1024 / 8;
  const int cu1 = std::min(12, lds / g1.lds), cu4 = 4 * std::min(4, lds / g4.lds);
  const double tasks = n / 256.0;
  if (four && (prims >= MM_PRIMS || (g1.nrt > MM_NRT && work >= MM_WORK4) ||
               (prims >= 12 && std::min<double>(cu4, 4 * tasks) >= 2 * std::min<double>(cu1, tasks))))
    return 4;
  if (!g1.waves || (n >= MM_TASKS / 2 && ((cu1 <= 4 && prims >= MM_PRIMS) || (cu1 <= 2 && prims >= 8)))) return 0;
  return 1;
}

// One matrix to lay out: the bra matrix of the virtual pair (a, b) or the
// ket matrix of (a, b) (three-centre kinds: b = a, no transfer), at off.
struct XferItem {
  int a, b, ket, rows, ks;  // rows: tiles of 16; ks: k steps of 4
  int64_t off;
};
// Matrices of a plan's pairs, by ordered virtual pair.
struct XferView {
  const double* m;
  const int64_t* bra;
  const int64_t* ket;
  int nv;
};
// max_rows, max_ks: the largest among the items
hipError_t launch_xfer(const VShell* vsh, int kind, int sph, const XferItem* items, int n, int max_rows, int max_ks,
                       double* m, hipStream_t stream);
// The matrix kernel on waves per task (1 or 4; mm_layout(..., waves).waves != 0).
hipError_t launch_matrix(const BasisView& B, const BucketArgs& A, const XferView& X, int waves,
                         hipStream_t stream);

// Waves from which on a workgroup takes several tasks, one after another: where
// a primitive quartet's products are few, the set-up of a workgroup weighs more
// than an even load (30 000 (s|s): 170 -> 146 us on the generic kernel; 30 000
// (pf|dg) second derivatives 29.0 -> 30.8 ms).
inline int64_t gen_share(const GenLayout& g) { return g.nE * g.nF * g.nrt <= 2000 ? 8192 : 16384; }

// Whether the kernel's tables hold the class.
inline bool gen_fits(const GenLayout& g) {
  return g.nE <= GEN_ECAP && g.nF <= GEN_FCAP && 3 * g.nrt * (g.E + 1) * (g.F + 1) <= GEN_VCAP;
}

}  // namespace mcint
