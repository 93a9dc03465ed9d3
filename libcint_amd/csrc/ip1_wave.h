// Gradient digest of the i-derivative classes, and their wave kernel.
//
// The digest is the adjoint of the passes that form (d/dA_x a b|c d): per
// quartet the weights W = fkl [-2 D_ab D_cd + (D_ac D_bd + D_ad D_bc)/2] are
// taken back through the ket's spherical transform and transfer once for the
// three directions (G[ab][f], one lane per row ab), then through the bra's
// transform and transfer (one lane per column f) and meet the raised and
// lowered sets there:
//   g_x = sum_f sum_u ( sum_a a_x H_a[u+1_x-a] X-[u][f] - H[u] X+[u+1_x][f] ).
// Against forming the three derivative blocks first it transforms one ket
// instead of three.  Gradient of 58 shells: 13.7 -> 12.3 ms with both.
#pragma once
#include <algorithm>

#include "eri_fast.h"

namespace mcint {

// G[(ao, bo)][f] for the rows r0, r0 + rs, ...
template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void ip1_weights(const BasisView& Bv, const Task& tk, const BucketArgs& A,
                                            double* __restrict__ G, int r0, int rs) {
  using C = FastClass<LA, LB, LC, LD, 1>;
  constexpr int NF = C::NF, NC = C::NC, ND = C::ND;
  constexpr int NAo = C::NAo, NBo = C::NBo, NCo = C::NCo, NDo = C::NDo;
  const VShell& sa = Bv.vsh[tk.sh[0]];
  const VShell& sb = Bv.vsh[tk.sh[1]];
  const VShell& sc = Bv.vsh[tk.sh[2]];
  const VShell& sd = Bv.vsh[tk.sh[3]];
  const double cd[3] = {sc.r[0] - sd.r[0], sc.r[1] - sd.r[1], sc.r[2] - sd.r[2]};
  double cdp[3][LD + 1];
  sfor<3>([&](auto DI) {
    constexpr int d = decltype(DI)::value;
    cdp[d][0] = 1.0;
    sfor<LD>([&](auto K) { cdp[d][decltype(K)::value + 1] = cdp[d][decltype(K)::value] * cd[d]; });
  });
  const double fkl = sc.shell != sd.shell ? 2.0 : 1.0;
  const int64_t N = A.nao;
  const double* __restrict__ D = A.dm;
  const double* __restrict__ DR = D + (int64_t)sc.ao * N + sd.ao;
  for (int row = r0; row < NAo * NBo; row += rs) {
    const int ao = row / NBo, bo = row % NBo;
    const double* __restrict__ DP = D + (int64_t)(sa.ao + ao) * N;
    const double* __restrict__ DQ = D + (int64_t)(sb.ao + bo) * N;
    const double dpq = -2.0 * DP[sb.ao + bo];
    double pr[NCo], qr[NCo], ps[NDo], qs[NDo];
    sfor<NCo>([&](auto I) {
      constexpr int c = decltype(I)::value;
      pr[c] = 0.5 * DP[sc.ao + c];
      qr[c] = 0.5 * DQ[sc.ao + c];
    });
    sfor<NDo>([&](auto I) {
      constexpr int d = decltype(I)::value;
      ps[d] = DP[sd.ao + d];
      qs[d] = DQ[sd.ao + d];
    });
    double Zc[NC * ND];
    sfor<NC * ND>([&](auto I) { Zc[decltype(I)::value] = 0.0; });
    sfor<NCo * NDo>([&](auto OD) {
      constexpr int co = decltype(OD)::value / NDo, dd = decltype(OD)::value % NDo;
      const double w = fma(dpq, DR[co * N + dd], fma(pr[co], qs[dd], ps[dd] * qr[co]));
      sfor<NC * ND>([&](auto CD) {
        constexpr int c = decltype(CD)::value / ND, d = decltype(CD)::value % ND;
        constexpr double cc = c2x(true, LC, co, c) * c2x(true, LD, dd, d);
        if constexpr (cc != 0.0) Zc[c * ND + d] = fma(cc, w, Zc[c * ND + d]);
      });
    });
    double R[NF];
    sfor<NF>([&](auto I) { R[decltype(I)::value] = 0.0; });
    sfor<NC * ND>([&](auto CD) {
      constexpr int c = decltype(CD)::value / ND, d = decltype(CD)::value % ND;
      constexpr int cx = cpx(LC, c), cy = cpy(LC, c), cz = cpz(LC, c);
      constexpr int dx = cpx(LD, d), dy = cpy(LD, d), dz = cpz(LD, d);
      sfor<(dx + 1) * (dy + 1) * (dz + 1)>([&](auto TT) {
        constexpr int tt = decltype(TT)::value;
        constexpr int tx = tt / ((dy + 1) * (dz + 1)), ty = (tt / (dz + 1)) % (dy + 1), tz = tt % (dz + 1);
        constexpr double cb = binomc(dx, tx) * binomc(dy, ty) * binomc(dz, tz);
        constexpr int f = cindex(LC, cx + tx, cy + ty, cz + tz);
        const double pw = cdp[0][dx - tx] * cdp[1][dy - ty] * cdp[2][dz - tz];
        R[f] = fma(cb * pw, Zc[c * ND + d], R[f]);
      });
    });
    sfor<NF>([&](auto I) { G[row * NF + decltype(I)::value] = fkl * R[decltype(I)::value]; });
  }
}

// Adds to g the contraction of the block X (raised rows, then lowered rows,
// NF columns) with G over the columns f0, f0 + fs, ...
template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void ip1_contract(const BasisView& Bv, const Task& tk,
                                             const double* __restrict__ X, const double* __restrict__ G,
                                             int f0, int fs, double (&g)[3]) {
  using C = FastClass<LA, LB, LC, LD, 1>;
  constexpr int NF = C::NF, NA = C::NA, NB = C::NB, NAo = C::NAo, NBo = C::NBo, NEP = C::NEP;
  constexpr int NU = csum(LA, LA + LB);
  const VShell& sa = Bv.vsh[tk.sh[0]];
  const VShell& sb = Bv.vsh[tk.sh[1]];
  const double ab[3] = {sa.r[0] - sb.r[0], sa.r[1] - sb.r[1], sa.r[2] - sb.r[2]};
  double abp[3][LB + 1];
  sfor<3>([&](auto DI) {
    constexpr int d = decltype(DI)::value;
    abp[d][0] = 1.0;
    sfor<LB>([&](auto K) { abp[d][decltype(K)::value + 1] = abp[d][decltype(K)::value] * ab[d]; });
  });
  for (int f = f0; f < NF; f += fs) {
    double Gc[NA * NB];
    sfor<NA * NB>([&](auto I) { Gc[decltype(I)::value] = 0.0; });
    sfor<NAo * NBo>([&](auto OB) {
      constexpr int ao = decltype(OB)::value / NBo, bo = decltype(OB)::value % NBo;
      const double v = G[decltype(OB)::value * NF + f];
      sfor<NA * NB>([&](auto AB) {
        constexpr int a = decltype(AB)::value / NB, b = decltype(AB)::value % NB;
        constexpr double cc = c2x(true, LA, ao, a) * c2x(true, LB, bo, b);
        if constexpr (cc != 0.0) Gc[a * NB + b] = fma(cc, v, Gc[a * NB + b]);
      });
    });
    // transfer: the weight of [a+t| from every (a, b), by u = a+t for the
    // raised set and per direction, times a_x, for the lowered one
    auto transfer = [&](auto&& add) {
      sfor<NA * NB>([&](auto AB) {
        constexpr int a = decltype(AB)::value / NB, b = decltype(AB)::value % NB;
        constexpr int ax = cpx(LA, a), ay = cpy(LA, a), az = cpz(LA, a);
        constexpr int bx = cpx(LB, b), by = cpy(LB, b), bz = cpz(LB, b);
        sfor<(bx + 1) * (by + 1) * (bz + 1)>([&](auto TT) {
          constexpr int tt = decltype(TT)::value;
          constexpr int tx = tt / ((by + 1) * (bz + 1)), ty = (tt / (bz + 1)) % (by + 1), tz = tt % (bz + 1);
          constexpr double cb = binomc(bx, tx) * binomc(by, ty) * binomc(bz, tz);
          const double pw = cb * (abp[0][bx - tx] * abp[1][by - ty] * abp[2][bz - tz]);
          add(std::integral_constant<int, a>{}, std::integral_constant<int, ax + tx>{},
              std::integral_constant<int, ay + ty>{}, std::integral_constant<int, az + tz>{}, pw,
              Gc[a * NB + b]);
        });
      });
    };
    double H[NU];
    sfor<NU>([&](auto I) { H[decltype(I)::value] = 0.0; });
    transfer([&](auto, auto UX, auto UY, auto UZ, double pw, double v) {
      constexpr int u = cindex(LA, decltype(UX)::value, decltype(UY)::value, decltype(UZ)::value);
      H[u] = fma(pw, v, H[u]);
    });
    const double* __restrict__ Xf = X + f;
    sfor<NU>([&](auto I) {
      constexpr int u = decltype(I)::value;
      constexpr int ux = cpx(LA, u), uy = cpy(LA, u), uz = cpz(LA, u);
      constexpr int ix = cindex(LA + 1, ux + 1, uy, uz), iy = cindex(LA + 1, ux, uy + 1, uz);
      constexpr int iz = cindex(LA + 1, ux, uy, uz + 1);
      g[0] = fma(-H[u], Xf[ix * NF], g[0]);
      g[1] = fma(-H[u], Xf[iy * NF], g[1]);
      g[2] = fma(-H[u], Xf[iz * NF], g[2]);
    });
    if constexpr (LA > 0) {
      constexpr int NM = C::NEM;
      sfor<3>([&](auto DI) {
        constexpr int x = decltype(DI)::value;
        double L[NM];
        sfor<NM>([&](auto I) { L[decltype(I)::value] = 0.0; });
        transfer([&](auto AI, auto UX, auto UY, auto UZ, double pw, double v) {
          constexpr int a = decltype(AI)::value;
          constexpr int ax = x == 0 ? cpx(LA, a) : (x == 1 ? cpy(LA, a) : cpz(LA, a));
          if constexpr (ax > 0) {
            constexpr int u = cindex(LA - 1, decltype(UX)::value - (x == 0), decltype(UY)::value - (x == 1),
                                     decltype(UZ)::value - (x == 2));
            L[u] = fma(ax == 1 ? pw : ax * pw, v, L[u]);
          }
        });
        sfor<NM>([&](auto I) {
          constexpr int u = decltype(I)::value;
          g[x] = fma(L[u], Xf[(NEP + u) * NF], g[x]);
        });
      });
    }
  }
}

// Digest of the chunk kernels' blocks: TE lanes per task, LDS for the block
// and the weights.
template <int LA, int LB, int LC, int LD>
struct Ip1GradCfg {
  using C = FastClass<LA, LB, LC, LD, 1>;
  static constexpr int BUDGET = 6144;  // LDS doubles
  static constexpr int NEF = C::NE * C::NF, ROWS = C::NAo * C::NBo;
  static constexpr int PER = NEF + ROWS * C::NF;
  static constexpr int TPB_LDS = BUDGET / PER > 0 ? BUDGET / PER : 1;
  // columns and rows are whole lanes' work; the lane count covers the larger
  // unless fewer lanes halve the estimated wave instructions per task
  static constexpr int COL = 4 * C::NA * xfer_terms(LB) + nnz_c2s(LA) * nnz_c2s(LB);
  static constexpr int ROW = C::NC * xfer_terms(LD) + nnz_c2s(LC) * nnz_c2s(LD) + 4 * C::NCo * C::NDo;
  static constexpr int WORK = C::NF > ROWS ? C::NF : ROWS;
  static constexpr int TE_COVER = WORK > 32 ? 64 : (WORK > 16 ? 32 : (WORK > 8 ? 16 : (WORK > 4 ? 8 : 4)));
  static constexpr int tpb(int te) {
    const int t = 256 / te < TPB_LDS ? 256 / te : TPB_LDS;
    const int q = te < 64 ? 64 / te : 1;  // tasks per full wave
    return t >= q ? t - t % q : t;
  }
  static constexpr int64_t cost(int te) {
    const int lanes = tpb(te) * te < 64 ? tpb(te) * te : 64;
    return ((int64_t)((C::NF + te - 1) / te) * COL + (int64_t)((ROWS + te - 1) / te) * ROW) * 64 * te / lanes;
  }
  static constexpr int pick_te() {
    int best = TE_COVER;
    for (int te = TE_COVER / 2; te >= 1; te /= 2) {
      if (tpb(te) * te % 64) continue;
      const int blocks = 163840 / (tpb(te) * PER * 8 + 1);
      if ((blocks < 8 ? blocks : 8) * (tpb(te) * te / 64) < 8) continue;  // waves per CU
      if (2 * cost(te) <= cost(TE_COVER) && cost(te) < cost(best)) best = te;
    }
    return best;
  }
  static constexpr int TE = pick_te();
  static constexpr int TPB = tpb(TE);
  static constexpr int THREADS = TPB * TE;
  static_assert(PER <= BUDGET, "gradient digest exceeds its LDS budget");
};

template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(256) eri_ip1_grad_kernel(BasisView Bv, BucketArgs A) {
  using P = Ip1GradCfg<LA, LB, LC, LD>;
  constexpr int NEF = P::NEF, TE = P::TE;
  __shared__ double sm[P::TPB * P::PER];
  __shared__ double s_g[P::TPB][3];
  __shared__ int s_atom[2][P::TPB];
  const int team = threadIdx.x / TE;
  const int tl = threadIdx.x % TE;
  const int64_t t = A.t0 + (int64_t)blockIdx.x * P::TPB + team;
  const bool valid = t < A.t1;
  double* X = sm + team * P::PER;
  double* G = X + NEF;
  int any = 0;
  Task tk;
  if (valid) {
    tk = A.tasks[t];
    const int64_t slot = t - A.t0;
    any = A.flags[slot];
    const double* src = A.scratch + slot * NEF;
    if (any) {
      for (int k = tl; k < NEF; k += TE) X[k] = src[k];
      ip1_weights<LA, LB, LC, LD>(Bv, tk, A, G, tl, TE);
    }
  }
  __syncthreads();
  double g[3] = {0.0, 0.0, 0.0};
  if (valid && any) ip1_contract<LA, LB, LC, LD>(Bv, tk, X, G, tl, TE, g);
  for (int off = 1; off < TE; off <<= 1)
    for (int x = 0; x < 3; ++x) g[x] += __shfl_xor(g[x], off);
  if (tl == 0) {
    for (int x = 0; x < 3; ++x) s_g[team][x] = g[x];
    s_atom[0][team] = (valid && any) ? Bv.vsh[tk.sh[0]].atom : -1;
    s_atom[1][team] = (valid && any) ? grad_ref(A, tk) : -1;
  }
  __syncthreads();
  grad_block_flush(A, s_g, s_atom[0], s_atom[1], P::TPB);
}

// Wave kernel of a derivative class (the walk of eri_wave_kernel): a lane
// owns one row of the raised or lowered set.  For (dd| (65 rows) a lane owns
// one of the 55 distinct rows and sums it with and without the weight 2 a_i.
// With a density it digests in place, else it stores the block.  A wave takes
// consecutive groups of quartets and adds its sums where the atom changes.
template <int LA, int LB, int LC, int LD>
struct Ip1WaveCfg {
  using C = FastClass<LA, LB, LC, LD, 1>;
  static constexpr bool DUAL = C::NE > 64;
  static constexpr int NROW = DUAL ? csum(LA - 1, C::E) : C::NE;
  static constexpr int LPT = NROW <= 16 ? 16 : (NROW <= 32 ? 32 : 64);
  static constexpr int TPW = 64 / LPT;
  static constexpr int VS = (C::E + 1) * (C::F + 1);
  static constexpr int PV = 3 * C::NR * VS;
  static constexpr int PB0 = 2560 / (TPW * PV);
  static constexpr int PB = PB0 < 1 ? 1 : (PB0 > LPT ? LPT : PB0);
  static constexpr int PER = C::NE * C::NF + C::NAo * C::NBo * C::NF;  // block and weights
  // Blocks of 360+ components with at least 9 columns (the digest gives a lane
  // whole columns).  Gradient lists of one class, chunk kernels -> wave
  // kernel: (dd|dd) of 1 primitive quartet 139 -> 24 us, (dp|dp) of 36
  // 426 -> 233 us, (pd|dp) of 36 305 -> 164 us; below, it loses: (dd|ds) of 1
  // 108 -> 270 us, (pp|dp) of 36 178 -> 234 us.
  static constexpr bool OK = C::NF >= 9 && C::NE * C::NF >= 360;
  // Few columns per lane on a list that fills the chip: the chunk kernels'
  // lanes have a primitive quartet each.  Lists of 200 000 of 1 and 16 primitive
  // quartets, chunk and wave kernels: (pd|pp) stored 1.00 / 1.55, 1.71 / 2.68
  // ms, digested 1.01 / 1.25, 1.75 / 2.41; (dd|pp) stored 2.04 / 2.36, 3.09 /
  // 3.72, digested 1.79 / 1.65, 2.86 / 3.08; (pd|dp) stored 1.76 / 2.04, 3.02 /
  // 3.35, digested 1.86 / 1.39, 3.15 / 2.73.  Of 300 to 3000 the wave kernel
  // takes 1.02 to 2.1 times less in all of them.
  static constexpr bool MANY_DIGEST = C::NF >= 16;
  static constexpr bool MANY_STORE = C::NF > 16 || (C::NF == 16 && LA >= LB);
};

template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(64) eri_ip1_wave_kernel(BasisView Bv, BucketArgs A) {
  using C = FastClass<LA, LB, LC, LD, 1>;
  using W = Ip1WaveCfg<LA, LB, LC, LD>;
  constexpr int NF = C::NF, E = C::E, F = C::F, NR = C::NR, NEF = C::NE * NF, NEP = C::NEP;
  constexpr int LPT = W::LPT, TPW = W::TPW, VS = W::VS, PV = W::PV, PB = W::PB;
  constexpr bool DUAL = W::DUAL;
  constexpr int WALK_D = TPW * (PB * PV + 2 * PB * NR + PB * ((int)(sizeof(WavePrim) / 8) + 1));
  constexpr int EPI_D = TPW * W::PER;
  __shared__ double s_mem[WALK_D > EPI_D ? WALK_D : EPI_D];
  const int lane = threadIdx.x;
  const int sub = lane / LPT, sl = lane - sub * LPT;
  double* const sV = s_mem + sub * (PB * PV);
  double* const su = s_mem + TPW * PB * PV + sub * (PB * NR);
  double* const sw = s_mem + TPW * PB * PV + TPW * PB * NR + sub * (PB * NR);
  double* const s2a = s_mem + TPW * (PB * PV + 2 * PB * NR) + sub * PB;  // 2 a_i
  WavePrim* const sp = reinterpret_cast<WavePrim*>(s_mem + TPW * (PB * PV + 2 * PB * NR + PB)) + sub * PB;
  // this lane's row
  const bool has = sl < W::NROW;
  const int e0 = has ? sl : 0;
  int ox, oy, oz;       // offsets of its recurrence rows
  bool up;              // in the raised set
  [[maybe_unused]] bool low = false;  // DUAL: in the lowered set
  if constexpr (DUAL) {
    ox = cpx(LA - 1, e0);
    oy = cpy(LA - 1, e0);
    oz = cpz(LA - 1, e0);
    up = e0 >= csum(LA - 1, LA);
    low = e0 < C::NEM;
  } else {
    up = e0 < NEP;
    const int lo = up ? LA + 1 : LA - 1, k = up ? e0 : e0 - NEP;
    ox = cpx(lo, k);
    oy = cpy(lo, k);
    oz = cpz(lo, k);
  }
  ox *= F + 1;
  oy *= F + 1;
  oz *= F + 1;
  const double Ecut = Bv.expcutoff_4c;
  const double omega = Bv.omega;
  constexpr double cfac = 34.986836655249725 *
                          (LA == 0 ? 0.282094791773878143 : LA == 1 ? 0.488602511902919921 : 1.0) *
                          (LB == 0 ? 0.282094791773878143 : LB == 1 ? 0.488602511902919921 : 1.0) *
                          (LC == 0 ? 0.282094791773878143 : LC == 1 ? 0.488602511902919921 : 1.0) *
                          (LD == 0 ? 0.282094791773878143 : LD == 1 ? 0.488602511902919921 : 1.0);
  const unsigned long long own = (LPT == 64 ? ~0ull : ((1ull << LPT) - 1)) << (sub * LPT);
  const bool digest = A.dm != nullptr;
  int cur = -1;      // lanes 0-2 of a quartet: x, y, z of its atom; 3-5: of the
  double cs = 0.0;   // reference atom, minus
  double* const gbase = digest ? A.grad + slot_offset(A) : nullptr;
  const int64_t ngrp = (A.t1 - A.t0 + TPW - 1) / TPW;
  const int64_t g0 = ngrp * blockIdx.x / gridDim.x, g1 = ngrp * (blockIdx.x + 1) / gridDim.x;
  for (int64_t grp = g0; grp < g1; ++grp) {
    const int64_t t_first = A.t0 + grp * TPW;
    const int64_t t = t_first + sub;
    const bool valid = t < A.t1;
    const Task tk = A.tasks[valid ? t : t_first];
    const VShell& sa = Bv.vsh[tk.sh[0]];
    const VShell& sb = Bv.vsh[tk.sh[1]];
    const VShell& sc = Bv.vsh[tk.sh[2]];
    const VShell& sd = Bv.vsh[tk.sh[3]];
    double acc[NF];
    [[maybe_unused]] double acc2[DUAL ? NF : 1];
    sfor<NF>([&](auto J) {
      acc[decltype(J)::value] = 0.0;
      if constexpr (DUAL) acc2[decltype(J)::value] = 0.0;
    });
    // libcint's screening, one candidate per lane in its order
    const int nij = sa.nprim * sb.nprim, nkl = sc.nprim * sd.nprim;
    const int64_t pab = (int64_t)tk.sh[0] * Bv.nv + tk.sh[1];
    const int64_t pcd = (int64_t)tk.sh[2] * Bv.nv + tk.sh[3];
    const int64_t oij = Bv.pair_off[pab], okl = Bv.pair_off[pcd];
    const PairPrim* __restrict__ pij = Bv.pp + oij;
    const PairPrim* __restrict__ pkl = Bv.pp + okl;
    const double dij = (LA + LB + 1) * Bv.pair_ld[pab], dkl = (LC + LD) * Bv.pair_ld[pcd];
    // each pair's records ascend in cce0: the first decides emptiness
    const bool live = valid && pij[0].cce0 - dij < Ecut && pkl[0].cce0 - dkl < Ecut;
    const int npq = live ? nij * nkl : 0;
    int maxpq = npq;
    for (int off = LPT; off < 64; off <<= 1) maxpq = max(maxpq, __shfl_xor(maxpq, off));
    int any = 0;
    for (int base = 0; base < maxpq; base += LPT) {
      const int p = base + sl;
      bool pass = false;
      WavePrim wp;
      double a2 = 0.0;
      if (p < npq) {
        const int kl = (int)((unsigned)p / (unsigned)nij);
        const PairPrim P = pij[p - kl * nij];
        const PairPrim Q = pkl[kl];
        const double cce_kl = Q.cce0 - dkl, cce_ij = P.cce0 - dij;
        if (!(cce_kl > Ecut) && !(cce_ij > Ecut - cce_kl)) {
          any = 1;
          pass = cce_ij < Ecut && cce_kl < Ecut;  // else the stored exp factor is 0
        }
        if (pass) {
          a2 = 2.0 * P.ai;
          wp.aij = P.aij;
          wp.akl = Q.aij;
          wp.a1 = P.aij * Q.aij;
          wp.a0 = wp.a1 * rcp_pos(P.aij + Q.aij);
          wp.pq[0] = P.px - Q.px;
          wp.pq[1] = P.py - Q.py;
          wp.pq[2] = P.pz - Q.pz;
          wp.pa[0] = P.px - sa.r[0];
          wp.pa[1] = P.py - sa.r[1];
          wp.pa[2] = P.pz - sa.r[2];
          wp.qc[0] = Q.px - sc.r[0];
          wp.qc[1] = Q.py - sc.r[1];
          wp.qc[2] = Q.pz - sc.r[2];
          const double rr = wp.pq[0] * wp.pq[0] + wp.pq[1] * wp.pq[1] + wp.pq[2] * wp.pq[2];
          wp.fac = sqrt_pos(wp.a0 * rcp_pos(wp.a1 * wp.a1 * wp.a1)) * cfac * P.kab * Q.kab;
          wp.x = wp.a0 * rr;
          wp.theta = 1.0;
          if (omega > 0) {
            wp.theta = omega * omega * rcp_pos(omega * omega + wp.a0);
            wp.x *= wp.theta;
            wp.fac *= sqrt_pos(wp.theta);
          }
        }
      }
      const unsigned long long mask = __ballot(pass) & own;
      const int nsurv = __popcll(mask);
      const int slot = __popcll(mask & ((1ull << lane) - 1));
      int maxsurv = nsurv;
      for (int off = LPT; off < 64; off <<= 1) maxsurv = max(maxsurv, __shfl_xor(maxsurv, off));
      for (int b0 = 0; b0 < maxsurv; b0 += PB) {
        const int np = nsurv - b0 < 0 ? 0 : (nsurv - b0 < PB ? nsurv - b0 : PB);
        if (pass && slot >= b0 && slot < b0 + PB) {
          sp[slot - b0] = wp;
          s2a[slot - b0] = a2;
        }
        __syncthreads();
        for (int it = sl; it < np * NR; it += LPT) {
          const int q = it / NR, r = it - q * NR;
          double u, w;
          rys_root_one(NR, r, sp[q].x, u, w);
          if (omega > 0) {
            const double ut = u * sp[q].theta;
            u = ut * rcp_pos(u + 1.0 - ut);
          }
          su[it] = u;
          sw[it] = w * sp[q].fac;
        }
        __syncthreads();
        for (int it = sl; it < np * 3 * NR; it += LPT) {
          const int q = it / (3 * NR), dr = it - q * 3 * NR, d = dr / NR, r = dr - d * NR;
          const WavePrim& P = sp[q];
          const double u2 = P.a0 * su[q * NR + r];
          const double tmp4 = 0.5 * rcp_pos(u2 * (P.aij + P.akl) + P.a1);
          const double b00 = u2 * tmp4, b10 = b00 + tmp4 * P.akl, b01 = b00 + tmp4 * P.aij;
          const double c00 = P.pa[d] - 2.0 * b00 * P.akl * P.pq[d];
          const double c0p = P.qc[d] + 2.0 * b00 * P.aij * P.pq[d];
          double V[E + 1][F + 1];
          vrr2d<E, F, double>(V, d == 2 ? sw[q * NR + r] : 1.0, c00, c0p, b10, b01, b00);
          double* dst = sV + q * PV + dr * VS;
          sfor<(E + 1) * (F + 1)>([&](auto I) {
            constexpr int i = decltype(I)::value;
            dst[i] = V[i / (F + 1)][i % (F + 1)];
          });
        }
        __syncthreads();
        if (has) {
          for (int q = 0; q < np; ++q) {
            const double s2 = s2a[q];
            const double sc1 = up ? s2 : 1.0;
            for (int r = 0; r < NR; ++r) {
              const double* Vx = sV + q * PV + r * VS + ox;
              const double* Vy = sV + q * PV + (NR + r) * VS + oy;
              const double* Vz = sV + q * PV + (2 * NR + r) * VS + oz;
              double vx[F + 1], vy[F + 1], vz[F + 1], wz[DUAL ? F + 1 : 1];
              sfor<F + 1>([&](auto K) {
                constexpr int k = decltype(K)::value;
                vx[k] = Vx[k];
                vy[k] = Vy[k];
                vz[k] = DUAL ? Vz[k] : Vz[k] * sc1;
                if constexpr (DUAL) wz[k] = vz[k] * s2;
              });
              sfor<NF>([&](auto J) {
                constexpr int j = decltype(J)::value;
                constexpr int fx = cpx(LC, j), fy = cpy(LC, j), fz = cpz(LC, j);
                const double xy = vx[fx] * vy[fy];
                acc[j] = fma(xy, vz[fz], acc[j]);
                if constexpr (DUAL) acc2[j] = fma(xy, wz[fz], acc2[j]);
              });
            }
          }
        }
        __syncthreads();
      }
    }
    any = (__ballot(any) & own) != 0 && live;
    // the block: raised rows, then lowered rows, in LDS or to the scratch
    const int64_t slot_t = t - A.t0;
    double* const X = digest ? s_mem + sub * W::PER : A.scratch + slot_t * NEF;
    if (has && valid) {
      if constexpr (DUAL) {
        if (up) sfor<NF>([&](auto J) {
          X[(e0 - csum(LA - 1, LA)) * NF + decltype(J)::value] = acc2[decltype(J)::value];
        });
        if (low) sfor<NF>([&](auto J) { X[(NEP + e0) * NF + decltype(J)::value] = acc[decltype(J)::value]; });
      } else {
        sfor<NF>([&](auto J) { X[e0 * NF + decltype(J)::value] = acc[decltype(J)::value]; });
      }
    }
    if (!digest) {
      if (valid && sl == 0) {
        A.flags[slot_t] = any;
        if (A.not0) A.not0[A.task_id ? A.task_id[t] : t] = any;
      }
      continue;
    }
    double* const G = X + NEF;
    if (valid && any) ip1_weights<LA, LB, LC, LD>(Bv, tk, A, G, sl, LPT);
    __syncthreads();
    double g[3] = {0.0, 0.0, 0.0};
    if (valid && any) ip1_contract<LA, LB, LC, LD>(Bv, tk, X, G, sl, LPT, g);
    for (int off = 1; off < LPT; off <<= 1)
      for (int x = 0; x < 3; ++x) g[x] += __shfl_xor(g[x], off);
    if (valid && any && sl < 6) {
      const int at = sl < 3 ? sa.atom : grad_ref(A, tk);
      const double gx = sl == 0 || sl == 3 ? g[0] : (sl == 1 || sl == 4 ? g[1] : g[2]);
      if (at != cur) {
        if (cur >= 0) atomicAdd(gbase + 3 * cur + sl % 3, cs);
        cur = at;
        cs = 0.0;
      }
      cs += sl < 3 ? gx : -gx;
    }
    __syncthreads();  // the next quartet's walk reuses the LDS
  }
  if (digest && sl < 6 && cur >= 0) atomicAdd(gbase + 3 * cur + sl % 3, cs);
}

// Whether a launch of a derivative class runs the wave kernel: teams of one
// (up to 128 primitive quartets), long lists as above.  With 216 the
// chunk kernels' lanes all have a primitive quartet of their own: (dp|pp)
// 420 us against 602, (pp|dp) 746 against 1071.
template <int LA, int LB, int LC, int LD>
bool ip1_on_wave(const BucketArgs& A, double omega) {
  using W = Ip1WaveCfg<LA, LB, LC, LD>;
  if (!W::OK || g_wave_kernels == 0 || omega < 0) return false;
  return g_wave_kernels == 2 || (A.tune_team == 1 && (!A.many || (A.dm ? W::MANY_DIGEST : W::MANY_STORE)));
}

template <int LA, int LB, int LC, int LD, int... GRPs>
hipError_t launch_ip1(const BasisView& B, const BucketArgs& A, hipStream_t stream,
                      std::integer_sequence<int, GRPs...>) {
  const int64_t n = A.t1 - A.t0;
  hipError_t e = hipSuccess;
  bool done = false;
  if constexpr (Ip1WaveCfg<LA, LB, LC, LD>::OK) {
    if (ip1_on_wave<LA, LB, LC, LD>(A, B.omega)) {
      constexpr int TPW = Ip1WaveCfg<LA, LB, LC, LD>::TPW;
      const int64_t grp = (n + TPW - 1) / TPW;
      // several groups per wave once the chip is full (16 waves per CU)
      const int64_t rounds = A.dm ? std::min<int64_t>(16, std::max<int64_t>(1, grp / 4096)) : 1;
      hipLaunchKernelGGL((eri_ip1_wave_kernel<LA, LB, LC, LD>), dim3((unsigned)((grp + rounds - 1) / rounds)),
                         dim3(64), 0, stream, B, A);
      if (A.dm) return hipGetLastError();
      e = hipGetLastError();
      done = true;
    }
  }
  if (!done) {
    const int64_t per = ChunkCfg<LA, LB, LC, LD, 1>::THREADS / A.team;
    const unsigned nblk = (unsigned)((n + per - 1) / per);
    ((e = (e == hipSuccess ? launch_chunk_group<LA, LB, LC, LD, GRPs, 1>(B, A, stream, nblk) : e)), ...);
  }
  if (e != hipSuccess) return e;
  if (A.dm) {
    if (!A.sph) return hipErrorInvalidValue;
    using P = Ip1GradCfg<LA, LB, LC, LD>;
    hipLaunchKernelGGL((eri_ip1_grad_kernel<LA, LB, LC, LD>), dim3((unsigned)((n + P::TPB - 1) / P::TPB)),
                       dim3(P::THREADS), 0, stream, B, A);
  } else if (A.sph) {
    using P = Ip1EpiCfg<LA, LB, LC, LD>;
    hipLaunchKernelGGL((eri_ip1_epi_kernel<LA, LB, LC, LD>), dim3((unsigned)((n + P::TPB - 1) / P::TPB)),
                       dim3(P::THREADS), 0, stream, B, A);
  } else {
    using P = Ip1EpiCfg<LA, LB, LC, LD, false>;
    hipLaunchKernelGGL((eri_ip1_epi_kernel<LA, LB, LC, LD, false>), dim3((unsigned)((n + P::TPB - 1) / P::TPB)),
                       dim3(P::THREADS), 0, stream, B, A);
  }
  return hipGetLastError();
}

#define MCINT_IP1_DEFINE(a, b, c, d)                                                       \
  template <>                                                                              \
  hipError_t launch_ip1_class<a, b, c, d>(const BasisView& B, const BucketArgs& A,         \
                                          hipStream_t stream) {                            \
    return launch_ip1<a, b, c, d>(                                                         \
        B, A, stream, std::make_integer_sequence<int, chunk_groups(ChunkCfg<a, b, c, d, 1>::NCH)>{});    \
  }

}  // namespace mcint
