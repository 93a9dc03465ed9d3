// Generic kernel: any class and kind, one 64-lane workgroup per contracted
// quartet, class known at run time.  It serves what has neither a register
// kernel nor a plan's transfer matrices (matrix.hip): single calls on an
// optimizer's device state, classes whose sums exceed the LDS or leave a CU too
// few waves, whose matrices outweigh their walk or exceed the plan's bound.
//
// The walk takes 64 candidate primitive quartets at a time (one per lane, in
// libcint's order and with its tests), compacts the survivors, and for a
// batch of them evaluates all roots (one (quartet, root) per lane), then all
// 2D recurrences (one (quartet, direction, root) per lane) into LDS; then
// each lane sums the batch's products of its components and adds them to the
// task's block once.  Blocks stay in LDS wherever they fit (gen_layout).
// The passes after contraction (bra derivative and transfer, bra transform,
// ket derivative and transfer, ket transform and store) read transfer terms
// whose weights are laid out once per task, and step through their elements
// by carries instead of divisions.
//
// What bounds it: latency (waves wait 0.6 of their cycles, VALU issue 0.18,
// a quarter of it FP64) at the index arithmetic and LDS reads of runtime
// classes, and few lanes in use for small classes.  Measured on all of
// int2e_ipip1 + int2e_ip1ip2 of 20 shells: 25.1 ms, 101 ms with the block in
// global memory, one primitive quartet at a time and binomials and powers
// recomputed for each transfer term.
#include <algorithm>

#include "gen_device.h"

namespace mcint {

// Three waves per SIMD: at two (216 VGPRs) the three-centre derivatives of
// 186 shells take 6.9 ms instead of 5.6, at four and five (spilling) 6.3 and
// 7.7 ms.
template <bool IN_LDS>
__global__ void __launch_bounds__(GEN_LANES)
__attribute__((amdgpu_waves_per_eu(3))) eri_generic_kernel(BasisView B, BucketArgs A, GenLayout G) {
  extern __shared__ double sm[];
  const int lane = threadIdx.x;
  const int kind = A.kind;
  const bool three = kind_three(kind);
  const bool noscreen = kind == KIND_2C2E;  // (i|k): no screening (src/cint2c2e.c:57-147)
  const int la = A.la, lb = A.lb, lc = A.lc, ld = three ? 0 : A.ld;
  double* const X = IN_LDS ? sm : A.scratch + (int64_t)blockIdx.x * G.nblk;
  double* const sV = sm + G.oV;
  GenPrim* const sp = reinterpret_cast<GenPrim*>(sm + G.oP);
  double* const su = sm + G.ou;
  double* const sw = sm + G.ow;
  double* const tbw = sm + G.oTb;  // weights of the bra / ket transfer terms
  double* const tkw = sm + G.oTk;
  int2* const sets = reinterpret_cast<int2*>(sm + G.oI);  // put_sets
  int* const code = reinterpret_cast<int*>(sets + GEN_SETS);
  const int ncode = tet((G.E > G.F ? G.E : G.F) + 1);
  const int ntb = xfer_count(lb), ntk = three ? 1 : xfer_count(ld);
  int* const tb = code + ncode;   // exponents t of the terms, x | y << 4 | z << 8 | (b - t) << 12 ..
  int* const tk_ = tb + ntb;
  int* const tbp = tk_ + ntk;     // first term of each component
  int* const tkp = tbp + G.ncb + 1;

  // ---- per wave: exponents of the Cartesian components, transfer terms ---
  if (lane == 0) put_sets(G, sets);
  for (int i = lane; i < ncode; i += GEN_LANES) {
    int l = 0, k = i;
    while (k >= ncart(l)) { k -= ncart(l); ++l; }
    int m = 0;
    while ((m + 1) * (m + 2) / 2 <= k) ++m;
    const int z = k - m * (m + 1) / 2;
    code[i] = (l - m) | ((m - z) << 4) | (z << 8);
  }
  __syncthreads();
  auto terms = [&](int l, int n, int* start, int* term) {
    for (int b = lane; b <= n; b += GEN_LANES) {
      int s = 0;
      for (int i = 0; i < b; ++i) {
        const int c = code[tet_d(l) + i];
        s += ((c & 15) + 1) * (((c >> 4) & 15) + 1) * (((c >> 8) & 15) + 1);
      }
      start[b] = s;
      if (b == n) continue;
      const int c = code[tet_d(l) + b];
      const int bx = c & 15, by = (c >> 4) & 15, bz = (c >> 8) & 15;
      for (int tx = 0; tx <= bx; ++tx)
        for (int ty = 0; ty <= by; ++ty)
          for (int tz = 0; tz <= bz; ++tz)
            term[s++] = tx | (ty << 4) | (tz << 8) | ((bx - tx) << 12) | ((by - ty) << 16) |
                        ((bz - tz) << 20);
    }
  };
  terms(lb, G.ncb, tbp, tb);
  terms(ld, three ? 1 : G.ncd, tkp, tk_);

  const double Ecut0 = three ? B.expcutoff_3c : B.expcutoff_4c;
  const double omega = B.omega;
  const bool sr = omega < 0;
  const int nr = G.nr, nrt = G.nrt;
  const int ER = G.E, FR = G.F, F1 = FR + 1, VS = (ER + 1) * F1;
  const double cfac = PI3_2_SQRTPI * common_fac_sp(la) * common_fac_sp(lb) * common_fac_sp(lc) *
                      (three ? 1.0 : common_fac_sp(ld));

  for (int64_t t = A.t0 + blockIdx.x; t < A.t1; t += gridDim.x) {
    const Task tk = A.tasks[t];
    const VShell& s0 = B.vsh[tk.sh[0]];
    const VShell& s1 = B.vsh[tk.sh[1]];
    const VShell& s2 = B.vsh[tk.sh[2]];
    const VShell& s3 = B.vsh[three ? tk.sh[2] : tk.sh[3]];
    __syncthreads();  // the last task's passes have read their terms and blocks

    // transfer weights: binomials times powers of A-B and C-D
    auto weights = [&](const VShell& p, const VShell& q, const int* term, int n, double* w) {
      const double r[3] = {p.r[0] - q.r[0], p.r[1] - q.r[1], p.r[2] - q.r[2]};
      for (int i = lane; i < n; i += GEN_LANES) {
        const int c = term[i];
        double v = 1.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int tt = (c >> (4 * d)) & 15, k = (c >> (12 + 4 * d)) & 15;
          for (int j = 0; j < k; ++j) v *= r[d];
          if (tt && k) v *= binom_small(tt + k, k);
        }
        w[i] = v;
      }
    };
    weights(s0, s1, tb, ntb, tbw);
    if (!three) weights(s2, s3, tk_, ntk, tkw);
    else if (lane == 0) tkw[0] = 1.0;
    for (int i = lane; i < G.nX; i += GEN_LANES) X[i] = 0.0;

    // ---- the walk ---------------------------------------------------------
    const int nij = s0.nprim * s1.nprim;
    const int nkl = three ? s2.nprim : s2.nprim * s3.nprim;
    const int64_t pab = (int64_t)tk.sh[0] * B.nv + tk.sh[1];
    const int64_t pcd = three ? 0 : (int64_t)tk.sh[2] * B.nv + tk.sh[3];
    const int64_t oij = B.pair_off[pab], okl = three ? 0 : B.pair_off[pcd];
    const PairPrim* __restrict__ pij = B.pp + oij;
    const PairPrim* __restrict__ pkl = B.pp + okl;
    const int* __restrict__ pos_ij = B.pp_pos + oij;
    const int* __restrict__ pos_kl = B.pp_pos + okl;
    const double* __restrict__ ek = B.env + s2.pexp;
    const double* __restrict__ ck = B.env + s2.pcoef;
    // distance terms of the screening estimate cce = cce0 - l * log(d + 1);
    // short range widens them to log(d + theta_pair r_guess + 1) and raises
    // the loop cutoff (src/optimizer.c:301-315, src/cint2e.c:358-380,
    // src/cint3c2e.c:279-296; r_guess = 8)
    const int lij = G.lij, lkl = G.lkl;
    double dij_term = lij * B.pair_ld[pab], dkl_term = three ? 0.0 : lkl * B.pair_ld[pcd];
    double Ecut = Ecut0;
    if (sr) {
      const double w2 = omega * omega;
      auto dist = [](const VShell& p, const VShell& q) {
        return sqrt((p.r[0] - q.r[0]) * (p.r[0] - q.r[0]) + (p.r[1] - q.r[1]) * (p.r[1] - q.r[1]) +
                    (p.r[2] - q.r[2]) * (p.r[2] - q.r[2]));
      };
      const double dab = dist(s0, s1);
      const double th_ij = w2 / (w2 + B.env[s0.pexp + s0.nprim - 1] + B.env[s1.pexp + s1.nprim - 1]);
      dij_term = lij > 0 ? lij * log(dab + th_ij * 8.0 + 1.0) : 0.0;
      if (nr > 1 && lij > 0) Ecut += lij * log((dab + th_ij * 8.0 + 1.0) / (dab + 1.0));
      if (three) {
        const double th_k = w2 / (w2 + B.env[s2.pexp + s2.nprim - 1]);
        if (nr > 1 && lkl > 0) Ecut += lkl * log(th_k * 8.0 + 1.0);
      } else {
        const double dcd = dist(s2, s3);
        const double th_kl = w2 / (w2 + B.env[s2.pexp + s2.nprim - 1] + B.env[s3.pexp + s3.nprim - 1]);
        dkl_term = lkl > 0 ? lkl * log(dcd + th_kl * 8.0 + 1.0) : 0.0;
        if (nr > 1 && lkl > 0) Ecut += lkl * log((dcd + th_kl * 8.0 + 1.0) / (dcd + 1.0));
      }
    }
    // pair emptiness (libcint returns early when a pair has no primitive
    // below the cutoff: src/cint2e.c:96-109)
    bool live_ij = noscreen, live_kl = three;
    if (!noscreen)
      for (int p = lane; p < nij; p += GEN_LANES) live_ij |= (pij[p].cce0 - dij_term) < Ecut0;
    if (!three)
      for (int p = lane; p < nkl; p += GEN_LANES) live_kl |= (pkl[p].cce0 - dkl_term) < Ecut0;
    const bool live = __ballot(live_ij) != 0 && __ballot(live_kl) != 0;
    const int npq = live ? nij * nkl : 0;
    bool any = false;
    for (int base = 0; base < npq; base += GEN_LANES) {
      // one candidate per lane, in libcint's order (ip fastest)
      const int p = base + lane;
      bool pass = false;
      GenPrim wp;
      if (p < npq) {
        const int kl = (int)((unsigned)p / (unsigned)nij), ij = p - kl * nij;
        const PairPrim P = pij[pos_ij[ij]];
        double cce_kl = 0.0, akl, kkl, ak, q[3];
        if (three) {
          akl = ak = ek[kl];
          kkl = ck[kl];
          q[0] = s2.r[0]; q[1] = s2.r[1]; q[2] = s2.r[2];
        } else {
          const PairPrim Q = pkl[pos_kl[kl]];
          cce_kl = Q.cce0 - dkl_term;
          akl = Q.aij;
          ak = Q.ai;
          kkl = Q.kab;
          q[0] = Q.px; q[1] = Q.py; q[2] = Q.pz;
        }
        const double cce_ij = noscreen ? -1e300 : P.cce0 - dij_term;
        const double room = three ? Ecut : Ecut - cce_kl;
        if ((three || !(cce_kl > Ecut)) && !(cce_ij > room)) {
          // beyond the unwidened cutoff the stored exp factor is 0
          const bool kept = noscreen || (cce_ij < Ecut0 && cce_kl < Ecut0);
          wp.aij = P.aij;
          wp.akl = akl;
          wp.a1 = P.aij * akl;
          wp.a0 = wp.a1 * rcp_pos(P.aij + akl);
          wp.pq[0] = P.px - q[0];
          wp.pq[1] = P.py - q[1];
          wp.pq[2] = P.pz - q[2];
          wp.pa[0] = P.px - s0.r[0];
          wp.pa[1] = P.py - s0.r[1];
          wp.pa[2] = P.pz - s0.r[2];
          wp.qc[0] = q[0] - s2.r[0];
          wp.qc[1] = q[1] - s2.r[1];
          wp.qc[2] = q[2] - s2.r[2];
          const double rr = wp.pq[0] * wp.pq[0] + wp.pq[1] * wp.pq[1] + wp.pq[2] * wp.pq[2];
          wp.fac = sqrt_pos(wp.a0 * rcp_pos(wp.a1 * wp.a1 * wp.a1)) * cfac * P.kab * kkl;
          wp.x = wp.a0 * rr;
          wp.theta = 1.0;
          wp.w[0] = 2.0 * P.ai;
          wp.w[1] = wp.w[0] * wp.w[0];
          wp.w[2] = 2.0 * ak;
          if (sr) {
            // pairs beyond the unwidened cutoff carry no data, and tiny erfc
            // tails are dropped: src/g2e.c:4449-4453 (EXPCUTOFF_SR)
            if (kept) {
              wp.theta = omega * omega * rcp_pos(omega * omega + wp.a0);
              const double tx = wp.theta * wp.x;
              pass = !(tx > room - cce_ij || tx > 40.0);
              any |= pass;
            }
          } else {
            any = true;
            pass = kept;
            if (omega > 0) {
              wp.theta = omega * omega * rcp_pos(omega * omega + wp.a0);
              wp.x *= wp.theta;
              wp.fac *= sqrt_pos(wp.theta);
            }
          }
        }
      }
      const unsigned long long mask = __ballot(pass);
      const int nsurv = __popcll(mask);
      const int slot = __popcll(mask & ((1ull << lane) - 1));
      for (int b0 = 0; b0 < nsurv; b0 += G.PB) {
        const int np = min(nsurv - b0, G.PB);
        if (pass && slot >= b0 && slot < b0 + np) sp[slot - b0] = wp;
        __syncthreads();
        // roots: short range takes the full rule on nr roots minus the
        // theta-scaled rule on nr more (src/g2e.c:4455-4476; exact for the
        // polynomial integrand, as is the rule on [sqrt(theta), 1])
        for (int it = lane; it < np * nrt; it += GEN_LANES) {
          const int q = (int)((unsigned)it / (unsigned)nrt), r = it - q * nrt;
          const double th = sp[q].theta, x = sp[q].x;
          const bool lr = sr && r >= nr;
          double u, w;
          rys_root_one(nr, lr ? r - nr : r, lr ? x * th : x, u, w);
          if (omega > 0 || lr) {
            const double ut = u * th;
            u = ut * rcp_pos(u + 1.0 - ut);
          }
          if (lr) w *= -sqrt_pos(th);
          su[it] = u;
          sw[it] = w * sp[q].fac;
        }
        __syncthreads();
        // 2D recurrence of every (primitive quartet, direction, root)
        for (int it = lane; it < np * 3 * nrt; it += GEN_LANES) {
          const int q = (int)((unsigned)it / (unsigned)(3 * nrt)), dr = it - q * 3 * nrt;
          const int d = dr >= 2 * nrt ? 2 : (dr >= nrt ? 1 : 0), r = dr - d * nrt;
          const GenPrim& P = sp[q];
          const double u2 = P.a0 * su[q * nrt + r];
          const double tmp4 = 0.5 * rcp_pos(u2 * (P.aij + P.akl) + P.a1);
          const double b00 = u2 * tmp4, b10 = b00 + tmp4 * P.akl, b01 = b00 + tmp4 * P.aij;
          const double c00 = P.pa[d] - 2.0 * b00 * P.akl * P.pq[d];
          const double c0p = P.qc[d] + 2.0 * b00 * P.aij * P.pq[d];
          double* V = sV + q * 3 * nrt * VS + dr * VS;
          V[0] = d == 2 ? sw[q * nrt + r] : 1.0;
          double v1 = V[0], v0 = 0.0;
          for (int e = 0; e < ER; ++e) {
            const double v = fma(e * b10, v0, c00 * v1);
            V[(e + 1) * F1] = v;
            v0 = v1;
            v1 = v;
          }
          for (int f = 0; f < FR; ++f) {
            double prev = 0.0;
            for (int e = 0; e <= ER; ++e) {
              const double cur = V[e * F1 + f];
              double v = fma(e * b00, prev, c0p * cur);
              if (f > 0) v = fma(f * b01, V[e * F1 + f - 1], v);
              V[e * F1 + f + 1] = v;
              prev = cur;
            }
          }
        }
        __syncthreads();
        // products: each lane's components, the batch summed, then added to
        // the sets the component belongs to
        const int nEF = G.nE * G.nF;
        const int te = tet_d(G.e_lo), tf = tet_d(G.f_lo);
        Odo<2> o(lane, {G.nF, G.nE});
        for (int c = lane; c < nEF; c += GEN_LANES, o.next()) {
          const int jf = o.d[0], ie = o.d[1];
          const int ec = code[te + ie], fc = code[tf + jf];
          const double* Vx = sV + (ec & 15) * F1 + (fc & 15);
          const double* Vy = sV + nrt * VS + ((ec >> 4) & 15) * F1 + ((fc >> 4) & 15);
          const double* Vz = sV + 2 * nrt * VS + ((ec >> 8) & 15) * F1 + ((fc >> 8) & 15);
          // weight 1, 2a_i, 4a_i^2; the same times 2a_k
          double g0 = 0, g1 = 0, g2 = 0, h0 = 0, h1 = 0;
          for (int q = 0; q < np; ++q) {
            // one root's values are on their way while the last one's are used
            // (25.2 -> 23.4 ms for the lists of add_to_sets)
            double g = 0, vx = Vx[0], vy = Vy[0], vz = Vz[0];
            for (int o = VS; o < nrt * VS; o += VS) {
              const double nx = Vx[o], ny = Vy[o], nz_ = Vz[o];
              g = fma(vx * vy, vz, g);
              vx = nx;
              vy = ny;
              vz = nz_;
            }
            g = fma(vx * vy, vz, g);
            g0 += g;
            if (G.nbs > 1) {
              g1 = fma(g, sp[q].w[0], g1);
              if (G.nbc == 9) g2 = fma(g, sp[q].w[1], g2);
            } else if (G.nbc > 1) {  // a lone raised set (no lowered shell)
              g1 = fma(g, sp[q].w[0], g1);
              g2 = fma(g, sp[q].w[1], g2);
            }
            if (G.nkc > 1) {
              const double h = g * sp[q].w[2];
              h0 += h;
              h1 = fma(h, sp[q].w[0], h1);
            }
            Vx += 3 * nrt * VS;
            Vy += 3 * nrt * VS;
            Vz += 3 * nrt * VS;
          }
          add_to_sets(sets, G.KF, X, ie, jf, g0, g1, g2, h0, h1);
        }
        __syncthreads();
      }
    }
    __syncthreads();  // the zeroed block, also where nothing survived
    const int nz = __ballot(any) != 0 && live;
    if (lane == 0 && A.not0) A.not0[A.task_id ? A.task_id[t] : t] = nz;

    // ---- output addressing: canonical axis A holds the original axis
    // (perm >> 2A) & 3; strides of the packed Fortran block ------------------
    int64_t st0, st1, st2, st3, stc;
    {
      const int perm = task_perm(tk);
      const int naxes = three ? 3 : 4;
      int dorig[4] = {1, 1, 1, 1};
      for (int a = 0; a < naxes; ++a) {
        const VShell& v = B.vsh[tk.sh[a]];
        dorig[(perm >> (2 * a)) & 3] = A.sph ? v.dsph : v.dcart;
      }
      const int64_t so[4] = {1, dorig[0], (int64_t)dorig[0] * dorig[1],
                             (int64_t)dorig[0] * dorig[1] * dorig[2]};
      st0 = so[perm & 3];
      st1 = so[(perm >> 2) & 3];
      st2 = so[(perm >> 4) & 3];
      st3 = three ? 0 : so[(perm >> 6) & 3];
      stc = so[3] * dorig[3];
    }
    double* const out = A.out + task_out(tk);
    const int nD = three ? 1 : G.nDo;
    if (!nz) {
      if (A.dm) continue;  // nothing to contract
      Odo<5> o(lane, {G.nAo, G.nBo, G.nCo, nD, G.ncomp});
      const int n = G.ncomp * G.nAo * G.nBo * G.nCo * nD;
      for (int i = lane; i < n; i += GEN_LANES, o.next())
        out[o.d[4] * stc + o.d[0] * st0 + o.d[1] * st1 + o.d[2] * st2 + o.d[3] * st3] = 0.0;
      continue;
    }

    const bool bra_c2s = A.sph && (la > 1 || lb > 1);
    const bool ket_x = !(three && G.nkc == 1);
    double* const H1 = X + G.oH1;
    double* const H2 = bra_c2s ? X + G.oH2 : H1;
    double* const H3 = ket_x ? (bra_c2s ? H1 : X + G.oH2) : H2;
    const int tla = tet_d(la), tlc = tet_d(lc);
    // row of set r at exponents (x, y, z), column f
    auto row = [&](int r, int x, int y, int z) { return G.ox[r] + (cart_all(x, y, z) - tet_d(G.blo[r])) * G.KF; };
    const bool jk = A.jk_j != nullptr || A.jk_k != nullptr;
    const bool digest = A.dm != nullptr && !jk;
    const double fjk = jk ? jk_degeneracy(s0.shell, s1.shell, s2.shell, s3.shell) : 0.0;
    const double fkl = (!three && s2.shell != s3.shell) ? 2.0 : 1.0;
    double gpart[3] = {0.0, 0.0, 0.0};

    for (int bc0 = 0; bc0 < G.nbc; bc0 += G.nbg) {
      const int nb = min(G.nbg, G.nbc - bc0);
      // bra derivative and transfer (a,b| = sum_t w(b,t) [a+t|, H1[bc][a][b][kf]
      {
        Odo<4> o(lane, {G.KF, G.ncb, G.nca, nb});
        const int n = nb * G.nca * G.ncb * G.KF;
        for (int i = lane; i < n; i += GEN_LANES, o.next()) {
          const int kf = o.d[0], b = o.d[1];
          const int ca = code[tla + o.d[2]];
          const int ax = ca & 15, ay = (ca >> 4) & 15, az = (ca >> 8) & 15;
          const int i0 = tbp[b], i1 = tbp[b + 1];
          const double* Xk = X + kf;
          double v = 0.0;
          if (G.nbc == 1) {
            for (int it = i0; it < i1; ++it) {
              const int tt = tb[it];
              v = fma(tbw[it], Xk[row(0, ax + (tt & 15), ay + ((tt >> 4) & 15), az + ((tt >> 8) & 15))], v);
            }
          } else if (G.nbc == 3) {
            // a_p [a-1_p+t| - [2a] [a+1_p+t|; raised set last, lowered first
            const int p = bc0 + o.d[3];
            const int px = p == 0, py = p == 1, pz = p == 2;
            const int ap = p == 0 ? ax : (p == 1 ? ay : az);
            for (int it = i0; it < i1; ++it) {
              const int tt = tb[it];
              const int x = ax + (tt & 15), y = ay + ((tt >> 4) & 15), z = az + ((tt >> 8) & 15);
              double s = -Xk[row(G.nbs - 1, x + px, y + py, z + pz)];
              if (ap > 0) s = fma((double)ap, Xk[row(0, x - px, y - py, z - pz)], s);
              v = fma(tbw[it], s, v);
            }
          } else {
            // D_p D_q (sets: la-2 only for la >= 2)
            const int bc = bc0 + o.d[3];
            const int p = bc >= 6 ? 2 : (bc >= 3 ? 1 : 0), q = bc - 3 * p;
            const int s4 = G.nbs - 1, s2_ = G.nbs - 2;
            const int px = p == 0, py = p == 1, pz = p == 2, qx = q == 0, qy = q == 1, qz = q == 2;
            const int ap = p == 0 ? ax : (p == 1 ? ay : az), aq = q == 0 ? ax : (q == 1 ? ay : az);
            for (int it = i0; it < i1; ++it) {
              const int tt = tb[it];
              const int x = ax + (tt & 15), y = ay + ((tt >> 4) & 15), z = az + ((tt >> 8) & 15);
              double s = Xk[row(s4, x + px + qx, y + py + qy, z + pz + qz)];
              if (p == q) {
                s = fma(-(double)(2 * ap + 1), Xk[row(s2_, x, y, z)], s);
                if (ap > 1)
                  s = fma((double)(ap * (ap - 1)), Xk[row(0, x - 2 * px, y - 2 * py, z - 2 * pz)], s);
              } else {
                if (aq > 0) s = fma(-(double)aq, Xk[row(s2_, x + px - qx, y + py - qy, z + pz - qz)], s);
                if (ap > 0) s = fma(-(double)ap, Xk[row(s2_, x + qx - px, y + qy - py, z + qz - pz)], s);
                if (ap > 0 && aq > 0)
                  s = fma((double)(ap * aq), Xk[row(0, x - px - qx, y - py - qy, z - pz - qz)], s);
              }
              v = fma(tbw[it], s, v);
            }
          }
          H1[i] = v;
        }
      }
      __syncthreads();
      // bra Cartesian -> spherical, H2[bc][ao][bo][kf]
      if (bra_c2s) {
        Odo<4> o(lane, {G.KF, G.nBo, G.nAo, nb});
        const int n = nb * G.nAo * G.nBo * G.KF;
        for (int i = lane; i < n; i += GEN_LANES, o.next()) {
          const double* h = H1 + o.d[3] * G.nH1 + o.d[0];
          const int ra = la * la + o.d[2], rb = lb * lb + o.d[1];
          double v = 0.0;
          for (int ia = c2s_sparse.ptr[ra]; ia < c2s_sparse.ptr[ra + 1]; ++ia) {
            const double* ha = h + c2s_sparse.k[ia] * G.ncb * G.KF;
            double s = 0.0;
            for (int ib = c2s_sparse.ptr[rb]; ib < c2s_sparse.ptr[rb + 1]; ++ib)
              s = fma(c2s_sparse.v[ib], ha[c2s_sparse.k[ib] * G.KF], s);
            v = fma(c2s_sparse.v[ia], s, v);
          }
          H2[i] = v;
        }
        __syncthreads();
      }
      // ket derivative and transfer, H3[bc][kc][ao][bo][c][d]
      const int nab = G.nAo * G.nBo;
      if (ket_x) {
        Odo<5> o(lane, {G.ncd, G.ncc, nab, G.nkc, nb});
        const int n = nb * G.nH3;
        for (int i = lane; i < n; i += GEN_LANES, o.next()) {
          const int cc = code[tlc + o.d[1]];
          const int cx = cc & 15, cy = (cc >> 4) & 15, cz = (cc >> 8) & 15;
          const double* h2 = H2 + (o.d[4] * nab + o.d[2]) * G.KF;
          const int i0 = tkp[o.d[0]], i1 = tkp[o.d[0] + 1];
          double v = 0.0;
          if (G.nkc == 1) {
            const int lo = tet_d(G.klo[0]);
            for (int it = i0; it < i1; ++it) {
              const int tt = tk_[it];
              v = fma(tkw[it], h2[cart_all(cx + (tt & 15), cy + ((tt >> 4) & 15), cz + ((tt >> 8) & 15)) - lo], v);
            }
          } else {
            const int q = o.d[3], up = G.nks - 1;
            const int qx = q == 0, qy = q == 1, qz = q == 2;
            const int cq = q == 0 ? cx : (q == 1 ? cy : cz);
            const int lo0 = tet_d(G.klo[0]), lo1 = tet_d(G.klo[up]);
            for (int it = i0; it < i1; ++it) {
              const int tt = tk_[it];
              const int x = cx + (tt & 15), y = cy + ((tt >> 4) & 15), z = cz + ((tt >> 8) & 15);
              double s = -h2[G.cf[up] + cart_all(x + qx, y + qy, z + qz) - lo1];
              if (cq > 0) s = fma((double)cq, h2[cart_all(x - qx, y - qy, z - qz) - lo0], s);
              v = fma(tkw[it], s, v);
            }
          }
          H3[i] = v;
        }
        __syncthreads();
      }
      // ket Cartesian -> spherical, then the store, the J/K digest (six block
      // updates of jk_degeneracy, device_common.h) or the gradient digest
      {
        const int nc = ket_x ? G.ncc * G.ncd : G.KF;
        const int nk = nb * G.nkc;
        Odo<5> o(lane, {G.nAo, G.nBo, G.nCo, nD, nk});
        const int n = nk * nab * G.nCo * nD;
        for (int i = lane; i < n; i += GEN_LANES, o.next()) {
          const int ao = o.d[0], bo = o.d[1], co = o.d[2], dd = o.d[3];
          const int comp = bc0 * G.nkc + o.d[4];
          const double* h = H3 + ((o.d[4] * G.nAo + ao) * G.nBo + bo) * nc;
          double v;
          if (!A.sph) {
            v = h[co * (three ? 1 : G.ncd) + dd];
          } else {
            const int rc = lc * lc + co, rd = ld * ld + dd;
            v = 0.0;
            for (int ic = c2s_sparse.ptr[rc]; ic < c2s_sparse.ptr[rc + 1]; ++ic) {
              const double* hc = h + c2s_sparse.k[ic] * (three ? 1 : G.ncd);
              double s = 0.0;
              for (int id = c2s_sparse.ptr[rd]; id < c2s_sparse.ptr[rd + 1]; ++id)
                s = fma(c2s_sparse.v[id], hc[c2s_sparse.k[id]], s);
              v = fma(c2s_sparse.v[ic], s, v);
            }
          }
          if (jk) {
            const int64_t N = A.nao;
            const int64_t P = s0.ao + ao, Q = s1.ao + bo, R = s2.ao + co, S = s3.ao + dd;
            const double* D = A.dm;
            const int64_t slot = slot_offset(A);
            if (A.jk_j) {
              atomicAdd(A.jk_j + slot + P * N + Q, 2.0 * fjk * v * D[R * N + S]);
              atomicAdd(A.jk_j + slot + R * N + S, 2.0 * fjk * v * D[P * N + Q]);
            }
            if (A.jk_k) {
              atomicAdd(A.jk_k + slot + P * N + R, fjk * v * D[Q * N + S]);
              atomicAdd(A.jk_k + slot + P * N + S, fjk * v * D[Q * N + R]);
              atomicAdd(A.jk_k + slot + Q * N + R, fjk * v * D[P * N + S]);
              atomicAdd(A.jk_k + slot + Q * N + S, fjk * v * D[P * N + R]);
            }
          } else if (digest) {
            // dE/dA = sum (d/dr i j|kl) [-2 D_ij D_kl + (D_ik D_jl + D_il D_jk)/2],
            // times 2 when k and l are different shells (the list holds k >= l)
            const int64_t N = A.nao;
            const int64_t P = s0.ao + ao, Q = s1.ao + bo, R = s2.ao + co, S = s3.ao + dd;
            const double* D = A.dm;
            const double w = fkl * (-2.0 * D[P * N + Q] * D[R * N + S] +
                                    0.5 * (D[P * N + R] * D[Q * N + S] + D[P * N + S] * D[Q * N + R]));
            if (comp == 0) gpart[0] = fma(v, w, gpart[0]);
            else if (comp == 1) gpart[1] = fma(v, w, gpart[1]);
            else gpart[2] = fma(v, w, gpart[2]);
          } else {
            out[comp * stc + ao * st0 + bo * st1 + co * st2 + dd * st3] = v;
          }
        }
      }
      __syncthreads();
    }
    if (digest) {
      double* gs = A.grad + slot_offset(A);
      const int ref = grad_ref(A, tk);
      for (int c = 0; c < 3; ++c) {
        double g = gpart[c];
        for (int off = 1; off < GEN_LANES; off <<= 1) g += __shfl_xor(g, off);
        if (lane == 0) atomicAdd(gs + 3 * s0.atom + c, g);
        if (lane == 0 && ref >= 0) atomicAdd(gs + 3 * ref + c, -g);
      }
    }
  }
}

hipError_t launch_generic(const BasisView& B, const BucketArgs& A, hipStream_t stream) {
  const int64_t n = A.t1 - A.t0;
  if (n <= 0) return hipSuccess;
  const GenLayout G = gen_layout(A.kind, A.sph, A.la, A.lb, A.lc, A.ld, B.omega);
  if (!gen_fits(G)) return hipErrorInvalidValue;
  if (A.scratch_stride < G.nblk) return hipErrorInvalidValue;
  // several tasks per wave share its tables once the chip is full
  const int64_t per = std::min<int64_t>(8, std::max<int64_t>(1, n / gen_share(G)));
  const dim3 grid((unsigned)((n + per - 1) / per));
  const size_t lds = sizeof(double) * G.lds;
  if (G.in_lds)
    hipLaunchKernelGGL(eri_generic_kernel<true>, grid, dim3(GEN_LANES), lds, stream, B, A, G);
  else
    hipLaunchKernelGGL(eri_generic_kernel<false>, grid, dim3(GEN_LANES), lds, stream, B, A, G);
  return hipGetLastError();
}

}  // namespace mcint
