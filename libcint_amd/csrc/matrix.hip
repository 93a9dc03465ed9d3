// Matrix kernel: any class and kind of a plan, class known at run time, one
// or four waves per contracted quartet.  It serves what has no register kernel
// (second derivatives, three-centre and short-range derivatives, two-centre
// integrals, high auxiliary shells) wherever a plan has laid out its pairs'
// transfer matrices; generic.hip serves the rest.
//
// The walk takes one candidate primitive quartet per lane, compacts the
// survivors, and for a batch of them evaluates all roots (one (quartet, root)
// per lane), all 2D recurrences (one (quartet, direction, root) per lane) and
// the products of their components; components too few for the lanes are
// shared by lanes that take every S-th primitive quartet.  What follows on
// contracted data is linear in the primitive sums X (row sets by column
// sets, gen_layout.h) with coefficients of the two shell pairs alone: the
// derivative rules, both transfers and both spherical transforms of the bra
// are one matrix of its pair, those of the ket another,
//   block = B_bra X B_ket^T,
// two products on the matrix cores, 16 rows of the block at a time.
//
// What bounds it: the walk's latency (root tables, recurrences and barriers
// per batch) where tasks hold hundreds of primitive quartets, the set-up per
// task where they hold one.  Measured against the generic kernel, whose
// passes go term by term and whose tasks have one wave:
//   int2e_ipip1 + int2e_ip1ip2 of 20 shells (168 000 quartets): 25.1 -> 10.7 ms
//   int3c2e_ip1 + int3c2e_ip2 of 186 shells: 5.25 -> 4.83 ms
// Where the generic kernel is the better one: mm_waves (gen_layout.h).
#include <algorithm>

#include "gen_device.h"

namespace mcint {

typedef double v4d __attribute__((ext_vector_type(4)));

// LDS of this wave written by some of its lanes, made visible to the others
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waves per SIMD: one-wave workgroups at three (at two, 186 VGPRs and no
// spills, second derivatives of 20 shells took 16.9 ms instead of 12.6),
// four-wave workgroups at four (11.2 ms, 11.7 at three).
// W waves per task; NRT roots (0: G.nrt, known at run time).
template <int W, int NRT>
__global__ void __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(W == 4 ? 4 : 3)))
eri_matrix_kernel(BasisView B, BucketArgs A, GenLayout G, XferView XV) {
  constexpr int TH = 64 * W;
  extern __shared__ double sm[];
  const int tid = threadIdx.x, ln = tid & 63, wave = tid >> 6;
  const int kind = A.kind;
  const bool three = kind_three(kind);
  const bool noscreen = kind == KIND_2C2E;  // (i|k): no screening (src/cint2c2e.c:57-147)
  const int la = A.la, lb = A.lb, lc = A.lc, ld = three ? 0 : A.ld;
  double* const X = sm;
  double* const sV = sm + G.oV;
  GenPrim* const sp = reinterpret_cast<GenPrim*>(sm + G.oP);
  double* const su = sm + G.ou;
  double* const sw = sm + G.ow;
  const int ncode = tet((G.E > G.F ? G.E : G.F) + 1);
  int2* const sets = reinterpret_cast<int2*>(sm + G.oI);  // put_sets
  int* const rt = reinterpret_cast<int*>(sets + GEN_SETS);  // output functions and component of each block row
  int* const ct = rt + G.nrow;     // ... and column, a | b << 8 | component << 16
  int* const scnt = ct + G.ncol;   // survivors of each wave, twice
  uint16_t* const code = reinterpret_cast<uint16_t*>(scnt + 2 * W);  // exponents of the components
  if (tid == 0) put_sets(G, sets);
  for (int i = tid; i < ncode; i += TH) {
    int l = 0, k = i;
    while (k >= ncart(l)) { k -= ncart(l); ++l; }
    int m = 0;
    while ((m + 1) * (m + 2) / 2 <= k) ++m;
    const int z = k - m * (m + 1) / 2;
    code[i] = (l - m) | ((m - z) << 4) | (z << 8);
  }
  for (int i = tid; i < G.nrow + G.ncol; i += TH) {
    const bool row = i < G.nrow;
    const int k = row ? i : i - G.nrow, n0 = row ? G.nAo : G.nCo;
    const int n1 = row ? G.nBo : (three ? 1 : G.nDo);
    const int q = (int)((unsigned)k / (unsigned)n0), c = (int)((unsigned)q / (unsigned)n1);
    rt[i] = (k - q * n0) | ((q - c * n1) << 8) | (c << 16);
  }

  const double Ecut0 = three ? B.expcutoff_3c : B.expcutoff_4c;
  const double omega = B.omega;
  const bool sr = omega < 0;
  const int nr = G.nr, nrt = NRT ? NRT : G.nrt;
  const int ER = G.E, FR = G.F, F1 = FR + 1, VS = (ER + 1) * F1;
  // recurrence tables: [primitive][direction][e][f][root]
  const int VD = VS * nrt, VP = 3 * VD;
  const double cfac = PI3_2_SQRTPI * common_fac_sp(la) * common_fac_sp(lb) * common_fac_sp(lc) *
                      (three ? 1.0 : common_fac_sp(ld));
  const int nEF = G.nE * G.nF;
  const int te = tet_d(G.e_lo), tf = tet_d(G.f_lo);
  // weights the row sets need: 2a_i, 4a_i^2 (bits 0, 1), 2a_k (bit 2)
  const int wt = (G.nbc > 1 ? 1 : 0) | (G.nbc == 9 ? 2 : 0) | (G.nkc > 1 ? 4 : 0);

  for (int64_t t = A.t0 + blockIdx.x; t < A.t1; t += gridDim.x) {
    const Task tk = A.tasks[t];
    const VShell& s0 = B.vsh[tk.sh[0]];
    const VShell& s1 = B.vsh[tk.sh[1]];
    const VShell& s2 = B.vsh[tk.sh[2]];
    const VShell& s3 = B.vsh[three ? tk.sh[2] : tk.sh[3]];
    __syncthreads();  // the last task's products have read their blocks
    for (int i = tid; i < G.nXz; i += TH) X[i] = 0.0;

    // ---- the walk ---------------------------------------------------------
    const int nij = s0.nprim * s1.nprim;
    const int nkl = three ? s2.nprim : s2.nprim * s3.nprim;
    const int64_t pab = (int64_t)tk.sh[0] * B.nv + tk.sh[1];
    const int64_t pcd = three ? 0 : (int64_t)tk.sh[2] * B.nv + tk.sh[3];
    const PairPrim* __restrict__ pij = B.pp + B.pair_off[pab];
    const PairPrim* __restrict__ pkl = B.pp + (three ? 0 : B.pair_off[pcd]);
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
    // pair emptiness (src/cint2e.c:96-109): a pair's first record has its
    // smallest estimate
    const bool live = (noscreen || pij[0].cce0 - dij_term < Ecut0) && (three || pkl[0].cce0 - dkl_term < Ecut0);
    const int npq = live ? nij * nkl : 0;
    int any = 0;
    // components shared by lanes: this lane's component and its turn
    const int S = G.spread ? (int)((unsigned)TH / (unsigned)nEF) : 1;
    const int mys = G.spread ? (int)((unsigned)tid / (unsigned)nEF) : 0;
    double g0 = 0, g1 = 0, g2 = 0, h0 = 0, h1 = 0;
    // products of one component over the batch's quartets q0, q0 + step, ...,
    // with weights 1, 2a_i, 4a_i^2; the same times 2a_k: those that the row
    // sets need (WT, uniform)
    auto products = [&](int ie, int jf, int q0, int step, int np) {
      const int ec = code[te + ie], fc = code[tf + jf];
      const int vx = ((ec & 15) * F1 + (fc & 15)) * nrt;
      const int vy = VD + (((ec >> 4) & 15) * F1 + ((fc >> 4) & 15)) * nrt;
      const int vz = 2 * VD + (((ec >> 8) & 15) * F1 + ((fc >> 8) & 15)) * nrt;
      auto run = [&](auto WT) {
        constexpr int wt = decltype(WT)::value;
        const double* V = sV + q0 * VP;
#pragma unroll 2
        for (int q = q0; q < np; q += step) {
          double g = 0;
          if constexpr (NRT != 0) {
#pragma unroll
            for (int r = 0; r < NRT; ++r) g = fma(V[vx + r] * V[vy + r], V[vz + r], g);
          } else {
            double x = V[vx], y = V[vy], z = V[vz];
            for (int r = 1; r < nrt; ++r) {
              const double nx = V[vx + r], ny = V[vy + r], nz_ = V[vz + r];
              g = fma(x * y, z, g);
              x = nx;
              y = ny;
              z = nz_;
            }
            g = fma(x * y, z, g);
          }
          g0 += g;
          if constexpr (wt & 1) g1 = fma(g, sp[q].w[0], g1);
          if constexpr (wt & 2) g2 = fma(g, sp[q].w[1], g2);
          if constexpr (wt & 4) {
            const double h = g * sp[q].w[2];
            h0 += h;
            if constexpr (wt & 1) h1 = fma(h, sp[q].w[0], h1);
          }
          V += step * VP;
        }
      };
      switch (wt) {
        case 0: run(std::integral_constant<int, 0>{}); break;
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        case 4: run(std::integral_constant<int, 4>{}); break;
        default: run(std::integral_constant<int, 5>{}); break;
      }
    };
    auto scatter = [&](int ie, int jf) { add_to_sets(sets, G.KF, X, ie, jf, g0, g1, g2, h0, h1); };
    for (int base = 0, odd = 0; base < npq; base += TH, odd ^= W) {
      // one candidate per lane, libcint's tests
      const int p = base + tid;
      bool pass = false;
      if (p < npq) {
        const int kl = (int)((unsigned)p / (unsigned)nij), ij = p - kl * nij;
        const double cce_kl = three ? 0.0 : pkl[kl].cce0 - dkl_term;
        const double cce_ij = noscreen ? -1e300 : pij[ij].cce0 - dij_term;
        const double room = three ? Ecut : Ecut - cce_kl;
        if ((three || !(cce_kl > Ecut)) && !(cce_ij > room)) {
          // beyond the unwidened cutoff the stored exp factor is 0
          pass = noscreen || (cce_ij < Ecut0 && cce_kl < Ecut0);
          if (!sr) {
            any = 1;
          } else if (pass) {
            // tiny erfc tails are dropped: src/g2e.c:4449-4453 (EXPCUTOFF_SR)
            const PairPrim &P = pij[ij], &Q = pkl[kl];
            const double akl = three ? ek[kl] : Q.aij;
            const double a0 = P.aij * akl * rcp_pos(P.aij + akl);
            const double x = P.px - (three ? s2.r[0] : Q.px), y = P.py - (three ? s2.r[1] : Q.py);
            const double z = P.pz - (three ? s2.r[2] : Q.pz);
            const double tx = omega * omega * rcp_pos(omega * omega + a0) * a0 * (x * x + y * y + z * z);
            pass = !(tx > room - cce_ij || tx > 40.0);
            any |= pass;
          }
        }
      }
      const unsigned long long mask = __ballot(pass);
      int nsurv = __popcll(mask);
      int slot = __popcll(mask & ((1ull << ln) - 1));
      if constexpr (W > 1) {
        // counts of these candidates; the next ones go beside them, since a wave
        // may be one barrier ahead of another's reads
        int* const cnt = scnt + odd;
        if (ln == 0) cnt[wave] = nsurv;
        __syncthreads();
        nsurv = 0;
        for (int w = 0; w < W; ++w) {
          if (w < wave) slot += cnt[w];
          nsurv += cnt[w];
        }
      }
      for (int b0 = 0; b0 < nsurv; b0 += G.PB) {
        const int np = min(nsurv - b0, G.PB);
        if (pass && slot >= b0 && slot < b0 + np) {
          const int kl = (int)((unsigned)p / (unsigned)nij);
          const PairPrim P = pij[p - kl * nij];
          double akl, kkl, ak, q[3];
          if (three) {
            akl = ak = ek[kl];
            kkl = ck[kl];
            q[0] = s2.r[0]; q[1] = s2.r[1]; q[2] = s2.r[2];
          } else {
            const PairPrim Q = pkl[kl];
            akl = Q.aij;
            ak = Q.ai;
            kkl = Q.kab;
            q[0] = Q.px; q[1] = Q.py; q[2] = Q.pz;
          }
          GenPrim& w = sp[slot - b0];
          const double a1 = P.aij * akl, a0 = a1 * rcp_pos(P.aij + akl);
          w.aij = P.aij;
          w.akl = akl;
          w.a1 = a1;
          w.a0 = a0;
          const double pq[3] = {P.px - q[0], P.py - q[1], P.pz - q[2]};
          w.pq[0] = pq[0];
          w.pq[1] = pq[1];
          w.pq[2] = pq[2];
          w.pa[0] = P.px - s0.r[0];
          w.pa[1] = P.py - s0.r[1];
          w.pa[2] = P.pz - s0.r[2];
          w.qc[0] = q[0] - s2.r[0];
          w.qc[1] = q[1] - s2.r[1];
          w.qc[2] = q[2] - s2.r[2];
          double fac = sqrt_pos(a0 * rcp_pos(a1 * a1 * a1)) * cfac * P.kab * kkl;
          double x = a0 * (pq[0] * pq[0] + pq[1] * pq[1] + pq[2] * pq[2]), theta = 1.0;
          if (omega != 0) theta = omega * omega * rcp_pos(omega * omega + a0);
          if (omega > 0) {
            x *= theta;
            fac *= sqrt_pos(theta);
          }
          w.x = x;
          w.fac = fac;
          w.theta = theta;
          w.w[0] = 2.0 * P.ai;
          w.w[1] = 4.0 * P.ai * P.ai;
          w.w[2] = 2.0 * ak;
        }
        __syncthreads();
        // roots: short range takes the full rule on nr roots minus the
        // theta-scaled rule on nr more (src/g2e.c:4455-4476; exact for the
        // polynomial integrand, as is the rule on [sqrt(theta), 1])
        for (int it = tid; it < np * nrt; it += TH) {
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
        for (int it = tid; it < np * 3 * nrt; it += TH) {
          const int q = (int)((unsigned)it / (unsigned)(3 * nrt)), dr = it - q * 3 * nrt;
          const int d = dr >= 2 * nrt ? 2 : (dr >= nrt ? 1 : 0), r = dr - d * nrt;
          const GenPrim& P = sp[q];
          const double u2 = P.a0 * su[q * nrt + r];
          const double tmp4 = 0.5 * rcp_pos(u2 * (P.aij + P.akl) + P.a1);
          const double b00 = u2 * tmp4, b10 = b00 + tmp4 * P.akl, b01 = b00 + tmp4 * P.aij;
          const double c00 = P.pa[d] - 2.0 * b00 * P.akl * P.pq[d];
          const double c0p = P.qc[d] + 2.0 * b00 * P.aij * P.pq[d];
          double* V = sV + q * VP + d * VD + r;
          const int se = F1 * nrt;  // step in e; nrt in f
          double v1 = d == 2 ? sw[q * nrt + r] : 1.0, v0 = 0.0;
          V[0] = v1;
          for (int e = 0; e < ER; ++e) {
            const double v = fma(e * b10, v0, c00 * v1);
            V[(e + 1) * se] = v;
            v0 = v1;
            v1 = v;
          }
          for (int f = 0; f < FR; ++f) {
            // the next element is read before this one's result is stored
            double* Vf = V + f * nrt;
            double prev = 0.0, cur = Vf[0], low = f > 0 ? Vf[-nrt] : 0.0;
            const double fb = f * b01;
            for (int e = 0; e <= ER; ++e) {
              double nc = 0.0, nl = 0.0;
              if (e < ER) {
                nc = Vf[se];
                if (f > 0) nl = Vf[se - nrt];
              }
              Vf[nrt] = fma(fb, low, fma(e * b00, prev, c0p * cur));
              prev = cur;
              cur = nc;
              low = nl;
              Vf += se;
            }
          }
        }
        __syncthreads();
        if (G.spread) {
          if (mys < S) {
            const int c = tid - mys * nEF;
            const int ie = (int)((unsigned)c / (unsigned)G.nF);
            products(ie, c - ie * G.nF, mys, S, np);
          }
        } else {
          Odo<2> o(tid, {G.nF, G.nE}, TH);
          for (int c = tid; c < nEF; c += TH, o.next()) {
            g0 = g1 = g2 = h0 = h1 = 0.0;
            products(o.d[1], o.d[0], 0, 1, np);
            scatter(o.d[1], o.d[0]);
          }
        }
        __syncthreads();
      }
    }
    int nz;
    if constexpr (W > 1) nz = __syncthreads_or(any) && live;
    else nz = __ballot(any) != 0 && live;
    if (G.spread) {
      double* const part = sV;
      if (mys < S) {
        part[tid] = g0;
        part[TH + tid] = g1;
        part[2 * TH + tid] = g2;
        part[3 * TH + tid] = h0;
        part[4 * TH + tid] = h1;
      }
      __syncthreads();
      if (tid < nEF) {
        g0 = g1 = g2 = h0 = h1 = 0.0;
        for (int s = 0; s < S; ++s) {
          const double* q = part + s * nEF + tid;
          g0 += q[0];
          g1 += q[TH];
          g2 += q[2 * TH];
          h0 += q[3 * TH];
          h1 += q[4 * TH];
        }
        const int ie = (int)((unsigned)tid / (unsigned)G.nF);
        scatter(ie, tid - ie * G.nF);
      }
    }
    __syncthreads();
    if (tid == 0 && A.not0) A.not0[A.task_id ? A.task_id[t] : t] = nz;

    // ---- output addressing: canonical axis A holds the original axis
    // (perm >> 2A) & 3; strides of the packed Fortran block ------------------
    int64_t st0, st1, st2, st3, stc;
    {
      const int perm = task_perm(tk);
      const int naxes = three ? 3 : 4;
      int64_t so[4] = {1, 1, 1, 1};  // widths of the original axes, then strides
      for (int a = 0; a < naxes; ++a) {
        const VShell& v = B.vsh[tk.sh[a]];
        const int w = A.sph ? v.dsph : v.dcart, o = (perm >> (2 * a)) & 3;
#pragma unroll
        for (int k = 0; k < 4; ++k) so[k] = k == o ? w : so[k];
      }
      stc = so[0] * so[1] * so[2] * so[3];
      const int64_t d1 = so[0], d2 = so[0] * so[1], d3 = d2 * so[2];
      auto stride = [&](int o) { return o == 0 ? (int64_t)1 : (o == 1 ? d1 : (o == 2 ? d2 : d3)); };
      st0 = stride(perm & 3);
      st1 = stride((perm >> 2) & 3);
      st2 = stride((perm >> 4) & 3);
      st3 = three ? 0 : stride((perm >> 6) & 3);
    }
    double* const out = A.out + task_out(tk);
    if (!nz) {
      if (A.dm) continue;  // nothing to contract
      Odo<5> o(tid, {G.nAo, G.nBo, G.nCo, three ? 1 : G.nDo, G.ncomp}, TH);
      const int n = G.ncomp * G.nAo * G.nBo * G.nCo * (three ? 1 : G.nDo);
      for (int i = tid; i < n; i += TH, o.next())
        out[o.d[4] * stc + o.d[0] * st0 + o.d[1] * st1 + o.d[2] * st2 + o.d[3] * st3] = 0.0;
      continue;
    }

    const bool jk = A.jk_j != nullptr || A.jk_k != nullptr;
    const double fjk = jk ? jk_degeneracy(s0.shell, s1.shell, s2.shell, s3.shell) : 0.0;
    const double fkl = (!three && s2.shell != s3.shell) ? 2.0 : 1.0;
    double gpart[3] = {0.0, 0.0, 0.0};
    // J/K digest (six block updates of jk_degeneracy, device_common.h) or
    // gradient digest of one element
    auto contract = [&](int comp, int ao, int bo, int co, int dd, double v) {
      const int64_t N = A.nao;
      const int64_t P = s0.ao + ao, Q = s1.ao + bo, R = s2.ao + co, Sd = s3.ao + dd;
      const double* D = A.dm;
      if (jk) {
        const int64_t slot = slot_offset(A);
        if (A.jk_j) {
          atomicAdd(A.jk_j + slot + P * N + Q, 2.0 * fjk * v * D[R * N + Sd]);
          atomicAdd(A.jk_j + slot + R * N + Sd, 2.0 * fjk * v * D[P * N + Q]);
        }
        if (A.jk_k) {
          atomicAdd(A.jk_k + slot + P * N + R, fjk * v * D[Q * N + Sd]);
          atomicAdd(A.jk_k + slot + P * N + Sd, fjk * v * D[Q * N + R]);
          atomicAdd(A.jk_k + slot + Q * N + R, fjk * v * D[P * N + Sd]);
          atomicAdd(A.jk_k + slot + Q * N + Sd, fjk * v * D[P * N + R]);
        }
        return;
      }
      // dE/dA = sum (d/dr i j|kl) [-2 D_ij D_kl + (D_ik D_jl + D_il D_jk)/2],
      // times 2 when k and l are different shells (the list holds k >= l)
      const double w = fkl * (-2.0 * D[P * N + Q] * D[R * N + Sd] +
                              0.5 * (D[P * N + R] * D[Q * N + Sd] + D[P * N + Sd] * D[Q * N + R]));
      if (comp == 0) gpart[0] = fma(v, w, gpart[0]);
      else if (comp == 1) gpart[1] = fma(v, w, gpart[1]);
      else gpart[2] = fma(v, w, gpart[2]);
    };

    // ---- block = B_bra X B_ket^T.  Operand layout of the 16x16x4 product:
    // lane l holds row (column) l % 16 at k = l / 16; result element j of
    // lane l is row l / 16 + 4 j, column l % 16.
    const double* __restrict__ MB = XV.m + XV.bra[(int64_t)tk.sh[0] * XV.nv + tk.sh[1]] + ln;
    const double* __restrict__ MK = XV.m + XV.ket[(int64_t)tk.sh[2] * XV.nv + tk.sh[three ? 2 : 3]] + ln;
    double* const Y = sm + G.nXz + wave * 16 * G.YS;
    const int l16 = ln & 15, l4 = ln >> 4;
    for (int tr = wave; tr < G.RT; tr += W) {
      const double* Ab = MB + (int64_t)tr * G.KS * 64;
      for (int tc = 0; tc < G.CT1; tc += 2) {
        const int c0 = tc * 16 + l16, c1 = c0 + 16;
        const bool ok0 = c0 < G.KF, ok1 = c1 < G.KF;
        const double* x0 = X + l4 * G.KF + (ok0 ? c0 : 0);
        const double* x1 = X + l4 * G.KF + (ok1 ? c1 : 0);
        v4d acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
        if (tc + 1 < G.CT1) {
#pragma unroll 4
          for (int s = 0; s < G.KS; ++s) {
            const double a = Ab[s * 64], b0 = x0[s * 4 * G.KF], b1 = x1[s * 4 * G.KF];
            acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b0, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, ok1 ? b1 : 0.0, acc1, 0, 0, 0);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) Y[(l4 + 4 * j) * G.YS + c1] = acc1[j];
        } else {
#pragma unroll 4
          for (int s = 0; s < G.KS; ++s) {
            const double a = Ab[s * 64], b0 = x0[s * 4 * G.KF];
            acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, ok0 ? b0 : 0.0, acc0, 0, 0, 0);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) Y[(l4 + 4 * j) * G.YS + c0] = acc0[j];
      }
      wave_sync();
      // this lane's four rows of the tile and their output offsets
      int rc[4];
      int64_t ro[4], ro2[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = tr * 16 + l4 + 4 * j;
        rc[j] = r < G.nrow ? rt[r] : -1;
        ro[j] = ro2[j] = 0;
        if (rc[j] < 0) continue;
        const int64_t o = (rc[j] & 255) * st0 + ((rc[j] >> 8) & 255) * st1;
        const int bc = rc[j] >> 16;
        if (G.nbu == 6) {  // (p, q), p <= q, and its mirror
          const int p = bc < 3 ? 0 : (bc < 5 ? 1 : 2), q = bc < 3 ? bc : (bc < 5 ? bc - 2 : 2);
          ro[j] = o + (3 * p + q) * stc;
          ro2[j] = o + (3 * q + p) * stc;
        } else {
          ro[j] = o + (int64_t)bc * G.nkc * stc;
        }
      }
      for (int tc = 0; tc < G.CT2; ++tc) {
        const double* Bk = MK + tc * G.KS2 * 64;
        const double* y = Y + l16 * G.YS + l4;
        v4d acc = {0, 0, 0, 0};
#pragma unroll 4
        for (int s = 0; s < G.KS2; ++s)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(y[s * 4], Bk[s * 64], acc, 0, 0, 0);
        const int c = tc * 16 + l16;
        if (c >= G.ncol) continue;
        const int cc = ct[c];
        const int co = cc & 255, dd = (cc >> 8) & 255, kc = cc >> 16;
        if (A.dm) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (rc[j] >= 0)
              contract((rc[j] >> 16) * G.nkc + kc, rc[j] & 255, (rc[j] >> 8) & 255, co, dd, acc[j]);
        } else {
          const int64_t o = co * st2 + dd * st3 + kc * stc;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (rc[j] < 0) continue;
            out[ro[j] + o] = acc[j];
            if (G.nbu == 6 && ro2[j] != ro[j]) out[ro2[j] + o] = acc[j];
          }
        }
      }
      wave_sync();  // Y is rewritten
    }
    if (A.dm && !jk) {
      double* gs = A.grad + slot_offset(A);
      const int ref = grad_ref(A, tk);
      for (int c = 0; c < 3; ++c) {
        double g = gpart[c];
        for (int off = 1; off < 64; off <<= 1) g += __shfl_xor(g, off);
        if (ln == 0) atomicAdd(gs + 3 * s0.atom + c, g);
        if (ln == 0 && ref >= 0) atomicAdd(gs + 3 * ref + c, -g);
      }
    }
  }
}

hipError_t launch_matrix(const BasisView& B, const BucketArgs& A, const XferView& XV, int waves,
                         hipStream_t stream) {
  const int64_t n = A.t1 - A.t0;
  if (n <= 0) return hipSuccess;
  const GenLayout G = mm_layout(A.kind, A.sph, A.la, A.lb, A.lc, A.ld, B.omega, waves);
  if (!gen_fits(G) || !G.waves || !XV.m) return hipErrorInvalidValue;
  // several tasks per workgroup share its tables once the chip is full
  const int64_t per = std::min<int64_t>(8, std::max<int64_t>(1, n * waves / gen_share(G)));
  const dim3 grid((unsigned)((n + per - 1) / per));
  const size_t lds = sizeof(double) * G.lds;
  auto go = [&](auto W, auto N) {
    constexpr int w = decltype(W)::value;
    hipLaunchKernelGGL((eri_matrix_kernel<w, decltype(N)::value>), grid, dim3(64 * w), lds, stream, B, A, G, XV);
  };
  auto roots = [&](auto W) {
    switch (G.nrt) {
      case 1: return go(W, std::integral_constant<int, 1>{});
      case 2: return go(W, std::integral_constant<int, 2>{});
      case 3: return go(W, std::integral_constant<int, 3>{});
      case 4: return go(W, std::integral_constant<int, 4>{});
      case 5: return go(W, std::integral_constant<int, 5>{});
      case 6: return go(W, std::integral_constant<int, 6>{});
      default: return go(W, std::integral_constant<int, 0>{});
    }
  };
  if (waves == 4) roots(std::integral_constant<int, 4>{});
  else roots(std::integral_constant<int, 1>{});
  return hipGetLastError();
}

// Row sets of a pair's matrix columns (the sets of gen_layout): first shell,
// position of its first component, component count.
struct PairSets {
  int n, lo[3], pos[3];
};
__device__ __forceinline__ PairSets pair_sets(int kind, bool ket, int l1, int l2) {
  PairSets s{};
  int at = 0;
  auto add = [&](int shift) {
    if (l1 + shift < 0) return;
    s.lo[s.n] = l1 + shift;
    s.pos[s.n++] = at;
    at += tet(l1 + shift + l2 + 1) - tet(l1 + shift);
  };
  const bool one = ket ? kind_ket_der(kind) || kind == KIND_2E_IP1IP2
                       : kind_bra_der(kind) || kind == KIND_2E_IP1IP2;
  if (!ket && kind == KIND_2E_IPIP1) {
    add(-2);
    add(0);
    add(2);
  } else if (one) {
    add(-1);
    add(1);
  } else {
    add(0);
  }
  return s;
}

// One row of a pair's matrix: the output function (ao, bo) and derivative
// component bc of shells la, lb as a sum over the pair's primitive sums:
// spherical transform of both shells, transfer (a,b| = sum_t C(b,t)
// (A-B)^(b-t) [a+t|, and the derivative rules of gen_layout.h.
// add(set, x, y, z, value).
template <typename Add>
__device__ __forceinline__ void xfer_row(int sph, bool one, bool two, int top, int la, int lb, int ao, int bo, int bc,
                                         const double (*binom)[LMAX + 1], const double (*pw)[LMAX + 1], Add&& add) {
  const int p = two ? (bc < 3 ? 0 : (bc < 5 ? 1 : 2)) : bc;
  const int q = two ? (bc < 3 ? bc : (bc < 5 ? bc - 2 : 2)) : 0;
  const int ra = la * la + ao, rb = lb * lb + bo;
  const int ia1 = sph ? c2s_sparse.ptr[ra + 1] : ao + 1, ib1 = sph ? c2s_sparse.ptr[rb + 1] : bo + 1;
  for (int ia = sph ? c2s_sparse.ptr[ra] : ao; ia < ia1; ++ia) {
    const int ka = sph ? c2s_sparse.k[ia] : ia;
    int ma = 0;
    while ((ma + 1) * (ma + 2) / 2 <= ka) ++ma;
    const int az = ka - ma * (ma + 1) / 2, ay = ma - az, ax = la - ma;
    const int px = p == 0, py = p == 1, pz = p == 2, qx = q == 0, qy = q == 1, qz = q == 2;
    const int ap = p == 0 ? ax : (p == 1 ? ay : az), aq = q == 0 ? ax : (q == 1 ? ay : az);
    for (int ib = sph ? c2s_sparse.ptr[rb] : bo; ib < ib1; ++ib) {
      const int kb = sph ? c2s_sparse.k[ib] : ib;
      int mb = 0;
      while ((mb + 1) * (mb + 2) / 2 <= kb) ++mb;
      const int bz = kb - mb * (mb + 1) / 2, by = mb - bz, bx = lb - mb;
      const double cc = sph ? c2s_sparse.v[ia] * c2s_sparse.v[ib] : 1.0;
      for (int tx = 0; tx <= bx; ++tx)
        for (int ty = 0; ty <= by; ++ty)
          for (int tz = 0; tz <= bz; ++tz) {
            const double w = cc * (binom[bx][tx] * binom[by][ty] * binom[bz][tz]) *
                             (pw[0][bx - tx] * pw[1][by - ty] * pw[2][bz - tz]);
            const int x = ax + tx, y = ay + ty, z = az + tz;
            if (!one && !two) {
              add(0, x, y, z, w);
              continue;
            }
            if (one) {
              add(top, x + px, y + py, z + pz, -w);
              if (ap > 0) add(0, x - px, y - py, z - pz, ap * w);
              continue;
            }
            add(top, x + px + qx, y + py + qy, z + pz + qz, w);
            if (p == q) {
              add(top - 1, x, y, z, -(2 * ap + 1) * w);
              if (ap > 1) add(0, x - 2 * px, y - 2 * py, z - 2 * pz, ap * (ap - 1) * w);
            } else {
              if (aq > 0) add(top - 1, x + px - qx, y + py - qy, z + pz - qz, -aq * w);
              if (ap > 0) add(top - 1, x + qx - px, y + qy - py, z + qz - pz, -ap * w);
              if (ap > 0 && aq > 0) add(0, x - px - qx, y - py - qy, z - pz - qz, (double)(ap * aq) * w);
            }
          }
    }
  }
}

// The matrices of a plan's pairs (blockIdx.x), laid out as the 16 x 4 tiles of
// the matrix instruction, lane order, zero padded.  A lane sums one row; a
// workgroup the 2^k rows that fit its LDS, then writes them, and the rows of
// a matrix are spread over gridDim.y workgroups.  What bounds it: a row is a
// chain of hundreds to thousands of small additions.  Made in global memory by
// one workgroup per matrix they took 2.1 ms for 16 (gg| pairs' i-derivatives.
__global__ void __launch_bounds__(64)
xfer_kernel(const VShell* __restrict__ vsh, int kind, int sph, const XferItem* __restrict__ items,
            double* __restrict__ m, int lds) {
  extern __shared__ double acc[];  // lds doubles, [column][row]
  __shared__ double binom[LMAX + 1][LMAX + 1], pw[3][LMAX + 1];
  const int tid = threadIdx.x;
  const XferItem it = items[blockIdx.x];
  const bool ket = it.ket, three = kind_three(kind);
  const VShell &a = vsh[it.a], &b = vsh[it.b];
  const int la = a.l, lb = ket && three ? 0 : b.l;
  if (tid <= LMAX)
    for (int k = 0; k <= tid; ++k) binom[tid][k] = binom_small(tid, k);
  if (tid < 3) {
    double v = 1.0;
    for (int k = 0; k <= lb; ++k) {
      pw[tid][k] = v;
      v *= a.r[tid] - b.r[tid];
    }
  }
  const PairSets S = pair_sets(kind, ket, la, lb);
  const bool two = !ket && kind == KIND_2E_IPIP1;
  const bool one = !two && (ket ? kind_ket_der(kind) || kind == KIND_2E_IP1IP2
                                : kind_bra_der(kind) || kind == KIND_2E_IP1IP2);
  const int nA = sph ? 2 * la + 1 : ncart(la), nB = sph ? 2 * lb + 1 : ncart(lb);
  const int n = nA * nB * (two ? 6 : (one ? 3 : 1));
  const int ncol = it.ks * 4;
  int rw = 64;
  while (rw > 1 && rw * ncol > lds) rw >>= 1;
  double* const M = m + it.off;
  for (int r0 = blockIdx.y * rw; r0 < it.rows * 16; r0 += gridDim.y * rw) {
    for (int i = tid; i < rw * ncol; i += 64) acc[i] = 0.0;
    __syncthreads();
    const int row = r0 + tid;
    if (tid < rw && row < n)
      xfer_row(sph, one, two, S.n - 1, la, lb, row % nA, (row / nA) % nB, row / (nA * nB), binom, pw,
               [&](int r, int x, int y, int z, double v) {
                 acc[(S.pos[r] + cart_all(x, y, z) - tet_d(S.lo[r])) * rw + tid] += v;
               });
    __syncthreads();
    // column k: k step k / 4, lane group k % 4
    for (int i = tid; i < rw * ncol; i += 64) {
      const int k = i / rw, r = r0 + i % rw;
      if (r < it.rows * 16) M[((int64_t)(r >> 4) * it.ks + (k >> 2)) * 64 + (k & 3) * 16 + (r & 15)] = acc[i];
    }
    __syncthreads();
  }
}

hipError_t launch_xfer(const VShell* vsh, int kind, int sph, const XferItem* items, int n, int max_rows, int max_ks,
                       double* m, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const int lds = std::max(4000, 4 * max_ks);
  int rw = 64;  // rows at a time of the largest matrix, as in the kernel
  while (rw > 1 && rw * 4 * max_ks > lds) rw >>= 1;
  const int split = std::min(64, (max_rows * 16 + rw - 1) / rw);
  hipLaunchKernelGGL(xfer_kernel, dim3((unsigned)n, (unsigned)split), dim3(64), sizeof(double) * lds,
                     stream, vsh, kind, sph, items, m, lds);
  return hipGetLastError();
}

}  // namespace mcint
