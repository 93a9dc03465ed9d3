"""The work a user of this framework has it do, as timed cases.

Every case goes through the public entry points of ``libcint_amd`` (libcint's
data model, shell lists, device-resident plans, J/K builders, gradient plans)
on molecules cut from the seeded workloads of ``libcint_amd.synthetic`` (their
heavy atoms and hydrogens, displaced by the case's seed) in three bases:

* ``dz``: 3s2p1d on heavy atoms, 2s1p1d on hydrogen, two shells contracted
  over six primitives (the basis of the gradient workload);
* ``tz``: 4s3p2d1f / 3s1p, contractions of 8-10 primitives (the basis of the
  throughput workload); with ``aux`` an even-tempered fitting basis up to g;
* ``gc``: a generally contracted split-valence basis (one 8-primitive s shell
  with two contraction columns per heavy atom).

Kinds of case (``case["kind"]``):

* ``call``   one libcint-style call of one shell quartet, host arrays;
* ``batch``  the drop-in for a loop over such calls: host lists, host blocks;
* ``eri``    a plan over the Schwarz-screened unique quartets, device blocks;
* ``jk``     Coulomb and exchange matrices of one SCF iteration;
* ``grad``   the two-electron nuclear gradient for one density;
* ``energy`` energy and its gradients by autograd, from coordinates (every
  plan is built inside the call, as in a geometry step);
* ``df``     three- and two-centre integrals of density fitting;
* ``dfgrad`` their derivatives on the orbital and on the fitting function;
* ``hess``   second-derivative integrals for a Hessian.
"""
import math

import numpy as np
import torch

import libcint_amd as mc
from libcint_amd import flops
from libcint_amd import jk as mjk
from libcint_amd.synthetic import (ANG_OF, ATOM_OF, ATM_SLOTS, BAS_SLOTS, NCTR_OF, NPRIM_OF, PTR_COEFF,
                                   PTR_COORD, PTR_ENV_START, PTR_EXP, PTR_RANGE_OMEGA, Molecule,
                                   make_molecule, normalized_coefficients, random_density,
                                   screened_quartets, unique_quartets)

SCHWARZ = 1e-12


def listed():
    return [
        # one call of the libcint API, as code ported call by call makes them
        {"name": "call_dpps", "kind": "call", "basis": "dz", "heavy": 2, "hyd": 2, "cls": "dpps"},
        # a caller's loop over quartets turned into one host batch; general contraction
        {"name": "batch_gc", "kind": "batch", "basis": "gc", "heavy": 3, "hyd": 4, "intor": "int2e_sph"},
        # ERIs of a small molecule: many short launches
        {"name": "eri_dz_small", "kind": "eri", "basis": "dz", "heavy": 2, "hyd": 4, "intor": "int2e_sph",
         "omega": 0.0},
        # the throughput workload's basis, f functions and deep contractions
        {"name": "eri_tz", "kind": "eri", "basis": "tz", "heavy": 6, "hyd": 6, "intor": "int2e_sph",
         "omega": 0.0},
        # short-range part of a range-separated functional
        {"name": "eri_tz_erfc", "kind": "eri", "basis": "tz", "heavy": 4, "hyd": 5, "intor": "int2e_sph",
         "omega": -0.3},
        # one SCF iteration of a medium molecule in a double-zeta basis
        {"name": "jk_dz", "kind": "jk", "basis": "dz", "heavy": 8, "hyd": 12, "fp32": 0.0},
        # one SCF iteration in the triple-zeta basis on the mixed-precision tier
        {"name": "jk_tz_mixed", "kind": "jk", "basis": "tz", "heavy": 7, "hyd": 7, "fp32": 1e-7},
        # nuclear gradient of one density
        {"name": "grad_dz", "kind": "grad", "basis": "dz", "heavy": 5, "hyd": 7, "fp32": 0.0},
        # energy, forces and dE/dD through autograd: a geometry step from scratch
        {"name": "energy_dz", "kind": "energy", "basis": "dz", "heavy": 2, "hyd": 3},
        # density fitting: (ij|P) and (P|Q)
        {"name": "df_tz", "kind": "df", "basis": "tz", "heavy": 7, "hyd": 10, "omega": 0.0},
        # density-fitted gradient: derivatives on the orbital and the fitting function
        {"name": "dfgrad_tz", "kind": "dfgrad", "basis": "tz", "heavy": 3, "hyd": 4},
        # second-derivative integrals of a small molecule
        {"name": "hess_dz", "kind": "hess", "basis": "dz", "heavy": 2, "hyd": 2},
    ]


def draw(rng):
    """One more case: the kinds above over their ranges of size, basis and option."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))

    kind = rng.choice(["call", "batch", "eri", "eri", "jk", "jk", "grad", "energy", "df", "dfgrad", "hess"])
    basis = rng.choice(["dz", "tz", "gc"])
    case = {"kind": kind, "basis": basis}
    if kind == "call":
        heavy = log_int(1, 4)
        case["cls"] = "".join(rng.choice("spd") for _ in range(4))
    elif kind == "batch":
        heavy = rng.randint(1, 2 if basis == "tz" else 3)
        case["intor"] = rng.choice(["int2e_sph", "int2e_cart"])
    elif kind == "eri":
        heavy = log_int(1, {"tz": 5, "dz": 7, "gc": 8}[basis])
        case["intor"] = rng.choice(["int2e_sph", "int2e_sph", "int2e_cart"])
        case["omega"] = rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.6), 3)])
        if case["intor"] == "int2e_sph" and heavy <= 4 and rng.random() < 0.3:
            case["omega"] = -round(rng.uniform(0.1, 0.6), 3)
    elif kind == "jk":
        heavy = log_int(1, {"tz": 6, "dz": 8, "gc": 9}[basis])
        case["fp32"] = rng.choice([0.0, 0.0, 1e-7])
    elif kind == "grad":
        case["basis"] = basis = rng.choice(["dz", "gc"])
        heavy = log_int(1, 4)
        case["fp32"] = rng.choice([0.0, 0.0, 1e-7])
    elif kind == "energy":
        case["basis"] = basis = rng.choice(["dz", "gc"])
        heavy = rng.randint(1, 2)
    elif kind == "df":
        case["basis"] = basis = "tz"
        heavy = log_int(1, 7)
        case["omega"] = rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.6), 3), -round(rng.uniform(0.1, 0.6), 3)])
    elif kind == "dfgrad":
        case["basis"] = basis = "tz"
        heavy = rng.randint(1, 3)
    else:
        case["basis"] = basis = rng.choice(["dz", "gc"])
        heavy = rng.randint(1, 2)
    case["heavy"] = heavy
    case["hyd"] = rng.randint(1, heavy + 2)
    return case


# ---- molecules ------------------------------------------------------------

def _gc_shells(rng, heavy):
    """(l, exponents, coefficient columns) of the generally contracted basis."""
    even = [0.16 * 3.4 ** k for k in range(8)]
    if heavy:
        return [(0, even, 1.1 - rng.uniform(0.1, 1.0, (2, 8))), (0, [rng.uniform(0.1, 0.3)], np.ones((1, 1))),
                (1, even[:3], 1.1 - rng.uniform(0.1, 1.0, (1, 3))), (1, [rng.uniform(0.1, 0.3)], np.ones((1, 1))),
                (2, [rng.uniform(0.4, 1.2)], np.ones((1, 1)))]
    return [(0, even[:3], 1.1 - rng.uniform(0.1, 1.0, (1, 3))), (0, [rng.uniform(0.1, 0.3)], np.ones((1, 1))),
            (1, [rng.uniform(0.5, 1.0)], np.ones((1, 1)))]


def _gc_molecule(base):
    """base's atoms with the generally contracted basis."""
    rng = np.random.default_rng(77)
    env, atm, bas = [0.0] * PTR_ENV_START, [], []
    for sym, xyz in zip(base.symbols, base.coords):
        atm.append([int(base.atm[len(atm), 0]), len(env), 1, 0, 0, 0][:ATM_SLOTS])
        env.extend(float(v) for v in xyz)
    for ia, sym in enumerate(base.symbols):
        for l, exps, cols in _gc_shells(rng, sym != "H"):
            pe = len(env)
            env.extend(exps)
            pc = len(env)
            for col in cols:
                env.extend(normalized_coefficients(l, exps, col).tolist())
            bas.append([ia, l, len(exps), len(cols), 0, pe, pc, 0][:BAS_SLOTS])
    return Molecule("gc", np.array(atm, np.int32), np.array(bas, np.int32), np.array(env), list(base.symbols),
                    base.coords.copy())


def molecule(case, seed, displace=0.1):
    """The case's molecule: the first heavy atoms of the workload and hydrogens
    bonded to them, every coordinate displaced by up to 0.1 Bohr by the seed."""
    aux = case["kind"] in ("df", "dfgrad")
    full = make_molecule({"dz": "c3", "tz": "c4" if aux else "c1", "gc": "c1"}[case["basis"]])
    nheavy_full = sum(s != "H" for s in full.symbols)
    bonded = [nheavy_full + k for k in range(full.natm - nheavy_full) if k % nheavy_full < case["heavy"]]
    spare = [nheavy_full + k for k in range(full.natm - nheavy_full) if k % nheavy_full >= case["heavy"]]
    atoms = list(range(case["heavy"])) + (bonded + spare)[:case["hyd"]]
    index = {a: i for i, a in enumerate(atoms)}
    rows = [b for b in full.bas if int(b[ATOM_OF]) in index]
    orbital = [b for i, b in enumerate(full.bas) if int(b[ATOM_OF]) in index and not 0 <= full.aux_start <= i]
    bas = np.array(rows, np.int32)
    bas[:, ATOM_OF] = [index[int(a)] for a in bas[:, ATOM_OF]]
    coords = full.coords[atoms] + np.random.default_rng(seed).uniform(-displace, displace, (len(atoms), 3))
    mol = Molecule(case["basis"], full.atm[atoms].copy(), bas, full.env.copy(), [full.symbols[a] for a in atoms],
                   full.coords[atoms], len(orbital) if aux else -1)
    if case["basis"] == "gc":
        mol = _gc_molecule(mol)
    mol = mol.with_coords(coords)
    mol.env[PTR_RANGE_OMEGA] = case.get("omega", 0.0)
    return mol


def _eri_list(case):
    """Unique quartets of a plan that stores its blocks.  Beyond the smallest
    molecules they are Schwarz-screened, with the bounds of the undisplaced
    molecule, so that the list and the layout of the blocks outlive a move."""
    mol = molecule(case, 0, displace=0.0)
    if mol.nbas <= 40:
        return unique_quartets(mol.nbas)
    db = mc.DeviceBasis(mc.Basis(mol.atm, mol.bas, mol.env))
    quartets, _ = screened_quartets(db.schwarz(), mol.nbas, SCHWARZ)
    db.close()
    return quartets


def _call_shells(mol, cls):
    """A quartet of the wanted angular momenta, on the molecule's last shells of each."""
    out = []
    for i, ch in enumerate(cls):
        l = "spd".index(ch)
        have = [s for s in range(mol.nbas) if int(mol.bas[s, ANG_OF]) == l]
        out.append(have[(5 * i + 1) % len(have)])
    return out


def _tuples(ii, jj, kk):
    """(i, j, k) triples: every listed pair with every k, as rows of four."""
    out = np.zeros((len(ii) * len(kk), 4), np.int32)
    out[:, 0] = np.repeat(ii, len(kk))
    out[:, 1] = np.repeat(jj, len(kk))
    out[:, 2] = np.tile(kk, len(ii))
    return out


def _lists(case, mol):
    """(integral, shell tuples) of the case's plans, without Schwarz screening."""
    kind = case["kind"]
    if kind == "call":
        return [("int2e_sph", np.array([_call_shells(mol, case["cls"])], np.int32))]
    if kind in ("batch", "eri"):
        return [(case["intor"], unique_quartets(mol.nbas))]
    if kind == "jk":
        return [("int2e_sph", unique_quartets(mol.nbas))]
    if kind == "grad":
        return [("int2e_ip1_sph", mjk.gradient_quartets(mol.nbas))]
    if kind == "energy":
        return [("int2e_sph", unique_quartets(mol.nbas)), ("int2e_ip1_sph", mjk.gradient_quartets(mol.nbas))]
    if kind == "hess":
        return [("int2e_ipip1_sph", mjk.gradient_quartets(mol.nbas)),
                ("int2e_ip1ip2_sph", mjk.gradient_quartets(mol.nbas))]
    ns = mol.aux_start
    aux = np.arange(ns, mol.nbas)
    ii, jj = np.tril_indices(ns)
    pp, qq = np.tril_indices(len(aux))
    if kind == "df":
        metric = np.zeros((len(pp), 4), np.int32)
        metric[:, 0], metric[:, 1] = aux[pp], aux[qq]
        return [("int3c2e_sph", _tuples(ii, jj, aux)), ("int2c2e_sph", metric)]
    fi, fj = (a.ravel() for a in np.meshgrid(np.arange(ns), np.arange(ns), indexing="ij"))
    return [("int3c2e_ip1_sph", _tuples(fi, fj, aux)), ("int3c2e_ip2_sph", _tuples(ii, jj, aux))]


# ---- the passes -----------------------------------------------------------

def prepare(case, seed):
    mol = molecule(case, seed)
    basis = mc.Basis(mol.atm, mol.bas, mol.env)
    kind = case["kind"]
    state = {"kind": kind, "mol": mol, "basis": basis}
    if kind == "call":
        state["shells"] = _call_shells(mol, case["cls"])
    elif kind == "batch":
        state["intor"], state["quartets"] = _lists(case, mol)[0]
    elif kind == "energy":
        state["coords"] = torch.tensor(mol.coords, dtype=torch.float64, device="cuda")
        state["dm"] = torch.tensor(random_density(mol.nao_sph(), seed), device="cuda")
    elif kind == "jk":
        db = mc.DeviceBasis(basis)
        quartets, _ = screened_quartets(db.schwarz(), mol.nbas, SCHWARZ)
        db.close()
        dm = random_density(mol.nao_sph(), seed)
        state["builder"] = mjk.JKBuilder(basis, quartets, fp32_threshold=case["fp32"], dmax=float(np.abs(dm).max()))
        state["dm"] = torch.tensor(dm, device="cuda")
    elif kind == "grad":
        dm = random_density(mol.nao_sph(), seed)
        state["plan"] = mjk.GradientPlan(basis, mol.natm, fp32_threshold=case["fp32"], dmax=float(np.abs(dm).max()))
        state["dm"] = torch.tensor(dm, device="cuda")
    else:
        db = mc.DeviceBasis(basis)
        state["db"] = db
        state["stream"] = torch.cuda.Stream()
        state["plans"] = []
        for name, tuples in _lists(case, mol):
            if kind == "eri":
                tuples = _eri_list(case)
            plan = mc.Plan(db, name, tuples)
            out = torch.empty(plan.out_size, dtype=torch.float64, device="cuda")
            state["plans"].append((plan, out))
    return state


def run(state):
    kind = state["kind"]
    if kind == "call":
        return list(mc.intor("int2e_sph", state["shells"], state["basis"]))
    if kind == "batch":
        out, _, not0 = mc.batch(state["intor"], state["quartets"], state["basis"])
        return [out, not0]
    if kind == "jk":
        return list(state["builder"].run(state["dm"]))
    if kind == "grad":
        return [state["plan"].run(state["dm"])]
    if kind == "energy":
        coords = state["coords"].clone().requires_grad_(True)
        dm = state["dm"].clone().requires_grad_(True)
        e = mjk.TwoElectronEnergy.apply(coords, dm, state["mol"])
        e.backward()
        return [e, coords.grad, dm.grad]
    for plan, out in state["plans"]:
        plan.execute(out.data_ptr(), stream_ptr=state["stream"].cuda_stream)
    return [out for _, out in state["plans"]]


# ---- the work a pass cannot do without --------------------------------------

def _pair_estimates(mol, raise_l=0):
    """{(li, lj): (exponent estimates of every primitive pair, shell pairs)} over
    the unordered orbital pairs: libcint's screening measure of a pair."""
    n = mol.aux_start if mol.aux_start >= 0 else mol.nbas
    out = {}
    for i in range(n):
        for j in range(i + 1):
            a, b = mol.bas[i], mol.bas[j]
            ea = mol.env[a[PTR_EXP]:a[PTR_EXP] + a[NPRIM_OF]]
            eb = mol.env[b[PTR_EXP]:b[PTR_EXP] + b[NPRIM_OF]]
            d2 = float(((mol.coords[a[ATOM_OF]] - mol.coords[b[ATOM_OF]]) ** 2).sum())
            key = tuple(sorted((int(a[ANG_OF]), int(b[ANG_OF])), reverse=True))
            est = (d2 * np.outer(ea, eb) / np.add.outer(ea, eb)).ravel()
            out.setdefault(key, [[], 0, 0])
            out[key][0].append(np.tile(est, int(a[NCTR_OF] * b[NCTR_OF])))
            out[key][1] += int(a[NCTR_OF] * b[NCTR_OF])
    return {k: (np.sort(np.concatenate(v[0])), v[1]) for k, v in out.items()}


def work(case):
    mol = molecule(case, 0)
    kind = case["kind"]
    cut = 60.0  # exponents beyond which libcint neglects a primitive quartet
    total = 0.0
    if kind == "call":
        sh = _call_shells(mol, case["cls"])
        nprim = int(np.prod([mol.bas[s, NPRIM_OF] for s in sh]))
        ls = [int(mol.bas[s, ANG_OF]) for s in sh]
        total = flops.bucket_flops(ls, nprim, 1)
        return {"bytes": 8.0 * float(np.prod([2 * l + 1 for l in ls])), "flops": float(total)}
    pairs = _pair_estimates(mol)
    nbytes = 8.0 * sum(_out_size(name, t, mol) for name, t in _lists(case, mol))
    if kind in ("jk", "grad", "energy"):
        nao = mol.nao_sph()
        nbytes = 8.0 * (3 if kind == "jk" else 2) * nao * nao
    if kind in ("df", "dfgrad"):
        naux = sum(int(b[NPRIM_OF]) for b in mol.bas[mol.aux_start:])
        for (la, lb), (est, npair) in pairs.items():
            nprim = int((est < cut).sum())
            for lc in range(5):
                aux = sum(1 for b in mol.bas[mol.aux_start:] if int(b[ANG_OF]) == lc)
                if kind == "df":
                    total += flops.bucket_flops((la, lb, lc, 0), nprim * aux, npair * aux)
                else:
                    total += 3 * flops.bucket_flops((la + 1, lb, lc, 0), nprim * aux, npair * aux)
        return {"bytes": nbytes, "flops": float(total + 500.0 * naux * naux)}
    keys = sorted(pairs)
    for x, p in enumerate(keys):
        for q in keys[:x + 1]:
            (ep, np_), (eq, nq) = pairs[p], pairs[q]
            prims = float(np.searchsorted(eq, cut - ep).sum())
            quart = float(np_ * nq)
            if p == q:
                prims, quart = prims / 2, quart / 2
            cls = p + q
            plain = flops.prim_flops(*cls) * prims + flops.c2s_flops(*cls) * quart
            # derivatives on three of the four centres; nine components of
            # each second-derivative kind
            up = (p[0] + 1, p[1]) + q
            total += {"grad": 9.0 * flops.prim_flops(*up) * prims / 3,
                      "energy": plain + 3.0 * flops.prim_flops(*up) * prims,
                      "hess": 18.0 * flops.prim_flops(*up) * prims}.get(kind, plain)
    return {"bytes": nbytes, "flops": total}


def _out_size(name, tuples, mol):
    return int(mc.Basis(mol.atm, mol.bas, mol.env).block_sizes(name, tuples).sum())


# ---- 64-bit values by plain torch -------------------------------------------
#
# McMurchie-Davidson: the Cartesian product of two Gaussians expanded in
# Hermite Gaussians, (ab|cd) = sum E_ab E_cd R, vectorised over the quartets of
# one class and over their primitive pairs.

_EXACT_PRIMS = 1e8  # primitive quartets that take well under 20 seconds


def _cart(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _sph(l):
    """Real solid harmonics over the Cartesian components: [2l+1, ncart]."""
    if l == 0:
        return np.array([[math.sqrt(1 / (4 * math.pi))]])
    if l == 1:
        return np.eye(3) * math.sqrt(3 / (4 * math.pi))
    comps = _cart(l)
    f, c = math.factorial, math.comb
    out = np.zeros((2 * l + 1, len(comps)))
    for m in range(-l, l + 1):
        am = abs(m)
        norm = math.sqrt((2 * l + 1) / (4 * math.pi) * f(l - am) / f(l + am)) * (math.sqrt(2) if m else 1)
        for k in range((l - am) // 2 + 1):
            ck = (-1) ** k * 2.0 ** -l * c(l, k) * c(2 * l - 2 * k, l) * f(l - 2 * k) / f(l - 2 * k - am)
            # z^(l-2k-|m|) (x^2+y^2+z^2)^k times Re or Im of (x+iy)^|m|
            for a in range(k + 1):
                for b in range(k - a + 1):
                    r2 = c(k, a) * c(k - a, b)
                    for t in range(am + 1):
                        if (t % 2 == 0) != (m >= 0):
                            continue
                        sign = (-1) ** (t // 2) if m >= 0 else (-1) ** ((t - 1) // 2)
                        e = (am - t + 2 * a, t + 2 * b, l - 2 * k - am + 2 * (k - a - b))
                        out[m + l, comps.index(e)] += norm * ck * r2 * sign * c(am, t)
    return out


def _cart_fac(l):
    """libcint's Cartesian functions carry the angular factor of s and p only."""
    return np.eye((l + 1) * (l + 2) // 2) * {0: math.sqrt(1 / (4 * math.pi)),
                                             1: math.sqrt(3 / (4 * math.pi))}.get(l, 1.0)


def _boys(nmax, x):
    """F_0..F_nmax of a tensor x >= 0."""
    big = x > 40.0
    xs = torch.where(big, torch.zeros_like(x), x)
    ex = torch.exp(-xs)
    term = torch.full_like(xs, 1.0 / (2 * nmax + 1))
    s = term.clone()
    for i in range(1, 140):
        term = term * (2 * xs) / (2 * nmax + 2 * i + 1)
        s += term
    down = [None] * (nmax + 1)
    down[nmax] = ex * s
    for n in range(nmax, 0, -1):
        down[n - 1] = (2 * xs * down[n] + ex) / (2 * n - 1)
    xb = torch.where(big, x, torch.full_like(x, 41.0))
    exb = torch.exp(-xb)
    up = [0.5 * torch.sqrt(math.pi / xb) * torch.erf(torch.sqrt(xb))]
    for n in range(nmax):
        up.append(((2 * n + 1) * up[n] - exb) / (2 * xb))
    return [torch.where(big, u, d) for u, d in zip(up, down)]


def _hermites(l):
    return [(t, u, v) for n in range(l + 1) for t in range(n + 1) for u in range(n - t + 1) for v in [n - t - u]]


def _pair_data(mol, i, j, sph, dev):
    """Of one shell pair: centres [p,3], exponents [p], Hermite expansions
    [p, functions of i, functions of j, hermites], contraction columns folded in.
    j < 0: the constant function."""
    a = mol.bas[i]
    la, A = int(a[ANG_OF]), mol.coords[a[ATOM_OF]]
    ea = mol.env[a[PTR_EXP]:a[PTR_EXP] + a[NPRIM_OF]]
    ca = mol.env[a[PTR_COEFF]:a[PTR_COEFF] + a[NPRIM_OF] * a[NCTR_OF]].reshape(a[NCTR_OF], -1)
    if j < 0:
        lb, B, eb, cb, tb = 0, A, np.zeros(1), np.ones((1, 1)), np.ones((1, 1))
    else:
        b = mol.bas[j]
        lb, B = int(b[ANG_OF]), mol.coords[b[ATOM_OF]]
        eb = mol.env[b[PTR_EXP]:b[PTR_EXP] + b[NPRIM_OF]]
        cb = mol.env[b[PTR_COEFF]:b[PTR_COEFF] + b[NPRIM_OF] * b[NCTR_OF]].reshape(b[NCTR_OF], -1)
        tb = _sph(lb) if sph else _cart_fac(lb)
    ta = _sph(la) if sph else _cart_fac(la)
    p = np.add.outer(ea, eb).ravel()
    mu = (np.multiply.outer(ea, eb)).ravel() / p
    P = (np.repeat(ea, len(eb))[:, None] * A + np.tile(eb, len(ea))[:, None] * B) / p[:, None]
    E = np.zeros((3, len(p), la + 1, lb + 1, la + lb + 1))
    for d in range(3):
        pa, pb = P[:, d] - A[d], P[:, d] - B[d]
        e = E[d]
        e[:, 0, 0, 0] = np.exp(-mu * (A[d] - B[d]) ** 2)
        for x in range(la + 1):
            for y in range(lb + 1):
                if x == y == 0:
                    continue
                src, sh = (e[:, x - 1, y], pa) if x else (e[:, x, y - 1], pb)
                for t in range(x + y + 1):
                    v = sh * src[:, t]
                    if t:
                        v = v + src[:, t - 1] / (2 * p)
                    if t + 1 <= la + lb:
                        v = v + (t + 1) * src[:, t + 1]
                    e[:, x, y, t] = v
    herm = _hermites(la + lb)
    H = np.zeros((len(p), len(_cart(la)), len(_cart(lb)), len(herm)))
    for m, (ax, ay, az) in enumerate(_cart(la)):
        for n, (bx, by, bz) in enumerate(_cart(lb)):
            for h, (t, u, v) in enumerate(herm):
                if t <= ax + bx and u <= ay + by and v <= az + bz:
                    H[:, m, n, h] = E[0][:, ax, bx, t] * E[1][:, ay, by, u] * E[2][:, az, bz, v]
    H = np.einsum("pmnh,am,bn->pabh", H, ta, tb)
    cc = np.einsum("ap,bq->pqab", ca, cb).reshape(len(p), len(ca), len(cb))
    H = np.einsum("pabh,pxy->pxaybh", H, cc).reshape(len(p), len(ca) * ta.shape[0], len(cb) * tb.shape[0], -1)
    return tuple(torch.tensor(v, device=dev) for v in (P, p, H.reshape(len(p), -1, len(herm))))


def _exact_blocks(mol, tuples, sph, axes):
    """Packed Fortran blocks of plain integrals over 4 (ij|kl), 3 (ij|k) or 2 (i|k) shells."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    omega = float(mol.env[PTR_RANGE_OMEGA])
    dims = ((2 * mol.bas[:, ANG_OF] + 1) if sph else (mol.bas[:, ANG_OF] + 1) * (mol.bas[:, ANG_OF] + 2) // 2)
    dims = (dims * mol.bas[:, NCTR_OF]).astype(np.int64)
    bra = [(int(t[0]), int(t[1]) if axes > 2 else -1) for t in tuples]
    ket = [(int(t[2] if axes > 2 else t[1]), int(t[3]) if axes == 4 else -1) for t in tuples]

    def size(pr):
        return int(dims[pr[0]] * (dims[pr[1]] if pr[1] >= 0 else 1))

    def sig(pr):
        b = mol.bas
        return (int(b[pr[0], ANG_OF]), int(b[pr[0], NPRIM_OF]), int(b[pr[0], NCTR_OF])) + (
            (int(b[pr[1], ANG_OF]), int(b[pr[1], NPRIM_OF]), int(b[pr[1], NCTR_OF])) if pr[1] >= 0 else (0, 1, 0))

    off = np.concatenate([[0], np.cumsum([size(p) * size(q) for p, q in zip(bra, ket)])]).astype(np.int64)
    out = torch.zeros(int(off[-1]), dtype=torch.float64, device=dev)
    slot, data, groups = {}, {}, {}  # pair -> row of its signature's stacked data
    for p in sorted(set(bra) | set(ket)):
        rows = data.setdefault(sig(p), [])
        slot[p] = len(rows)
        rows.append(_pair_data(mol, p[0], p[1], sph, dev))
    data = {s: tuple(torch.stack(v) for v in zip(*rows)) for s, rows in data.items()}
    for n, (p, q) in enumerate(zip(bra, ket)):
        groups.setdefault((sig(p), sig(q)), []).append(n)
    for (sp, sq), members in groups.items():
        lb, lk = sp[0] + sp[3], sq[0] + sq[3]
        hb, hk = _hermites(lb), _hermites(lk)
        npq = sp[1] * sp[4] * sq[1] * sq[4]
        step = max(1, int(3e7 / (npq * (len(hb) * len(hk) + 12 * (lb + lk + 1) ** 2))))
        for n0 in range(0, len(members), step):
            part = members[n0:n0 + step]
            P, ep, Hp = (v[torch.tensor([slot[bra[n]] for n in part], device=dev)] for v in data[sp])
            Q, eq, Hq = (v[torch.tensor([slot[ket[n]] for n in part], device=dev)] for v in data[sq])
            R = (P[:, :, None, :] - Q[:, None, :, :])
            x2 = (R * R).sum(-1)
            pq = ep[:, :, None] * eq[:, None, :]
            rho = pq / (ep[:, :, None] + eq[:, None, :])
            pref = 2 * math.pi ** 2.5 / (pq * torch.sqrt(ep[:, :, None] + eq[:, None, :]))

            def tables(alpha, fac):
                F = _boys(lb + lk, alpha * x2)
                r = {}

                def get(t, u, v, n):
                    key = (t, u, v, n)
                    if min(t, u, v) < 0:
                        return None
                    if key not in r:
                        if t == u == v == 0:
                            r[key] = (-2 * alpha) ** n * F[n]
                        else:
                            d = 0 if t else 1 if u else 2
                            low = [t, u, v]
                            low[d] -= 1
                            val = R[..., d] * get(*low, n + 1)
                            if low[d] > 0:
                                lower = list(low)
                                lower[d] -= 1
                                val = val + low[d] * get(*lower, n + 1)
                            r[key] = val
                    return r[key]

                return lambda t, u, v: fac * get(t, u, v, 0)

            fulls = []
            if omega <= 0:
                fulls.append((1.0, tables(rho, pref)))
            if omega != 0:
                th = omega ** 2 / (omega ** 2 + rho)
                fulls.append((1.0 if omega > 0 else -1.0, tables(rho * th, pref * torch.sqrt(th))))
            acc = None
            for sign, get in fulls:
                M = torch.stack([torch.stack([(-1.0) ** sum(k) * get(*(a + c for a, c in zip(b, k))) for k in hk], -1)
                                 for b in hb], -2)  # [n, p, q, hb, hk]
                T = torch.einsum("npqbk,nqck->npbc", M, Hq)
                val = sign * torch.einsum("npbc,npab->nac", T, Hp)
                acc = val if acc is None else acc + val
            di, dk = int(dims[bra[part[0]][0]]), int(dims[ket[part[0]][0]])
            blk = acc.reshape(len(part), di, acc.shape[1] // di, dk, acc.shape[2] // dk).permute(0, 4, 3, 2, 1)
            blk = blk.reshape(len(part), -1)
            to = torch.tensor(off[part], device=dev)[:, None] + torch.arange(blk.shape[1], device=dev)
            out[to] = blk
    return out


def exact(case, seed):
    """Plain integrals by the Hermite expansion; derivatives and the larger cases have no value here."""
    if case["kind"] not in ("call", "batch", "df", "eri"):
        return None
    mol = molecule(case, seed)
    if case["kind"] == "eri" and mol.nbas > 40:  # its list follows the framework's Schwarz bounds
        return None
    lists = _lists(case, mol)
    for name, t in lists:
        slots, _ = mc.intor_shape(name)
        prims = np.prod([mol.bas[t[:, s], NPRIM_OF].astype(np.float64) for s in slots], axis=0)
        if prims.sum() > _EXACT_PRIMS or len(t) > 100000:
            return None
    vals = [_exact_blocks(mol, t, name.endswith("sph"), len(mc.intor_shape(name)[0])) for name, t in lists]
    if case["kind"] == "call":
        shape = [int((2 * mol.bas[s, ANG_OF] + 1) * mol.bas[s, NCTR_OF]) for s in lists[0][1][0]]
        return [vals[0].cpu().numpy().reshape(shape, order="F"), None]
    if case["kind"] == "batch":
        return [vals[0].cpu().numpy(), None]
    return vals
