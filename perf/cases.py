"""The work that users of this package have it do, as cases to be timed.

Each case is one call that a program makes again and again through the
package's public entry points: the J/K build of an SCF iteration (exact, mixed
precision, batched, density fitted, captured in a graph), the digestion of raw
ERI batches, the one-electron matrices, the nuclear gradient, and the energy
and force of a new geometry.  Geometries, densities and orbitals are seeded;
no two seeds give the same inputs.

`exact` evaluates the same quantities in plain torch at 64 bits from the
Hermite-Gaussian (McMurchie-Davidson) expansion, with nothing of this package
but the basis-set data.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "libaccint-public_amd"))

import libaccint as lai  # noqa: E402
from libaccint import _cabi, autograd, systems  # noqa: E402

DEV = "cuda"
THR = 1e-12  # Schwarz threshold of every screened build (the package's default)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest SCF iteration there is: launches and copies
        {"name": "jk_h2o_sto3g", "kind": "fock", "system": "water", "n": 1, "basis": "sto-3g"},
        # a small polyatomic in a triple-zeta basis with f shells, one engine,
        # pointers in HBM as an SCF driver on torch holds them
        {"name": "jk_molecule_ccpvtz", "kind": "jk", "system": "random", "n": 9, "basis": "cc-pvtz"},
        # a small cluster whose iterations replay one captured graph (serving loops, MD)
        {"name": "jk_3water_graph", "kind": "jk_graph", "system": "water", "n": 3, "basis": "cc-pvdz"},
        # an ordinary cluster: the package's headline build
        {"name": "jk_16water_ccpvdz", "kind": "jk", "system": "water", "n": 16, "basis": "cc-pvdz"},
        # the largest: a long chain, sparse bra/ket lists, 1010 functions
        {"name": "jk_c40h82_def2svp", "kind": "jk", "system": "alkane", "n": 40, "basis": "def2-svp"},
        # mixed precision through the host consumer, on a ragged chain length
        {"name": "jk_mixed_c17h36", "kind": "mixed", "system": "alkane", "n": 17, "basis": "def2-svp"},
        # many molecules of unequal sizes in one engine (screening of data sets)
        {"name": "jk_batch_ccpvtz", "kind": "batch", "system": "batch", "n": 7, "basis": "cc-pvtz"},
        # density-fitted iteration, ordinary cluster: fitted tensor in HBM
        {"name": "df_16water_ccpvdz", "kind": "df", "system": "water", "n": 16, "basis": "cc-pvdz"},
        # density-fitted iteration of a small molecule through the host consumer
        {"name": "df_2water_ccpvdz", "kind": "df_host", "system": "water", "n": 2, "basis": "cc-pvdz"},
        # unscreened raw ERI batches digested on the device (the work-unit route)
        {"name": "eri_1water_ccpvdz", "kind": "eri", "system": "water", "n": 1, "basis": "cc-pvdz"},
        # forces of a converged density, the largest gradient
        {"name": "grad_32water_def2svp", "kind": "grad", "system": "water", "n": 32, "basis": "def2-svp"},
        # a geometry step: new engine, lists, energy and backward pass
        {"name": "force_2water_def2svp", "kind": "force", "system": "water", "n": 2, "basis": "def2-svp"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fock", "jk", "jk", "jk_graph", "mixed", "batch", "df", "df_host", "eri", "grad", "force"])
    system, basis = "water", rng.choice(["cc-pvdz", "def2-svp"])
    if kind == "fock":
        n, basis = _log_int(rng, 1, 8), rng.choice(["sto-3g", "cc-pvdz", "def2-svp"])
    elif kind == "jk":
        system = rng.choice(["water", "alkane", "random"])
        if system == "random":
            n, basis = rng.randint(4, 11), rng.choice(["cc-pvtz", "cc-pvdz", "def2-svp"])
        else:
            n = _log_int(rng, 1, 20 if system == "water" else 30)
    elif kind == "jk_graph":
        n = _log_int(rng, 1, 10)
    elif kind == "mixed":
        system, n = "alkane", _log_int(rng, 2, 24)
    elif kind == "batch":
        system, n, basis = "batch", rng.randint(2, 7), rng.choice(["cc-pvtz", "cc-pvdz"])
    elif kind == "df":
        n = _log_int(rng, 3, 18)
    elif kind == "df_host":
        n = _log_int(rng, 1, 6)
    elif kind == "eri":
        system, n = "random", rng.randint(2, 3)
    elif kind == "grad":
        n = _log_int(rng, 1, 28 if basis == "def2-svp" else 14)
    else:
        n = rng.randint(1, 6)
    return {"kind": kind, "system": system, "n": n, "basis": basis}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _waters(n, seed):
    cube = 14.0 * (n / 16.0) ** (1.0 / 3.0) if n > 1 else 1.0
    while True:
        try:
            return systems.water_cluster(n, cube, seed=seed)
        except RuntimeError:
            cube *= 1.1


def _molecules(case, seed):
    """The molecules of a case: one, or the unequal ones of a batch."""
    n, rng = case["n"], np.random.default_rng(seed)
    if case["system"] == "water":
        return [_waters(n, seed)]
    if case["system"] == "alkane":
        # a chain off its ideal geometry by thermal displacements
        return [[(z, tuple(np.asarray(p) + 0.02 * rng.standard_normal(3))) for z, p in systems.alkane(n)]]
    sizes = [n] if case["system"] == "random" else [3 + (5 * k) % 11 for k in range(n)]
    return [_grown(k, rng) for k in sizes]


def _grown(n, rng):
    """n atoms of H, C, N and O (as many of each for every seed) bonded by a
    random walk at 2.0-2.9 bohr."""
    Z = np.random.default_rng(n).choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1])
    at = [np.zeros(3)]
    while len(at) < n:
        step = rng.standard_normal(3)
        p = at[int(rng.integers(len(at)))] + rng.uniform(2.0, 2.9) * step / np.linalg.norm(step)
        if all(np.linalg.norm(p - q) >= 1.8 for q in at):
            at.append(p)
    return [(int(z), tuple(p)) for z, p in zip(Z, at)]


def _density(basis, atoms, seed):
    """D = 2 C C^T of one localised orbital per electron pair: amplitudes fall
    off with the distance from an atom, as occupied orbitals do."""
    rng = np.random.default_rng(seed + 77)
    shells = basis.shells()
    at = np.concatenate([np.tile(_xyz(s), (s.n_functions(), 1)) for s in shells])
    n = len(at)
    n_occ = max(1, min(n, sum(z for z, _ in atoms) // 2))
    home = np.array([p for z, p in atoms for _ in range(z)])[::2][:n_occ]
    home = home + 0.3 * rng.standard_normal(home.shape)
    r = np.linalg.norm(at[:, None, :] - home[None, :, :], axis=2)
    C = rng.standard_normal(r.shape) * np.exp(-r / 2.5)
    C /= np.linalg.norm(C, axis=0)
    D = C @ C.T
    return D + D.T  # exactly symmetric


def _xyz(shell):
    p = shell.center()
    return [p.x, p.y, p.z]


def _options(mixed=False):
    return lai.JKOptions(schwarz_threshold=THR, mixed_precision=True) if mixed else lai.JKOptions(schwarz_threshold=THR)


def prepare(case, seed):
    kind = case["kind"]
    mols = _molecules(case, seed)
    atoms = mols[0]
    bases = [lai.basis_set(case["basis"], m) for m in mols]
    D = [_density(b, m, seed + 1000 * k) for k, (b, m) in enumerate(zip(bases, mols))]
    basis, n = bases[0], bases[0].n_basis_functions()
    s = {"kind": kind, "basis": basis, "D": D[0], "atoms": atoms, "n": n}
    if kind in ("fock", "eri", "mixed"):
        s["engine"] = lai.Engine(basis)
        if kind != "eri":
            s["engine"].prepare_worklist(_options(kind == "mixed"), D[0])
        s["op"] = lai.Operator.coulomb()
        if kind == "eri":  # every shell quartet in every order, as the plain digestion takes them
            s["quartets"] = np.indices((basis.n_shells(),) * 4).reshape(4, -1).T.copy()
        s["builder"] = (lai.MixedPrecisionFockBuilder if kind == "mixed" else lai.GpuFockBuilder)(n)
    elif kind in ("jk", "jk_graph"):
        s["engine"], s["options"] = lai.Engine(basis), _options()
        s["engine"].prepare_worklist(s["options"])
        s["dD"] = torch.from_numpy(D[0]).to(DEV)
        s["dJ"], s["dK"] = torch.zeros_like(s["dD"]), torch.zeros_like(s["dD"])
        if kind == "jk_graph":
            s["stream"] = torch.cuda.Stream()
            torch.cuda.synchronize()
            s["engine"].capture_jk_graph(s["dD"].data_ptr(), s["dJ"].data_ptr(), s["dK"].data_ptr(), s["options"],
                                         s["stream"].cuda_stream)
    elif kind == "batch":
        s["engine"], s["options"], s["bases"] = lai.BatchEngine(bases), _options(), bases
        s["engine"].prepare_worklist(s["options"])
        s["dD"] = torch.from_numpy(np.concatenate([d.ravel() for d in D])).to(DEV)
        s["dJ"], s["dK"] = torch.zeros_like(s["dD"]), torch.zeros_like(s["dD"])
    elif kind in ("df", "df_host"):
        aux = "def2-SVP-RI" if case["basis"] == "def2-svp" else "cc-pVDZ-RI"
        s["builder"] = lai.make_df_fock_builder(basis, [z for z, _ in atoms], [list(p) for _, p in atoms], aux)
        s["builder"].initialize()
        if kind == "df":
            s["dD"] = torch.from_numpy(D[0]).to(DEV)
            s["dJ"], s["dK"] = torch.zeros_like(s["dD"]), torch.zeros_like(s["dD"])
    elif kind == "grad":
        s["engine"] = lai.Engine(basis)
        s["engine"].prepare_worklist(_options())
        s["n_atoms"] = len(atoms)
    else:
        s["name"] = case["basis"]
        s["xyz"] = torch.tensor([p for _, p in atoms], dtype=torch.float64, device=DEV, requires_grad=True)
        s["Z"] = [z for z, _ in atoms]
        s["dD"] = torch.from_numpy(D[0]).to(DEV)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind in ("fock", "mixed"):
        fb = s["builder"]
        fb.reset()
        fb.set_density(s["D"])
        s["engine"].compute_and_consume(s["op"], fb)
        return {"J": fb.get_coulomb_matrix(), "K": fb.get_exchange_matrix()}
    if kind == "eri":
        fb = s["builder"]
        fb.reset()
        fb.set_density(s["D"])
        batch = s["engine"].compute_eri_batch_device(s["quartets"])
        fb.accumulate_device_eri_batch(batch)
        return {"J": fb.get_coulomb_matrix(), "K": fb.get_exchange_matrix()}
    if kind in ("jk", "batch"):
        s["dJ"].zero_()
        s["dK"].zero_()
        s["engine"].build_jk_device(s["dD"].data_ptr(), s["dJ"].data_ptr(), s["dK"].data_ptr(), s["options"],
                                    torch.cuda.current_stream().cuda_stream)
        return {"J": s["dJ"], "K": s["dK"]}
    if kind == "jk_graph":
        st = s["stream"]
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            s["dJ"].zero_()
            s["dK"].zero_()
            s["engine"].launch_jk_graph(st.cuda_stream)
        torch.cuda.current_stream().wait_stream(st)
        return {"J": s["dJ"], "K": s["dK"]}
    if kind == "df":
        # J and K of a symmetric density, as the package's own SCF driver asks for them
        _cabi.check(_cabi.lib().lai_dev_df_jk(s["builder"].device_handle(), s["dD"].data_ptr(), s["dJ"].data_ptr(),
                                              s["dK"].data_ptr(), 1 | 2 | 4, torch.cuda.current_stream().cuda_stream))
        return {"J": s["dJ"], "K": s["dK"]}
    if kind == "df_host":
        s["builder"].set_density(s["D"])
        s["builder"].compute()
        return {"J": s["builder"].coulomb_matrix(), "K": s["builder"].exchange_matrix()}
    if kind == "grad":
        return {"grad": s["engine"].compute_jk_gradient(s["D"], 1.0, s["n_atoms"])}
    s["xyz"].grad = None
    E = autograd.jk_energy(s["xyz"], s["Z"], s["name"], s["dD"])
    E.backward()
    return {"E": E.detach(), "grad": s["xyz"].grad}


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
_work = {}


def _jk_flops(case, thr, grad):
    """Flops of the Rys recursion over the primitive quartets of the screened
    canonical list (and of the derivative recursion), from the list's own
    statistics for one geometry of the case."""
    flops = 0.0
    for m in _molecules(case, 0):
        eng = lai.Engine(lai.basis_set(case["basis"], m))
        eng.prepare_worklist(lai.JKOptions(schwarz_threshold=thr))
        a, b = (torch.zeros(55, dtype=torch.float64) for _ in range(2))
        fn = _cabi.lib().lai_dev_worklist_grad_flops if grad else _cabi.lib().lai_dev_worklist_class_flops
        ptr = lambda t: np.ctypeslib.as_ctypes(t.numpy())  # noqa: E731
        _cabi.check(fn(eng.device_basis_handle(), ptr(a), ptr(b)))
        flops += float(b.sum()) if grad else float(a.sum() + b.sum())
    return flops


def work(case):
    key = (case["kind"], case["system"], case["n"], case["basis"])
    if key not in _work:
        kind = case["kind"]
        mols = _molecules(case, 0)
        nbf = [lai.basis_set(case["basis"], m).n_basis_functions() for m in mols]
        io = 24.0 * sum(n * n for n in nbf)  # D in, J and K out
        if kind in ("df", "df_host"):
            aux = "def2-SVP-RI" if case["basis"] == "def2-svp" else "cc-pVDZ-RI"
            naux = lai.load_auxiliary_basis(aux, [z for z, _ in mols[0]], [list(p) for _, p in mols[0]]).n_functions()
            n, occ = nbf[0], sum(z for z, _ in mols[0]) // 2
            # the fitted tensor once; exchange through the occupied space (2 n^2
            # n_aux n_occ, then half of as much) and the two Coulomb contractions
            io += 8.0 * n * n * naux
            flops = 3.0 * n * n * naux * occ + 4.0 * n * n * naux
        else:
            flops = 0.0 if kind == "grad" else _jk_flops(case, 0.0 if kind == "eri" else THR, False)
            if kind in ("grad", "force"):
                flops += _jk_flops(case, THR, True)
                io = 8.0 * sum(n * n for n in nbf) + 48.0 * len(mols[0])
        _work[key] = {"bytes": io, "flops": flops}
    return _work[key]


def tolerance(case):
    kind = case["kind"]
    if kind == "eri":  # nothing is screened: the order of the sums only
        return {"rel": 2e-13}
    if kind in ("grad", "force"):
        return {"rel": 1e-12}
    # quartets below the Schwarz threshold, the float recursion of the mixed
    # build (1e-12 against the FP64 one), the condition of the fitting metric
    return {"rel": 5e-12}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _cart(L):
    return [(x, y, L - x - y) for x in range(L, -1, -1) for y in range(L - x, -1, -1)]


def _hermite(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


class _Boys(torch.autograd.Function):
    """F_0..F_M(T), with dF_m/dT = -F_{m+1}."""

    @staticmethod
    def forward(ctx, T, M):
        F = _boys(T, M + 1)
        ctx.save_for_backward(F)
        return F[: M + 1]

    @staticmethod
    def backward(ctx, g):
        (F,) = ctx.saved_tensors
        return -(g * F[1:]).sum(0), None


def _boys(T, M):
    small = T < 40.0
    t = torch.where(small, T, torch.zeros_like(T))
    e = torch.exp(-t)
    term = e / (2 * M + 1)
    top = term.clone()
    for k in range(1, 170):
        term = term * (2.0 * t) / (2 * M + 2 * k + 1)
        top += term
    low = [None] * (M + 1)
    low[M] = top
    for m in range(M, 0, -1):
        low[m - 1] = (2.0 * t * low[m] + e) / (2 * m - 1)
    b = torch.where(small, torch.full_like(T, 40.0), T)
    eb = torch.exp(-b)
    high = [0.5 * torch.sqrt(math.pi / b)]
    for m in range(M):
        high.append(((2 * m + 1) * high[m] - eb) / (2.0 * b))
    return torch.stack([torch.where(small, x, y) for x, y in zip(low, high)])


def _expansion(la, lb, p, PA, PB, mu_R2):
    """Hermite coefficients E[i][j][t] of one axis."""
    E = {(0, 0, 0): torch.exp(-mu_R2)}
    get = lambda i, j, t: E.get((i, j, t), 0.0)  # noqa: E731
    for i in range(la + 1):
        for j in range(lb + 1):
            if i == j == 0:
                continue
            for t in range(i + j + 1):
                if i > 0:
                    a, b, X = i - 1, j, PA
                else:
                    a, b, X = i, j - 1, PB
                v = X * get(a, b, t)
                if t > 0:
                    v = v + get(a, b, t - 1) / (2.0 * p)
                if t + 1 <= a + b:
                    v = v + (t + 1) * get(a, b, t + 1)
                E[(i, j, t)] = v
    return E


class _Shells:
    def __init__(self, basis, xyz=None, unit=False):
        self.L, self.f, self.ex, self.co, self.at = [], [], [], [], []
        rows = []
        for s in basis:
            self.L.append(s.angular_momentum())
            self.f.append(s.function_index())
            keep = [k for k, c in enumerate(s.coefficients()) if c != 0.0]
            self.ex.append([s.exponents()[k] for k in keep])
            self.co.append([s.coefficients()[k] for k in keep])
            self.at.append(s.atom_index())
            rows.append(_xyz(s))
        self.xyz = torch.tensor(rows, dtype=torch.float64, device=DEV) if xyz is None else xyz[torch.tensor(self.at, device=DEV)]
        self.n = max(f + (L + 1) * (L + 2) // 2 for f, L in zip(self.f, self.L))


def _norm(c):
    odd = lambda k: math.prod(range(1, 2 * k, 2))  # noqa: E731
    return 1.0 / math.sqrt(odd(c[0]) * odd(c[1]) * odd(c[2]))


def _pair_blocks(S, single=False):
    """Per class of shell pairs: exponents and centres of its primitive pairs,
    which pair each belongs to, their Hermite coefficients [prim, component,
    Hermite function], and the two functions of each (pair, component)."""
    blocks = {}
    for i in range(len(S.L)):
        if single:
            blocks.setdefault((S.L[i], 0), []).append((i, None))
            continue
        for j in range(i + 1):
            a, b = (i, j) if S.L[i] >= S.L[j] else (j, i)
            blocks.setdefault((S.L[a], S.L[b]), []).append((a, b))
    out = []
    for (La, Lb), prs in sorted(blocks.items()):
        ia, ib, al, be, cc, own = [], [], [], [], [], []
        for k, (a, b) in enumerate(prs):
            for x, cx in zip(S.ex[a], S.co[a]):
                for y, cy in zip(*((S.ex[b], S.co[b]) if b is not None else ([0.0], [1.0]))):
                    ia.append(a), ib.append(a if b is None else b), al.append(x), be.append(y), cc.append(cx * cy), own.append(k)
        T = lambda v: torch.tensor(v, dtype=torch.float64, device=DEV)  # noqa: E731
        al, be, cc, own = T(al), T(be), T(cc), torch.tensor(own, device=DEV)
        A, B = S.xyz[torch.tensor(ia, device=DEV)], S.xyz[torch.tensor(ib, device=DEV)]
        p = al + be
        P = (al[:, None] * A + be[:, None] * B) / p[:, None]
        mu = al * be / p
        E = [_expansion(La, Lb, p, P[:, x] - A[:, x], P[:, x] - B[:, x], mu * (A[:, x] - B[:, x]) ** 2) for x in range(3)]
        herm = _hermite(La + Lb)
        comps = [(ca, cb) for ca in _cart(La) for cb in _cart(Lb)]
        zero = torch.zeros_like(p)
        H = torch.stack([torch.stack([
            cc * _norm(ca) * _norm(cb) * E[0].get((ca[0], cb[0], t), zero) * E[1].get((ca[1], cb[1], u), zero)
            * E[2].get((ca[2], cb[2], v), zero) for t, u, v in herm], 1) for ca, cb in comps], 1)
        nb = (Lb + 1) * (Lb + 2) // 2
        fa = torch.tensor([S.f[a] + c // nb for a, b in prs for c in range(len(comps))], device=DEV)
        fb = torch.tensor([-1 if b is None else S.f[b] + c % nb for a, b in prs for c in range(len(comps))], device=DEV)
        out.append({"L": La + Lb, "p": p, "P": P, "own": own, "n": len(prs), "H": H, "fa": fa, "fb": fb})
    return out


def _coulomb_R(L, alpha, X):
    """R_tuv of the Hermite Coulomb integrals, t + u + v <= L, for the
    displacements X[..., 3]."""
    F = _Boys.apply(alpha * (X * X).sum(-1), L)
    level = {}
    s = torch.ones_like(alpha)
    base = []
    for m in range(L + 1):
        base.append(F[m] * s)
        s = s * (-2.0 * alpha)
    level = {(0, 0, 0): base}  # R^(m) for m = 0 .. L - (t + u + v)
    for t, u, v in sorted(_hermite(L), key=sum):
        if t + u + v == 0:
            continue
        ax = 0 if t > 0 else (1 if u > 0 else 2)
        k = [t, u, v]
        k[ax] -= 1
        down = level[tuple(k)]
        q = k[ax]
        k2 = list(k)
        k2[ax] -= 1
        rows = []
        for m in range(L - (t + u + v) + 1):
            r = X[..., ax] * down[m + 1]
            if q > 0:
                r = r + q * level[tuple(k2)][m + 1]
            rows.append(r)
        level[(t, u, v)] = rows
    return {k: v[0] for k, v in level.items()}


def _two_electron(bra, ket, take):
    """take(bra rows, ERIs [bra pair, bra comp, ket pair, ket comp]) over chunks
    of one bra block's pairs against one ket block."""
    hb, hk = _hermite(bra["L"]), _hermite(ket["L"])
    sign = torch.tensor([(-1.0) ** sum(h) for h in hk], dtype=torch.float64, device=DEV)
    Hk = ket["H"] * sign
    nk, ck = len(ket["p"]), ket["H"].shape[1]
    order = torch.argsort(bra["own"], stable=True)
    counts = torch.bincount(bra["own"], minlength=bra["n"]).tolist()
    room = int(3e7 // max(1, nk * (len(_hermite(bra["L"] + ket["L"])) + len(hk)))) + 1
    k = 0
    start = 0
    while k < bra["n"]:
        k1, rows = k, 0
        while k1 < bra["n"] and (k1 == k or rows + counts[k1] <= room):
            rows += counts[k1]
            k1 += 1
        sel = order[start:start + rows]
        p, q = bra["p"][sel][:, None], ket["p"][None, :]
        alpha = p * q / (p + q)
        pre = 2.0 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
        R = _coulomb_R(bra["L"] + ket["L"], alpha, bra["P"][sel][:, None, :] - ket["P"][None, :, :])
        out = torch.zeros((k1 - k, bra["H"].shape[1], ket["n"], ck), dtype=torch.float64, device=DEV)
        for i, h in enumerate(hb):
            G = torch.stack([R[(h[0] + g[0], h[1] + g[1], h[2] + g[2])] for g in hk], 2) * pre[:, :, None]
            V = (G[:, :, None, :] * Hk[None]).sum(3)  # [bra prim, ket prim, ket comp]
            V = torch.zeros((rows, ket["n"], ck), dtype=torch.float64, device=DEV).index_add(1, ket["own"], V)
            W = bra["H"][sel][:, :, i][:, :, None, None] * V[:, None]
            out = out.index_add(0, bra["own"][sel] - k, W)
        take(slice(k, k1), out)
        start += rows
        k = k1


def _eri_tensor(S):
    """(mu nu|la si) of all functions."""
    n = S.n
    T = torch.zeros((n * n, n * n), dtype=torch.float64, device=DEV)
    blocks = _pair_blocks(S)
    for x, bra in enumerate(blocks):
        for ket in blocks[: x + 1]:
            nc = bra["H"].shape[1]

            def take(rows, v):
                at = slice(rows.start * nc, rows.stop * nc)
                fa, fb = bra["fa"][at], bra["fb"][at]
                v = v.reshape(len(fa), -1)
                for r in (fa * n + fb, fb * n + fa):
                    for c in (ket["fa"] * n + ket["fb"], ket["fb"] * n + ket["fa"]):
                        T[r[:, None], c[None, :]] = v
                        T[c[:, None], r[None, :]] = v.T
            _two_electron(bra, ket, take)
    return T.reshape(n, n, n, n)


def _jk_exact(basis, D):
    T = _eri_tensor(_Shells(basis.shells()))
    D = torch.from_numpy(D).to(DEV)
    n = len(D)
    J = (T.reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    K = (T.permute(0, 2, 1, 3).reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    return {"J": J, "K": K}


def _force_exact(atoms, name, D):
    """E = 1/2 tr(DJ) - 1/4 tr(DK) and its gradient by reverse mode, block by block."""
    basis = lai.basis_set(name, atoms)
    xyz = torch.tensor([p for _, p in atoms], dtype=torch.float64, device=DEV, requires_grad=True)
    D = torch.from_numpy(D).to(DEV)
    E = 0.0
    with torch.no_grad():
        n_blocks = len(_pair_blocks(_Shells(basis.shells(), xyz)))
    for x in range(n_blocks):
        for y in range(n_blocks):
            blocks = _pair_blocks(_Shells(basis.shells(), xyz))
            bra, ket = blocks[x], blocks[y]
            nc = bra["H"].shape[1]
            parts = []

            def take(rows, v):
                at = slice(rows.start * nc, rows.stop * nc)
                a, b = bra["fa"][at][:, None], bra["fb"][at][:, None]
                c, d = ket["fa"][None, :], ket["fb"][None, :]
                own = torch.arange(bra["n"], device=DEV).repeat_interleave(nc)[at]
                # each unordered shell pair stands for both orders of its functions
                wb = torch.where(_same(bra, own), 1.0, 2.0)[:, None]
                wk = torch.where(_same(ket, torch.arange(ket["n"], device=DEV).repeat_interleave(ket["H"].shape[1])), 1.0, 2.0)[None, :]
                W = 0.5 * D[a, b] * D[c, d] - 0.125 * (D[a, c] * D[b, d] + D[a, d] * D[b, c])
                e = (wb * wk * W * v.reshape(len(a), -1)).sum()
                e.backward(retain_graph=True)
                parts.append(float(e.detach()))
            _two_electron(bra, ket, take)
            E += math.fsum(parts)
    return {"E": torch.tensor(E, dtype=torch.float64), "grad": xyz.grad}


def _same(block, own):
    """Whether the pair of each row is a shell with itself."""
    nc = block["H"].shape[1]
    fa, fb = block["fa"].reshape(-1, nc)[:, 0], block["fb"].reshape(-1, nc)[:, 0]
    return (fa == fb)[own]


def _df_exact(basis, atoms, aux_name, D):
    n = basis.n_basis_functions()
    aux = lai.load_auxiliary_basis(aux_name, [z for z, _ in atoms], [list(p) for _, p in atoms])
    first, shells = 0, []
    for s in aux.shells():
        shells.append(_AuxShell(s, first))
        first += s.n_functions()
    A, B = _pair_blocks(_Shells(shells), single=True), _pair_blocks(_Shells(basis.shells()))
    V = torch.zeros((first, first), dtype=torch.float64, device=DEV)
    T = torch.zeros((n * n, first), dtype=torch.float64, device=DEV)
    for ket in A:
        for bra, out, rows in [(b, V, (lambda f, g: (f,))) for b in A] + [(b, T, (lambda f, g: (f * n + g, g * n + f))) for b in B]:
            nc = bra["H"].shape[1]

            def take(sl, v):
                at = slice(sl.start * nc, sl.stop * nc)
                f, g = bra["fa"][at], bra["fb"][at]
                for r in rows(f, g):
                    out[r[:, None], ket["fa"][None, :]] = v.reshape(len(f), -1)
            _two_electron(bra, ket, take)
    D = torch.from_numpy(D).to(DEV)
    V = 0.5 * (V + V.T)
    L = torch.linalg.cholesky(V)
    Bt = torch.linalg.solve_triangular(L, T.T.contiguous(), upper=False)  # [P, ab]
    J = (Bt.T @ (Bt @ D.reshape(-1))).reshape(n, n)
    Bp = Bt.reshape(first, n, n)
    K = sum(Bp[q] @ D @ Bp[q].T for q in range(first))
    return {"J": J, "K": K}


class _AuxShell:
    """A fitting shell with its first function."""

    def __init__(self, s, first):
        self._s, self._first = s, first

    def function_index(self):
        return self._first

    def __getattr__(self, name):
        return getattr(self._s, name)


def exact(case, seed):
    kind = case["kind"]
    mols = _molecules(case, seed)
    bases = [lai.basis_set(case["basis"], m) for m in mols]
    D = [_density(b, m, seed + 1000 * k) for k, (b, m) in enumerate(zip(bases, mols))]
    n = max(b.n_basis_functions() for b in bases)
    if kind in ("fock", "eri", "jk", "jk_graph", "mixed", "batch"):
        if n > 80 or len(mols) > 1:
            return None
        return _jk_exact(bases[0], D[0])
    if kind in ("df", "df_host"):
        if n > 160:
            return None
        return _df_exact(bases[0], mols[0], "def2-SVP-RI" if case["basis"] == "def2-svp" else "cc-pVDZ-RI", D[0])
    if n > 50:
        return None
    g = _force_exact(mols[0], case["basis"], D[0])
    return {"grad": g["grad"]} if kind == "grad" else g
