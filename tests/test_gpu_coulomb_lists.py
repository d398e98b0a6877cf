"""The Coulomb accumulators in list order (blocks of the shell pairs in the
order of the worklist, added whole cache lines at a time) against the oracle,
at the sizes where the list arithmetic can go wrong: one pair; ket runs just
below, at and above the 2048 quartets that are sorted at a time (in one chunk
where the chunk cap is raised, else in chunks of equal length); (ss| kets,
whose elements are summed by run position, beside kets of 3 to 10 Coulomb
elements, which go through the wavefront tiles; runs shortened by the density
screen; molecules of different sizes in one list.  Bar: 1e-10 relative, the J/K
bar of test_gpu_parity.py (FP64 sums in another order)."""
import numpy as np
import pytest

import oracle
from libaccint import systems
import libaccint as lai

pytestmark = pytest.mark.gpu
TOL = 1e-10


def rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def hydrogens(n):
    """n H atoms on a jittered cubic grid of 2.2 bohr: n s shells, n (n + 1) / 2
    (ss| pairs, few of them negligible."""
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    jit = np.random.default_rng(n).uniform(-0.2, 0.2, (n, 3))
    grid = [(x, y, z) for x in range(m) for y in range(m) for z in range(m)][:n]
    return [(1, tuple(2.2 * np.array(g) + j)) for g, j in zip(grid, jit)]


def case(name):
    if name.startswith("h"):
        return "sto-3g", hydrogens(int(name[1:]))
    if name == "water_tz":
        return "cc-pvtz", systems.h2o_sto3g_geometry()
    return name, systems.water_cluster(2, 8.0, seed=3)


@pytest.mark.parametrize("name", ["h1", "h2", "h63", "h64", "h91", "sto-3g", "def2-svp", "water_tz"])
@pytest.mark.parametrize("weighted", [False, True])
def test_jk_matches_oracle(name, weighted):
    print("coulomb lists", name, weighted, flush=True)
    basis_name, atoms = case(name)
    basis = lai.basis_set(basis_name, atoms)
    n = basis.n_basis_functions()
    D = systems.density(n, max(1, n // 4), 7, 1.0 / np.sqrt(n))
    J, K = lai.Engine(basis).build_jk(D, lai.JKOptions(schwarz_threshold=1e-12, density_weighted=weighted))
    Jo, Ko = oracle.Oracle(oracle.RawBasis(basis_name, atoms)).jk_canonical(D)
    assert rel(J, Jo) < TOL and rel(K, Ko) < TOL


def test_batch_of_unequal_molecules():
    mols = [("sto-3g", hydrogens(64)), ("cc-pvdz", systems.h2o_sto3g_geometry()), ("sto-3g", hydrogens(1)),
            ("def2-svp", systems.random_molecule(np.random.default_rng(3), 5, 5))]
    bases = [lai.basis_set(b, a) for b, a in mols]
    be = lai.BatchEngine(bases)
    off = be.matrix_offsets()
    Ds = [systems.density(b.n_basis_functions(), 1, 3 + k, 0.3) for k, b in enumerate(bases)]
    J, K = be.build_jk(np.concatenate([d.ravel() for d in Ds]), lai.JKOptions(schwarz_threshold=1e-12))
    for k, (b, a) in enumerate(mols):
        Jo, Ko = oracle.Oracle(oracle.RawBasis(b, a)).jk_canonical(Ds[k])
        sl = slice(off[k], off[k + 1])
        assert rel(J[sl].reshape(Jo.shape), Jo) < TOL and rel(K[sl].reshape(Ko.shape), Ko) < TOL


def contracted(n, n_prim, seed):
    """n atoms, each with one s and one p shell of n_prim primitives."""
    rng = np.random.default_rng(seed)
    ex = list(0.15 * 2.1 ** np.arange(n_prim))
    at = rng.uniform(0.0, 3.0 * n ** (1.0 / 3.0), (n, 3))
    return [(l, tuple(p), ex, list(rng.uniform(0.2, 1.0, n_prim))) for p in at for l in (0, 1)]


@pytest.mark.parametrize("n_atoms, n_prim", [(1, 1), (1, 2), (2, 5), (3, 10), (1, 13), (9, 4)])
def test_divided_kets_match_oracle(n_atoms, n_prim):
    """Few quartets of long contractions: a quartet's ket primitives are divided
    over lanes (n_prim^2 pairs a ket: 1 to 169, so one part, several, more than
    the 127 a quartet may have), in J, K and the gradient."""
    print("divided kets", n_atoms, n_prim, flush=True)
    sh = contracted(n_atoms, n_prim, 5)
    basis = lai.BasisSet([lai.Shell(l, list(p), e, c) for l, p, e, c in sh])
    n = basis.n_basis_functions()
    D = systems.density(n, 2, 11, 1.0 / np.sqrt(n))
    raw = oracle.RawBasis.__new__(oracle.RawBasis)
    raw.L = np.array([s[0] for s in sh], dtype=np.int32)
    raw.centers = np.array([s[1] for s in sh])
    raw.nprim = np.array([n_prim] * len(sh), dtype=np.int32)
    raw.exps = np.concatenate([s[2] for s in sh])
    raw.raw_coefs = np.concatenate([s[3] for s in sh])
    raw.nbf, raw.n_shells = n, len(sh)
    opts = lai.JKOptions(schwarz_threshold=0.0)
    e = lai.Engine(basis)
    J, K = e.build_jk(D, opts)
    Jo, Ko = oracle.Oracle(raw).jk_canonical(D)
    assert rel(J, Jo) < TOL and rel(K, Ko) < TOL
    # dE/dx of the first shell against fourth-order central differences of the
    # same energy: with h = 1e-4 and exponents up to 0.15 * 2.1^12 = 1100 the
    # truncation h^4/30 E^(5) ~ h^4/30 |g| (2 * 1100)^2 is below 1e-9 (second
    # order leaves h^2/6 |g| 2200 ~ 1e-4), rounding 1e-15 |E| / h below 1e-10
    g = e.compute_jk_gradient(D, 1.0, len(sh))

    def energy(dx):
        moved = [(l, (p[0] + (dx if k == 0 else 0.0), p[1], p[2]), x, c) for k, (l, p, x, c) in enumerate(sh)]
        J, K = lai.Engine(lai.BasisSet([lai.Shell(l, list(p), x, c) for l, p, x, c in moved])).build_jk(D, opts)
        return 0.5 * np.sum(D * J) - 0.25 * np.sum(D * K)
    fd = (8.0 * (energy(1e-4) - energy(-1e-4)) - (energy(2e-4) - energy(-2e-4))) / 12e-4
    assert abs(g[0, 0] - fd) < 1e-6 * max(1.0, abs(energy(0.0)))


@pytest.mark.parametrize("name", ["h63", "h64", "h91"])
@pytest.mark.parametrize("chunk", [2047, 2048, 4096, 8192])
def test_chunks_beyond_one_sort(name, chunk):
    """(ss|ss) chunks of up to 2016, 2080 and 4186 kets (every length below them
    as the bra goes through its list, 2048 among them): one pass of the sort,
    two, and three, the Coulomb elements added and cleared between them."""
    print("coulomb lists, chunk cap", name, chunk, flush=True)
    basis_name, atoms = case(name)
    basis = lai.basis_set(basis_name, atoms)
    n = basis.n_basis_functions()
    D = systems.density(n, max(1, n // 4), 7, 1.0 / np.sqrt(n))
    e = lai.Engine(basis)
    e.set_dispatch_table(lai.DispatchTable([lai.DispatchEntry(0, lai.GpuExecutionStrategy(0), chunk, 0)]))
    Jo, Ko = oracle.Oracle(oracle.RawBasis(basis_name, atoms)).jk_canonical(D)
    for weighted in (False, True):
        J, K = e.build_jk(D, lai.JKOptions(schwarz_threshold=0.0 if not weighted else 1e-12, density_weighted=weighted))
        assert rel(J, Jo) < TOL and rel(K, Ko) < TOL
