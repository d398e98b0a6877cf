"""The exchange of a symmetric density from its factor (LAI_DF_SYMMETRIC,
lai_dev_df_jk) against the general products (no flag), for the densities that
decide which of the two runs: low rank, rank about and above half of the
functions, full rank, indefinite (a difference of densities; a zero diagonal
with non-zero elements), zero, not finite.  225 and 250 functions (rows and
columns that do not fill tiles), and 200, where no factor is tried.  Bar: both
are FP64 sums of the same terms in another order, and the factor reproduces D to
7e-15; 1e-12 relative."""
import ctypes

import numpy as np
import pytest
import torch

from libaccint import _cabi, systems
import libaccint as lai

pytestmark = pytest.mark.gpu

_builders = {}


def builder(n_water):
    if n_water not in _builders:
        atoms = systems.water_cluster(n_water, 12.0, seed=4)
        basis = lai.basis_set("cc-pvdz", atoms)
        fb = lai.make_df_fock_builder(basis, [z for z, _ in atoms], [list(p) for _, p in atoms], "cc-pVDZ-RI")
        fb.initialize()
        _builders[n_water] = (basis, fb)
    return _builders[n_water][1]


def jk(fb, D, flags):
    n = D.shape[0]
    d = torch.from_numpy(np.ascontiguousarray(D)).cuda()
    J, K = torch.full((n, n), 7.0, dtype=torch.float64, device="cuda"), torch.full((n, n), 7.0, dtype=torch.float64, device="cuda")
    _cabi.check(_cabi.lib().lai_dev_df_jk(ctypes.c_void_p(fb.device_handle()), d.data_ptr(), J.data_ptr(), K.data_ptr(),
                                          flags, torch.cuda.current_stream().cuda_stream))
    return J.cpu().numpy(), K.cpu().numpy()


def density(kind, n):
    rng = np.random.default_rng(n)
    C = rng.standard_normal((n, n)) / np.sqrt(n)
    if kind.startswith("rank"):
        r = int(kind[4:])
        return C[:, :r] @ C[:, :r].T
    if kind == "half":
        return C[:, :n // 2] @ C[:, :n // 2].T
    if kind == "full":
        return C @ C.T
    if kind == "difference":
        return C[:, :40] @ C[:, :40].T - C[:, 40:80] @ C[:, 40:80].T
    if kind == "zero_diagonal":
        D = C + C.T
        np.fill_diagonal(D, 0.0)
        return D
    if kind == "graded":  # columns of very different size
        G = C[:, :30] * 10.0 ** (-0.25 * np.arange(30))
        return G @ G.T
    return np.zeros((n, n))


@pytest.mark.parametrize("n_water", [8, 9, 10])
@pytest.mark.parametrize("kind", ["rank1", "rank40", "rank81", "half", "rank130", "full", "difference", "zero_diagonal",
                                  "graded", "zero"])
def test_symmetric_density_matches_general_products(n_water, kind):
    print("df factor", n_water, kind, flush=True)
    fb = builder(n_water)
    D = density(kind, fb.n_orb())
    D = 0.5 * (D + D.T)
    J0, K0 = jk(fb, D, 3)
    for flags in (7, 6, 5):
        J, K = jk(fb, D, flags)
        if flags & 1:
            assert np.max(np.abs(J - J0)) <= 1e-12 * np.max(np.abs(J0))
        if flags & 2:
            assert np.max(np.abs(K - K0)) <= 1e-12 * np.max(np.abs(K0))
            assert np.array_equal(K, K.T)


def test_density_that_is_not_finite_gives_nan():
    fb = builder(9)
    n = fb.n_orb()
    for bad in (np.nan, np.inf):
        D = density("rank40", n)
        D[3, 3] = bad
        J, K = jk(fb, D, 7)
        assert not np.isfinite(J).all() and not np.isfinite(K).all()


def info(fb):
    ok, rank = ctypes.c_int(), ctypes.c_int()
    _cabi.check(_cabi.lib().lai_dev_df_factor_info(ctypes.c_void_p(fb.device_handle()), ctypes.byref(ok),
                                                   ctypes.byref(rank)))
    return ok.value, rank.value


@pytest.mark.parametrize("n_water", [8, 9, 10])
@pytest.mark.parametrize("kind, rank", [("rank1", 1), ("rank40", 40), ("rank81", 81), ("half", None), ("graded", 30),
                                        ("rank130", 0), ("full", 0), ("difference", 0), ("zero_diagonal", 0),
                                        ("zero", 0)])
def test_form_of_the_exchange(n_water, kind, rank):
    """Which of the two forms ran: the factor's columns for a semidefinite D of
    at most n/2 of them, the general products for the others (and always below
    224 functions)."""
    print("df form", n_water, kind, flush=True)
    fb = builder(n_water)
    n = fb.n_orb()
    rank = n // 2 if rank is None else rank
    D = density(kind, n)
    D = 0.5 * (D + D.T)
    jk(fb, D, 7)
    if n_water == 8:
        assert info(fb)[0] == -1
    elif rank == 0:
        assert info(fb)[0] == 0
    else:  # (a few columns of D's rounding may be among them)
        assert info(fb)[0] == 1 and rank - 2 <= info(fb)[1] <= min(rank + 4, n // 2)


EPS = 2.220446049250313e-16


def orbitals(kind, n, r):
    Q, _ = np.linalg.qr(np.random.default_rng(n).standard_normal((n, r)))
    return Q * 10.0 ** (-4.0 * np.arange(r) / r) if kind == "graded" else Q


@pytest.mark.parametrize("kind", ["orthonormal", "graded"])
@pytest.mark.parametrize("n, r", [(2, 1), (31, 5), (32, 16), (33, 6), (225, 45), (400, 80), (512, 102), (513, 102),
                                  (640, 128), (645, 129), (1023, 204), (1024, 205), (1025, 205), (2048, 409)])
def test_factor_reproduces_density(kind, n, r):
    """L L^T against D, summed in long double over every row or 64 of them: at
    most 4 eps of the norm (the bound that the device applies; twice as much for
    a part of the rows), in one row per lane and two, one correction and two, the
    inverse in registers and in memory.  Without the correction: 12 to 190 eps."""
    print("df factor alone", kind, n, r, flush=True)
    Q = orbitals(kind, n, r)
    D = Q @ Q.T
    D = 0.5 * (D + D.T)
    d = torch.from_numpy(D).cuda()
    Lt = torch.zeros((n // 2, n), dtype=torch.float64, device="cuda")
    ok, rank, res = ctypes.c_int(), ctypes.c_int(), ctypes.c_double()
    _cabi.check(_cabi.lib().lai_dev_df_factor(d.data_ptr(), n, Lt.data_ptr(), ctypes.byref(ok), ctypes.byref(rank),
                                              ctypes.byref(res)))
    assert ok.value == 1 and r <= rank.value <= r + 4 and res.value <= 4 * EPS
    L = Lt[:rank.value].cpu().numpy().astype(np.longdouble)
    rows = np.arange(0, n, max(1, n // 64))
    E = (D[rows].astype(np.longdouble) - L[:, rows].T @ L).astype(float)
    assert np.linalg.norm(E) <= (4 if len(rows) == n else 8) * EPS * np.linalg.norm(D[rows])


@pytest.mark.parametrize("n, kind", [(33, "over"), (400, "over"), (1025, "over"), (400, "difference"),
                                     (2048, "difference"), (400, "nan"), (64, "zero")])
def test_factor_refuses(n, kind):
    print("df factor alone", n, kind, flush=True)
    rng = np.random.default_rng(n)
    C = rng.standard_normal((n, n)) / np.sqrt(n)
    A = C[:, :n // 2 + 1]
    D = A @ A.T
    if kind == "difference":
        D = C[:, :n // 5] @ C[:, :n // 5].T - C[:, n // 5:n // 3] @ C[:, n // 5:n // 3].T
    elif kind == "zero":
        D = np.zeros((n, n))
    D = 0.5 * (D + D.T)
    if kind == "nan":
        D = C[:, :40] @ C[:, :40].T
        D[3, 7] = D[7, 3] = np.nan
    d = torch.from_numpy(np.ascontiguousarray(D)).cuda()
    Lt = torch.zeros((n // 2, n), dtype=torch.float64, device="cuda")
    ok, rank, res = ctypes.c_int(), ctypes.c_int(), ctypes.c_double()
    _cabi.check(_cabi.lib().lai_dev_df_factor(d.data_ptr(), n, Lt.data_ptr(), ctypes.byref(ok), ctypes.byref(rank),
                                              ctypes.byref(res)))
    assert ok.value == 0


@pytest.mark.parametrize("kind", ["orthonormal", "graded"])
def test_exchange_is_as_exact_as_the_general_products(kind):
    """16 waters (400 functions, 80 orbitals).  Against long double the general
    products have a relative error of 1.2 to 1.5e-15 and the factored form 0.8 to
    1.1e-15, 1.8e-15 in quadrature; a third more is allowed.  (The uncorrected
    factor of the graded orbitals: 3.7e-15.)"""
    print("df exact", kind, flush=True)
    fb = builder(16)
    n = fb.n_orb()
    Q = orbitals(kind, n, 80)
    D = Q @ Q.T
    D = 0.5 * (D + D.T)
    K0 = jk(fb, D, 3)[1]
    K = jk(fb, D, 7)[1]
    assert info(fb)[0] == 1
    assert np.linalg.norm(K - K0) <= 2.4e-15 * np.linalg.norm(K0)


def test_captured_build_follows_its_density():
    """One captured build replayed on densities of both forms, with eager builds
    between: the device decides in every replay."""
    print("df captured", flush=True)
    fb = builder(9)
    n = fb.n_orb()
    dD = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    J, K = torch.zeros_like(dD), torch.zeros_like(dD)
    st = torch.cuda.Stream()

    def build():
        _cabi.check(_cabi.lib().lai_dev_df_jk(ctypes.c_void_p(fb.device_handle()), dD.data_ptr(), J.data_ptr(),
                                              K.data_ptr(), 7, st.cuda_stream))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        build()
    for kind, form in (("rank40", 1), ("difference", 0), ("graded", 1), ("full", 0), ("rank81", 1)):
        D = density(kind, n)
        D = 0.5 * (D + D.T)
        J0, K0 = jk(fb, D, 3)
        dD.copy_(torch.from_numpy(D))
        for _ in range(2):
            J.fill_(7.0)
            K.fill_(7.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert info(fb)[0] == form
            assert np.max(np.abs(J.cpu().numpy() - J0)) <= 1e-12 * np.max(np.abs(J0))
            assert np.max(np.abs(K.cpu().numpy() - K0)) <= 1e-12 * np.max(np.abs(K0))
