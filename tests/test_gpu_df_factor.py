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
