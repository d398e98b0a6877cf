"""The gradient kernels class by class: four contracted shells of given angular
momenta (every quartet class among them), their forces against fourth-order
central differences of the energy of the device J/K build, and translational
invariance.  Geometries: spread out, all four shells on two centres (T = 0 in
the Boys argument, AB = 0), and one shell far away (T beyond the table cuts).
Bar: with h = 1e-3 and exponents up to 4 the truncation h^4/30 E^(5) ~ h^4/30
|g| 8^2 is 2e-12 |g|, rounding 1e-15 |E| / h ~ 1e-12 |E|; 1e-9 of the larger of
|E| and |g| leaves room for the J/K sums' own 1e-13 errors over h."""
import numpy as np
import pytest

from libaccint import systems
import libaccint as lai

pytestmark = pytest.mark.gpu

OPTS = lai.JKOptions(schwarz_threshold=0.0)
PLACES = {
    "spread": [(0.0, 0.0, 0.0), (1.1, 0.3, -0.4), (-0.5, 1.4, 0.6), (0.2, -0.9, 1.3)],
    "two_centres": [(0.0, 0.0, 0.0), (0.0, 0.0, 0.0), (0.7, 0.8, -0.9), (0.7, 0.8, -0.9)],
    "far": [(0.0, 0.0, 0.0), (0.4, 0.1, 0.2), (9.0, 2.0, -1.0), (9.3, 2.2, -1.1)],
}


def basis_of(ls, places):
    ex = [[0.6, 2.7], [0.9], [0.5, 1.7, 4.0], [1.2, 0.4]]
    co = [[0.7, 0.4], [1.0], [0.5, 0.3, 0.4], [0.6, 0.5]]
    return lai.BasisSet([lai.Shell(l, list(p), e, c) for l, p, e, c in zip(ls, places, ex, co)])


@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("ls", [(0, 0, 0, 0), (1, 0, 0, 0), (1, 1, 0, 0), (1, 1, 1, 1), (2, 0, 1, 0), (2, 1, 1, 0),
                                (2, 1, 1, 1), (2, 2, 0, 1), (2, 2, 1, 1), (2, 2, 2, 1), (2, 2, 2, 2)])
def test_forces_match_energy_differences(ls, place):
    print("gradient classes", ls, place, flush=True)
    where = [np.array(p) for p in PLACES[place]]
    basis = basis_of(ls, where)
    n = basis.n_basis_functions()
    D = systems.density(n, n, 9, 1.0 / np.sqrt(n))  # full rank: every block of D takes part
    g = lai.Engine(basis).compute_jk_gradient(D, 0.7, 4)

    def energy(k, x, dx):
        moved = [p + (dx if k == m else 0.0) * np.eye(3)[x] for m, p in enumerate(where)]
        J, K = lai.Engine(basis_of(ls, moved)).build_jk(D, OPTS)
        return 0.5 * np.sum(D * J) - 0.25 * 0.7 * np.sum(D * K)
    h = 1e-3
    fd = np.array([[(8.0 * (energy(k, x, h) - energy(k, x, -h)) - (energy(k, x, 2 * h) - energy(k, x, -2 * h)))
                    / (12.0 * h) for x in range(3)] for k in range(4)])
    bar = 1e-9 * max(abs(energy(0, 0, 0.0)), float(np.max(np.abs(g))))
    assert np.max(np.abs(g - fd)) < bar
    assert np.max(np.abs(g.sum(axis=0))) < 1e-12 * max(1.0, float(np.max(np.abs(g))))
