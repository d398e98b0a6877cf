"""The f classes that run a lane per quartet with the bra in four or five slices
((fp|pp), (fs|dp), (fp|ds), (fd|ps), (fp|fs)) in each of their three strategies
(a saved table may name any): one water in cc-pVTZ against the oracle, with the
default chunk cap and one quartet per chunk (10 to 70 kets a bra), and three
waters (90 to 630 kets a bra) against the workgroup kernel, with caps just off a
wavefront and just off the lanes of a group of slices.  Bar: 1e-10 relative, the
J/K bar of test_gpu_parity.py, against the oracle; 1e-12 between strategies (FP64
sums in another order)."""
import ctypes

import numpy as np
import pytest

import oracle
from libaccint import _cabi, systems
import libaccint as lai

pytestmark = pytest.mark.gpu
PAIRS = ["ss", "ps", "pp", "ds", "dp", "dd", "fs", "fp", "fd", "ff"]
CLASSES = [b * (b + 1) // 2 + k for b, k in
           ((PAIRS.index(x), PAIRS.index(y)) for x, y in
            (("fp", "pp"), ("fs", "dp"), ("fp", "ds"), ("fd", "ps"), ("fp", "fs")))]
_case = {}


def case():
    if not _case:
        atoms = systems.h2o_sto3g_geometry()
        basis = lai.basis_set("cc-pvtz", atoms)
        n = basis.n_basis_functions()
        D = systems.density(n, 5, 11, 1.0 / np.sqrt(n))
        _case["v"] = basis, D, oracle.Oracle(oracle.RawBasis("cc-pvtz", atoms)).jk_canonical(D)
    return _case["v"]


def test_classes_have_three_strategies():
    for c in CLASSES:
        s, a = ctypes.c_int(), ctypes.c_int()
        _cabi.check(_cabi.lib().lai_dev_class_strategies(c, ctypes.byref(s), ctypes.byref(a)))
        assert (s.value, a.value) == (0, 1)


@pytest.mark.parametrize("strategy", [0, 1, 2])
@pytest.mark.parametrize("chunk", [0, 1, 65, 300])
def test_strategies_match_oracle(strategy, chunk):
    print("f slices", strategy, chunk, flush=True)
    basis, D, (Jo, Ko) = case()
    e = lai.Engine(basis)
    S = lai.GpuExecutionStrategy
    e.set_dispatch_table(lai.DispatchTable([lai.DispatchEntry(c, S(strategy), chunk, 0) for c in CLASSES]))
    for mixed in (False, True):
        J, K = e.build_jk(D, lai.JKOptions(schwarz_threshold=1e-12, mixed_precision=mixed, fp32_threshold=1e-12))
        assert np.max(np.abs(J - Jo)) < 1e-10 * np.max(np.abs(Jo))
        assert np.max(np.abs(K - Ko)) < 1e-10 * np.max(np.abs(Ko))


@pytest.mark.parametrize("chunk", [0, 63, 65, 255, 257, 321])
def test_strategies_match_on_long_runs(chunk):
    print("f slices, long runs", chunk, flush=True)
    basis = lai.basis_set("cc-pvtz", systems.water_cluster(3, 10.0, seed=5))
    n = basis.n_basis_functions()
    D = systems.density(n, 15, 11, 1.0 / np.sqrt(n))
    e = lai.Engine(basis)
    S = lai.GpuExecutionStrategy
    opts = lai.JKOptions(schwarz_threshold=1e-12)
    got = []
    for strategy in (2, 0, 1):
        cap = 0 if strategy == 2 else chunk
        e.set_dispatch_table(lai.DispatchTable([lai.DispatchEntry(c, S(strategy), cap, 0) for c in CLASSES]))
        got.append(e.build_jk(D, opts))
    for J, K in got[1:]:
        assert np.max(np.abs(J - got[0][0])) < 1e-12 * np.max(np.abs(got[0][0]))
        assert np.max(np.abs(K - got[0][1])) < 1e-12 * np.max(np.abs(got[0][1]))
