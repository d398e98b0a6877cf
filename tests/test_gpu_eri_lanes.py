"""Raw ERI blocks whose primitive quartets are divided over lanes, against the
oracle: one quartet to a few (64 lanes each), just below and above a workgroup,
and lists long enough for one lane each; contracted and uncontracted shells (1
to 64 primitive pairs, fewer and more than the lanes on either side) in one
list, quartets in every shell order, s to f.  Bar: FP64 sums of at most 4096
terms, each good to some 1e-15, in another order: 1e-12 of the largest
integral."""
import numpy as np
import pytest

import oracle
from libaccint import systems
import libaccint as lai

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis_name", ["sto-3g", "cc-pvdz", "cc-pvtz"])
@pytest.mark.parametrize("n", [1, 2, 3, 127, 129, 2049, 300000])
def test_blocks_match_oracle(basis_name, n):
    print("eri lanes", basis_name, n, flush=True)
    atoms = systems.h2o_sto3g_geometry()
    basis = lai.basis_set(basis_name, atoms)
    rng = np.random.default_rng(n)
    quartets = rng.integers(0, basis.n_shells(), (n, 4)).astype(np.int32)
    if n < 4:
        quartets[0] = 0  # the most contracted
    blocks, offsets = lai.Engine(basis).compute_eri_blocks(quartets)
    blocks, offsets = np.asarray(blocks), np.asarray(offsets)
    orc = oracle.Oracle(oracle.RawBasis(basis_name, atoms))
    scale = max(np.max(np.abs(blocks)), 1e-300)
    known = {}
    for t in range(n) if n < 3000 else rng.integers(0, n, 1500):
        q = tuple(int(x) for x in quartets[t])
        if q not in known:
            known[q] = orc.eri_quartet(*q).ravel()
        got = blocks[offsets[t]:offsets[t] + known[q].size]
        assert np.max(np.abs(got - known[q])) <= 1e-12 * scale, (q, known[q].size)
