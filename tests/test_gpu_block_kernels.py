"""Halo fill and boundary ramp (k_buffer_exchange, k_smooth_ramp) against the
oracle at every block size: copies, and products in the oracle's order, so
the values agree exactly."""
import numpy as np
import pytest

from iblgf_amd import PoissonSolver, setups

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extent", [6, 8, 10, 14, 16])
def test_halo_and_ramp_match_oracle(oracle_mod, extent):
    print(f"case: halo fill and boundary ramp, {extent}^3 blocks", flush=True)
    v = setups.VortexRings(seed=7, block_extent=extent, base_blocks=4, nref=1, nrings=1, centre_range=2.0,
                           radius=(3.0, 4.0), core=(1.5, 2.0), refinement_factor=0.3)
    a = np.random.default_rng(extent).standard_normal((v.info["nblocks"],) + (v.tree.n,) * 3)
    ot = oracle_mod.Tree(v.arrays, v.info, v.tree.n)
    s = PoissonSolver(v.tree)
    f = s.field()
    s.upload(f, a)
    for level in range(v.info["base_level"], v.info["depth"]):
        s.buffer_exchange(f, level)
        ot.buffer_exchange(a, level)
        assert np.array_equal(s.download(f), a)
        for leaf_only in (False, True):
            s.smooth_boundary(f, level, leaf_only)
            ot.smooth_boundary(a, level, leaf_only)
            assert np.array_equal(s.download(f), a)
