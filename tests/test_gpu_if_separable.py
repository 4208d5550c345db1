"""Integrating-factor passes as separable sums (csrc/if_separable.hip) against
the oracle's block convolutions: every block size, meshes whose blocks miss
neighbours on some or all sides, an adaptive tree, several components, and a
tree whose Morton keys wrap, which keeps the spectral path.  The device sums
in FP64 without transforms and the oracle through FP64 transforms, each within
a few rounding errors of sums of at most 27 (n - 2)^3 positive products that
add up to one: 1e-13 relative."""
import numpy as np
import pytest

from iblgf_amd import PREC_MIXED, PoissonSolver, Tree, lib, setups

pytestmark = pytest.mark.gpu


def _uniform(extent, region, box=8):
    lo = -(box // 2) * extent
    t = Tree((lo,) * 3, (box * extent,) * 3, extent, 1.0 / extent,
             [(0, 0, 0) + tuple(r * extent for r in region)])
    return t.init_refine(0).build_masks()


def _wrapped(extent):
    """All eight blocks of level 1 as the base level: every neighbour offset wraps onto one of them."""
    L = lib()
    keys = [L.iblgf_key_make(x, y, z, 1) for z in range(2) for y in range(2) for x in range(2)]
    t = Tree.from_keys((0, 0, 0), extent, 1, 1.0, keys, [1] * 8)
    return t.build_masks()


def _check(oracle_mod, tree, alpha, ncomp=1, precision=0):
    rng = np.random.default_rng(3)
    info, a = tree.info(), tree.export()
    shape = (info["nblocks"],) + (tree.n,) * 3
    src = [rng.standard_normal(shape) for _ in range(ncomp)]
    s = PoissonSolver(tree)
    s.set_precision(precision)
    fi, fo = [s.field() for _ in src], [s.field() for _ in src]
    for f, x in zip(fi, src):
        s.upload(f, x)
    s.apply_lgf_batch(fi, fo, kernel=1, alpha_base=alpha)
    ot = oracle_mod.Tree(a, info, tree.n)
    for f, x in zip(fo, src):
        ref, got = ot.apply_if(x, alpha), s.download(f)
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"relL2 {err:.2e}", flush=True)
        assert err < 1e-13


@pytest.mark.parametrize("extent", [6, 8, 10, 14, 16])
@pytest.mark.parametrize("region", [(1, 1, 1), (3, 2, 1), (4, 3, 3)])
def test_uniform_regions(oracle_mod, extent, region):
    print(f"case: separable IF, {extent}^3 blocks, region {region}", flush=True)
    _check(oracle_mod, _uniform(extent, region), 0.8)


@pytest.mark.parametrize("alpha", [0.0, 0.05, 40.0])
def test_adaptive_tree_components_and_alphas(oracle_mod, alpha):
    print(f"case: separable IF, adaptive tree, alpha {alpha}, two components", flush=True)
    v = setups.VortexRings(seed=7, block_extent=8, base_blocks=4, nref=2, nrings=3, centre_range=4.0,
                           radius=(4.0, 8.0), core=(1.5, 2.5), refinement_factor=0.5)
    _check(oracle_mod, v.tree, alpha, ncomp=2, precision=PREC_MIXED)


def test_wrapped_keys_keep_the_spectral_path(oracle_mod):
    print("case: IF on a level whose keys wrap", flush=True)
    _check(oracle_mod, _wrapped(8), 0.3)
