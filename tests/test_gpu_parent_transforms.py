"""Laplace levels by transforms of whole parents (csrc/parent_fft.hip) against
the oracle's block convolutions: every block size, meshes whose parents lack
children or neighbours, components in FP64 and with FP32 spectra, and trees
that keep the block path (wrapped keys).  FP64 transforms of up to 65 points a
side leave errors of a few 1e-15 of the largest contribution to a target: 1e-12
relative to the whole field.  FP32 spectra carry 6e-8 a value: 1e-6."""
import numpy as np
import pytest

from iblgf_amd import FLAG_LEAF, PREC_FP16X3_FORWARD, PREC_FP64, PREC_MIXED, PoissonSolver, Tree, lib, setups

pytestmark = pytest.mark.gpu


def _uniform(extent, region, box=8):
    lo = -(box // 2) * extent
    t = Tree((lo,) * 3, (box * extent,) * 3, extent, 1.0 / extent, [(0, 0, 0) + tuple(r * extent for r in region)])
    return t.init_refine(0).build_masks()


def _check(oracle_mod, tree, ncomp, precision, bound):
    rng = np.random.default_rng(11)
    info, a = tree.info(), tree.export()
    src = [rng.standard_normal((info["nblocks"],) + (tree.n,) * 3) for _ in range(ncomp)]
    s = PoissonSolver(tree)
    s.set_precision(precision)
    fi, fo = [s.field() for _ in src], [s.field() for _ in src]
    for f, x in zip(fi, src):
        s.upload(f, x)
    s.apply_lgf_batch(fi, fo)
    ot = oracle_mod.Tree(a, info, tree.n)
    lv = (a["flags"] & FLAG_LEAF) != 0
    for f, x in zip(fo, src):
        ref, got = ot.apply_lgf(x)[lv], s.download(f)[lv]
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"relL2 {err:.2e}", flush=True)
        assert err < bound
        assert np.max(np.abs(got - ref)) < 10 * bound * np.max(np.abs(ref))  # rings of the blocks too


@pytest.mark.parametrize("extent", [6, 8, 10, 14, 16])
@pytest.mark.parametrize("region", [(1, 1, 1), (2, 3, 1), (4, 3, 3)])
def test_uniform_regions(oracle_mod, extent, region):
    print(f"case: whole-parent transforms, {extent}^3 blocks, region {region}", flush=True)
    _check(oracle_mod, _uniform(extent, region), 1, PREC_FP64, 1e-12)


@pytest.mark.parametrize("extent, precision, bound", [(6, PREC_FP64, 1e-12), (8, PREC_FP64, 1e-12), (6, PREC_MIXED, 1e-6)])
def test_groups_of_targets(oracle_mod, extent, precision, bound):
    """4 x 3 x 2 parents: groups of four targets, of two, and shared sources
    that reach some of a group only."""
    print(f"case: whole-parent products in groups, {extent}^3 blocks, precision {precision}", flush=True)
    _check(oracle_mod, _uniform(extent, (7, 5, 3), box=16), 2, precision, bound)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED, PREC_FP16X3_FORWARD])
@pytest.mark.parametrize("extent", [6, 10])
def test_adaptive_tree_two_components(oracle_mod, extent, precision):
    print(f"case: whole-parent transforms, adaptive tree, {extent}^3 blocks, precision {precision}", flush=True)
    v = setups.VortexRings(seed=7, block_extent=extent, base_blocks=4, nref=2, nrings=3, centre_range=4.0,
                           radius=(4.0, 8.0), core=(1.5, 2.5), refinement_factor=0.5)
    _check(oracle_mod, v.tree, 2, precision, 1e-12 if precision == PREC_FP64 else 1e-6)


def test_wrapped_keys_keep_the_block_path(oracle_mod):
    print("case: Laplace on a level whose keys wrap", flush=True)
    keys = [lib().iblgf_key_make(x, y, z, 1) for z in range(2) for y in range(2) for x in range(2)]
    t = Tree.from_keys((0, 0, 0), 8, 1, 1.0, keys, [1] * 8).build_masks()
    _check(oracle_mod, t, 1, PREC_FP64, 1e-12)
