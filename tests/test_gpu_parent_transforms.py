"""Laplace levels by transforms of whole parents (csrc/parent_fft.hip) against
the oracle's block convolutions: every block size, meshes whose parents lack
children or neighbours, components in FP64 and with FP32 spectra, and trees
that keep the block path (wrapped keys).  FP64 transforms of up to 65 points a
side leave errors of a few 1e-15 of the largest contribution to a target: 1e-12
relative to the whole field.  FP32 spectra carry 6e-8 a value: 1e-6."""
import numpy as np
import pytest
import torch

from iblgf_amd import (FLAG_LEAF, PREC_FP16X3_FORWARD, PREC_FP64, PREC_INT8X4, PREC_MIXED, PoissonSolver, Tree, lib,
                       setups)

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


@pytest.mark.parametrize("precision", [PREC_MIXED, PREC_FP16X3_FORWARD, PREC_INT8X4])
@pytest.mark.parametrize("extent", [6, 8, 10, 14, 16])
def test_spectra_kept_in_fp64(oracle_mod, extent, precision):
    """With FP32 spectra, FP64 ones below the base level (all coarser levels of
    this mesh, in transforms of either kind) and for the first planes of whole
    parents.  What is left is stored to 2^-24 of each value, once as a source and
    once as a target: 1.2e-7."""
    print(f"case: FP64 among FP32 spectra, {extent}^3 blocks, precision {precision}", flush=True)
    _check(oracle_mod, _uniform(extent, (7, 5, 3), box=16), 2, precision, 1.2e-7)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED, PREC_FP16X3_FORWARD])
@pytest.mark.parametrize("extent", [6, 10])
def test_adaptive_tree_two_components(oracle_mod, extent, precision):
    print(f"case: whole-parent transforms, adaptive tree, {extent}^3 blocks, precision {precision}", flush=True)
    v = setups.VortexRings(seed=7, block_extent=extent, base_blocks=4, nref=2, nrings=3, centre_range=4.0,
                           radius=(4.0, 8.0), core=(1.5, 2.5), refinement_factor=0.5)
    _check(oracle_mod, v.tree, 2, precision, 1e-12 if precision == PREC_FP64 else 1e-6)


def _solver(tree, precision, ncomp):
    s = PoissonSolver(tree)
    s.set_precision(precision)
    rng = np.random.default_rng(12)
    src, dst = [s.field() for _ in range(ncomp)], [s.field() for _ in range(ncomp)]
    for f in src:
        s.upload(f, rng.standard_normal(s.shape))
    return s, src, dst


@pytest.mark.parametrize("extent", [6, 8, 10, 14, 16])
@pytest.mark.parametrize("region", [(1, 1, 1), (2, 3, 1), (4, 3, 3), None])
def test_scratch_in_rounds(extent, region):
    """The spectra of whole parents in the memory that block spectra leave: at
    once, in rounds of some frequencies (FP64 solves of as many components as
    the work arrays hold, here, on every mesh but the one of a single block),
    and, for a single block, outside it.  Frequencies are independent, so the
    results are equal bit for bit."""
    print(f"case: scratch of whole parents, {extent}^3 blocks, region {region}", flush=True)
    if region:
        t = _uniform(extent, region)
    else:
        t = setups.VortexRings(seed=7, block_extent=extent, base_blocks=4, nref=1, nrings=1, centre_range=2.0,
                               radius=(3.0, 4.0), core=(1.5, 2.0), refinement_factor=0.3).tree
    s, src, dst = _solver(t, PREC_FP64, 3)
    for f, d in zip(src, dst):
        s.apply_lgf(f, d)  # one component in work arrays of one
    one = [s.download(d) for d in dst]
    s.apply_lgf_batch(src, dst)  # three in arrays of three
    assert all(np.array_equal(s.download(d), x) for d, x in zip(dst, one))
    s.apply_lgf(src[0], dst[0])  # one in arrays of three: at once
    assert np.array_equal(s.download(dst[0]), one[0])


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("region", [(1, 1, 1), None])
def test_graphs_across_component_counts(region, precision):
    """Solves of one, three and one component captured as graphs: each replay,
    with other solves and growing work arrays in between, equals the eager result."""
    print(f"case: graphs of one and three components, region {region}, precision {precision}", flush=True)
    t = _uniform(10, region) if region else setups.VortexRings(
        seed=7, block_extent=10, base_blocks=4, nref=2, nrings=3, centre_range=4.0, radius=(4.0, 8.0), core=(1.5, 2.5),
        refinement_factor=0.5).tree
    s, src, dst = _solver(t, precision, 3)
    s.apply_lgf_batch(src, dst)
    ref = [s.download(d) for d in dst]

    def same(k):
        return all(np.array_equal(s.download(d), x) for d, x in zip(dst[:k], ref))

    s, src, dst = _solver(t, precision, 3)
    s.set_graphs(True)
    for k in (1, 1, 3, 1, 3, 1):
        for d in dst:
            s.upload(d, np.zeros(s.shape))
        s.apply_lgf_batch(src[:k], dst[:k])
        assert same(k), k
        s.apply_lgf_batch(src, dst, kernel=1, alpha_base=0.3)  # grows the work arrays, before a solve does
    s.set_graphs(False)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED])
def test_memory_of_a_component(precision):
    """A solve takes the memory of its work arrays, four fields and two
    block spectra of FP64 a component, and nothing beside them however its
    parents lie.  (Allocations come in whole pages of 2 MiB.)"""
    print(f"case: memory a component, precision {precision}", flush=True)
    t = setups.VortexRings(seed=7, block_extent=16, base_blocks=4, nref=2, nrings=3, centre_range=4.0,
                           radius=(4.0, 8.0), core=(1.5, 2.5), refinement_factor=0.5).tree
    s, src, dst = _solver(t, precision, 6)
    s.prepare()
    s.apply_lgf(src[0], dst[0])
    n, nb = t.n, s.shape[0]
    P = 2 * n - 1
    per = nb * (4 * n**3 * 8 + 2 * P * P * (P // 2 + 1) * 16)

    def used(k):
        s.apply_lgf_batch(src[:k], dst[:k])
        s.sync()
        free, total = torch.cuda.mem_get_info()
        return total - free

    at = [used(k) for k in (1, 3, 6)]
    assert at[1] - at[0] <= 2 * per + (16 << 20)
    assert at[2] - at[0] <= 5 * per + (16 << 20)


def test_wrapped_keys_keep_the_block_path(oracle_mod):
    print("case: Laplace on a level whose keys wrap", flush=True)
    keys = [lib().iblgf_key_make(x, y, z, 1) for z in range(2) for y in range(2) for x in range(2)]
    t = Tree.from_keys((0, 0, 0), 8, 1, 1.0, keys, [1] * 8).build_masks()
    _check(oracle_mod, t, 1, PREC_FP64, 1e-12)
