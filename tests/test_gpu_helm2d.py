"""Screened 2-D LGF tables and their free-space convolution on the device
(needs an MI355X), through the C ABI, against the FP64 oracle: tables within
1e-13 of G(0, 0), convolutions within relative L2 1e-12; at a 256 x 256 patch
the identity (Lap_h - c^2) u = scale * src at interior cells, relative 1e-9."""
import numpy as np
import pytest

from iblgf_amd import IblgfError, helm2d_convolve, helm2d_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _lap(u, c):
    return u[..., 1:-1, :-2] + u[..., 1:-1, 2:] + u[..., :-2, 1:-1] + u[..., 2:, 1:-1] - (4.0 + c * c) * u[..., 1:-1, 1:-1]


def test_tables_match_oracle():
    print("case: tables of 3 modes (c = 0.02, 0.4, 2.5) on a 48 x 40 patch", flush=True)
    cs = np.array([0.02, 0.4, 2.5])
    nx, ny = 48, 40
    t = torch.empty((3, ny, nx), dtype=torch.float64, device="cuda")
    helm2d_table(cs, nx, ny, t)
    got = t.cpu().numpy()
    for k, c in enumerate(cs):
        ref = O.helm2d_table(c, nx, ny)
        assert np.max(np.abs(got[k] - ref)) <= 1e-13 * abs(ref[0, 0]), c


def test_convolution_matches_oracle_per_mode():
    print("case: convolution of 4 modes on a 24 x 17 patch, scale 0.7", flush=True)
    cs = np.array([0.05, 0.3, 1.0, 3.0])
    nx, ny = 24, 17
    rng = np.random.default_rng(21)
    src = rng.standard_normal((4, ny, nx))
    t = torch.empty((4, ny, nx), dtype=torch.float64, device="cuda")
    helm2d_table(cs, nx, ny, t)
    s = torch.from_numpy(src).cuda()
    d = torch.empty_like(s)
    helm2d_convolve(t, s, d, 0.7)
    got, tab = d.cpu().numpy(), t.cpu().numpy()
    for k in range(4):
        ref = O.helm2d_convolve(tab[k], src[k], 0.7)
        assert np.linalg.norm(got[k] - ref) <= 1e-12 * np.linalg.norm(ref), k


@pytest.mark.parametrize("nx,ny", [(64, 3), (72, 5), (300, 2), (1024, 1), (1025, 1)])
def test_row_staged_widths_match_oracle(nx, ny):
    print(f"case: convolution of 2 modes on a {nx} x {ny} patch (row-staged widths and the edges)", flush=True)
    cs = np.array([0.08, 1.5])
    rng = np.random.default_rng(nx + ny)
    src = rng.standard_normal((2, ny, nx))
    t = torch.empty((2, ny, nx), dtype=torch.float64, device="cuda")
    helm2d_table(cs, nx, ny, t)
    s = torch.from_numpy(src).cuda()
    d = torch.empty_like(s)
    helm2d_convolve(t, s, d, -1.25)
    got, tab = d.cpu().numpy(), t.cpu().numpy()
    for k in range(2):
        ref = O.helm2d_convolve(tab[k], src[k], -1.25)
        assert np.linalg.norm(got[k] - ref) <= 1e-12 * np.linalg.norm(ref), k


def test_full_patch_satisfies_screened_poisson():
    print("case: 8 modes on a 256 x 256 patch, (Lap_h - c^2) u = src", flush=True)
    nx = ny = 256
    cs = 2.0 * np.pi * np.arange(1, 9) / 64.0 * (1.0 / 8.0)  # k dx for spanwise modes 1..8
    torch.manual_seed(5)
    s = torch.randn((8, ny, nx), dtype=torch.float64, device="cuda")
    t = torch.empty_like(s)
    d = torch.empty_like(s)
    helm2d_table(cs, nx, ny, t)
    helm2d_convolve(t, s, d, 1.0)
    u, f = d.cpu().numpy(), s.cpu().numpy()
    for k, c in enumerate(cs):
        r = _lap(u[k], c) - f[k, 1:-1, 1:-1]
        assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(f[k]), (k, c)


def test_argument_errors():
    print("case: argument errors of the 2-D Helmholtz entry points", flush=True)
    t = torch.empty((1, 8, 8), dtype=torch.float64, device="cuda")
    with pytest.raises(IblgfError):
        helm2d_table([0.0], 8, 8, t)  # no screening: the Laplace kernel, not this one
    with pytest.raises(IblgfError):
        helm2d_table([1e-5], 8, 8, t)
    with pytest.raises(IblgfError):
        helm2d_table(np.full(257, 0.5), 1, 1, torch.empty(257, dtype=torch.float64, device="cuda"))
    big = torch.empty((1, 1, 65537), dtype=torch.float64, device="cuda")
    with pytest.raises(IblgfError):
        helm2d_table([0.5], 65537, 1, big)
    with pytest.raises(IblgfError):
        helm2d_convolve(t, t, t)  # source and target must differ
    with pytest.raises(ValueError):
        helm2d_table([0.5], 8, 8, t.float())


@pytest.mark.parametrize("nx,ny", [(8, 32), (15, 18), (31, 9), (32, 8), (33, 40), (63, 5), (64, 17), (65, 33), (128, 2),
                                   (129, 7), (256, 9), (257, 16), (511, 3), (512, 8)])
def test_transformed_widths_match_oracle(nx, ny):
    """Patches whose x direction is transformed: the edges of the transform lengths and of the target-row
    groups, rows of very different size next to each other, a scale.  FP64 transforms of up to 1024 points and sums
    over at most 65 536 products: 1e-12 of the field."""
    print(f"case: transformed convolution of 3 modes on a {nx} x {ny} patch", flush=True)
    cs = np.array([0.05, 0.7, 3.0])
    rng = np.random.default_rng(nx * ny)
    src = rng.standard_normal((3, ny, nx)) * 10.0 ** rng.integers(-3, 4, (3, ny, 1))
    t = torch.empty((3, ny, nx), dtype=torch.float64, device="cuda")
    helm2d_table(cs, nx, ny, t)
    s = torch.from_numpy(src).cuda()
    d = torch.full_like(s, float("nan"))
    helm2d_convolve(t, s, d, 0.6)
    got, tab = d.cpu().numpy(), t.cpu().numpy()
    for k in range(3):
        ref = O.helm2d_convolve(tab[k], src[k], 0.6)
        assert np.linalg.norm(got[k] - ref) <= 1e-12 * np.linalg.norm(ref), k


@pytest.mark.parametrize("nx,ny", [(16, 16), (32, 40), (100, 60), (200, 31), (300, 40), (512, 20)])
def test_far_cells_of_a_compact_source_within_the_stated_bound(nx, ny):
    """Screened kernels fall off by many powers of ten within a patch.  Cell by
    cell, the transformed convolution of a compact source stays within the bound
    that the header states, relative to the source and table rows: three
    transforms of log2(P) steps, one rounding of 2^-53 a step (measured: at most
    0.02 of it)."""
    print(f"case: compact source, strong screening, {nx} x {ny} patch", flush=True)
    cs = np.array([0.05, 1.0, 3.0])
    src = np.zeros((3, ny, nx))
    src[:, ny // 2 - 1:ny // 2 + 2, nx // 3:nx // 3 + 4] = np.random.default_rng(nx).standard_normal((3, 3, 4))
    t = torch.empty((3, ny, nx), dtype=torch.float64, device="cuda")
    helm2d_table(cs, nx, ny, t)
    s = torch.from_numpy(src).cuda()
    d = torch.full_like(s, float("nan"))
    helm2d_convolve(t, s, d)
    got, tab = d.cpu().numpy(), t.cpu().numpy()
    steps = 3 * max(6, int(np.ceil(np.log2(2 * nx))))
    for k in range(3):
        # two neighbouring rows share a transform: a source row with the one beside it, a table row (both sides) likewise
        def pair(a):
            n = np.linalg.norm(np.pad(a, ((1, 1), (0, 0))), axis=1)
            return np.sqrt(n[1:-1] ** 2 + np.maximum(n[:-2], n[2:]) ** 2)

        sn, tn = pair(src[k]), np.sqrt(2.0) * pair(tab[k])
        j = np.arange(ny)
        bound = steps * 2.0 ** -53 * (tn[abs(j[:, None] - j[None, :])] @ sn)
        # target rows are transformed back in pairs too
        bound = np.maximum(bound, np.maximum(np.append(bound[1:], 0), np.insert(bound[:-1], 0, 0)))
        err = np.max(np.abs(got[k] - O.helm2d_convolve(tab[k], src[k], 1.0)), axis=1)
        print(f"mode {k}: largest error / bound {np.max(err / bound):.2f}", flush=True)
        assert np.all(err <= bound), k
