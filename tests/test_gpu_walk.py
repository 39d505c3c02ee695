"""The volume adjoint's cell walk on the GPU, at the sizes where it branches.

``vol_walk_kernel`` forms each cell's corner sums in closed form from the
cell's run of samples: singleton axes and half-cell borders, less than one
sample per cell, thousands of samples per cell, axes beyond 2^18 grid samples
(FP64 coordinates instead of biased ones), slabs that fit no brick, and rays
too sparse for one.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests import scenes

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dpt import _native  # noqa: E402

from .test_gpu_parity import NativeScene, _rel  # noqa: E402


def _volume(grid, samples, precision, seed=0, views=3, rows=19, cols=21, rays=None):
    panels = None if rays is not None else scenes.cone_panels(grid, views, rows, cols, sod=120.0, sdd=200.0, offset=0.3)
    geometry = dict(rays=rays) if rays is not None else dict(panels=panels)
    count = len(rays[0]) if rays is not None else views * rows * cols
    seeds = np.random.default_rng(seed).uniform(-1.0, 1.0, count)
    values = np.full(grid.voxels, 0.02, dtype=np.float32)
    if precision == "float32":
        seeds = seeds.astype(np.float32)
    expected, _, _, _ = O.Scene(grid, samples, **geometry).vjp(
        values, seeds, precision="fp32" if precision == "float32" else "fp64", pose=False)
    actual, _, status = NativeScene(grid, samples, precision=precision, **geometry).vjp(values, seeds, pose_grad=False)
    assert not any(status)
    assert np.linalg.norm(expected) > 0
    return actual, expected


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("shape,samples", [((1, 26, 28), 97), ((24, 1, 28), 97), ((24, 26, 1), 97), ((2, 2, 2), 5),
                                           ((24, 26, 28), 3), ((24, 26, 28), 31), ((3, 4, 5), 4001)])
def test_cell_sums_match_the_per_sample_scatter(shape, samples, precision):
    print(f"case walk {shape} S={samples} {precision}", flush=True)
    grid = O.Grid(shape, (1.0, 0.9, 1.1), tuple(-0.5 * (n - 1) * h for n, h in zip(shape[::-1], (1.0, 0.9, 1.1))))
    actual, expected = _volume(grid, samples, precision)
    # FP32: the oracle rounds each sample's position, |p| <= 200 mm at 2^-24
    # (1.2e-5 voxel), and increments to FP32; FP64: FP32-rounded increments
    # and one FP32 rounding of the result
    assert _rel(actual, expected) <= (1e-5 if precision == "float32" else 1e-7)


def _blocky():
    return O.Grid((40, 44, 48), (1.0, 1.0, 1.0), (-23.5, -21.5, -19.5))


@pytest.mark.parametrize("precision", ["float32", "float64"])
def test_slabs_that_fit_no_brick_use_device_atomics(precision, monkeypatch):
    """Dense rays (1.6 voxels apart) whose tiles cover 26 x 26 voxels: a slab of
    one sample holds more than 512 entries."""
    print(f"case walk cap=512 {precision}", flush=True)
    monkeypatch.setenv("DPT_AMD_BRICK_CAP", "512")
    actual, expected = _volume(_blocky(), 61, precision, rows=40, cols=40)
    assert _rel(actual, expected) <= (1e-5 if precision == "float32" else 1e-7)


@pytest.mark.parametrize("views_per_block", ["1", "2", "4"])
@pytest.mark.parametrize("samples", [1, 7, 61, 900])
@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("rows,cols", [(16, 15), (9, 10)])
def test_sparse_rays_add_by_pairs_of_lanes(rows, cols, samples, precision, views_per_block, monkeypatch):
    """Rays four (along x) and seven voxels apart (along any axis) walk without
    bricks, the wave as one, until its last ray ends."""
    print(f"case walk sparse {rows}x{cols} S={samples} {precision} vb={views_per_block}", flush=True)
    monkeypatch.setenv("DPT_AMD_VIEWS_PER_BLOCK", views_per_block)
    actual, expected = _volume(_blocky(), samples, precision, views=5, rows=rows, cols=cols)
    assert _rel(actual, expected) <= (1e-5 if precision == "float32" else 1e-7)


@pytest.mark.parametrize("shape", [(1, 44, 48), (40, 1, 48), (40, 44, 1), (40, 44, 48)])
@pytest.mark.parametrize("mode", ["float32", "float64", "cell_gauss"])
def test_random_rays_match_the_oracle(shape, mode):
    """Bundles of random directions, a partial last wave, rays that miss and zero
    cotangents among them, singleton axes."""
    print(f"case walk random {shape} {mode}", flush=True)
    grid = O.Grid(shape, (1.0, 0.9, 1.1), tuple(-0.5 * (n - 1) * h for n, h in zip(shape[::-1], (1.0, 0.9, 1.1))))
    rng = np.random.default_rng(11)
    ends = rng.normal(size=(2, 333, 3))
    ends *= 40.0 / np.linalg.norm(ends, axis=2, keepdims=True)
    if 1 in shape:  # rays near the plane of the grid
        ends[..., 2 - shape.index(1)] *= 0.01
    rays = (ends[0], ends[1])
    seeds = rng.uniform(-1.0, 1.0, 333)
    seeds[::7] = 0.0
    values = np.full(grid.voxels, 0.02, np.float32)
    precision = "float32" if mode == "float32" else "float64"
    seeds = seeds.astype(precision)
    gauss = mode == "cell_gauss"
    expected, _, _, _ = O.Scene(grid, 97, rays=rays).vjp(values, seeds, precision="fp32" if mode == "float32" else "fp64",
                                                         pose=False, **(dict(integration=mode) if gauss else {}))
    gpu = NativeScene(grid, 97, rays=rays, precision=precision, extra_needs=_native.CELL_GAUSS if gauss else 0)
    actual, _, status = gpu.vjp(values, seeds, pose_grad=False)
    assert not any(status)
    assert np.linalg.norm(expected) > 0
    # the oracle's FP32 positions (|p| <= 40 mm at 2^-24: 2.4e-6 voxel) and FP32 increments
    assert _rel(actual, expected) <= (1e-5 if mode == "float32" else 1e-7)


@pytest.mark.parametrize("precision", ["float32", "float64"])
def test_axes_beyond_the_biased_coordinates(precision):
    """2^18 + 40 grid samples along x: FP32 sampling resolves positions to
    2^18 * 2^-24 = 1/64 voxel, so its gradient is compared through its total
    (each ray's weights sum to one per sample); FP64 element by element."""
    print(f"case walk wide {precision}", flush=True)
    n = (1 << 18) + 40
    grid = O.Grid((3, 2, n), (1.0, 1.0, 1.0))
    src = np.array([[n - 80.25, 0.5, 1.0], [n - 90.0, -0.2, 0.4], [-3.0, 0.4, 1.1]])
    end = np.array([[n + 30.0, 0.6, 1.2], [n - 20.0, 1.2, 1.7], [50.0, 0.7, 0.9]])
    actual, expected = _volume(grid, 257, precision, rays=(src, end))
    if precision == "float64":
        assert _rel(actual, expected) <= 1e-7
    else:
        assert abs(actual.sum(dtype=np.float64) / expected.sum(dtype=np.float64) - 1.0) <= 1e-5
        assert _rel(actual, expected) <= 5e-2


def test_more_samples_than_the_float_counter_holds():
    print("case walk S=5e6", flush=True)
    grid = O.Grid((3, 3, 3), (1.0, 1.0, 1.0))
    rays = (np.array([[-4.0, 0.3, 0.9]]), np.array([[7.0, 1.4, 1.6]]))
    actual, expected = _volume(grid, 5_000_000, "float32", rays=rays)
    assert _rel(actual, expected) <= 1e-5


@pytest.mark.parametrize("scale", [1.0, 1e-33])
@pytest.mark.parametrize("shape", [(24, 26, 28), (1, 26, 28), (24, 26, 1)])
def test_cell_gauss_pieces_match_the_oracle(shape, scale):
    """Factors in the walk's range, and below 2^-102, whose rays take the
    reference's products piece by piece."""
    print(f"case walk gauss {shape} {scale}", flush=True)
    grid = O.Grid(shape, (1.0, 0.9, 1.1), tuple(-0.5 * (n - 1) * h for n, h in zip(shape[::-1], (1.0, 0.9, 1.1))))
    panels = scenes.cone_panels(grid, 3, 19, 21, sod=120.0, sdd=200.0, offset=0.3)
    seeds = scale * np.random.default_rng(2).uniform(-1.0, 1.0, 3 * 19 * 21)
    values = np.full(grid.voxels, 0.02, dtype=np.float32)
    expected, _, _, _ = O.Scene(grid, 7, panels=panels).vjp(values, seeds, precision="fp64", pose=False,
                                                           integration="cell_gauss")
    gpu = NativeScene(grid, 7, panels=panels, precision="float64", extra_needs=_native.CELL_GAUSS)
    actual, _, status = gpu.vjp(values, seeds, pose_grad=False)
    assert not any(status)
    # FP32-rounded increments, then one FP32 rounding of each sum
    assert _rel(actual / scale, expected / scale) <= 1e-7


@pytest.mark.parametrize("offset", [2e-2, 2e-3, 1e-4])
def test_chords_near_the_rounding_of_a_sample(offset):
    """Rays that clip a vertical edge with chords down to the FP32 rounding of a
    sample's position: their end samples fall outside the support, the others
    are one run, added with the rest."""
    print(f"case walk grazing {offset}", flush=True)
    grid = O.Grid((6, 20, 20), (1.0, 1.0, 1.0), (-9.5, -9.5, -2.5))
    z = np.linspace(-2.0, 2.0, 64)
    corner = 10.0 - offset
    src = np.stack([np.full(64, corner - 700.0), np.full(64, corner + 700.0), z], 1)
    end = np.stack([np.full(64, corner + 500.0), np.full(64, corner - 500.0), z], 1)
    actual, expected = _volume(grid, 1024, "float32", rays=(src, end))
    # the oracle drops the same end samples; a chord of 2 offset holds the
    # rounding of its positions, 1e-4 voxel, in weights near one
    assert _rel(actual, expected) <= 2e-3


def _corner_rays(exponents, seed):
    """512 rays of 1/8 mm along x, one in every second cell of a 16^3 unit grid,
    whose midpoints lie 2^-e short of the cell's far corner on every axis."""
    rng = np.random.default_rng(seed)
    k, j, i = (2 * a.ravel() for a in np.meshgrid(*[np.arange(8)] * 3, indexing="ij"))
    cell = np.stack([i, j, k], 1).astype(np.float64)
    short = 2.0 ** -rng.integers(*exponents, cell.shape)
    short[:, 0] += 0.0625  # the whole segment inside the cell
    middle = cell + 1.0 - short
    half = np.array([0.0625, 0.0, 0.0])
    return cell.astype(int), middle - half, middle + half


@pytest.mark.parametrize("mode", ["float32", "float64", "cell_gauss"])
def test_small_corner_sums_keep_sign_and_relative_accuracy(mode):
    """Corner weights down to the product of three distances 2^-e: the sums of a
    positive image are positive and accurate to their own size, not to that of
    the largest corner."""
    print(f"case walk corners {mode}", flush=True)
    grid = O.Grid((16, 16, 16), (1.0, 1.0, 1.0))
    cell, src, end = _corner_rays((4, 12) if mode == "float32" else (4, 24), 1)
    precision = "float32" if mode == "float32" else "float64"
    gpu = NativeScene(grid, 1, rays=(src, end), precision=precision,
                      extra_needs=_native.CELL_GAUSS if mode == "cell_gauss" else 0)
    actual, _, status = gpu.vjp(np.full(grid.voxels, 0.02, np.float32), np.ones(len(src)), pose_grad=False)
    assert not any(status)
    actual = actual.reshape(grid.shape).astype(np.float64)
    fraction = 0.5 * (src + end) - cell  # exact
    for corner in range(8):
        bits = [corner >> a & 1 for a in range(3)]
        weight = np.prod([fraction[:, a] if bits[a] else 1.0 - fraction[:, a] for a in range(3)], axis=0)
        at = cell + np.array(bits)
        got = actual[at[:, 2], at[:, 1], at[:, 0]]
        assert np.all(got >= 0.0), (corner, got.min())
        # three products, the factor and the gradient, rounded to 24 bits each
        np.testing.assert_allclose(got, 0.125 * weight, rtol=6 * 2.0 ** -24, atol=0, err_msg=str(bits))


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("samples", [2, 3, 8, 500])
def test_corner_sums_of_oblique_runs_stay_non_negative(samples, precision):
    """Runs from near one corner of a cell to near the opposite one, where the
    covariances cancel the products of the mean fractions."""
    print(f"case walk oblique runs S={samples} {precision}", flush=True)
    grid = O.Grid((16, 16, 16), (1.0, 1.0, 1.0))
    rng = np.random.default_rng(samples)
    cell = _corner_rays((4, 5), 0)[0].astype(np.float64)
    near = rng.integers(0, 2, cell.shape)
    slack = 2.0 ** -rng.integers(3, 13, (2, *cell.shape))
    src = cell + np.where(near, 1.0 - slack[0], slack[0])
    end = cell + np.where(near, slack[1], 1.0 - slack[1])
    gpu = NativeScene(grid, samples, rays=(src, end), precision=precision)
    actual, _, status = gpu.vjp(np.full(grid.voxels, 0.02, np.float32), np.ones(len(src)), pose_grad=False)
    assert not any(status)
    actual = actual.reshape(grid.shape).astype(np.float64)
    assert actual.min() >= 0.0
    at = (np.arange(samples) + 0.5)[:, None, None] / samples
    fraction = src + at * (end - src) - cell
    length = np.linalg.norm(end - src, axis=1)
    for corner in range(8):
        bits = [corner >> a & 1 for a in range(3)]
        weight = np.prod([fraction[..., a] if bits[a] else 1.0 - fraction[..., a] for a in range(3)], axis=0).mean(0)
        v = cell.astype(int) + np.array(bits)
        # FP32 rays: positions up to 16 at 2^-24 in origin and direction; the
        # covariances leave at least an eighth of the products at these slacks
        np.testing.assert_allclose(actual[v[:, 2], v[:, 1], v[:, 0]], length * weight, rtol=1e-6,
                                   atol=6e-7 if precision == "float32" else 1e-15, err_msg=str(bits))


@pytest.mark.parametrize("distance", [1e15, 3e16, 4e17])
def test_cell_gauss_pieces_that_do_not_advance_flag_the_view(distance):
    """Rays from so far away that neighbouring planes share a ray parameter (one
    ulp of it is 0.2, 7 and 90 grid samples): the volume adjoint alone reports
    what the image and the joint adjoint report."""
    print(f"case walk gauss progress {distance}", flush=True)
    grid = O.Grid((6, 7, 4000), (1.0, 1.0, 1.0))
    values = np.full(grid.voxels, 0.02, np.float32)
    rng = np.random.default_rng(3)
    for _ in range(12):
        y0, y1, z = rng.uniform(0.0, 6.0), rng.uniform(0.0, 6.0), rng.uniform(0.0, 5.0)
        rays = (np.array([[-distance, y0, z]]), np.array([[distance, y1, z]]))
        _, expected = O.Scene(grid, 7, rays=rays).forward(values, precision="fp64", integration="cell_gauss")
        assert bool(expected[0]) == (distance > 1e15)
        gpu = NativeScene(grid, 7, rays=rays, precision="float64", extra_needs=_native.CELL_GAUSS)
        for pose_grad in (False, True):
            _, _, status = gpu.vjp(values, np.ones(1), pose_grad=pose_grad)
            assert status.tolist() == expected.tolist(), (y0, y1, z, pose_grad)
