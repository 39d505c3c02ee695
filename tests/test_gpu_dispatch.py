"""How launches are laid over the chip: rows of tiles dealt to the XCDs in turn,
against the oracle where the last round of rows is partial and where blank rows
pad a view, and by time where a layout once left most XCDs idle.
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

POSE = scenes.compose(scenes.IDENTITY12, (0.5, -0.7, 0.3, 0.02, -0.015, 0.03))


# rows of tiles a view: 16 (a multiple of 8), 17, 9 and 33 of 16 pixels; 1 view
# alone, views below, at and above the eight of a contiguous run each
@pytest.mark.parametrize("views,rows", [(1, 270), (1, 521), (2, 256), (3, 137), (6, 40), (7, 64), (7, 51), (8, 64),
                                        (15, 33)])
@pytest.mark.parametrize("precision", ["float32", "float64"])
def test_rows_in_turn_match_the_oracle(views, rows, precision):
    print(f"case rows {views} x {rows} {precision}", flush=True)
    grid = O.Grid((21, 22, 25), (1.0, 0.9, 1.1), (-12.0, -10.0, -11.0))
    panels = scenes.cone_panels(grid, views, rows, 37, sod=120.0, sdd=200.0, offset=0.3)
    values = scenes.smooth_field(grid, 3)
    fp = "fp32" if precision == "float32" else "fp64"
    ref, gpu = O.Scene(grid, 41, panels=panels), NativeScene(grid, 41, panels=panels, precision=precision)
    expected, _ = ref.forward(values, POSE, precision=fp)
    actual, status = gpu.forward(values, POSE)
    assert not any(status)
    # every ray's own sum, in the oracle's order
    np.testing.assert_allclose(actual.ravel(), expected.ravel(), rtol=1e-6 if precision == "float32" else 1e-12,
                               atol=1e-7 if precision == "float32" else 1e-15)
    seeds = np.random.default_rng(5).uniform(-1.0, 1.0, expected.size).astype(actual.dtype)
    g_ref, p_ref, _, _ = ref.vjp(values, seeds, POSE, precision=fp)
    g_gpu, p_gpu, status = gpu.vjp(values, seeds, POSE)
    assert not any(status)
    # the bars of the parity tests: FP32 positions rounded by the oracle, and
    # FP32-rounded FP64 increments; FP64 sums over rays in another order
    assert _rel(g_gpu, g_ref) <= (1e-5 if precision == "float32" else 1e-7)
    assert _rel(p_gpu, p_ref) <= (1e-12 if precision == "float32" else 1e-10)


def _milliseconds(call, repeats=7):
    call()
    times = []
    for _ in range(repeats):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        call()
        end.record()
        end.synchronize()
        times.append(begin.elapsed_time(end))
    return min(times)


class Timed:
    """A scene of random density and its three launches."""

    def __init__(self, shape, views, rows, cols, samples, spacing=1.0, distances=(1000.0, 1500.0),
                 one_angle=False):
        origin = tuple(-(n - 1) * spacing / 2 for n in reversed(shape))
        self.grid = O.Grid(shape, (spacing,) * 3, origin)
        panels = scenes.cone_panels(self.grid, views, rows, cols, *distances, offset=0.1)
        panels = panels[:1] * views if one_angle else panels
        self.scene = NativeScene(self.grid, samples, panels=panels)
        generator = torch.Generator("cuda").manual_seed(1)
        self.field = 0.02 * torch.rand(shape, generator=generator, device="cuda")
        self.seeds = torch.rand((views, rows, cols), generator=generator, device="cuda") - 0.5
        self.image, self.volume = torch.empty_like(self.seeds), torch.empty_like(self.field)
        self.pose = torch.empty((views, 12), dtype=torch.float64, device="cuda")
        self.poses = self.scene._poses(POSE)

    def forward(self):
        self.scene.plan.forward(self.field.data_ptr(), self.poses.data_ptr(), self.image.data_ptr(), self.scene.stream)

    def vjp(self, flags):
        self.scene.plan.vjp(self.field.data_ptr(), self.poses.data_ptr(), self.seeds.data_ptr(),
                            self.volume.data_ptr() if flags & _native.VOLUME else None,
                            self.pose.data_ptr() if flags & _native.POSE else None, flags, self.scene.stream)


def test_fewer_views_take_no_longer():
    """10 views of 16 rows of tiles, of which the middle four meet the grid: dealt
    to the same four XCDs by every view they took 4.4 ms, where 16 views in
    contiguous runs take 1.7."""
    few, more = (Timed((139, 512, 512), views, 256, 256, 1024) for views in (10, 16))
    for call in (Timed.forward, lambda t: t.vjp(_native.POSE)):
        times = [_milliseconds(lambda: call(t)) for t in (few, more)]
        print(f"10 and 16 views: {times}", flush=True)
        assert times[0] <= 1.8 * times[1]


def test_few_samples_take_no_longer_than_more_rays():
    """One sample a ray: two 512^2 views with eight waves to set up each ray took
    58 us for the image and 134 us for the pose adjoint, where three views with
    one took 20 and 46."""
    few, more = (Timed((32, 32, 32), views, 512, 512, 1) for views in (2, 3))
    for call in (Timed.forward, lambda t: t.vjp(_native.POSE)):
        times = [_milliseconds(lambda: call(t), 15) for t in (few, more)]
        print(f"2 and 3 views, one sample: {times}", flush=True)
        assert times[0] <= 1.4 * times[1]


def test_views_that_share_cells_keep_a_workgroup():
    """2000 views of 16^2 a fifth of a degree apart: the four views of a workgroup
    share cells; a workgroup per wave tile took 0.33 ms of the pose adjoint, twice
    2080 views (above the split kernels' range)."""
    few, more = (Timed((32, 32, 32), views, 16, 16, 128) for views in (2000, 2080))
    times = [_milliseconds(lambda: t.vjp(_native.POSE), 15) for t in (few, more)]
    print(f"2000 and 2080 views: {times}", flush=True)
    assert times[0] <= 1.4 * times[1]


def test_views_at_one_angle_take_no_longer():
    """32 views of 48^2 and 1000 samples a ray fill a seventh of the chip's waves:
    at one angle, four views a workgroup, a lane per ray took 0.28 ms for the image
    and 0.39 for the pose adjoint, split 0.10 and 0.13."""
    few, more = (Timed((97, 181, 203), 32, 48, 48, 1000, one_angle=one) for one in (True, False))
    for call in (Timed.forward, lambda t: t.vjp(_native.POSE)):
        times = [_milliseconds(lambda: call(t), 15) for t in (few, more)]
        print(f"one angle and a circle: {times}", flush=True)
        assert times[0] <= 1.4 * times[1]


def test_fewer_rays_take_no_longer():
    """24 views over 192^3, pixels eight voxels apart (48^2) and 1.5 (256^2): with
    a slab of LDS for a handful of rays the sparse panels took 6.1 ms, the dense
    ones 1.8."""
    few, more = (Timed((192, 192, 192), 24, side, side, 48) for side in (48, 256))
    times = [_milliseconds(lambda: t.vjp(_native.VOLUME)) for t in (few, more)]
    print(f"48^2 and 256^2: {times}", flush=True)
    assert times[0] <= times[1]
