"""The gather's edge lines (quads of lanes, four samples a step) at the sizes
where their layout changes: the least axis that has lines (4), the step from two
to four band samples (16), axes that leave a line's last wave partly empty, and
sample counts that are no multiple of four: bit for bit the oracle's gather.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests import scenes

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from .test_gpu_gather import _gather  # noqa: E402
from .test_gpu_parity import NativeScene  # noqa: E402


@pytest.mark.parametrize("samples", [1, 30, 67])
@pytest.mark.parametrize("shape", [(4, 5, 6), (3, 9, 9), (15, 16, 18), (16, 16, 16), (17, 24, 33)])
def test_edge_lines_are_bitwise_the_oracle_gather(shape, samples):
    print(f"case gather edges {shape} S={samples}", flush=True)
    grid = O.Grid(shape, (1.0, 0.9, 1.1), tuple(-0.5 * (n - 1) * h for n, h in zip(shape[::-1], (1.0, 0.9, 1.1))))
    panels = scenes.cone_panels(grid, 4, 19, 23, sod=80.0, sdd=130.0, offset=0.3)
    pose = scenes.compose(scenes.IDENTITY12, (0.3, -0.4, 0.2, 0.02, -0.015, 0.03))
    gpu = NativeScene(grid, samples, panels=panels, precision="float64")
    seeds = np.random.default_rng(6).uniform(-1.0, 1.0, int(np.prod(gpu.shape)))
    expected, _ = O.Scene(grid, samples, panels=panels).gather(seeds, pose)
    actual, status = _gather(gpu, seeds, pose)
    assert not any(status)
    np.testing.assert_array_equal(actual.view(np.int64), expected.view(np.int64))
