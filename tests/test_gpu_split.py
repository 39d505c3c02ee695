"""Small FP32 launches sample a ray in several waves and add in one: images and
pose gradients carry the same bits as a large launch's one-lane march, at sample
counts around the rounds of 28 samples, for linear and copied gathers, FP32 and
16-bit storage, panels that are no multiple of a wave tile, and explicit rays.
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

GRID = O.Grid((21, 22, 25), (1.0, 0.9, 1.1), (-12.0, -10.0, -11.0))
FEW, MANY = 5, 620  # 620 views of 2 x 2 tiles: 9920 waves, above the 8192 of a small launch


@pytest.mark.parametrize("cells", [False, True])
@pytest.mark.parametrize("storage", ["float32", "bfloat16"])
@pytest.mark.parametrize("samples", [1, 3, 27, 28, 29, 57, 1000])
def test_small_and_large_launches_agree_bit_for_bit(samples, storage, cells):
    print(f"case split S={samples} {storage} cells={cells}", flush=True)
    few = scenes.cone_panels(GRID, FEW, 19, 27, sod=120.0, sdd=200.0, offset=0.3)
    many = [few[k % FEW] for k in range(MANY)]
    values = scenes.smooth_field(GRID, 3)
    pose = scenes.compose(scenes.IDENTITY12, (0.5, -0.7, 0.3, 0.02, -0.015, 0.03))
    needs = _native.GATHER_CELLS if cells else 0
    seeds = np.random.default_rng(4).uniform(-1.0, 1.0, (FEW, 19, 27)).astype(np.float32)
    out = {}
    for name, panels in (("few", few), ("many", many)):
        gpu = NativeScene(GRID, samples, panels=panels, storage=storage, extra_needs=needs)
        image, status = gpu.forward(values, pose)
        assert not any(status)
        _, grad, status = gpu.vjp(values, np.tile(seeds, (len(panels) // FEW, 1, 1)), pose, volume=False)
        assert not any(status)
        out[name] = image[:FEW], grad[:FEW]
    np.testing.assert_array_equal(out["few"][0].view(np.int32), out["many"][0].view(np.int32))
    np.testing.assert_array_equal(out["few"][1].view(np.int64), out["many"][1].view(np.int64))


@pytest.mark.parametrize("shape", [(1, 22, 25), (21, 1, 25), (21, 22, 1)])
def test_singleton_axes_match_the_oracle(shape):
    print(f"case split singleton {shape}", flush=True)
    grid = O.Grid(shape, (1.0, 0.9, 1.1), tuple(-0.5 * (n - 1) * h for n, h in zip(shape[::-1], (1.0, 0.9, 1.1))))
    panels = scenes.cone_panels(grid, 3, 17, 9, sod=120.0, sdd=200.0, offset=0.3)
    values = scenes.smooth_field(grid, 3)
    ref, gpu = O.Scene(grid, 61, panels=panels), NativeScene(grid, 61, panels=panels)
    expected, _ = ref.forward(values)
    actual, status = gpu.forward(values)
    assert not any(status)
    np.testing.assert_array_equal(actual.view(np.int32), expected.view(np.int32).reshape(actual.shape))
    seeds = np.random.default_rng(5).uniform(-1.0, 1.0, expected.size).astype(np.float32)
    _, p_ref, _, _ = ref.vjp(values, seeds, volume=False)
    _, p_gpu, _ = gpu.vjp(values, seeds, volume=False)
    # the same FP32 sums a ray; FP64 sums over rays in another order
    assert _rel(p_gpu, p_ref) <= 1e-12
