"""The tiled first sweep of the device NaN fill against the host sweep, bit for
bit, at the sizes where a tile ends (interiors of 1 to 9 planes, 7 to 17 rows,
15 to 33 columns, and long thin ones) and with the values a median can trip
over: both signed zeros, infinities of both signs, denormals, and regions with
nothing to fill from."""
import numpy as np
import pytest

import pseudoctimaging_amd as pct

pytestmark = pytest.mark.gpu

# interior extents (z, x, y)
SHAPES = [(1, 1, 1), (1, 7, 15), (3, 8, 16), (4, 9, 17), (5, 17, 33), (9, 6, 31), (70, 3, 5),
          (2, 90, 4), (3, 4, 130)]


def _volume(rng, shape, kind):
    v = rng.normal(size=shape).astype(np.float32)
    if kind == "zeros":
        v = rng.choice(np.array([0.0, -0.0, 1e-45, -1e-45, 1.0, -1.0], np.float32), shape)
    elif kind == "infinities":
        v = np.where(rng.random(shape) < 0.4,
                     rng.choice(np.array([np.inf, -np.inf], np.float32), shape), v)
    return np.ascontiguousarray(v.astype(np.float32))


@pytest.mark.parametrize("nh", [3, 5])
@pytest.mark.parametrize("kind", ["normal", "zeros", "infinities"])
@pytest.mark.parametrize("interior", SHAPES)
def test_tiled_fill_matches_host(gpu, interior, kind, nh):
    import torch
    lo = (nh - 1) // 2 + 1
    shape = tuple(n + 2 * lo for n in interior)
    rng = np.random.default_rng(hash((interior, nh)) % (1 << 31))
    for density in (0.02, 0.6, 1.0):
        v = _volume(rng, shape, kind)
        v[rng.random(shape) < density] = np.nan   # the border's NaN stay
        dev = torch.from_numpy(v.copy()).cuda()
        pct.regularization_step_device(dev, nh)
        got = dev.cpu().numpy()
        pct.regularization_step(v, nh)
        nan = np.isnan(v)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got.view(np.uint32)[~nan], v.view(np.uint32)[~nan])


# fewer than 256 tiles (one kernel scans and lists them), more (a scan kernel
# first), and more than 4096 diagonals (clear, scan, places and list as kernels)
@pytest.mark.parametrize("interior", [(9, 40, 150), (12, 40, 150), (2, 3, 70000)])
def test_tile_list_paths(gpu, interior):
    import torch
    nh, lo = 3, 2
    shape = tuple(n + 2 * lo for n in interior)
    rng = np.random.default_rng(interior[0])
    for density in (0.001, 0.5):
        v = rng.normal(size=shape).astype(np.float32)
        v[rng.random(shape) < density] = np.nan
        dev = torch.from_numpy(v.copy()).cuda()
        pct.regularization_step_device(dev, nh)
        got = dev.cpu().numpy()
        pct.regularization_step(v, nh)
        assert np.array_equal(got.view(np.uint32), v.view(np.uint32))
