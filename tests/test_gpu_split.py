"""Small problems split the window over work items, by dz and then by dy.  The default
configuration against the FP64 oracle and against one forced configuration
without a split, for every window at sizes below a tile, one tile and just past
it; host and device calls bit for bit.

The bounds: each of up to 3 * 15^3 weighted terms is summed in FP32 in some
order, a relative error of at most 2^-24 * 10125 = 6e-4 and about 2^-24 * 100 =
6e-6 when roundings are independent; 1e-4 is the bar of the other parity tests."""
import numpy as np
import pytest

import oracle
import pseudoctimaging_amd as pct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh", [3, 5, 7, 9, 11, 13, 15])
@pytest.mark.parametrize("interior", [(1, 1, 1), (2, 8, 30), (3, 9, 31), (5, 17, 61)])
@pytest.mark.parametrize("data,sigma", [("tissue", 2.5), ("tissue", 0.3), ("uniform", 2.5)])
def test_default_configuration_on_small_volumes(gpu, nh, interior, data, sigma):
    import torch
    r = (nh - 1) // 2 + 1
    nz, nx, ny = (n + 2 * r for n in interior)
    n = 1 + nh % 3
    if data == "tissue":
        img, amri, lab = pct.synth_tissue(nx, ny, nz, n, 2, False, nh)
    else:
        img, amri, lab = pct.synth_uniform(nx, ny, nz, n, nh)
    pct.normalize_labels(lab)
    ref = oracle.fuse(img, amri, lab, nh, sigma, 1.0)

    def run():
        d = [torch.from_numpy(a).cuda() for a in (img, amri, lab)]
        out = torch.full_like(d[0], -1.0)
        pct.fuse_device(*d, out, nh, sigma)
        return out.cpu().numpy()

    got = run()
    host = pct.multi_patch_based_segmentation_gpu(img, amri, lab, nh, sigma, 1.0)
    try:
        pct.force_tile_config(11, 1)
        whole = run()
    finally:
        pct.force_tile_config(-1, 0)
    nan = np.isnan(ref)
    for v in (got, whole):
        assert np.array_equal(np.isnan(v), nan)
        assert np.allclose(v[~nan], ref[~nan], rtol=1e-4, atol=1e-6)
    assert np.array_equal(got.view(np.uint32), host.view(np.uint32))
