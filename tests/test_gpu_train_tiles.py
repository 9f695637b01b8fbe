"""The training gradient at the sizes where its 16-slot tiles and its waves end:
slot counts below, at and past a tile, anchors that share a tile (NH 1), one
wave and several workgroups, against the FP64 gradient.  NH 2 has eight offsets
for a window of one, so its slots leave the window and take the loads that
check the volume's bounds.

The bound: logits of up to about 100 carry FP32 errors of 6e-8 relative, 6e-6
absolute, into p and q, and the sums add roundings of the same size; 1e-4 of
the gradient's norm leaves a factor of ten."""
import numpy as np
import pytest

import mlp_ref
from pseudoctimaging_amd import api as pct
from pseudoctimaging_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,n_anchors", [(1, 1), (1, 7), (1, 8), (1, 9), (1, 200), (3, 1), (3, 4),
                                          (3, 5), (5, 9), (7, 21), (2, 1), (2, 16), (2, 33)])
def test_gradient_at_tile_edges(gpu, monkeypatch, nh, n_anchors):
    import torch
    nz, nx, ny, n = 24, 21, 19, 3
    img, amri, _ = pct.synth_tissue(nx, ny, nz, n, 2, False, 40 + nh)
    rng = np.random.default_rng(nh * 100 + n_anchors)
    mu, inv_sd = learned.intensity_stats(img)
    p = learned.mlp_init(3, mu, inv_sd)
    for lo, hi in ((learned.OFF_B1, learned.OFF_W2), (learned.OFF_B2, learned.OFF_W3),
                   (learned.OFF_B3, learned.OFF_MU)):
        p[lo:hi] = rng.normal(scale=0.1, size=hi - lo)
    r = (nh - 1) // 2 + 1
    z_end = nz - r
    if nh == 2:   # offsets (0 .. 7, 0, 0)
        z_end = nz - 8
        monkeypatch.setattr(mlp_ref, "_offsets",
                            lambda _: (np.arange(8), np.zeros(8, int), np.zeros(8, int)))
    anchors = np.stack([rng.integers(r, z_end, n_anchors), rng.integers(r, nx - r, n_anchors),
                        rng.integers(r, ny - r, n_anchors), rng.integers(0, n, n_anchors)], 1)
    loss, g = learned.mlp_loss_grad(torch.from_numpy(img).cuda(), torch.from_numpy(amri).cuda(),
                                    nh, 2.5, 1.0, p, anchors, 1.0, 0.5)
    loss64, g64 = mlp_ref.loss_grad(p, img, amri, [tuple(a) for a in anchors], nh, 0.5, 1.0)
    assert abs(loss - loss64) <= 1e-4 * abs(loss64) + 1e-6
    assert np.linalg.norm(g - g64) <= 1e-4 * np.linalg.norm(g64) + 1e-6
    assert np.all(g[30 * 64:2048] == 0) and np.all(g[7312:] == 0)
