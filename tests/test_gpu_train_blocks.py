"""The gradient of many anchors, block by block (the weights and biases of each layer),
so that an error in a block with small entries shows.  40 anchors and the same 40 a
thousand times (1.1e6 slots, 35 tiles of 16 to each of 2048 waves) have one FP64
gradient: both are means over the anchors.

The bound: a wave's accumulators add 35 * 16 = 560 slots, a workgroup 8 waves, the last
pass 64 workgroups and 4 parts: 636 FP32 additions, 636 * 2^-24 = 4e-5 of the terms at
worst and sqrt(636) * 2^-24 = 1.5e-6 when roundings are independent; logits of up to 100
carry 6e-6 into every term.  1e-4 of the block's norm leaves room for terms of both
signs.  The last bias shifts all embeddings alike, so its gradient is zero and what is
left are roundings: 2e-6 of the whole gradient's norm, which every block is allowed."""
import numpy as np
import pytest

import mlp_ref
import pseudoctimaging_amd as pct
from pseudoctimaging_amd import learned

pytestmark = pytest.mark.gpu


def test_gradient_by_block(gpu):
    import torch
    nh, n = 3, 2
    img, amri, _ = pct.synth_tissue(24, 20, 18, n, 2, False, 5)
    dimg, dam = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (img, amri))
    p = learned.mlp_init(3, *learned.intensity_stats(img))
    rng = np.random.default_rng(1)
    few = np.stack([rng.integers(2, m - 2, 40) for m in img.shape] + [rng.integers(0, n, 40)], 1)
    loss64, g64 = mlp_ref.loss_grad(p, img, amri, [tuple(a) for a in few], nh, 0.5, 1.0)
    whole = np.linalg.norm(g64)
    L = learned
    blocks = {"W1": (0, 30 * 64), "b1": (L.OFF_B1, L.OFF_W2), "W2": (L.OFF_W2, L.OFF_B2),
              "b2": (L.OFF_B2, L.OFF_W3), "W3": (L.OFF_W3, L.OFF_B3), "b3": (L.OFF_B3, L.OFF_MU)}
    for repeat in (1, 1000):
        loss, g = learned.mlp_loss_grad(dimg, dam, nh, 2.5, 1.0, p, np.tile(few, (repeat, 1)),
                                        tau=1.0, teacher_t=0.5)
        assert abs(loss - loss64) <= 1e-4 * abs(loss64)
        for name, (lo, hi) in blocks.items():
            err = np.linalg.norm(g[lo:hi] - g64[lo:hi])
            assert err <= 1e-4 * np.linalg.norm(g64[lo:hi]) + 2e-6 * whole, (repeat, name)
