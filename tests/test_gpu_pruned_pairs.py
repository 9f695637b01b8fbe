"""The pruned kernel's pair slabs: every window, both tile shapes, with one offset
per atlas that fits.

Atlas a is the image moved by an offset d_a, in uniform noise: the patch distance
is exactly zero at d_a, so its weight is exactly one, and at any other offset it
is so large that the weight underflows.  d_a has the smallest embedding distance
(zero), so it is kept, and lies off the sample lattice, so the mean sample weight
and with it the tail are zero: the fusion is the mean of the atlases' CT at d_a.
With whole-number CT the sums are exact and only the last division rounds."""
import numpy as np
import pytest

from pseudoctimaging_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape_id", [8, 13])
@pytest.mark.parametrize("nh", [5, 7, 9, 11, 13, 15])
@pytest.mark.parametrize("interior", [(1, 2, 3), (4, 17, 31)])
def test_one_fitting_offset_is_copied(gpu, interior, nh, shape_id):
    import torch
    hw = (nh - 1) // 2
    r = hw + 1
    shape = tuple(n + 2 * r for n in interior)
    rng = np.random.default_rng(100 * nh + shape_id)
    big = (rng.random(tuple(n + 2 * hw for n in shape)) * 1000.0).astype(np.float32)

    def part(d):   # the image at p - d, so that the atlas at p + d is the image at p
        return big[tuple(slice(hw - o, hw - o + n) for o, n in zip(d, shape))]

    # (z, x, y); never all of a lattice coordinate
    offsets = [(hw, -hw, hw - 1), (-hw, hw - 1, -hw), (1, -hw, hw)]
    img = np.ascontiguousarray(part((0, 0, 0)))
    amri = np.stack([part(d) for d in offsets])
    lab = rng.integers(0, 200, amri.shape).astype(np.float32)
    p = learned.mlp_init(1, *learned.intensity_stats(img))
    out = torch.full(shape, -3.0, device="cuda:0")
    print(f"case {interior} NH={nh} shape {shape_id}", flush=True)
    frac = learned.fuse_pruned_device(_dev(img), _dev(amri), _dev(lab), out, nh, 2.5, 1.0, p,
                                      topk=32, samples=27, margin=0.0, max_slabs=0,
                                      shape_id=shape_id, max_err=0.0)
    torch.cuda.synchronize()
    assert frac == 0.0
    got = out.cpu().numpy()[tuple(slice(r, n - r) for n in shape)]
    want = np.zeros(interior)
    for a, d in enumerate(offsets):
        want += lab[a][tuple(slice(r + o, n - r + o) for o, n in zip(d, shape))]
    want /= len(offsets)
    np.testing.assert_allclose(got, want, rtol=3 * 2.0 ** -24, atol=0)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
