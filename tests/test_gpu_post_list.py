"""Each way the NaN fill lists its tiles, against the host sweep bit for bit: scanned and
listed by one kernel, listed by one kernel after a scan (tiles up to and past the
first 8192, whose flags a second round reads), and by four kernels.  Which way a
volume goes is worked out from the constants of the source, so that a change of the
tiles cannot leave one untested."""
import os
import re

import numpy as np
import pytest

import pseudoctimaging_amd as pct

pytestmark = pytest.mark.gpu

SRC = open(os.path.join(os.path.dirname(pct.__file__), "csrc", "pct_post.hip")).read()


def _const(name):
    v = re.search(r"\b%s = (\d+(?: << \d+)?)[,;]" % name, SRC).group(1)
    return eval(v)


def _list_path(interior):
    tz, tx, ty = (_const(c) for c in ("kTZ", "kTX", "kTY"))
    iz, ix, iy = interior
    ni, nj, nk = -(-iz // tz), (tz + ix - 2) // tx + 2, (tz + tx + iy - 3) // ty + 2
    tiles = ni * nj * nk
    j_end = tz * (ni - 1) // tx + nj
    diags = ni + j_end + (tz * (ni - 1) + tx * j_end) // ty + nk
    if diags > _const("kPlanDiags") or tiles > _const("kPlanTiles"):
        return "kernels"
    if tiles <= _const("kPlanScan"):
        return "one"
    return "scan" if tiles <= 8 * _const("kPlanThreads") else "scan, two rounds"


@pytest.mark.parametrize("interior,path", [((9, 40, 150), "one"), ((16, 40, 150), "scan"),
                                           ((100, 160, 200), "scan, two rounds"),
                                           ((2, 3, 70000), "kernels")])
def test_each_list_path(gpu, interior, path):
    import torch
    assert _list_path(interior) == path
    nh, lo = 3, 2
    shape = tuple(n + 2 * lo for n in interior)
    rng = np.random.default_rng(interior[0])
    inner = tuple(slice(lo, lo + n) for n in interior)
    for density in (0.0, 0.0005, 0.5):
        v = rng.normal(size=shape).astype(np.float32)
        v[inner][rng.random(interior) < density] = np.nan
        # the ends of the list: both corners and the last rows
        v[inner][0, 0, 0] = v[inner][-1, -1, -1] = np.nan
        v[inner][-1, -1, -20:] = np.nan
        dev = torch.from_numpy(v.copy()).cuda()
        pct.regularization_step_device(dev, nh)
        got = dev.cpu().numpy()
        pct.regularization_step(v, nh)
        assert np.array_equal(got.view(np.uint32), v.view(np.uint32)), density
