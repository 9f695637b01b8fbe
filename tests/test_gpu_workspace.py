"""A window split over work items has a partial sum per part.  With a workspace that
does not hold them all the parts run in rounds, and every output keeps its bits:
the least workspace, one slot more, all but one, and all of them, for splits by dz and
by dy, both forms of the kernel, and slabs out of the cross-term range in a part."""
import ctypes

import numpy as np
import pytest

import oracle
import pseudoctimaging_amd as pct
from pseudoctimaging_amd import _lib
from parity import compare

pytestmark = pytest.mark.gpu


def _split(shape, n, nh, sigma):
    """The form and the number of parts of the configuration in use."""
    c = _lib.TileConfig()
    pb = pct.problem(shape, n, nh, sigma, 1.0)
    assert _lib.lib().pct_tile_config_choose(ctypes.byref(pb), ctypes.byref(c)) == 0
    c = c.as_dict()
    r = (nh - 1) // 2 + 1
    iz, ix, iy = (m - 2 * r for m in shape)
    tiles = -(-iz // c["bz"]) * -(-ix // (c["waves"] * (64 // c["seg_width"]) * c["bx"])) * \
        -(-iy // (c["seg_width"] - 2))
    if tiles <= 0:   # no interior
        return c["form"], 1
    assert c["items"] % (tiles * n) == 0
    return c["form"], c["items"] // (tiles * n)


# volume (z, x, y), atlases, NH, sigma, form, whether dy is split too
CASES = [((24, 31, 12), 4, 9, 0.3, 0, False), ((13, 16, 23), 1, 7, 2.5, 0, True),
         ((44, 25, 23), 1, 15, 2.5, 0, True), ((33, 82, 18), 9, 8, 2.5, 1, False),
         ((71, 73, 19), 2, 9, 2.5, 1, False), ((88, 46, 20), 2, 11, 2.5, 1, False),
         ((94, 40, 16), 1, 14, 2.5, 1, False), ((53, 33, 48), 1, 15, 2.5, 1, False)]


@pytest.mark.parametrize("spike", [False, True])
@pytest.mark.parametrize("shape,n,nh,sigma,form,dy", CASES)
def test_any_accepted_workspace_gives_the_same_bits(gpu, shape, n, nh, sigma, form, dy, spike):
    import torch
    used, parts = _split(shape, n, nh, sigma)
    assert used == form and parts > 1 and (parts > nh // 2 * 2 + 1) == dy
    nz, nx, ny = shape
    img, amri, lab = pct.synth_tissue(nx, ny, nz, n, 2, False, nh)
    pct.normalize_labels(lab)
    if spike:   # values out of the cross-term range: a few of an atlas, one of the target
        amri[n - 1, nz // 2, nx // 2 - 1:nx // 2 + 2, ny // 2] = 40.0
        img[nz // 2 - 2, nx - nx // 3, ny // 2] = 9.0
    d = [torch.from_numpy(a).cuda() for a in (img, amri, lab)]
    out = torch.full_like(d[0], -1.0)
    pct.fuse_device(*d, out, nh, sigma)
    compare(out.cpu().numpy(), oracle.fuse(img, amri, lab, nh, sigma, 1.0))

    L = _lib.lib()
    pb = pct.problem(shape, n, nh, sigma, 1.0)
    least = L.pct_fuse_workspace_size(ctypes.byref(pb), pct.CHOICE_SM)
    slot = 8 * n * img.size
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(nbytes):
        ws = torch.full((nbytes // 4 + 64,), float("nan"), device="cuda")
        got = torch.full_like(out, -2.0)
        rc = L.pct_fuse_dev_ws(ctypes.byref(pb), *(ctypes.c_void_p(t.data_ptr()) for t in d),
                               ctypes.c_void_p(got.data_ptr()), pct.CHOICE_SM,
                               ctypes.c_void_p(ws.data_ptr()), nbytes, stream)
        torch.cuda.synchronize()
        return rc, got

    for more in sorted({0, 1, 2, parts // 2, parts - 2, parts - 1, parts, 4 * parts}):
        rc, got = run(least + more * (slot + 256) // 256 * 256)
        assert rc == 0
        assert torch.equal(got.view(torch.int32), out.view(torch.int32)), more
    rc, got = run(least - 256)
    assert rc == _lib.PCT_ERR_INVALID and bool((got == -2.0).all())


# volume, atlases, NH of a call, and of one that is recorded in the workspace it left:
# more than whole windows' sums of the second, and less (but more than one sum)
@pytest.mark.parametrize("first,recorded", [(((48, 80, 96), 4, 3), ((60, 60, 60), 1, 15)),
                                            (((4, 60, 60), 1, 3), ((24, 31, 12), 4, 9))])
def test_graph_in_a_workspace_too_small_for_all_parts(gpu, first, recorded):
    """A recorded call cannot grow the library's workspace: it runs in what an earlier
    call left.  Later calls that outgrow it leave the graph its memory."""
    import torch

    def inputs(shape, n, nh):
        img, amri, lab = pct.synth_tissue(shape[1], shape[2], shape[0], n, 2, False, nh)
        pct.normalize_labels(lab)
        d = [torch.from_numpy(a).cuda() for a in (img, amri, lab)]
        return d, torch.full_like(d[0], -1.0)

    assert _split(*first, 2.5) == (0, 1)
    left = 8 * first[1] * int(np.prod(first[0]))
    form, parts = _split(*recorded, 2.5)
    volume = 8 * int(np.prod(recorded[0]))
    pairs = form * recorded[1] * volume
    assert volume + pairs < left < parts * recorded[1] * volume + pairs
    d1, o1 = inputs(*first)
    d2, o2 = inputs(*recorded)
    # the recorded problem's output, in a workspace of the test's own
    L = _lib.lib()
    pb = pct.problem(*recorded, 2.5, 1.0)
    nbytes = L.pct_fuse_workspace_size(ctypes.byref(pb), pct.CHOICE_SM)
    ws = torch.empty(nbytes // 4 + 64, device="cuda")
    want = torch.full_like(o2, -3.0)
    assert L.pct_fuse_dev_ws(ctypes.byref(pb), *(ctypes.c_void_p(t.data_ptr()) for t in d2),
                             ctypes.c_void_p(want.data_ptr()), pct.CHOICE_SM,
                             ctypes.c_void_p(ws.data_ptr()), nbytes,
                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    pct.release()
    pct.fuse_device(*d1, o1, first[2], 2.5)   # leaves a workspace between the two sizes
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pct.fuse_device(*d2, o2, recorded[2], 2.5)
    for replay in range(4):
        o2.fill_(-2.0)
        if replay == 2:   # outgrows the workspace; the next calls use the new one
            grown = torch.full_like(o2, -4.0)
            pct.fuse_device(*d2, grown, recorded[2], 2.5)
            pct.fuse_device(*d1, o1, first[2], 2.5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o2.view(torch.int32), want.view(torch.int32)), replay
    assert torch.equal(grown.view(torch.int32), want.view(torch.int32))
    del graph
    pct.release()
