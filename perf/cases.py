"""The workloads whose speed this framework is measured by.

Each case is one call that a program makes in earnest: a fusion of one
subject (device tensors or host arrays), a batch of subjects, the
learned-pruned fusion, one evaluation of the embedding network's training
objective, and the NaN fill with rounding and HU rescale that follows a
fusion.  Sizes are those of the repository's tests and benchmark, and odd ones
between them.
"""
import math

import torch

import pseudoctimaging_amd as pct
from pseudoctimaging_amd import learned


def listed():
    return [
        # the smoke-test volume: one call's launches and host work
        {"name": "fuse_30x34x22_n2_nh7", "kind": "fuse", "nx": 30, "ny": 34, "nz": 22, "n": 2,
         "nh": 7, "sigma": 2.5, "data": "tissue"},
        # a region of interest with two atlases, too small to fill the chip
        {"name": "fuse_64x64x32_n2_nh7", "kind": "fuse", "nx": 64, "ny": 64, "nz": 32, "n": 2,
         "nh": 7, "sigma": 2.5, "data": "tissue"},
        # a whole head against one atlas
        {"name": "fuse_160x160x96_n1_nh7", "kind": "fuse", "nx": 160, "ny": 160, "nz": 96, "n": 1,
         "nh": 7, "sigma": 2.5, "data": "tissue"},
        # an odd-sized acquisition at the reference program's default sigma
        {"name": "fuse_181x149x83_n3_nh9", "kind": "fuse", "nx": 181, "ny": 149, "nz": 83, "n": 3,
         "nh": 9, "sigma": 1.0, "data": "tissue"},
        # selective weights (small sigma), a small window
        {"name": "fuse_128x128x64_n4_nh5_selective", "kind": "fuse", "nx": 128, "ny": 128,
         "nz": 64, "n": 4, "nh": 5, "sigma": 0.25, "data": "tissue"},
        # the reference program's random mode: every value 10 U[0, 1)
        {"name": "fuse_128x128x64_n10_nh7_random", "kind": "fuse", "nx": 128, "ny": 128, "nz": 64,
         "n": 10, "nh": 7, "sigma": 2.5, "data": "uniform"},
        # the headline: a whole head against ten atlases with the widest usual window
        {"name": "fuse_222x222x112_n10_nh11", "kind": "fuse", "nx": 222, "ny": 222, "nz": 112,
         "n": 10, "nh": 11, "sigma": 2.5, "data": "tissue"},
        # host arrays in and out, as the reference's wrapper is called
        {"name": "host_160x160x96_n4_nh7", "kind": "host", "nx": 160, "ny": 160, "nz": 96, "n": 4,
         "nh": 7, "sigma": 2.5, "data": "tissue"},
        # uneven subjects of a cohort in one call ("nx ny nz n nh" each)
        {"name": "batch_four_uneven", "kind": "batch", "sigma": 2.5, "data": "tissue",
         "subjects": "160 160 96 1 7, 128 128 64 10 7, 192 192 96 3 9, 96 112 64 2 11"},
        # the learned-pruned fusion of the headline volume
        {"name": "pruned_222x222x112_n10_nh11", "kind": "pruned", "nx": 222, "ny": 222, "nz": 112,
         "n": 10, "nh": 11, "sigma": 2.5, "data": "tissue"},
        # forward and backward of the embedding network, one training step's anchors
        {"name": "grad_96x96x64_n3_nh11_a256", "kind": "grad", "nx": 96, "ny": 96, "nz": 64, "n": 3,
         "nh": 11, "sigma": 2.5, "anchors": 256, "data": "tissue"},
        # the chain after a random-mode fusion with most weights exhausted: NaN fill,
        # rounding, HU rescale
        {"name": "post_222x222x112_nan76", "kind": "post", "nx": 222, "ny": 222, "nz": 112, "nh": 3,
         "nan": 0.76, "data": "uniform"},
    ]


#: candidate-voxel pairs of the largest listed fusion
_MOST_PAIRS = 210 * 210 * 100 * 10 * 11 ** 3


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pairs(c):
    r = (c["nh"] - 1) // 2 + 1
    v = 1
    for d in ("nx", "ny", "nz"):
        v *= max(0, c[d] - 2 * r)
    return v * c["n"] * c["nh"] ** 3


def _volume(rng, nh, most):
    """Dimensions from 24 voxels (or just above the window's border) to `most`."""
    lo = max(24, nh + 9)
    nx = _log_int(rng, lo, most)
    ny = min(most, max(lo, int(nx * rng.uniform(0.7, 1.4))))
    nz = min(128, max(lo, int(nx * rng.uniform(0.4, 0.9))))
    return {"nx": nx, "ny": ny, "nz": nz}


def _subject(rng, windows, most, limit):
    while True:
        nh = rng.choice(windows)
        c = {**_volume(rng, nh, most), "n": _log_int(rng, 1, 10), "nh": nh}
        if _pairs(c) <= limit:
            return c


def draw(rng):
    kind = rng.choice(["fuse"] * 7 + ["host", "batch", "pruned", "grad", "post", "post"])
    if kind in ("fuse", "host"):
        c = _subject(rng, [3, 5, 7, 7, 9, 9, 11, 11, 13, 15], 256,
                     _MOST_PAIRS if kind == "fuse" else _MOST_PAIRS // 20)
        data = rng.choice(["tissue"] * 4 + ["uniform"])
        sigma = 2.5 if data == "uniform" else rng.choice([0.25, 0.5, 1.0, 2.5, 2.5])
        return {"kind": kind, **c, "sigma": sigma, "data": data}
    if kind == "batch":
        subs = [_subject(rng, [5, 7, 9, 11], 192, _MOST_PAIRS // 8)
                for _ in range(rng.randint(2, 6))]
        return {"kind": kind, "sigma": rng.choice([1.0, 2.5]), "data": "tissue",
                "subjects": ", ".join("%d %d %d %d %d" % (s["nx"], s["ny"], s["nz"], s["n"],
                                                          s["nh"]) for s in subs)}
    if kind == "pruned":
        return {"kind": kind, **_subject(rng, [7, 9, 11], 222, _MOST_PAIRS), "sigma": 2.5,
                "data": "tissue"}
    if kind == "grad":
        c = {**_volume(rng, 11, 128), "n": rng.randint(1, 4), "nh": rng.choice([5, 7, 9, 11])}
        return {"kind": kind, **c, "sigma": 2.5, "anchors": _log_int(rng, 16, 300),
                "data": "tissue"}
    return {"kind": kind, **_volume(rng, 11, 222), "nh": rng.choice([3, 5, 7, 9, 11]),
            "nan": round(math.exp(rng.uniform(math.log(0.002), math.log(0.8))), 4),
            "data": rng.choice(["tissue", "uniform"])}


# ---- inputs ------------------------------------------------------------------

def _smooth(v):
    """Three passes of a 5^3 box filter: correlation lengths of a few voxels."""
    v = v[None, None]
    for _ in range(3):
        v = torch.nn.functional.avg_pool3d(
            torch.nn.functional.pad(v, (2,) * 6, mode="replicate"), 5, stride=1)
    return v[0, 0]


def _tissue(g, nx, ny, nz, n, max_shift=3):
    """A target of four tissue classes (air, fat, soft tissue, bone) with noise, and atlases
    whose anatomy is the target's, displaced by a few voxels, each with noise of its own."""
    dev = "cuda"
    m = max_shift
    field = _smooth(torch.randn((nz + 2 * m, nx + 2 * m, ny + 2 * m), generator=g, device=dev))
    field = (field - field.mean()) / field.std()
    cls = (field > -0.6745).long() + (field > 0).long() + (field > 0.6745).long()
    mri = torch.tensor([0.0, 0.8, 0.5, 0.2], device=dev)
    ct = torch.tensor([-1000.0, -100.0, 40.0, 1000.0], device=dev)

    def view(dz, dx, dy):
        return cls[m + dz:m + dz + nz, m + dx:m + dx + nx, m + dy:m + dy + ny]

    def noise(sd):
        return sd * torch.randn((nz, nx, ny), generator=g, device=dev)

    img = (mri[view(0, 0, 0)] + noise(0.03)).contiguous()
    shifts = torch.randint(-m, m + 1, (n, 3), generator=g, device=dev).tolist()
    atlas = torch.empty((n, nz, nx, ny), device=dev)
    label = torch.empty((n, nz, nx, ny), device=dev)
    for a, s in enumerate(shifts):
        atlas[a] = mri[view(*s)] + noise(0.03)
        label[a] = ct[view(*s)] + noise(20.0)
    return img, atlas, label


def _inputs(case, nx, ny, nz, n, g):
    """Target, atlas MRI and atlas CT normalised to [0, 255]."""
    if case["data"] == "uniform":
        img = 10 * torch.rand((nz, nx, ny), generator=g, device="cuda")
        atlas = 10 * torch.rand((n, nz, nx, ny), generator=g, device="cuda")
        label = 10 * torch.rand((n, nz, nx, ny), generator=g, device="cuda")
    else:
        img, atlas, label = _tissue(g, nx, ny, nz, n)
    label = 255.0 * ((label + 1024.0) / 4095.0)
    return img, atlas, label


def _subjects(case):
    return [tuple(int(v) for v in s.split()) for s in case["subjects"].split(",")]


def _anchors(case, g):
    r = (case["nh"] - 1) // 2 + 1
    cols = [torch.randint(r, case[d] - r, (case["anchors"],), generator=g, device="cuda")
            for d in ("nz", "nx", "ny")]
    cols.append(torch.randint(0, case["n"], (case["anchors"],), generator=g, device="cuda"))
    return torch.stack(cols, 1).int().cpu().numpy()


def _network(img, seed):
    return learned.mlp_init(seed, float(img.double().mean()), 1.0 / float(img.double().std()))


def _holes(case, g):
    """A fused volume (zero border, values of the CT scale inside) in which a share of the
    interior voxels is NaN: patches where a smooth field is low, and single voxels."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    r = (case["nh"] - 1) // 2 + 1
    if case["data"] == "uniform":
        vol = 60.0 + 5.0 * torch.rand((nz, nx, ny), generator=g, device="cuda")
        low = torch.rand((nz, nx, ny), generator=g, device="cuda")
    else:
        vol = _tissue(g, nx, ny, nz, 1)[2][0]
        vol = 255.0 * ((vol + 1024.0) / 4095.0)
        low = _smooth(torch.randn((nz, nx, ny), generator=g, device="cuda"))
        low = low + 0.3 * low.std() * torch.randn((nz, nx, ny), generator=g, device="cuda")
    k = max(1, int(case["nan"] * low.numel()))
    vol[low <= low.flatten().kthvalue(k).values] = float("nan")
    inside = torch.zeros_like(vol, dtype=torch.bool)
    inside[r:nz - r, r:nx - r, r:ny - r] = True
    return torch.where(inside, vol, torch.zeros_like(vol))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    if kind == "batch":
        subs = []
        for nx, ny, nz, n, nh in _subjects(case):
            img, atlas, label = _inputs(case, nx, ny, nz, n, g)
            subs.append({"img": img, "atlas": atlas, "label": label, "out": torch.empty_like(img),
                         "nh": nh, "sigma": case["sigma"], "beta": 1.0})
        return {"case": case, "subjects": subs}
    if kind == "post":
        holes = _holes(case, g)
        return {"case": case, "fused": holes, "out": torch.empty_like(holes)}
    img, atlas, label = _inputs(case, case["nx"], case["ny"], case["nz"], case["n"], g)
    if kind == "host":
        return {"case": case, "img": img.cpu().numpy(), "atlas": atlas.cpu().numpy(),
                "label": label.cpu().numpy()}
    s = {"case": case, "img": img, "atlas": atlas, "label": label, "out": torch.empty_like(img)}
    if kind in ("pruned", "grad"):
        s["params"] = _network(img, int(seed))
    if kind == "grad":
        s["anchors"] = _anchors(case, g)
    return s


# ---- one pass ----------------------------------------------------------------

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "fuse":
        pct.fuse_device(s["img"], s["atlas"], s["label"], s["out"], c["nh"], c["sigma"])
        return s["out"]
    if kind == "host":
        return pct.multi_patch_based_segmentation_gpu(s["img"], s["atlas"], s["label"], c["nh"],
                                                      c["sigma"])
    if kind == "batch":
        pct.fuse_batch(s["subjects"])
        return [x["out"] for x in s["subjects"]]
    if kind == "pruned":
        learned.fuse_pruned_device(s["img"], s["atlas"], s["label"], s["out"], c["nh"],
                                   c["sigma"], 1.0, s["params"], report_fallback=False)
        return s["out"]
    if kind == "grad":
        loss, grad = learned.mlp_loss_grad(s["img"], s["atlas"], c["nh"], c["sigma"], 1.0,
                                           s["params"], s["anchors"], tau=1.0, teacher_t=0.5)
        return {"loss": loss, "grad": grad}
    # the chain works in place: on a copy, as the fused volume is kept beside the HU volume
    s["out"].copy_(s["fused"])
    pct.postprocess_device(s["out"], c["nh"])
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------

def _fuse_work(nx, ny, nz, n, nh):
    """Volumes in and out once; per candidate and voxel the difference, its square, the
    separable 3x3x3 sum (two adds an axis), the weight and its two sums."""
    return {"bytes": 4 * nx * ny * nz * (2 + 2 * n),
            "flops": 12 * _pairs({"nx": nx, "ny": ny, "nz": nz, "n": n, "nh": nh})}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_fuse_work(*s) for s in _subjects(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    voxels = case["nx"] * case["ny"] * case["nz"]
    if kind in ("fuse", "host"):
        return _fuse_work(case["nx"], case["ny"], case["nz"], case["n"], case["nh"])
    if kind == "pruned":
        # 59 candidates (32 kept, 27 samples) a voxel and atlas, and the CT window sums
        r = (case["nh"] - 1) // 2 + 1
        inner = math.prod(max(0, case[d] - 2 * r) for d in ("nx", "ny", "nz"))
        return {"bytes": 4 * voxels * (2 + 2 * case["n"]),
                "flops": inner * case["n"] * (59 * 12 + 6)}
    if kind == "grad":
        # forward, and twice that for the gradients of inputs and weights; the patches once
        rows = case["anchors"] * (case["nh"] ** 3 + 1)
        macs = 30 * 64 + 64 * 64 + 64 * 16
        return {"bytes": 4 * (case["anchors"] * ((case["nh"] + 4) ** 3 + 125) + 2 * 7314),
                "flops": 6 * rows * macs}
    r = (case["nh"] - 1) // 2 + 1
    inner = math.prod(max(0, case[d] - 2 * r) for d in ("nx", "ny", "nz"))
    return {"bytes": 8 * voxels, "flops": 3 * voxels + case["nan"] * inner * 100}


# ---- 64-bit values -----------------------------------------------------------

def _exact_fuse(img, atlas, label, nh, sigma):
    """The fusion in float64: weighted mean over atlases and window offsets, NaN where the sums
    vanish, zero on the border."""
    hw = (nh - 1) // 2
    r = hw + 1
    nz, nx, ny = img.shape
    out = torch.zeros((nz, nx, ny), dtype=torch.float64, device=img.device)
    if min(nz, nx, ny) <= 2 * r:
        return out
    k = -1.0 / (2 * 27 * sigma * sigma)
    t = img.double()[hw:nz - hw, hw:nx - hw, hw:ny - hw]
    shape = (nz - 2 * r, nx - 2 * r, ny - 2 * r)
    P = torch.zeros(shape, dtype=torch.float64, device=img.device)
    S = torch.zeros_like(P)
    d = torch.empty_like(t)
    for a in range(atlas.shape[0]):
        A, L = atlas[a].double(), label[a].double()
        for dz in range(-hw, hw + 1):
            for dx in range(-hw, hw + 1):
                for dy in range(-hw, hw + 1):
                    torch.sub(t, A[hw + dz:nz - hw + dz, hw + dx:nx - hw + dx,
                                   hw + dy:ny - hw + dy], out=d)
                    e = d.square()
                    e = e[:, :, :-2] + e[:, :, 1:-1] + e[:, :, 2:]
                    e = e[:, :-2] + e[:, 1:-1] + e[:, 2:]
                    e = (e[:-2] + e[1:-1]).add_(e[2:]).mul_(k).exp_()
                    S += e
                    P.addcmul_(e, L[r + dz:nz - r + dz, r + dx:nx - r + dx, r + dy:ny - r + dy])
    eps = 2.0 ** -52
    v = torch.where((P.abs() > eps) & (S.abs() > eps), P / S, float("nan"))
    out[r:nz - r, r:nx - r, r:ny - r] = v
    return out


def _exact_grad(s):
    """Loss and gradient of the training objective in float64, by torch's autograd."""
    c = s["case"]
    img, atlas = s["img"].double(), s["atlas"].double()
    nz, nx, ny = img.shape
    hw = (c["nh"] - 1) // 2
    p = torch.tensor(s["params"], dtype=torch.float64, device=img.device)
    leaf = p[:learned.OFF_MU].clone().requires_grad_()
    mu, inv_sd = p[learned.OFF_MU], p[learned.OFF_SD]
    W1 = leaf[:learned.OFF_B1].view(32, 64)[:30]
    b1 = leaf[learned.OFF_B1:learned.OFF_W2]
    W2 = leaf[learned.OFF_W2:learned.OFF_B2].view(64, 64)
    b2 = leaf[learned.OFF_B2:learned.OFF_W3]
    W3 = leaf[learned.OFF_W3:learned.OFF_B3].view(64, 16)
    b3 = leaf[learned.OFF_B3:]

    def padded(v):
        return torch.nn.functional.pad((v - mu) * inv_sd, (1, 1, 1, 1, 1, 1))

    def embed(vol, z, x, y):
        f = [vol[z + 1 + dz, x + 1 + dx, y + 1 + dy]
             for dz in (-1, 0, 1) for dx in (-1, 0, 1) for dy in (-1, 0, 1)]
        f += [(vol[z + 1 + a, x + 1 + b, y + 1 + e] - vol[z + 1 - a, x + 1 - b, y + 1 - e]) / 2
              for a, b, e in ((1, 0, 0), (0, 1, 0), (0, 0, 1))]
        h = torch.relu(torch.stack(f, -1) @ W1 + b1)
        return torch.relu(h @ W2 + b2) @ W3 + b3

    off = torch.arange(-hw, hw + 1, device=img.device)
    oz, ox, oy = (v.reshape(-1) for v in torch.meshgrid(off, off, off, indexing="ij"))
    anchors = torch.tensor(s["anchors"], dtype=torch.int64, device=img.device)
    gi, ga = padded(img), [padded(v) for v in atlas]
    patch = [(a, b, e) for a in (-1, 0, 1) for b in (-1, 0, 1) for e in (-1, 0, 1)]
    loss, grad = 0.0, torch.zeros_like(leaf)
    for z, x, y, at in anchors.tolist():
        zz, xx, yy = z + oz, x + ox, y + oy
        ssd = sum((img[z + a, x + b, y + e] - atlas[at][zz + a, xx + b, yy + e]).square()
                  for a, b, e in patch)
        t = torch.tensor([z], device=img.device)
        eT = embed(gi, t, torch.tensor([x], device=img.device), torch.tensor([y], device=img.device))
        dist = (eT - embed(ga[at], zz, xx, yy)).square().sum(-1)
        logp = torch.log_softmax(-ssd / 0.5, 0)
        one = (logp.exp() * (logp - torch.log_softmax(-dist, 0))).sum() / len(anchors)
        grad += torch.autograd.grad(one, leaf)[0]
        loss += float(one.detach())
    full = torch.zeros_like(p)
    full[:learned.OFF_MU] = grad
    return {"loss": loss, "grad": full}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("pruned", "post"):
        # the pruned fusion has no closed value without its 16-bit selection; the post chain
        # gives whole numbers
        return None
    s = prepare(case, seed)
    if kind == "fuse":
        return _exact_fuse(s["img"], s["atlas"], s["label"], case["nh"], case["sigma"])
    if kind == "host":
        img, atlas, label = (torch.from_numpy(s[k]).cuda() for k in ("img", "atlas", "label"))
        return _exact_fuse(img, atlas, label, case["nh"], case["sigma"])
    if kind == "batch":
        return [_exact_fuse(x["img"], x["atlas"], x["label"], x["nh"], x["sigma"])
                for x in s["subjects"]]
    return _exact_grad(s)
