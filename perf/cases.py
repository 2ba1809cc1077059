"""The measured work of this framework: what a program that renders with the
adaptive sampler has it do, through the public entry points (pmdas_amd.kdgrid
and the C ABI behind it), from the smallest images to 1920x1080.

A case is a dict of plain values; `path` says which entry points a pass goes
through:

  run        KDGrid.Run to the sample target, Integrate, ConvertToBytes
             (optionally with the learned proposal scoring the leaves)
  preview    the step-by-step loop of an interactive viewer: SamplingPass,
             EvalNewSamples, Integrate, ConvertToBytes per frame
  integrate  reconstruction and byte conversion of a tree that is kept
  batch      many images advanced together and reconstructed (graph replay)
  collect    KDGrid.Run that gathers training rows for the learned proposal
  train      Mlp.train on collected rows
  qmc        the plain (non-adaptive) sampler's image, FP32 or FP64
"""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

import pmdas_amd
from pmdas_amd import _lib, kdgrid
from pmdas_amd._lib import check
from pmdas_amd.learned import extra_bits

DISKS = pmdas_amd.SCENE_DISKS_MB          # (x, y, t)
DOF = pmdas_amd.SCENE_SPHERES_DOF         # (x, y, u, v)
MBDOF = pmdas_amd.SCENE_SPHERES_MBDOF     # (x, y, t, u, v)
AO = pmdas_amd.SCENE_AO                   # (x, y, u, v, h1, h2)
DIM = {DISKS: 3, DOF: 4, MBDOF: 5, AO: 6}


def _run(name, kind, W, H, spp, b=1, alpha=0.25, cand=4, learned=False):
    return dict(name=name, path="run", kind=kind, W=W, H=H, spp=spp, b=b, alpha=alpha, cand=cand, learned=learned)


def listed():
    return [
        # a thumbnail, where launches and host round trips are all there is
        _run("run-5d-64x48", MBDOF, 64, 48, 8),
        # 3D motion-blurred disks at 256x256 (initial cells of whole pixels)
        _run("run-3d-disks-256", DISKS, 256, 256, 8, b=0),
        # an odd, portrait-format image with a flatter selection and 2 candidates
        _run("run-5d-odd-333x517", MBDOF, 333, 517, 16, alpha=0.125, cand=2),
        # 4D depth of field, 1920x1080, 16 spp (the benchmark's 4D line)
        _run("run-4d-dof-1080p", DOF, 1920, 1080, 16),
        # 5D motion blur + depth of field, 1920x1080, 32 spp (the headline)
        _run("run-5d-mbdof-1080p", MBDOF, 1920, 1080, 32),
        # 6D ambient occlusion with the network scoring the leaves, one
        # quarter-HD frame of the animation workload
        _run("run-6d-ao-learned-960x540", AO, 960, 540, 32, learned=True),
        # an interactive viewer: 12 frames of one pass each at 640x360
        dict(name="preview-5d-640x360", path="preview", kind=MBDOF, W=640, H=360, frames=12),
        # re-reconstruction of a finished 1080p tree into another resolution
        dict(name="integrate-5d-1280x719", path="integrate", kind=MBDOF, W=1920, H=1080, spp=16, out_W=1280, out_H=719),
        # eight images of uneven sizes in one batch
        dict(name="batch-8", path="batch", kind=MBDOF, images=8, p_lo=65536, p_hi=1048576, spp=16),
        # training rows from a small scene (the data gathering runs 200 of these)
        dict(name="collect-5d-160x90", path="collect", kind=MBDOF, W=160, H=90, spp=32),
        # four Adam steps on about the batch the training uses (65536 rows)
        dict(name="train-60k-rows", path="train", rows=60013, batch=65536, epochs=4),
        # FP64 ground truth of a small validation image
        dict(name="qmc-fp64-240x135", path="qmc", kind=MBDOF, W=240, H=135, spp=64, first=0, fp64=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, p_lo, p_hi):
    p = _log_uniform(rng, p_lo, p_hi)
    aspect = rng.uniform(0.6, 1.9)
    W = max(16, int(round(math.sqrt(p * aspect))))
    return W, max(16, int(round(p / W)))


def draw(rng):
    path = rng.choice(["run", "run", "run", "run", "preview", "integrate", "batch", "collect", "train", "qmc"])
    kind = rng.choice([DISKS, DOF, MBDOF, AO])
    if path == "run":
        learned = rng.random() < 0.25
        # samples in all stay below those of the largest listed run of the scene
        spp = rng.choice([6, 8, 12, 16, 24, 32])
        most = {DISKS: 24e6, DOF: 33e6, MBDOF: 50e6, AO: 14e6}[kind]
        W, H = _size(rng, 3072, min(2.0e6, most / spp))
        c = _run("", kind, W, H, spp, b=rng.choice([0, 1, 1]), alpha=rng.choice([0.25, 0.25, 0.125]),
                 cand=rng.choice([4, 4, 2, 8]), learned=learned)
        del c["name"]
        return c
    if path == "preview":
        W, H = _size(rng, 8192, 262144)
        return dict(path=path, kind=kind, W=W, H=H, frames=rng.randint(4, 14))
    if path == "integrate":
        W, H = _size(rng, 16384, 1.0e6)
        return dict(path=path, kind=kind, W=W, H=H, spp=rng.choice([8, 12, 16]),
                    out_W=max(16, int(W * rng.uniform(0.5, 1.5))), out_H=max(16, int(H * rng.uniform(0.5, 1.5))))
    if path == "batch":
        hi = _log_uniform(rng, 65536, 524288)
        return dict(path=path, kind=kind, images=rng.randint(2, 10), p_lo=max(4096, hi // 16), p_hi=hi,
                    spp=rng.choice([8, 12]))
    if path == "collect":
        W, H = _size(rng, 4096, 65536)
        return dict(path=path, kind=rng.choice([DOF, MBDOF, AO]), W=W, H=H, spp=rng.choice([8, 16, 32]))
    if path == "train":
        return dict(path=path, rows=_log_uniform(rng, 3000, 200000), batch=65536, epochs=rng.randint(1, 4))
    W, H = _size(rng, 8192, 131072)
    return dict(path="qmc", kind=kind, W=W, H=H, spp=rng.randint(4, 48), first=rng.choice([0, 64]),
                fp64=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs --
class _Memory:
    """A device range of a grid as something torch can view; the views keep
    the grid, which owns the range, alive."""

    def __init__(self, grid, ptr, shape):
        self.grid = grid
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(int(ptr), False), version=2)


def _view(grid, ptr, shape):
    return torch.as_tensor(_Memory(grid, ptr, shape), device="cuda")


def _network(seed):
    """A scoring network: the default initialisation with the feature scales
    the sampler's leaves have (log2 extents, counts, luminances, depth)."""
    m = kdgrid.Mlp(seed)
    p = m.params()
    mu = [-6.0] * 6 + [3.0, 0.4, 0.02, 0.3, 0.5, 4.0, -12.0, 0.0, -18.0, 5.0]
    sd = [3.0] * 6 + [0.7, 0.3, 0.04, 0.3, 0.3, 3.0, 6.0, 3.0, 6.0, 1.0]
    p[_lib.MLP_PARAMS:_lib.MLP_PARAMS + 16] = mu
    p[_lib.MLP_PARAMS + 16:] = [1.0 / s for s in sd]
    m.set_params(p)
    return m


def _grid(kind, W, H, spp, seed, b=1, alpha=0.25, cand=4):
    """Grid, scene and target as a program sets them up: about 4 initial
    samples per pixel and room for the passes' overshoot."""
    D = DIM[kind]
    e = extra_bits(W, H, D, b)
    target = spp * W * H
    cap = int(target * 1.5) + 4 * (1 << (b * D + 2 * e)) + 1024
    g = kdgrid.KDGrid(D, cap, cand, b, e, alpha, float(W), float(H))
    sc = kdgrid.Scene(kind, 1 + seed % 1000003, D, float(W), float(H))
    s = SimpleNamespace(grid=g, scene=sc, target=target, D=D)
    s.coords = _view(g, g.GetSampleCoordinates(), (cap, D))
    s.values = _view(g, g.GetSampleValues(), (cap, 3))
    return s


def _image(s, W, H):
    s.W, s.H = W, H
    s.pixels = torch.empty((H, W, 4), device="cuda")
    s.bytes = torch.empty((H, W, 4), dtype=torch.uint8, device="cuda")


def batch_sizes(case):
    """Image sizes of a batch: pixel counts evenly spaced in their logarithm,
    16:9 and its odd neighbours."""
    out = []
    for i in range(case["images"]):
        f = i / max(1, case["images"] - 1)
        p = math.exp(math.log(case["p_lo"]) * (1 - f) + math.log(case["p_hi"]) * f)
        W = int(math.sqrt(p * 16.0 / 9.0)) | (i & 1)
        out.append((W, max(16, int(p / W))))
    return out


def _training_set(case, seed):
    """Feature rows, labels and the parameters training starts from (uniform
    in +-1/sqrt(fan in), then the rows' mean and 1/deviation).  Rows and labels have the values that collection writes: log2 extents, 2..4 samples,
    luminances, depth, log2 errors."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = case["rows"]

    def u(lo, hi, k=1):
        return lo + (hi - lo) * torch.rand((n, k), device="cuda", generator=gen)

    ext = -torch.floor(u(0, 11, 2)) - 1
    oth = -torch.floor(u(0, 4, 3)) - 1
    cnt = torch.floor(u(2, 4.999))
    mean = u(0, 1)
    spread = u(0, 0.5) * (u(0, 1) < 0.6)
    lo, hi = (mean - spread).clamp(min=0), mean + spread
    depth = torch.floor(u(0, 12))
    vol = ext.sum(1, keepdim=True) + oth.sum(1, keepdim=True) + 21
    err = vol - 8 * u(0, 1) - 6 * (spread == 0)
    X = torch.cat([ext, oth, torch.zeros_like(vol), cnt, mean, spread * spread / 3, lo, hi, depth, err, err - vol, vol,
                   torch.full_like(vol, 5.0)], 1).contiguous()
    noise = torch.randn((n, 1), device="cuda", generator=gen)
    Y = (-1.5 - 4 * (spread == 0) + 2 * spread - 0.2 * depth + 2.5 * noise).clamp(-10, 0)[:, 0].contiguous()
    rng = np.random.default_rng(seed)
    p = np.zeros(_lib.MLP_FLOATS, np.float32)
    for at, count, fan in ((0, 1088, 16), (1088, 4225, 64)):
        p[at:at + count] = rng.uniform(-1, 1, count) / math.sqrt(fan)
    sd = X.double().std(0, unbiased=False)
    p[_lib.MLP_PARAMS:_lib.MLP_PARAMS + 16] = X.double().mean(0).float().cpu().numpy()
    p[_lib.MLP_PARAMS + 16:] = torch.where(sd > 1e-6, 1 / sd, 1.0).float().cpu().numpy()
    return X, Y, p


def prepare(case, seed):
    path = case["path"]
    if path == "train":
        X, Y, p0 = _training_set(case, seed)
        s = SimpleNamespace(X=X, Y=Y, p0=p0, mlp=kdgrid.Mlp(), seed=seed % 1000)
    elif path == "qmc":
        s = SimpleNamespace(scene=kdgrid.Scene(case["kind"], 1 + seed % 1000003, DIM[case["kind"]],
                                               float(case["W"]), float(case["H"])))
        s.out = torch.empty((case["H"], case["W"], 4), device="cuda",
                            dtype=torch.float64 if case["fp64"] else torch.float32)
        s.frame = seed % 4096
    elif path == "batch":
        s = SimpleNamespace(sizes=batch_sizes(case))
        s.members = [_grid(case["kind"], W, H, case["spp"], seed * 64 + i) for i, (W, H) in enumerate(s.sizes)]
        for m, (W, H) in zip(s.members, s.sizes):
            _image(m, W, H)
        s.batch = kdgrid.Batch([m.grid for m in s.members], [m.scene for m in s.members])
        s.targets = [m.target for m in s.members]
        s.ptrs = [m.pixels.data_ptr() for m in s.members]
    elif path == "preview":
        # room for every frame to select every leaf that the frames before made
        s = _grid(case["kind"], case["W"], case["H"], 64, seed)
        _image(s, case["W"], case["H"])
    elif path == "integrate":
        s = _grid(case["kind"], case["W"], case["H"], case["spp"], seed)
        s.grid.Run(s.scene, s.target)
        _image(s, case["out_W"], case["out_H"])
    elif path == "collect":
        s = _grid(case["kind"], case["W"], case["H"], case["spp"], seed)
        # a row per split, about a third of the samples after the initial grid
        s.cap = case["spp"] * case["W"] * case["H"] // 4
        s.rows = torch.zeros((s.cap, _lib.FEATURES), device="cuda")
        s.labels = torch.zeros((s.cap,), device="cuda")
    else:
        s = _grid(case["kind"], case["W"], case["H"], case["spp"], seed, case["b"], case["alpha"], case["cand"])
        _image(s, case["W"], case["H"])
        if case["learned"]:
            s.mlp = _network(seed % 4093)
            s.grid.set_learned(_lib.LEARN_SCORE, s.mlp)
            s.grid.set_learned_exponent(0.125)
    s.case = dict(case)
    return s


# ------------------------------------------------------------------- passes --
def _counts(s):
    return dict(samples=s.grid.GetNumberOfSamples(), leaves=s.grid.GetNumberOfNodes())


def _reconstruct(s):
    s.grid.Integrate(s.pixels.data_ptr(), s.W, s.H)
    s.grid.ConvertToBytes(s.pixels.data_ptr(), s.bytes.data_ptr(), s.W, s.H)
    return dict(image=s.pixels, bytes=s.bytes)


def run(s):
    case = s.case
    path = case["path"]
    if path == "run":
        passes = s.grid.Run(s.scene, s.target)
        # the samples asked for (the last pass overshoots the target)
        return dict(passes=passes, coords=s.coords[:s.target], values=s.values[:s.target], **_reconstruct(s), **_counts(s))
    if path == "preview":
        g = s.grid
        g.InitialSampling()
        g.EvalIntegrand(s.scene, 0, g.GetNumberOfSamples())
        for _ in range(case["frames"]):
            g.SamplingPass()
            g.EvalNewSamples(s.scene)
            out = _reconstruct(s)
        return dict(**out, **_counts(s))
    if path == "integrate":
        return _reconstruct(s)
    if path == "batch":
        s.batch.run(s.targets, use_graph=True)
        s.batch.integrate(s.ptrs, [w for w, _ in s.sizes], [h for _, h in s.sizes], use_graph=True)
        return [dict(image=m.pixels, samples=m.grid.GetNumberOfSamples(), leaves=m.grid.GetNumberOfNodes())
                for m in s.members]
    if path == "collect":
        s.grid.set_learned(_lib.LEARN_COLLECT, None, s.rows.data_ptr(), s.labels.data_ptr(), s.cap)
        passes = s.grid.Run(s.scene, s.target)
        return dict(passes=passes, rows=s.rows, labels=s.labels, offered=s.grid.learned_rows(), **_counts(s))
    if path == "train":
        s.mlp.set_params(s.p0)
        losses = s.mlp.train(SimpleNamespace(ptr=s.X.data_ptr()), SimpleNamespace(ptr=s.Y.data_ptr()), case["rows"],
                             case["epochs"], case["batch"], 1e-3, s.seed)
        return dict(params=s.mlp.params()[:_lib.MLP_PARAMS], losses=losses)
    check(_lib.load().mdas_render_qmc(s.scene.handle, case["W"], case["H"], case["spp"], case["first"],
                                      ctypes.c_uint32(s.frame), 1 if case["fp64"] else 0, s.out.data_ptr(), None))
    return s.out


def work(case):
    """Bytes and operations that a pass cannot do without: every sample's
    coordinates and value and every pixel written once; about 200 operations
    to shade a sample and the distances of its candidates."""
    path = case["path"]
    if path == "train":
        n = case["rows"] * case["epochs"]
        return dict(bytes=68.0 * n, flops=6.0 * 5184 * n)
    px = case.get("out_W", case.get("W", 0)) * case.get("out_H", case.get("H", 0))
    D = DIM[case["kind"]]
    if path == "qmc":
        return dict(bytes=px * (32.0 if case["fp64"] else 16.0), flops=200.0 * px * case["spp"])
    if path == "batch":
        px = sum(w * h for w, h in batch_sizes(case))
    if path == "integrate":
        n = case["W"] * case["H"] * case["spp"]  # the samples' values, and a box per 3 samples
        return dict(bytes=12.0 * n + 8.0 * D * n / 3 + 20.0 * px, flops=20.0 * n)
    spp = 4 + case["frames"] if path == "preview" else case["spp"]
    n = px * spp
    out = n / 3 * 68.0 if path == "collect" else 20.0 * px
    if path == "preview":
        out *= case["frames"]
    return dict(bytes=n * (4.0 * D + 12.0) + out, flops=n * (200.0 + 12.0 * case.get("cand", 4) * D))


# -------------------------------------------------------------- exact values --
# The adaptive paths have no 64-bit value of their own: every sample after the
# first pass is placed by comparisons of 32-bit errors with a 32-bit random
# stream, so a run in 64 bits is another run.
def exact(case, seed):
    if case["path"] == "qmc":
        return _exact_qmc(case, seed)
    if case["path"] == "train" and case["rows"] <= case["batch"]:
        return _exact_train(case, seed)
    return None


def _tea4(v0, v1):
    M = 0xFFFFFFFF
    s0 = 0
    for _ in range(4):
        s0 = (s0 + 0x9E3779B9) & M
        v0 = (v0 + (((v1 << 4) + 0xA341316C & M) ^ (v1 + s0 & M) ^ ((v1 >> 5) + 0xC8013EA4 & M))) & M
        v1 = (v1 + (((v0 << 4) + 0xAD90777D & M) ^ (v0 + s0 & M) ^ ((v0 >> 5) + 0x7E95761E & M))) & M
    return v0


def _scene_objects(kind, seed):
    """The seeded objects of a scene: rows of centre, radius, velocity, colour."""
    M = 0xFFFFFFFF
    v0, v1, s0 = seed & M, 0x5CE7E5, 0
    for _ in range(4):
        s0 = (s0 + 0x9E3779B9) & M
        v0 = (v0 + (((v1 << 4) + 0xA341316C & M) ^ (v1 + s0 & M) ^ ((v1 >> 5) + 0xC8013EA4 & M))) & M
        v1 = (v1 + (((v0 << 4) + 0xAD90777D & M) ^ (v0 + s0 & M) ^ ((v0 >> 5) + 0x7E95761E & M))) & M
    state = [v0]

    def u(lo=0.0, hi=1.0):
        state[0] = (1664525 * state[0] + 1013904223) & M
        r = np.float32(state[0] & 0xFFFFFF) / np.float32(16777216.0)
        return np.float32(lo) + (np.float32(hi) - np.float32(lo)) * r

    rows = []
    if kind == DISKS:
        for _ in range(16):
            rows.append([u(), u(), u(0.02, 0.1), u(-0.1, 0.1), u(-0.1, 0.1), u(), u(), u()])
    elif kind == AO:
        for _ in range(256):
            rows.append([u(-5, 5), u(-5, 5), u(-5, 5), u(0.1, 0.5), 0, 0, 0, 1, 1, 1])
    else:
        for _ in range(64):
            r = [u(-3, 3), u(-2, 2), u(3, 12), u(0.2, 0.8), u(-0.3, 0.3), u(-0.3, 0.3), u(-0.3, 0.3)]
            if kind == DOF:
                r[4:7] = [0, 0, 0]
            rows.append(r + [u(), u(), u()])
    return np.array(rows, dtype=np.float64)


def _disk(a, b):
    """Concentric map of the unit square onto the unit disk."""
    ox, oy = 2 * a - 1, 2 * b - 1
    wide = ox.abs() > oy.abs()
    r = torch.where(wide, ox, oy)
    q = torch.where(wide, oy / torch.where(wide, ox, 1.0), ox / torch.where(wide | (oy == 0), 1.0, oy)) * (math.pi / 4)
    th = torch.where(wide, q, math.pi / 2 - q)
    return r * torch.cos(th), r * torch.sin(th)


def _hits(o, d, objs, t, tmin, tmax):
    """Nearest sphere hit of each ray: distance (tmax on a miss) and index."""
    best = torch.full_like(d[0], tmax)
    idx = torch.full(d[0].shape, -2, dtype=torch.int64, device=d[0].device)
    for k, s in enumerate(objs):
        oc = [o[a] - (s[a] + s[4 + a] * t) for a in range(3)]
        b = sum(x * y for x, y in zip(oc, d))
        disc = b * b - (sum(x * x for x in oc) - s[3] * s[3])
        sq = disc.clamp(min=0).sqrt()
        th = torch.where(-b - sq > tmin, -b - sq, -b + sq)
        ok = (disc >= 0) & (th > tmin) & (th < best)
        best = torch.where(ok, th, best)
        idx = torch.where(ok, k, idx)
    return best, idx


def _shade(kind, objs, x, sx, sy):
    f32 = lambda v: float(np.float32(v))  # noqa: E731  (the scene's constants are 32-bit numbers)
    if kind == DISKS:
        u, v, t = x[0] / sx, x[1] / sy, x[2]
        col = [torch.zeros_like(u) for _ in range(3)]
        for s in objs:  # the highest index on top
            inside = (u - (s[0] + s[3] * t)) ** 2 + (v - (s[1] + s[4] * t)) ** 2 <= s[2] * s[2]
            col = [torch.where(inside, float(s[5 + c]), col[c]) for c in range(3)]
        return col
    ty = f32(0.41421356237)
    tx = float(np.float32(ty) * (np.float32(sx) / np.float32(sy)))
    eye_z = -12.0 if kind == AO else 0.0
    plane_y = -5.5 if kind == AO else -2.0
    lens = (x[3], x[4]) if kind == MBDOF else (x[2], x[3])
    t = x[2] if kind == MBDOF else torch.zeros_like(x[0])
    lx, ly = _disk(*lens)
    lx, ly = f32(0.05) * lx, f32(0.05) * ly
    dx, dy = 2 * (x[0] / sx) - 1, 2 * (x[1] / sy) - 1
    # the focus point lies at 5 / z along the unit direction, so z = 5 in the camera frame
    d = [5.0 * dx * tx - lx, 5.0 * dy * ty - ly, torch.full_like(dx, 5.0)]
    n = (d[0] ** 2 + d[1] ** 2 + d[2] ** 2).sqrt()
    d = [c / n for c in d]
    o = [lx, ly, torch.full_like(lx, eye_z)]
    th, idx = _hits(o, d, objs, t, 1e-3, 1e30)
    tp = torch.where(d[1] != 0, (plane_y - o[1]) / torch.where(d[1] != 0, d[1], 1.0), -1.0)
    plane = (tp > 1e-3) & (tp < th)
    th, idx = torch.where(plane, tp, th), torch.where(plane, -1, idx)
    miss = idx == -2
    th = torch.where(miss, 1.0, th)
    p = [o[a] + th * d[a] for a in range(3)]
    tab = torch.tensor(objs, device=th.device)[idx.clamp(min=0)]
    on = idx >= 0
    n = [torch.where(on, (p[a] - (tab[..., a] + tab[..., 4 + a] * t)) / tab[..., 3], 1.0 if a == 1 else 0.0)
         for a in range(3)]
    so = [p[a] + 1e-3 * n[a] for a in range(3)]
    if kind == AO:
        sign = torch.where(n[2] >= 0, 1.0, -1.0)
        a = -1 / (sign + n[2])
        b = n[0] * n[1] * a
        t1 = [1 + sign * n[0] * n[0] * a, sign * b, -sign * n[0]]
        t2 = [b, sign + n[1] * n[1] * a, -n[1]]
        hx, hy = _disk(x[4], x[5])
        hz = (1 - hx * hx - hy * hy).clamp(min=0).sqrt()
        w = [hx * t1[c] + hy * t2[c] + hz * n[c] for c in range(3)]
        hit = _hits(so, w, objs, t, 0.0, 1.0)[0] < 1.0
        q = torch.where(w[1] != 0, (plane_y - so[1]) / torch.where(w[1] != 0, w[1], 1.0), -1.0)
        hit |= (q > 0) & (q < 1.0)
        vis = torch.where(miss, 1.0, torch.where(hit, 0.0, 1.0))
        return [vis, vis, vis]
    light = [f32(-0.259160519), f32(0.863868415), f32(-0.431934208)]
    ndl = sum(n[c] * light[c] for c in range(3))
    dl = [torch.full_like(ndl, light[c]) for c in range(3)]
    lit = (ndl > 0) & (_hits(so, dl, objs, t, 0.0, 1e30)[0] >= 1e30)
    direct = torch.where(lit, ndl, 0.0)
    sky = 0.5 * (d[1] + 1)
    back = [1 - 0.5 * sky, 1 - 0.3 * sky, torch.ones_like(sky)]
    return [torch.where(miss, back[c], torch.where(on, tab[..., 7 + c], 0.5) *
                        (f32(0.1) + direct * f32([1.0, 0.95, 0.9][c]))) for c in range(3)]


def _exact_qmc(case, seed):
    """The Halton / Cranley-Patterson image in 64 bits."""
    kind, W, H = case["kind"], case["W"], case["H"]
    objs = _scene_objects(kind, 1 + seed % 1000003)
    pix = torch.arange(W * H, dtype=torch.int64, device="cuda")
    st = _tea4(pix, torch.full_like(pix, seed % 4096))
    off = []
    for _ in range(6):
        st = (1664525 * st + 1013904223) & 0xFFFFFFFF
        off.append((st & 0xFFFFFF).double() / 16777216.0)
    acc = [torch.zeros(W * H, dtype=torch.float64, device="cuda") for _ in range(3)]
    for s in range(case["first"], case["first"] + case["spp"]):
        x = []
        for d in range(DIM[kind]):
            base, r, f, j = (2, 3, 5, 7, 11, 13)[d], 0.0, 1.0, s
            while j > 0:
                f /= base
                r += f * (j % base)
                j //= base
            v = r + off[d]
            x.append(torch.where(v > 1, v - 1, v))
        x[0] = (pix % W + x[0]) * W / W
        x[1] = (pix // W + x[1]) * H / H
        acc = [a + c for a, c in zip(acc, _shade(kind, objs, x, float(W), float(H)))]
    img = torch.stack([a / case["spp"] for a in acc] + [torch.zeros_like(acc[0])], 1)
    return img.reshape(H, W, 4)


def _exact_train(case, seed):
    """Full-batch Adam on the 16 -> 64 -> 64 -> 1 network in 64 bits; weights,
    inputs and activations are rounded to bf16 where the network is defined
    to round them (gradients pass straight through)."""
    X, y, p0 = _training_set(case, seed)
    bf = lambda v: v.float().bfloat16().double()  # noqa: E731
    p = torch.tensor(p0, dtype=torch.float64, device="cuda")
    x = bf((X - p[5313:5329].float()) * p[5329:].float())
    y = y.double()
    p = p[:5313].clone()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    c0 = math.sqrt(2 / math.pi)

    def gelu(z):
        t = torch.tanh(c0 * (z + 0.044715 * z ** 3))
        return 0.5 * z * (1 + t), 0.5 * (1 + t) + 0.5 * z * (1 - t * t) * c0 * (1 + 3 * 0.044715 * z * z)

    losses = []
    for k in range(1, case["epochs"] + 1):
        W1, b1 = bf(p[:1024]).reshape(64, 16), p[1024:1088]
        W2, b2 = bf(p[1088:5184]).reshape(64, 64), p[5184:5248]
        w3, b3 = bf(p[5248:5312]), p[5312]
        a1, g1 = gelu(x @ W1.T + b1)
        a1 = bf(a1)
        a2, g2 = gelu(a1 @ W2.T + b2)
        a2 = bf(a2)
        diff = a2 @ w3 + b3 - y
        losses.append((diff * diff).mean())
        dy = diff * (2.0 / case["rows"])
        d2 = dy[:, None] * w3 * g2
        d1 = (d2 @ W2) * g1
        g = torch.cat([(d1.T @ x).reshape(-1), d1.sum(0), (d2.T @ a1).reshape(-1), d2.sum(0), dy @ a2, dy.sum()[None]])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** k)) / ((v / (1 - 0.999 ** k)).sqrt() + 1e-8)
    return dict(params=p, losses=torch.stack(losses))
