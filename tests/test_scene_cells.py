"""The integrand's sphere sets by cell (scenes.hpp: describe_cells, cell_word
and the lookups) give the same values as the plain loops over every sphere,
bit for bit, CPU only: the three sphere scenes over seeds and image sizes in
float and double, coordinates on cell and range edges and outside their ranges
(which take the groups), and hand-built scenes (a pinhole, a sphere around
the camera, spheres on the plane seen from far away, a sphere too large for
the tables)."""
import numpy as np
import pytest

from test_oracle_scene import F_EYE, F_LENS, F_PLANE, Scene
from test_scene_groups import _coords, _same


def _hold(orc, params, c, dim, cells=True):
    got, n = orc.eval_scene_cells(params, c, dim)
    assert (n > 0) == cells
    _same(orc.eval_scene(params, c, dim), got)
    c64 = c[:20000].astype(np.float64)
    _same(orc.eval_scene_f64(params, c64, dim), orc.eval_scene_cells(params, c64, dim, fp64=True)[0])


@pytest.mark.parametrize("kind,dim", [(2, 4), (3, 5), (4, 6)])
@pytest.mark.parametrize("seed,W,H", [(0, 1920.0, 1080.0), (1, 3840.0, 2160.0), (7, 64.0, 48.0), (12345, 333.0, 517.0)])
def test_cells_equal_plain(orc, kind, dim, seed, W, H):
    params = orc.make_scene(kind, seed, dim, W, H)
    rng = np.random.default_rng(100 * kind + seed)
    c = _coords(rng, 300000, dim, W, H)
    n = len(c) // 10
    # image positions on cell edges and their neighbours, shutter bin edges
    e = rng.integers(0, 65, (n, 2)) / 64.0 * (W, H)
    c[-n:, :2] = np.nextafter(e.astype(np.float32), rng.choice([-1, 0, 1, 1e9], (n, 2)).astype(np.float32)).clip(0, [W, H])
    c[-n:, 2:] = np.where(rng.random((n, dim - 2)) < 0.5, rng.integers(0, 5, (n, dim - 2)) / 4.0, c[-n:, 2:])
    # outside the ranges
    m = n // 4
    d = rng.integers(0, min(dim, 5), m)
    c[np.arange(m), d] = rng.choice([-0.25, -1e-6, 1.0000001, 1.5], m).astype(np.float32) * np.where(d == 0, W, np.where(d == 1, H, 1))
    if kind == 4:
        c[:m, 2:] = c[:m, 2:].clip(-0.2, 1.2)
    _hold(orc, params, c, dim)


def test_cells_hand_built_scenes(orc):
    rng = np.random.default_rng(6)
    rows = [[0.0, 0.0, 6.0, 1.0, 0.3, -0.2, 0.1, 0.2, 0.4, 0.6]]
    for lens in (0.05, 0.0, 0.4):
        s = Scene(orc, 3, 5)
        s.f[F_LENS] = lens
        # the second sphere holds the camera, the third passes close by it
        s.objects(rows + [[0.0, 0.1, 0.2, 0.5, 0, 0, 0, 1, 0, 0], [0.3, 0, 0.6, 0.2, -0.2, 0.1, -0.3, 0, 1, 0]])
        _hold(orc, bytes(s.buf), _coords(rng, 50000, 5, 1.0, 1.0), 5)
        s = Scene(orc, 2, 4)
        s.f[F_LENS] = lens
        s.objects(rows)  # moving, but this scene traces at t = 0
        _hold(orc, bytes(s.buf), _coords(rng, 50000, 4, 1.0, 1.0), 4)
    # the camera low over the plane and far away: shadow and occlusion rays
    # start far out on it
    s = Scene(orc, 3, 5, seed=3)
    plane = float(s.f[F_PLANE])
    s.f[F_EYE:F_EYE + 3] = (0.0, plane + 0.01, -50.0)
    c = _coords(rng, 50000, 5, 1.0, 1.0)
    c[:, 1] *= np.float32(0.5)
    _hold(orc, bytes(s.buf), c, 5)
    # small spheres and grazing hits: normals far from unit length
    s = Scene(orc, 4, 6)
    s.objects([[float(x), float(y), float(z), 0.01, 0, 0, 0, 1, 1, 1]
               for x, y, z in rng.uniform(-0.2, 0.2, (256, 3)) + (0, 0, -6)])
    c = _coords(rng, 100000, 6, 1.0, 1.0)
    c[:, :2] = 0.5 + (c[:, :2] - 0.5) * np.float32(0.1)
    _hold(orc, bytes(s.buf), c, 6)
    # too large for the tables
    s = Scene(orc, 4, 6)
    s.objects([[0.0, 1e4, 0.0, 1e4, 0, 0, 0, 1, 1, 1]])
    _hold(orc, bytes(s.buf), _coords(rng, 20000, 6, 1.0, 1.0), 6, cells=False)


def test_division_by_the_series_constants(orc):
    """The lens map's series and the Halton points divide by whole numbers
    with two fused operations on the GPU: the value of a division for squares of
    32-bit and 64-bit angles, mantissas next to powers of two and to
    multiples of the constants."""
    rng = np.random.default_rng(8)
    f = rng.uniform(0, np.pi / 4, 400000)
    x = [f ** 2, f.astype(np.float32).astype(np.float64) ** 2, np.exp(rng.uniform(-300, 0, 400000)), [0.0]]
    near = np.concatenate([np.ldexp(1.0, -np.arange(0, 900)), rng.integers(1, 1 << 50, 20000) * 342.0 / 2.0 ** 70,
                           rng.integers(1, 1 << 50, 20000) * 171.5 / 2.0 ** 70])
    x += [near, np.nextafter(near, 0), np.nextafter(near, 1e9)]
    assert orc.div_by_mismatches(np.concatenate(x)) == 0
