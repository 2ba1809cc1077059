"""Reconstruction of uploaded states that a run would not leave: trees that
do not cover the image, down to none at all."""
import numpy as np
import pytest

from oracle import pyoracle

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def mdas():
    import pmdas_amd
    from pmdas_amd import kdgrid
    pmdas_amd.load()
    return kdgrid


def _tree(dim, W, H, target, kind=1):
    """A grid's arguments and the state of an oracle's run on it."""
    args = (dim, 2 * target, 4, 0, 0, 0.25, float(W), float(H))
    o = pyoracle.OracleGrid(*args)
    o.run(pyoracle.make_scene(kind, 3, dim, float(W), float(H)), target)
    return args, o, o.state()


def _upload(g, st):
    g.upload_state(st["coords"], st["values"], st["idx"], st["box"], st["err"], st["seed"])


# 64 x 1 tiles of 40000 rows: tables of 2^32 tile ranges (16 GB each)
@pytest.mark.parametrize("size,tile", [((75, 50), (8, 8)), ((75, 50), (1, 16)), ((64, 40000), (64, 1))])
def test_tiles_without_a_leaf(mdas, size, tile):
    W, H = size
    _say(f"tiles without a leaf {size} {tile}")
    args, o, st = _tree(3, W, H, 2000)
    g = mdas.KDGrid(*args)
    g.set_recon_tile(*tile)
    upper = st["box"][:, 4] < 0.4 * H  # what ends in the image's first rows
    none = upper & False
    for keep in (~none, upper, none, ~upper):  # ranges of the tree before must not stay
        s = dict(st, **{k: st[k][keep] for k in ("idx", "box", "err", "seed")})
        o.set_state(s)
        _upload(g, s)
        want = o.integrate(W, H)
        assert np.array_equal(g.integrate_image(W, H).view(np.uint32), want.view(np.uint32)), keep.sum()
        assert (keep.sum() > 0) == bool(want.any())
    g.close()
    o.close()


def _overlaps_64(st, dim, W, H, sx, sy):
    """The image of kdgrid.cu:483-582 in 64 bits (sx, sy: the sample space)."""
    px = np.zeros((H, W, 3))
    val = np.where(st["idx"][..., None] >= 0, st["values"][np.maximum(st["idx"], 0)].astype(np.float64), 0.0)
    mean = val.sum(1) / (st["idx"] >= 0).sum(1)[:, None]
    box = st["box"].astype(np.float64)
    ext = box[:, dim:] - box[:, :dim]
    depth = ext[:, 2:].prod(1)  # volume over xy area
    ex, ey = (np.arange(n + 1) * s / n for n, s in ((W, sx), (H, sy)))
    for i in range(len(box)):
        ox = np.clip(np.minimum(ex[1:], box[i, dim]) - np.maximum(ex[:-1], box[i, 0]), 0, None)
        oy = np.clip(np.minimum(ey[1:], box[i, dim + 1]) - np.maximum(ey[:-1], box[i, 1]), 0, None)
        px += np.multiply.outer(np.multiply.outer(oy, ox) * depth[i], mean[i])
    return px * (W * H / (sx * sy))


@pytest.mark.parametrize("tile", [(8, 8), (4, 4), (64, 1), (1, 16)])
@pytest.mark.parametrize("off", [(-3.5, 0.0), (-6.25, -9.75), (-40.0, 2.5), (20.0, -11.0)])
def test_boxes_outside_the_image(mdas, tile, off):
    """Boxes moved off the image by some pixels, by both reconstructions."""
    W, H = 75, 50
    _say(f"boxes outside {tile} {off}")
    args, o, st = _tree(3, W, H, 2000)
    o.close()
    st["box"][:, 0::3] += np.float32(off[0])
    st["box"][:, 1::3] += np.float32(off[1])
    st["coords"][:, :2] += np.float32(off)
    g = mdas.KDGrid(*args)
    g.set_recon_tile(*tile)
    _upload(g, st)
    want = _overlaps_64(st, 3, W, H, W, H)
    # a pixel bound is a sum of at most 75 steps, each rounded below 75: within
    # 3.4e-4 pixels, an overlap within twice that; the depths of the leaves over
    # a point sum to 1 and a pixel has a few leaves side by side: 7 of them
    for scatter in (False, True):
        got = g.integrate_image(W, H, scatter=scatter)[..., :3]
        assert np.abs(got - want).max() < 5e-3 and want.max() > 0.1
    g.close()


@pytest.mark.parametrize("size", [(48, 32), (640, 360)])
def test_the_sorts_bytes(mdas, size):
    """The byte model of the sort's scan holds the counters that it had, those
    of the workgroups launched for the tree."""
    W, H = size
    g, sc = mdas.KDGrid(5, 40000, 4, 0, 2, 0.25, float(W), float(H)), mdas.Scene(3, 3, 5, float(W), float(H))
    g.set_timing(True)
    g.Run(sc, 20000)
    g.integrate_image(W, H)
    tiles = max(-(-W // 8), -(-H // 8))
    bits = 2 * (tiles - 1).bit_length()
    passes = -(-bits // 10)
    digit = max(4, -(-bits // passes))
    blocks = pyoracle.expected_keys(W, H, W, H, 8, 8, 5, 0, 2, g.GetNumberOfNodes())[1]
    assert g.kernel_stats()["k_rs_scan"][2] == 12.0 * 2 ** digit * blocks * passes
    g.close()
    sc.close()


def test_bytes_of_a_reconstruction_outlive_its_tree(mdas):
    """kernel_stats is of the last reconstruction, also once the grid has
    started over."""
    g, sc = mdas.KDGrid(3, 40000, 4, 0, 2, 0.25, 48.0, 32.0), mdas.Scene(1, 3, 3, 48.0, 32.0)
    g.set_timing(True)
    g.Run(sc, 20000)
    g.integrate_image(48, 32)
    before = g.kernel_stats()
    assert before["k_rs_hist"][2] == 8.0 * len(g.recon_keys()) * before["k_rs_hist"][0]
    g.InitialSampling()
    assert g.kernel_stats()["k_rs_hist"] == before["k_rs_hist"]
    g.close()
    sc.close()
