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
