"""Counts of the reconstruction's geometry (recon_geo.hpp) on the CPU, where
their tables need not exist: tiles of one pixel along an axis of up to 65535
make tables of 2^32 entries, every one of which has to be cleared."""
import numpy as np
import pytest


@pytest.mark.parametrize("size,tile", [((1, 1), (8, 8)), ((1920, 1080), (8, 8)), ((64, 32768), (64, 1)),
                                       ((64, 32769), (64, 1)), ((64, 40000), (16, 1)), ((40000, 64), (1, 16)),
                                       ((65535, 16), (1, 64)), ((65535, 32767), (8, 8))])
def test_every_tile_range_is_cleared(orc, size, tile):
    axis = max(-(-size[0] // tile[0]), -(-size[1] // tile[1]))
    n = orc.tile_entries(*size, *tile)
    assert n == 4 ** (axis - 1).bit_length()
    for threads in (256, 24 * 256, 4096 * 256):
        for tid in {0, 1, threads - 1, (n - 1) % threads}:
            first, last, count = orc.entries_of_thread(n, tid, threads)
            want = len(range(tid, n, threads))
            assert count == want
            if want:
                assert (first, last) == (tid, tid + (want - 1) * threads)
        assert orc.entries_of_thread(n, (n - 1) % threads, threads)[1] == n - 1


@pytest.mark.parametrize("size,tile,scale", [((75, 50), (8, 8), (75.0, 50.0)), ((201, 33), (4, 16), (1.0, 1.0)),
                                             ((64, 300), (64, 1), (64.0, 300.0)), ((17, 16), (1, 16), (2.0, 1.0))])
def test_a_box_touches_the_images_tiles_only(orc, size, tile, scale):
    """Boxes that begin or end outside the image (an uploaded state's may)."""
    (W, H), (TW, TH), (sx, sy) = size, tile, scale
    r = np.random.default_rng(W)
    n = 20000
    step = np.float32([sx / W, sy / H])
    lo = np.float32([-0.1, -0.1]) * (sx, sy) - 9 * TW * step * (r.random((n, 1)) < 0.3) * r.random((n, 2))
    mn = np.float32(lo + r.random((n, 2)) * 1.3 * (sx, sy))
    mx = np.float32(mn + r.random((n, 2)) ** 4 * (sx, sy))
    out, total = orc.box_tiles(W, H, sx, sy, TW, TH, np.stack([mn[:, 0], mx[:, 0], mn[:, 1], mx[:, 1]], 1))
    hit = out[:, 0] >= 0
    assert np.array_equal(hit, np.all(out >= 0, 1))
    assert total == ((out[:, 1] - out[:, 0] + 1) * (out[:, 3] - out[:, 2] + 1))[hit].sum()
    assert np.all(out[hit][:, [0, 2]] <= out[hit][:, [1, 3]])
    assert np.all(out[hit][:, 1] < -(-W // TW)) and np.all(out[hit][:, 3] < -(-H // TH))
    # in 64 bits, a thousandth of a pixel apart: the tiles that the box's part
    # of the image meets
    px = np.float64([W / sx, H / sy])
    a, b = mn * px, mx * px
    inside = np.all((b > 1e-3) & (a < np.float64([W, H]) - 1e-3), 1)
    assert np.all(hit[inside]) and not np.any(hit[np.any((b < -1 - 1e-3) | (a > np.float64([W, H]) + 1e-3), 1)])
    first = np.maximum(a[inside] - 1e-3, 0) // (TW, TH)
    last = np.minimum(b[inside] + 1e-3, np.float64([W, H]) - 1e-3) // (TW, TH)
    assert np.all(out[inside][:, [0, 2]] >= first) and np.all(out[inside][:, [1, 3]] <= last)
    first = np.maximum(a[inside] + 1e-3, 0) // (TW, TH)
    last = np.clip(b[inside] - 1e-3, 0, np.float64([W, H]) - 1e-3) // (TW, TH)
    assert np.all(out[inside][:, [0, 2]] <= first) and np.all(out[inside][:, [1, 3]] >= last)


# dim, scene, b, e, sample space (None: the image's pixels)
@pytest.mark.parametrize("dim,kind,b,e,scale", [(3, 1, 0, 0, 1.0), (5, 3, 0, 0, 1.0), (6, 4, 1, 0, 1.0), (4, 2, 0, 2, 1.0),
                                                (5, 3, 0, 0, None), (5, 3, 1, 3, None), (3, 1, 0, 5, None)])
def test_expected_keys(orc, dim, kind, b, e, scale):
    """The sort is launched for the keys that the host expects of a tree: of
    the order of its keys, from a leaf on the whole image to a leaf per tile."""
    sx, sy = (scale, scale) if scale else (320.0, 180.0)
    params = orc.make_scene(kind, 3, dim, sx, sy)
    for n in (300, 3000, 30000):
        o = orc.OracleGrid(dim, 4 * n + (8 << (b * dim + 2 * e)), 4, b, e, 0.25, sx, sy)
        o.run(params, n)
        for size, tile in (((320, 180), (8, 8)), ((1920, 1080), (8, 8)), ((80, 45), (4, 4)), ((320, 180), (64, 1))):
            keys = len(o.recon_keys(*size, *tile))
            want, blocks = orc.expected_keys(*size, sx, sy, *tile, dim, b, e, o.n_leaves)
            assert want / 4 < keys < want * 4, (n, size, tile, o.n_leaves)
            # no workgroup has more than 8 tiles of 4096 keys, unless all 1024 are at work
            assert 1 <= blocks <= 1024 and (blocks == 1024 or keys <= blocks * 8 * 4096)
        o.close()
