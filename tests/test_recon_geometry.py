"""Counts of the reconstruction's geometry (recon_geo.hpp) on the CPU, where
their tables need not exist: tiles of one pixel along an axis of up to 65535
make tables of 2^32 entries, every one of which has to be cleared."""
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
