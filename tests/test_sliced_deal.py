"""How the sliced CSR kernel's blocks and slices are dealt to workgroups (csrc/sliced_deal.h).  Host only."""
import ctypes

import pytest

import selftest_lib


@pytest.mark.parametrize("places", [224, 256])
@pytest.mark.parametrize("n", [1, 64, 65, 300, 1000, 1025, 7000, 18000, 72000, 300000])
def test_every_slice_of_every_block_once(n, places):
    """Every slice of every block is some workgroup's, once; no workgroup has to wait for another's place; and the longest run is within what
    an equal share of the slices, and of the tiles that have to be built, would be, a tile for ten slices."""
    L = selftest_lib.lib()
    slices = (n + 63) // 64
    for blocks in list(range(1, 33)) + [47, 63, 64, 111, 112, 127, 128, 200, 223, 224, 225, 247, 248, 249, 255, 256, 257, 313, 448, 500, 512, 625, 1250, 4096]:
        out = (ctypes.c_longlong * 3)()
        assert L.tsvm_selftest_sliced_deal(n, blocks, places, out) == 0, (n, blocks)
        workgroups, most_slices, most_tiles = out
        assert min(places, blocks) <= workgroups <= places
        share = -(-slices * blocks // places)
        # (one more tile where a run begins within a block, and another where it ends within one)
        assert most_slices + 10 * most_tiles <= 1.1 * (share + 10 * (share // slices + 3)), (n, blocks, out[:])
