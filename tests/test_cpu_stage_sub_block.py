"""The wide stage kernels' sub-block (kst_stage_sub_block): of the shapes that a
256-thread workgroup holds the one that covers a tile in the fewest
workgroups, then with the smallest halo, then the widest."""
import ctypes

import pytest

from kestrel_amd import runtime


def sub_block(nx, ny):
    w, h = ctypes.c_int32(), ctypes.c_int32()
    assert runtime.lib().kst_stage_sub_block(nx, ny, ctypes.byref(w), ctypes.byref(h)) == 0
    return w.value, h.value


@pytest.mark.parametrize("tile,shape", [((32, 32), (16, 16)), ((50, 50), (25, 10)), ((40, 40), (20, 10)),
                                        ((25, 25), (25, 9)), ((24, 24), (24, 8)), ((20, 20), (20, 10)),
                                        ((16, 16), (16, 16)), ((4, 4), (4, 4)), ((9, 37), (9, 19))])
def test_shapes(tile, shape):
    assert sub_block(*tile) == shape


def test_best_of_the_shapes_that_fit():
    def fits(w, h):   # threads, faces, region, beds, halo cells
        return (w * h <= 256 and (w + 1) * h <= 288 and w * (h + 1) <= 288 and (w + 4) * (h + 4) <= 432
                and h * (w + 3) <= 352 and w * (h + 3) <= 352 and 4 * (w + h) <= 160)
    shapes = [(w, h) for w in range(4, 33) for h in range(4, 33) if fits(w, h)]
    for nx in [*range(4, 34), 50, 64, 100]:
        for ny in [*range(4, 34, 3), 50, 64, 100]:
            best = min((s for s in shapes if s[0] <= nx and s[1] <= ny),
                       key=lambda s: (-(-nx // s[0]) * -(-ny // s[1]), s[0] + s[1], -s[0]))
            assert sub_block(nx, ny) == best, (nx, ny)


def test_tiles_too_small_are_refused():
    w = ctypes.c_int32()
    assert runtime.lib().kst_stage_sub_block(3, 8, ctypes.byref(w), ctypes.byref(w)) != 0
