"""The batched search's cell buffers: the DP and MAP sweeps load eight floats
past a row's end and before its start, so each matrix needs that much of the
allocation to either side of it."""
import ctypes

import pytest

import cother_amd

REACH = 8 * 4  # bytes a sweep's load reaches outside a matrix


@pytest.mark.parametrize("do_map", [0, 1])
@pytest.mark.parametrize("cells", [64, 64 * 63, 64 * 1000, 64 * ((1 << 31) + 5)])
def test_room_to_either_side_of_the_matrices(cells, do_map):
    out = (ctypes.c_uint64 * 5)()
    fn = cother_amd.lib().cth_selftest_batch_cells
    fn.argtypes = [ctypes.c_uint64, ctypes.c_int, ctypes.POINTER(ctypes.c_uint64)]
    fn.restype = None
    fn(cells, do_map, out)
    btck, scores, mods, post, size = out
    parts = [(btck, cells), (scores, 4 * cells), (mods, 4 * cells)] + ([(post, 4 * cells)] if do_map else [])
    # in order, without overlap, within the allocation
    for (a, n), (b, _) in zip(parts, parts[1:]):
        assert a + n <= b
    assert sum(parts[-1]) <= size
    # the matrices the sweeps read: the scores, and with MAP the modular scores and posteriors
    for a, n in parts[1:] if do_map else parts[1:2]:
        assert a >= REACH and a + n + REACH <= size
