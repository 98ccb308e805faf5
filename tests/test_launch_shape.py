"""The shape of a BM launch, a host calculation: what a caller or the autotuner
asks for is launched as asked at every size, and only what is left at 0 is chosen
by the number of blocks."""
import ctypes as C
import itertools
import os

import pytest

CUS = 256
SIZES = [1, 2, 256, 257, 300, 1000, 1024, 1025, 2000, 2048, 2049, 20480]


def _lib():
    from cochlearmodel_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    return _lib.lib()


def _shape(n, mode, waves, unroll, sections):
    s = [C.c_int(v) for v in (waves, unroll, sections)]
    assert _lib().cm_bm_launch_shape(n, CUS, mode, *(C.byref(v) for v in s)) == 0
    return tuple(v.value for v in s)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_what_is_asked_for_is_launched(n, mode):
    for asked in itertools.product((1, 2, 4), (1, 2, 4), (1, 2, 4)):
        assert _shape(n, mode, *asked) == asked
    for w in (1, 2, 4):
        assert _shape(n, mode, w, 0, 0)[0] == w


def test_what_is_left_open_follows_the_number_of_blocks():
    want = {1: (1, 4, 2), 256: (1, 4, 2), 257: (4, 4, 4), 1024: (4, 4, 4), 1025: (4, 2, 4), 2048: (4, 2, 4),
            2049: (1, 2, 4), 20480: (1, 2, 4)}
    for n, shape in want.items():
        assert _shape(n, 0, 0, 0, 0) == shape
    assert [_shape(n, 1, 0, 0, 0) for n in (1, 256, 257, 2048, 2049)] == [(1, 2, 4), (1, 2, 4), (4, 2, 4), (4, 2, 4),
                                                                          (1, 2, 4)]
    # a block over several waves is one workgroup
    assert _shape(1000, 0, 0, 0, 2)[0] == 1
    bad = [C.byref(C.c_int(0)) for _ in range(3)]
    assert _lib().cm_bm_launch_shape(-1, CUS, 0, *bad) == -3
