"""The shape of a BM launch, a host calculation: what a caller or the autotuner
asks for is launched as asked at every size, and only what is left at 0 is chosen
by the number of blocks.  The autotuner's sample is in the same range of blocks
per CU as the table that it tunes."""
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


@pytest.mark.parametrize("stride", [1, 2, 4, 8, 1000])
@pytest.mark.parametrize("n", SIZES + [4096, 4097, 9001])
def test_the_autotuner_samples_in_the_range_of_its_table(n, stride):
    got = _lib().cm_bm_trial_stride(n, CUS, stride)
    assert 1 <= got <= stride
    sample = len(range(0, n, got))
    band = lambda k: sum(k > edge * CUS for edge in (1, 4, 8))
    assert band(sample) == band(n)
    for mode in (0, 1):
        assert _shape(sample, mode, 0, 0, 0) == _shape(n, mode, 0, 0, 0)
    if n <= 8 * CUS:
        assert sample == n
    elif got < stride:   # no larger stride would do
        assert len(range(0, n, got + 1)) <= 8 * CUS


def test_a_sampling_stride_needs_a_table():
    assert _lib().cm_bm_trial_stride(0, CUS, 4) == -3
    assert _lib().cm_bm_trial_stride(100, CUS, 0) == -3


@pytest.mark.gpu
def test_a_tuned_batch_is_launched_as_it_was_measured():
    """600 short blocks, between one and eight per CU: tried at the full count, and
    the shape found is the one launched, with the untuned launch's results."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import numpy as np
    from cochlearmodel_amd import solver
    from cochlearmodel_amd.uneven import UnevenBatch
    fs, n = 44100.0, 600
    rng = np.random.default_rng(5)
    sigs = [(0.1 * rng.standard_normal(int(fs * 0.0004 * (1 + k % 3)))).astype(np.float32) for k in range(n)]
    ub = UnevenBatch(sigs, np.ones((n, 256), np.float32), [8.0] * n, fs, block_s=0.002, overlap_s=0.0005)
    print(f"case: {ub.TB} blocks tuned with a stride of 4", flush=True)
    sc = solver.default_scalars(fs)
    ub.run_bm(sc, timed=False)
    torch.cuda.synchronize()
    want = ub.d_speeds.cpu().numpy().tobytes(), ub.d_stats.cpu().numpy().tobytes()
    try:
        tune = ub.autotune(sc, trial_stride=4)
        assert tune["n_trial_items"] == ub.TB
        asked = int(tune["waves_per_block"]), int(tune["jacobi_unroll"]), int(tune["sections_per_lane"])
        assert ub.waves_per_block == asked[0] and _shape(ub.TB, 0, *asked) == asked
        ub.run_bm(sc, timed=False)
        torch.cuda.synchronize()
        assert (ub.d_speeds.cpu().numpy().tobytes(), ub.d_stats.cpu().numpy().tobytes()) == want
    finally:
        ub.clear_order()
    assert ub.waves_per_block == 0
