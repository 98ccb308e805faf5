"""A time block spread over 4 or 8 waves against the one-wave layout, bit for bit,
where the waves' reach matters: 31 (2 sections per lane) and 15 (1 per lane)
sweeps between exchanges, fixed counts below, at and beyond it, none, odd ones,
tolerance checks as far apart, a cap on the sweeps, and one pass per step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
FIXED = [(20, 2), (31, 15), (32, 16), (0, 1), (47, 0), (64, 33)]
TOL = [(1, 1000, 0), (15, 1000, 1), (16, 1000, 0), (31, 1000, 1), (33, 70, 0), (64, 1000, 1), (4, 0x7fffffff, 0)]


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _batch():
    from cochlearmodel_amd.uneven import UnevenBatch
    rng = np.random.default_rng(3)
    sigs = [(0.2 * 10.0 ** k * rng.standard_normal(int(FS * s))).astype(np.float32)
            for k, s in zip((-4, 0, 1), (0.012, 0.021, 0.008))]
    ohc = [np.ones(256, np.float32), np.linspace(1, 0, 256, dtype=np.float32), np.full(256, 0.5, np.float32)]
    ihc = [8.0] * 3
    return UnevenBatch(sigs, ohc, ihc, FS)


def _run(torch, ub, sc, layout):
    from cochlearmodel_amd import _lib
    L = _lib.lib()
    _lib.check(L.cm_set_bm_sections_per_lane(layout) if layout else L.cm_reset_bm_sections_per_lane())
    ub.d_speeds.fill_(7.0)
    ub.run_bm(sc, timed=False)
    torch.cuda.synchronize()
    _lib.check(L.cm_reset_bm_sections_per_lane())
    return ub.d_speeds.cpu().numpy().tobytes(), ub.d_stats.cpu().numpy().tobytes()


def _same(torch, sc, what):
    ub = _batch()
    print(f"case: {ub.TB} blocks, {what}", flush=True)
    want = _run(torch, ub, sc, 4)
    for layout in (2, 1, 0):
        assert _run(torch, ub, sc, layout) == want, (what, layout)


@pytest.mark.parametrize("slow,fast", FIXED)
@pytest.mark.parametrize("unroll", [1, 2, 4])
def test_fixed_sweeps(slow, fast, unroll):
    torch = _cuda()
    from cochlearmodel_amd import _lib, solver
    sc = solver.default_scalars(FS)
    sc.j_slow, sc.j_fast = slow, fast
    _lib.check(_lib.lib().cm_set_bm_jacobi_unroll(unroll))
    try:
        _same(torch, sc, f"{slow} and {fast} sweeps, unroll {unroll}")
        sc.max_passes = 1
        _same(torch, sc, f"one pass of {slow} sweeps, unroll {unroll}")
    finally:
        _lib.check(_lib.lib().cm_set_bm_jacobi_unroll(2))


@pytest.mark.parametrize("every,most,guess", TOL)
def test_tolerance(every, most, guess):
    torch = _cuda()
    from cochlearmodel_amd import solver
    sc = solver.default_scalars(FS)
    sc.jacobi_mode, sc.tol_rel, sc.check_every, sc.max_sweeps, sc.warm_start = 1, 1e-5, every, most, guess
    _same(torch, sc, f"checks every {every}, at most {most}, warm start {guess}")


@pytest.mark.parametrize("n", [250, 263, 1025, 2049])
@pytest.mark.parametrize("tol", [False, True])
def test_launch_shapes_chosen_by_size(n, tol):
    """The shapes that the number of blocks selects (either side of one, four and
    eight blocks per CU, of 256) against one that is asked for."""
    torch = _cuda()
    from cochlearmodel_amd import _lib, solver
    from cochlearmodel_amd.uneven import UnevenBatch
    L = _lib.lib()
    rng = np.random.default_rng(n)
    sigs = [(0.1 * rng.standard_normal(int(FS * 0.0004 * (1 + k % 3)))).astype(np.float32) for k in range(n)]
    ub = UnevenBatch(sigs, np.ones((n, 256), np.float32), [8.0] * n, FS, block_s=0.002, overlap_s=0.0005)
    print(f"case: {ub.TB} blocks, tolerance {tol}", flush=True)
    sc = solver.default_scalars(FS)
    if tol:
        sc.jacobi_mode, sc.tol_rel, sc.check_every, sc.max_sweeps, sc.warm_start = 1, 1e-5, 4, 1000, 1
    order = np.arange(ub.TB, dtype=np.int32)[::-1].copy()
    got = []
    try:
        for asked in (False, True):
            if asked:
                _lib.check(L.cm_set_bm_sections_per_lane(4))
                _lib.check(L.cm_set_bm_jacobi_unroll(2))
            _lib.check(L.cm_set_bm_order(_lib.ptr(order), len(order)))
            ub.d_speeds.fill_(7.0)
            ub.run_bm(sc, timed=False, waves_per_block=2 if asked else 1)
            torch.cuda.synchronize()
            got.append((ub.d_speeds.cpu().numpy().tobytes(), ub.d_stats.cpu().numpy().tobytes()))
    finally:
        ub.clear_order()
    assert got[0] == got[1]
