"""Launches with nothing pinned, as users make them: the VOICE run against the
committed known answers, and batches either side of one, four and eight blocks per
CU (of 256) against the one-wave layout with sweeps in pairs.  Settings that a
test leaves pinned do not reach the next one."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))
import make_oracle_fixtures as G  # noqa: E402


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _pin(waves, unroll, sections):
    from cochlearmodel_amd import _lib
    L = _lib.lib()
    for rc in (L.cm_set_bm_launch(waves, 0), L.cm_set_bm_jacobi_unroll(unroll),
               L.cm_set_bm_sections_per_lane(sections)):
        _lib.check(rc)


def _golden_voice():
    from cochlearmodel_amd import solver
    fx = dict(np.load(os.path.join(HERE, "golden", "oracle_c1.npz"), allow_pickle=False))
    lay = solver.voice_layout(G.FS, 5, 0.02, 0.005)
    g = solver.run_bm_voice(fx["input"][:lay.bufP1], lay)
    v = g["speeds"][G.ROW0:G.ROW1]
    np.testing.assert_array_equal(v[::G.STRIDE_V], fx["o1_rows"])
    st = g["stats"]
    np.testing.assert_array_equal(np.stack([st["steps"], st["passes"], st["sweeps"]], 1), fx["o1_stats"])


@pytest.mark.parametrize("pinned", [None, (1, 1, 4), (1, 4, 1), (4, 2, 4)])
def test_voice_run(pinned):
    _cuda()
    print(f"case: golden VOICE run, 5 blocks, {pinned or 'nothing'} pinned", flush=True)
    if pinned:
        _pin(*pinned)   # left pinned for the next test
    _golden_voice()


@pytest.mark.parametrize("blocks", [1, 2])
def test_no_setting_outlives_a_test(blocks):
    """Each run leaves its launch order behind, which the library refuses for a
    table of another size."""
    _cuda()
    from cochlearmodel_amd import _lib, batch, solver
    print(f"case: {blocks} blocks, launch order left installed", flush=True)
    tb = batch.ToneBatch([1000.0], [40.0], 0.02 * blocks, with_lambda=False)
    assert tb.TB == blocks
    tb.generate_input()
    tb.run_bm(solver.default_scalars(FS), timed=False)
    order = np.arange(blocks, dtype=np.int32)
    _lib.check(_lib.lib().cm_set_bm_order(_lib.ptr(order), blocks))


@pytest.mark.parametrize("n", [250, 263, 1025, 2049])
@pytest.mark.parametrize("tol", [False, True])
def test_batches_by_size(n, tol):
    torch = _cuda()
    from cochlearmodel_amd import solver
    from cochlearmodel_amd.uneven import UnevenBatch
    rng = np.random.default_rng(n)
    sigs = [(0.1 * rng.standard_normal(int(FS * 0.0004 * (1 + k % 3)))).astype(np.float32) for k in range(n)]
    ub = UnevenBatch(sigs, np.ones((n, 256), np.float32), [8.0] * n, FS, block_s=0.002, overlap_s=0.0005)
    print(f"case: {ub.TB} blocks, tolerance {tol}", flush=True)
    sc = solver.default_scalars(FS)
    if tol:
        sc.jacobi_mode, sc.tol_rel, sc.check_every, sc.max_sweeps, sc.warm_start = 1, 1e-5, 4, 1000, 1
    got = []
    for pinned in (False, True):
        if pinned:
            _pin(1, 2, 4)
        ub.d_speeds.fill_(7.0)
        ub.run_bm(sc, timed=False, waves_per_block=1 if pinned else None)
        torch.cuda.synchronize()
        got.append((ub.d_speeds.cpu().numpy().tobytes(), ub.d_stats.cpu().numpy().tobytes()))
    assert got[0] == got[1]
