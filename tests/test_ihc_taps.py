"""Tap counts of cm_ihc_lambda_run at their lower end: negative ones are refused on
the host, empty filters (AC or DC of zero taps) give the sums' empty value in one
pass and in two."""
import ctypes as C
import os

import numpy as np
import pytest

FS = 44100.0


@pytest.mark.parametrize("n_ac,n_dc", [(-1, 88), (76, -1), (-16, -16)])
def test_negative_tap_counts_are_refused_before_any_launch(n_ac, n_dc):
    from cochlearmodel_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    L = _lib.lib()
    f = C.c_void_p(0x1000)   # never dereferenced
    iv = np.zeros(1, _lib.IHC_INTERVAL_DTYPE)
    iv["len"], iv["L"], iv["tla"], iv["frdp"] = 100, 100, 100, 101
    sp = (C.c_float * 3)(0.0, 0.0, 0.0)
    for scratch in (None, f):
        rc = L.cm_ihc_lambda_run(f, 100, _lib.ptr(iv), 1, None, 0, f, None, n_ac, f, n_dc, f, f, sp, C.c_float(500),
                                 C.c_float(1), C.c_float(100), C.c_float(1), scratch, f, None)
        assert rc == -3 and "negative count" in L.cm_last_error().decode()


@pytest.mark.gpu
@pytest.mark.parametrize("n_ac,n_dc", [(0, 88), (76, 0), (0, 0), (1, 1)])
def test_empty_filters(n_ac, n_dc):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cochlearmodel_amd import stages
    print(f"case: {n_ac} AC taps, {n_dc} DC taps", flush=True)
    rows = 150
    bi = stages.BatchedIHC(FS)
    bi.n_ac, bi.n_dc = n_ac, n_dc
    ivs = stages.signal_intervals([0, 65], [65, 85])
    bm = torch.from_numpy((1e-3 * np.random.default_rng(n_ac + n_dc).standard_normal((rows, 256))).astype(np.float32))
    got = [bi.run(bm.cuda(), rows, ivs, stages=True, workspace=w) for w in (True, False)]
    # two passes: the velocity in the last lambda plane
    lam = torch.zeros((3, rows, 256), device="cuda")
    lam[2].copy_(bm)
    got.append(bi.run(lam[2], rows, ivs, d_lambda=lam, stages=True))
    torch.cuda.synchronize()
    for lam_k, st_k in got[1:]:
        assert torch.equal(lam_k, got[0][0]) and torch.equal(st_k, got[0][1])
    st = got[0][1].cpu()
    if n_ac == 0:
        assert not st[0].any()                            # AC
        assert torch.equal(st[1], bm * bm)                # dS = (BM - 0)^2
    if n_dc == 0:
        assert not st[2].any()                            # DC
    if n_ac == n_dc == 0:
        assert torch.equal(st[4], torch.full_like(st[4], -20.0))   # log10(0 + 1e-20)
