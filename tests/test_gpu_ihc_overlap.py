"""IHC/lambda whose outputs lie over the BM velocity, which a call with a workspace
may ask for: the velocity in each of the lambda planes, across two of them and in
the stage planes, with tables that do and do not travel with the launch."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
ROWS = 2600
TABLES = {"one interval": [2600], "six intervals": [700, 15, 16, 17, 1000, 852]}


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _iir():
    return np.array([0.02, 0.04, 0.02]), np.array([1.0, -1.56, 0.64])


@pytest.mark.parametrize("table", TABLES)
@pytest.mark.parametrize("filt", ["fir", "iir"])
@pytest.mark.parametrize("where", ["lambda 0", "lambda 1", "lambda 2", "lambda 0.5", "stages 0", "stages 3"])
def test_outputs_over_the_velocity(table, filt, where):
    torch = _cuda()
    from cochlearmodel_amd import stages
    print(f"case: {table}, {filt}, velocity in {where}", flush=True)
    lens = TABLES[table]
    ivs = stages.signal_intervals(np.cumsum([0] + lens[:-1]), lens)
    bi = stages.BatchedIHC(FS, ac=_iir() if filt == "iir" else None)
    bm = torch.from_numpy((1e-3 * np.random.default_rng(4).standard_normal((ROWS, 256))).astype(np.float32)).cuda()
    iir = ivs if filt == "iir" else None
    want, want_st = bi.run(bm, ROWS, ivs, iir, stages=True)
    lam = torch.full((3, ROWS, 256), 7.0, device="cuda")
    st = torch.full((5, ROWS, 256), 7.0, device="cuda")
    plane, k = where.split()
    flat = (lam if plane == "lambda" else st).view(-1)
    at = int(float(k) * ROWS) * 256
    over = flat[at:at + ROWS * 256].view(ROWS, 256)
    over.copy_(bm)
    scratch = torch.empty((2, ROWS, 256), device="cuda")
    L = stages.lib()
    ptr = stages.ptr
    L.cm_set_stream(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    tab = np.ascontiguousarray(ivs, stages.IHC_INTERVAL_DTYPE)
    stages.check(L.cm_ihc_lambda_run(ptr(over), ROWS, ptr(tab), len(tab), ptr(tab) if filt == "iir" else None,
                                     len(tab) if filt == "iir" else 0, ptr(bi.b), ptr(bi.a), bi.n_ac, ptr(bi.dc),
                                     bi.n_dc, ptr(bi.damage), ptr(bi.A), bi.spont, stages.LAMBDA_SAT, stages.ETA_AC,
                                     stages.ETA_DC, 1.0, ptr(scratch), ptr(lam), ptr(st)))
    torch.cuda.synchronize()
    assert torch.equal(lam, want)
    assert torch.equal(st, want_st)
