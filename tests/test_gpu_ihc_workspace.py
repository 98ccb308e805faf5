"""The AC/dS workspace (two planes of rows x 256 floats) is allocated for the calls
that read it and for no others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
ROWS = 20000
PLANE = ROWS * 256 * 4


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("case", ["fir", "iir", "kbase", "long dc", "over the velocity"])
def test_batched_calls(case):
    torch = _cuda()
    from cochlearmodel_amd import stages
    print(f"case: {case}, {ROWS} rows", flush=True)
    ac = (np.array([0.02, 0.04, 0.02]), np.array([1.0, -1.56, 0.64])) if case == "iir" else None
    bi = stages.BatchedIHC(96000.0 if case == "long dc" else FS, ac=ac or stages.load_ac_filter(FS))
    ivs = stages.signal_intervals([0, 9000], [9000, ROWS - 9000])
    if case == "kbase":
        ivs["kbase"], ivs["L"], ivs["tla"], ivs["frdp"] = [0, 9000], ROWS, ROWS, ROWS + 1
    lam = torch.empty((3, ROWS, 256), device="cuda")
    bm = lam[1] if case == "over the velocity" else torch.empty((ROWS, 256), device="cuda")
    bm.copy_(torch.from_numpy((1e-3 * np.random.default_rng(1).standard_normal((ROWS, 256))).astype(np.float32)))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    bi.run(bm, ROWS, ivs, ivs if ac else None, d_lambda=lam)
    torch.cuda.synchronize()
    grown = torch.cuda.max_memory_allocated() - before
    assert (grown >= 2 * PLANE) == (case != "fir"), grown


def test_tone_batches_hold_none():
    torch = _cuda()
    from cochlearmodel_amd import batch
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    tb = batch.ToneBatch([500.0, 2000.0], [60.0, 40.0], 0.2)
    assert torch.cuda.memory_allocated() - before < 4.5 * tb.rows * 1024
    with pytest.raises(ValueError):
        batch.ToneBatch([500.0], [60.0], 0.2, d_scratch=torch.empty(8, device="cuda"))


def test_tone_batches_give_one_when_asked():
    torch = _cuda()
    from cochlearmodel_amd import batch
    tb = batch.ToneBatch([500.0], [60.0], 0.04)
    ws = tb.d_scratch
    assert ws.shape == (2, tb.rows, 256) and ws.dtype == torch.float32 and ws.is_cuda
    assert tb.d_scratch is ws
    assert batch.ToneBatch([2000.0], [40.0], 0.04, d_scratch=ws).d_scratch is ws
