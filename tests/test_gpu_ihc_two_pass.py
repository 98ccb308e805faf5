"""The two-pass IHC/lambda kernels against the CPU oracle, bit for bit, with each
condition that selects them: DC filters of more than 97 taps (sampling rates above
48 kHz), FIR and IIR AC filters before them, intervals that continue the windows
of the one before (kbase > 0), and outputs that lie over the velocity.  Lengths
around a block of 16 rows and around the filters."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
LENS = [1, 15, 16, 17, 31, 97, 98, 99, 113, 201, 330]


def _field(rows, seed):
    """BM velocity with loud, quiet and silent sections and a silent stretch."""
    rng = np.random.default_rng(seed)
    scale = 10.0 ** np.linspace(-2, -12, 256)
    scale[200:210] = 0.0
    bm = (scale * rng.standard_normal((rows, 256))).astype(np.float32)
    bm[rows // 3:rows // 3 + 40] = 0.0
    return bm


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _check(oracle, torch, lam, st, bm, lens, b, a, dcv):
    from cochlearmodel_amd import stages
    s0 = 0
    for n in lens:
        lo, so = oracle.ihc_lambda(bm[s0:s0 + n], n, n + 1, b, dcv, stages.ihc_damage(8.0), stages.aihc_table(),
                                   np.array(stages.SPONT_DEFAULT, np.float32), stages=True, threads=8, ac_a=a)
        np.testing.assert_array_equal(st[:, s0:s0 + n].cpu().numpy(), so, err_msg=f"stages, {n} rows")
        np.testing.assert_array_equal(lam[:, s0:s0 + n].cpu().numpy(), lo, err_msg=f"{n} rows")
        s0 += n


@pytest.mark.parametrize("n_dc", [98, 112, 113, 200])
@pytest.mark.parametrize("filt", ["fir", "iir"])
def test_long_dc_filters(oracle, filt, n_dc):
    torch = _cuda()
    from scipy.signal import butter
    from cochlearmodel_amd import stages
    print(f"case: {n_dc} DC taps, {filt}", flush=True)
    b, a = butter(4, 0.3) if filt == "iir" else stages.load_ac_filter(FS)
    bm = _field(sum(LENS), n_dc)
    bi = stages.BatchedIHC(FS, ac=(b, a))
    dcv = np.linspace(1.0, 2.0, n_dc) / n_dc
    bi.dc, bi.n_dc = torch.from_numpy(dcv).cuda(), n_dc
    ivs = stages.signal_intervals(np.cumsum([0] + LENS[:-1]), LENS)
    lam, st = bi.run(torch.from_numpy(bm).cuda(), len(bm), ivs, ivs if filt == "iir" else None, stages=True)
    _check(oracle, torch, lam, st, bm, LENS, b, a, dcv)


@pytest.mark.parametrize("cuts", [[16], [1, 90], [75, 76, 77, 200], [15, 31, 300]])
def test_intervals_that_continue_a_window(oracle, cuts):
    torch = _cuda()
    from cochlearmodel_amd import stages
    print(f"case: 430 rows cut at {cuts}", flush=True)
    rows = 430
    bm = _field(rows, sum(cuts))
    at = np.array([0] + cuts + [rows])
    ivs = stages.signal_intervals(at[:-1], np.diff(at))
    ivs["kbase"], ivs["L"], ivs["tla"], ivs["frdp"] = at[:-1], rows, rows, rows + 1
    b, _ = stages.load_ac_filter(FS)
    lam, st = stages.BatchedIHC(FS).run(torch.from_numpy(bm).cuda(), rows, ivs, stages=True)
    _check(oracle, torch, lam, st, bm, [rows], b, None, stages.dc_filter(FS))


def test_outputs_over_the_velocity(oracle):
    torch = _cuda()
    from cochlearmodel_amd import stages
    print(f"case: velocity in the first lambda plane, lengths {LENS}", flush=True)
    bm = _field(sum(LENS), 9)
    b, _ = stages.load_ac_filter(FS)
    ivs = stages.signal_intervals(np.cumsum([0] + LENS[:-1]), LENS)
    lam = torch.zeros((3, len(bm), 256), device="cuda")
    lam[0].copy_(torch.from_numpy(bm))
    lam, st = stages.BatchedIHC(FS).run(lam[0], len(bm), ivs, d_lambda=lam, stages=True)
    _check(oracle, torch, lam, st, bm, LENS, b, None, stages.dc_filter(FS))
