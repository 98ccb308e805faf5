"""The one-pass IHC/lambda kernel against the CPU oracle, bit for bit, where its
tiles, blocks and windows have their edges: interval lengths around a block (16
rows), a trip (64) and a tile; AC taps around a chunk; DC filters around the
shortest and longest that it takes as a box car, and one with unequal taps;
windows that restart inside an interval, inside a block and on its first and
last row; the table in the launch (up to 4 intervals) and in device memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0


def _field(rows, seed):
    """BM velocity with loud, quiet and silent sections and a silent stretch."""
    rng = np.random.default_rng(seed)
    scale = 10.0 ** np.linspace(-2, -12, 256)
    scale[200:210] = 0.0
    bm = (scale * rng.standard_normal((rows, 256))).astype(np.float32)
    bm[rows // 3:rows // 3 + 40] = 0.0
    return bm


@pytest.mark.parametrize("lens,n_ac,dc", [
    ([1, 15, 16], 76, 88), ([17, 63, 64, 65], 76, 88), ([159, 160, 161, 2000, 31], 76, 88), ([700, 33], 1, 16),
    ([700], 4, 17), ([700], 15, 31), ([700], 16, 32), ([700], 17, 33), ([1100], 80, 96), ([1100], 129, 97),
    ([500], 76, 15), ([500, 90], 76, 1), ([900], 76, "ramp"),
])
def test_edges_of_tiles_and_windows(oracle, lens, n_ac, dc):
    import torch
    from cochlearmodel_amd import stages
    print(f"case: one-pass IHC/lambda, lengths {lens}, {n_ac} AC taps, DC {dc}", flush=True)
    rng = np.random.default_rng(n_ac + sum(lens))
    b = rng.standard_normal(n_ac) / n_ac
    dcv = np.linspace(0.001, 0.02, 40) if dc == "ramp" else np.full(dc, 1.0 / dc)
    starts = np.cumsum([0] + lens[:-1])
    bm = _field(sum(lens), 5)
    bi = stages.BatchedIHC(FS, ac=(b, None))
    bi.dc, bi.n_dc = torch.from_numpy(dcv).cuda(), len(dcv)
    lam, st = bi.run(torch.from_numpy(bm).cuda(), sum(lens), stages.signal_intervals(starts, lens), workspace=False,
                     stages=True)
    plain, _ = bi.run(torch.from_numpy(bm).cuda(), sum(lens), stages.signal_intervals(starts, lens), workspace=False)
    np.testing.assert_array_equal(plain.cpu().numpy(), lam.cpu().numpy())
    for s0, n in zip(starts, lens):
        lo, so = oracle.ihc_lambda(bm[s0:s0 + n], n, n + 1, b, dcv, stages.ihc_damage(8.0), stages.aihc_table(),
                                   np.array(stages.SPONT_DEFAULT, np.float32), stages=True, threads=8)
        np.testing.assert_array_equal(st[:, s0:s0 + n].cpu().numpy(), so, err_msg=f"stages, {n} rows")
        np.testing.assert_array_equal(lam[:, s0:s0 + n].cpu().numpy(), lo, err_msg=f"{n} rows")


@pytest.mark.parametrize("rows,L,frdp", [(900, 16, 901), (900, 7, 901), (900, 89, 901), (900, 300, 500),
                                         (1000, 160, 640), (640, 640, 320)])
def test_windows_that_restart_inside_an_interval(oracle, rows, L, frdp):
    import torch
    from cochlearmodel_amd import _lib, stages
    print(f"case: one-pass IHC/lambda, {rows} rows, period {L}, regular division up to row {frdp}", flush=True)
    bm = _field(rows, 6)
    iv = np.array([(0, rows, 0, L, rows, frdp, 0)], _lib.IHC_INTERVAL_DTYPE)
    bi = stages.BatchedIHC(FS)
    lam, _ = bi.run(torch.from_numpy(bm).cuda(), rows, iv, workspace=False)
    b, _ = stages.load_ac_filter(FS)
    lo = oracle.ihc_lambda(bm, L, frdp, b, stages.dc_filter(FS), stages.ihc_damage(8.0), stages.aihc_table(),
                           np.array(stages.SPONT_DEFAULT, np.float32), threads=8)
    np.testing.assert_array_equal(lam.cpu().numpy(), lo)


@pytest.mark.parametrize("taps", [2, 3, 5, 9, 10])
def test_iir_orders_and_lengths(oracle, taps):
    """The IIR AC filter of every register form and of the general one, over
    intervals around its blocks of 16 rows: the same values as the oracle's."""
    import torch
    from scipy.signal import butter
    from cochlearmodel_amd import stages
    print(f"case: IIR AC filter of {taps} taps", flush=True)
    lens = [1, 2, 15, 16, 17, 33, 700]
    b, a = butter(taps - 1, 0.3)
    starts = np.cumsum([0] + lens[:-1])
    bm = _field(sum(lens), 7)
    ivs = stages.signal_intervals(starts, lens)
    lam, st = stages.BatchedIHC(FS, ac=(b, a)).run(torch.from_numpy(bm).cuda(), sum(lens), ivs, ivs, stages=True)
    for s0, n in zip(starts, lens):
        lo, so = oracle.ihc_lambda(bm[s0:s0 + n], n, n + 1, b, stages.dc_filter(FS), stages.ihc_damage(8.0),
                                   stages.aihc_table(), np.array(stages.SPONT_DEFAULT, np.float32), stages=True,
                                   threads=8, ac_a=a)
        np.testing.assert_array_equal(st[:, s0:s0 + n].cpu().numpy(), so, err_msg=f"stages, {n} rows")
        np.testing.assert_array_equal(lam[:, s0:s0 + n].cpu().numpy(), lo, err_msg=f"{n} rows")
