"""The JND reductions' two forms, one thread per section for short bodies and tiles
for the others, against the CPU oracle, bit for bit: body lengths and numbers of
intervals on either side of the line between them, both sums and each alone, rates
that leave the range of the short division, and the stage dumps of short bodies."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("n,length", [(4, 1), (4, 2), (4, 16), (4, 17), (4, 45), (85, 33), (100, 47), (100, 48),
                                      (300, 94), (300, 95), (86, 515), (86, 517)])
@pytest.mark.parametrize("ai,rms", [(1, 1), (1, 0), (0, 1)])
def test_either_side_of_the_line(oracle, n, length, ai, rms):
    torch = _cuda()
    from cochlearmodel_amd import _lib
    if length > 500 and ai:
        pytest.skip("the line of rates alone")
    print(f"case: {n} bodies of {length} rows, AI {ai}, rate {rms}", flush=True)
    rng = np.random.default_rng(1000 * n + length)
    head, nodes = 3, length + 5
    lam = rng.uniform(0.1, 500.0, (3, n * nodes, 256)).astype(np.float32)
    at = lambda: (rng.integers(0, n * nodes, 30), rng.integers(0, 256, 30))
    for value in (0.0, 1e-38, 3e36):
        lam[(slice(None), *at())] = value
    dA = (10.0 ** rng.uniform(-4, 1, n)).astype(np.float32)
    dA[n // 2] = 0.0
    ref = rng.integers(0, n, n).astype(np.int32)
    nIHC, W = rng.uniform(50, 150, 256), np.array([0.61, 0.23, 0.16], np.float32)
    d = [torch.from_numpy(x).cuda() for x in (lam, dA, ref, np.arange(n, dtype=np.int32), nIHC)]
    mr = torch.empty((3, n, 256), device="cuda")
    fra, fai = torch.zeros((3, n), device="cuda"), torch.zeros((3, n), device="cuda")
    L, p = _lib.lib(), _lib.ptr
    L.cm_set_stream(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check(L.cm_jnd_run(p(d[0]), n * nodes, n, nodes, head, length, p(d[1]), p(d[2]), p(d[3]), n, p(d[4]),
                            (C.c_float * 3)(*W), FS, 0.2 * FS, ai, rms, p(mr), p(fra), p(fai)), "cm_jnd_run")
    mr_o, fra_o, fai_o = oracle.jnd(lam, n, nodes, head, length, dA, ref, nIHC, W, FS, 0.2 * FS, bool(ai), bool(rms))
    np.testing.assert_array_equal(mr.cpu().numpy(), mr_o)
    if ai:
        np.testing.assert_array_equal(fai.cpu().numpy(), fai_o)
    if rms:
        np.testing.assert_array_equal(fra.cpu().numpy(), fra_o)


@pytest.mark.parametrize("length", [1, 15, 16, 40])
def test_stage_dumps(oracle, length):
    _cuda()
    from cochlearmodel_amd import _lib, solver, stages
    from cochlearmodel_amd._lib import check, ptr
    from test_gpu_stages import _c4_small
    c = _c4_small()
    n, L = c["n_prof"], _lib.lib()
    print(f"case: stage dumps of {n} bodies of {length} rows", flush=True)
    rows = n * c["L"]
    rng = np.random.default_rng(length)
    # the library's own buffers: sized by a run of the stages, then loaded
    sec = solver.section_params()
    g = np.full(256, 0.5, np.float32)
    keep = [np.ascontiguousarray(x, np.float32) for x in (g, sec[0], sec[1], g, g, sec[2], sec[3], sec[4], sec[5],
                                                          sec[6], sec[7])]
    n_in = c["bufP1"] + 2 * c["ov"]
    check(L.BMOHCKernel_Init(*[ptr(k) for k in keep], 1.0, 0.0, n_in, n_in * 256, 0, 1, 0, 0), "init")
    check(L.InputProfilesArrayInitialization(n, c["L"], 0, 0, 0), "init")
    check(L.generateInputFromProfile(ptr(c["prof"]), ptr(c["WN"]), c["L"], None, 0, 0, 0, 0, 0.16, 0.0, 0, c["e1"],
                                     0, c["e1"], n, 0, 0, n, c["ov"], c["L"], c["head"], c["length"], FS, 0, None, 0,
                                     1, 1e-15, 1e-10, 0, 0.0, 0.0, c["DF"], 0, ptr(np.ones(1, np.float32)), 1,
                                     ptr(np.ones(1, np.float32)), 1), "generate")
    stages.run_ihc_reference(rows, c["block"], c["TB"], c["DF"])
    lam = rng.uniform(0.1, 500.0, (3, rows, 256)).astype(np.float32)
    check(L.ReverseKernel_Copy_Results_Float(ptr(lam), L.getCudaLambda(), 0, 3 * rows, 256), "load lambda")
    nIHC = rng.uniform(50, 150, 256)
    arg = {k: np.ascontiguousarray(c[k], np.int32) for k in ("serial", "to_ref", "refs", "calc")}
    ref_idx = stages.reference_index(n, arg["refs"], arg["serial"], arg["to_ref"])
    dA = c["prof"]["dA"].astype(np.float32)
    out = [np.zeros(3 * n, np.float32) for _ in range(2)]
    for k in range(1, 7):
        check(L.CudaCalculateJND(1, 1, 0, 3 * n, 2e-5, FS, 1.0, ptr(nIHC), ptr(arg["calc"]), len(arg["calc"]),
                                 ptr(arg["refs"]), len(arg["refs"]), 0, n, n, c["head"], c["ov"], c["L"], length,
                                 ptr(arg["serial"]), ptr(arg["to_ref"]), ptr(out[0]), ptr(out[1]), rows * 256,
                                 rows * 256, 0.2 * FS, 1, 0, 0, 0, k), f"stage {k}")
        want = oracle.jnd(lam, n, c["L"], c["head"], length, dA, ref_idx, nIHC,
                          np.array(stages.W_DEFAULT, np.float32), FS, 0.2 * FS, backup_stage=k)[3]
        got = np.zeros(want.size, np.float32)
        check(L.GeneralKernel_Copy_Results_Bytes(ptr(got), L.getCudaBuffer(), got.nbytes, 0), "stage copy")
        got = got.reshape(want.shape)
        if k in (3, 4):
            body = np.concatenate([np.arange(i * c["L"] + c["head"], i * c["L"] + c["head"] + length)
                                   for i in range(n)])
            got, want = got[:, body], want[:, body]
        np.testing.assert_array_equal(got, want, err_msg=f"stage {k}")


@pytest.mark.parametrize("n,length", [(100, 53), (100, 54), (256, 99), (256, 100), (257, 132), (257, 133), (300, 150),
                                      (300, 151), (600, 240), (600, 241), (85, 600), (86, 700)])
@pytest.mark.parametrize("ai,rms", [(1, 1), (0, 1)])
def test_either_side_of_the_lines_by_rounds(oracle, n, length, ai, rms):
    if length > 500 and ai:
        pytest.skip("the line of rates alone")
    test_either_side_of_the_line(oracle, n, length, ai, rms)
