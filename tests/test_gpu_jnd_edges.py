"""The JND reductions against the CPU oracle, bit for bit, at body lengths around
the kernel's 32-row tiles, for both sums and each alone, with rates that leave
the range of its short division (zeros, tiny and huge values) and an interval
without a signal increment (dA = 0)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FS = 44100.0


@pytest.mark.parametrize("length,ai,rms", [(1, 1, 1), (31, 1, 1), (32, 1, 1), (33, 1, 1), (64, 1, 1), (65, 1, 0),
                                           (97, 0, 1), (200, 1, 1)])
@pytest.mark.parametrize("extreme", [False, True])
def test_lengths_around_the_tiles(oracle, length, ai, rms, extreme):
    import torch
    from cochlearmodel_amd import _lib
    print(f"case: JND reductions, bodies of {length} rows, AI {ai}, rate {rms}, extreme rates {extreme}", flush=True)
    rng = np.random.default_rng(length)
    n, head, nodes = 4, 5, length + 9
    lam = rng.uniform(0.1, 500.0, (3, n * nodes, 256)).astype(np.float32)
    if extreme:
        lam[:, rng.integers(0, n * nodes, 40), rng.integers(0, 256, 40)] = 0.0
        lam[:, rng.integers(0, n * nodes, 40), rng.integers(0, 256, 40)] = 1e-38
        lam[:, rng.integers(0, n * nodes, 40), rng.integers(0, 256, 40)] = 3e36
    dA = np.array([0.02, 3e-4, 0.0, 7.0], np.float32)
    ref = np.array([3, 0, 3, 3], np.int32)
    nIHC, W = rng.uniform(50, 150, 256), np.array([0.61, 0.23, 0.16], np.float32)
    d = [torch.from_numpy(x).cuda() for x in (lam, dA, ref, np.arange(n, dtype=np.int32), nIHC)]
    mr = torch.empty((3, n, 256), device="cuda")
    fra, fai = torch.zeros((3, n), device="cuda"), torch.zeros((3, n), device="cuda")
    L = _lib.lib()
    L.cm_set_stream(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    p = _lib.ptr
    _lib.check(L.cm_jnd_run(p(d[0]), n * nodes, n, nodes, head, length, p(d[1]), p(d[2]), p(d[3]), n, p(d[4]),
                            (C.c_float * 3)(*W), FS, 0.2 * FS, ai, rms, p(mr), p(fra), p(fai)), "cm_jnd_run")
    mr_o, fra_o, fai_o = oracle.jnd(lam, n, nodes, head, length, dA, ref, nIHC, W, FS, 0.2 * FS, bool(ai), bool(rms))
    np.testing.assert_array_equal(mr.cpu().numpy(), mr_o)
    if ai:
        np.testing.assert_array_equal(fai.cpu().numpy(), fai_o)
    if rms:
        np.testing.assert_array_equal(fra.cpu().numpy(), fra_o)
