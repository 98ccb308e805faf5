"""BF16 product and column sums at the edges of their tiles: 64 x 32 and 64 x 64
tiles of C, K steps of 128 in pieces of 8, rows that start at odd elements,
leading dimensions wider than the matrix (what lies outside is NaN and must not
be read), more tiles than the narrow form takes (256 on 256 CUs), and columns
over many groups."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu
SIZES = [(1, 1, 1), (3, 5, 7), (63, 31, 127), (64, 32, 128), (65, 33, 129), (64, 64, 8), (130, 96, 136),
         (7, 70, 257), (1600, 1430, 9), (2048, 1090, 131), (1024, 512, 769), (1024, 513, 512)]


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _padded(torch, x, ld, shift):
    """Device BF16 rows of x at leading dimension ld from element `shift`, NaN elsewhere."""
    buf = np.full(shift + x.shape[0] * ld, np.nan, np.float32)
    buf[shift:].reshape(x.shape[0], ld)[:, :x.shape[1]] = x
    return torch.from_numpy(buf).cuda().to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
def test_gemm_tiles(tA, tB, M, N, K):
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    L = lib()
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    A = mo.bf16_round(rng.standard_normal((K, M) if tA else (M, K)).astype(np.float32))
    B = mo.bf16_round(rng.standard_normal((N, K) if tB else (K, N)).astype(np.float32))
    ref = (A.T if tA else A) @ (B.T if tB else B)
    # the sum of absolute products times 2^-24 for each of the K additions
    tol = K * 2.0 ** -24 * (np.abs(A.T if tA else A) @ np.abs(B.T if tB else B)) + 1e-30
    for pad, shift in ((0, 0), (5, 3), (8, 8)):
        print(f"gemm tA={tA} tB={tB} M={M} N={N} K={K} pad={pad} shift={shift}", flush=True)
        lda, ldb, ldc = A.shape[1] + pad, B.shape[1] + pad, N + pad
        dA = _padded(torch, A.astype(np.float32), lda, shift)
        dB = _padded(torch, B.astype(np.float32), ldb, shift)
        dC = torch.full((M, ldc), float("nan"), device="cuda")
        check(L.cm_gemm_bf16(tA, tB, M, N, K, dA.data_ptr() + 2 * shift, lda, dB.data_ptr() + 2 * shift, ldb,
                             dC.data_ptr(), ldc, None, 0.0))
        torch.cuda.synchronize()
        got = dC.cpu().numpy()
        assert np.all(np.abs(got[:, :N] - ref) <= tol)
        assert np.all(np.isnan(got[:, N:]))


@pytest.mark.parametrize("M,N", [(1, 1), (31, 33), (32, 32), (33, 31), (1025, 70), (2, 65536 * 32 + 5)])
def test_colsum_groups(M, N):
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    print(f"colsum M={M} N={N}", flush=True)
    x = np.random.default_rng(M + N).standard_normal((M, N)).astype(np.float32)
    d = torch.from_numpy(x).cuda()
    db = torch.full((N,), float("nan"), device="cuda")
    check(lib().cm_colsum(d.data_ptr(), db.data_ptr(), M, N))
    torch.cuda.synchronize()
    tol = M * 2.0 ** -24 * np.abs(x).sum(0, dtype=np.float64) + 1e-30
    assert np.all(np.abs(db.cpu().numpy() - x.sum(0, dtype=np.float64)) <= tol)
