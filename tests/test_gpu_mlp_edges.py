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


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 31, 40), (65, 97, 129), (1024, 512, 256), (2048, 1090, 9)])
def test_products_with_activation_equal_the_separate_kernels(M, N, K):
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    L = lib()
    print(f"gemm with gelu M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    dev = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    new = lambda t: torch.full((M, N), 7.0, dtype=t, device="cuda")
    p = lambda t: t.data_ptr()
    A, W, Wt, bias = dev(M, K).bfloat16(), dev(K, N).bfloat16(), dev(N, K).bfloat16(), dev(N)
    Z, G, Z2, G2 = new(torch.float32), new(torch.bfloat16), new(torch.float32), new(torch.bfloat16)
    check(L.cm_gemm_bf16(0, 0, M, N, K, p(A), K, p(W), N, p(Z), N, p(bias), 0.0))
    check(L.cm_gelu_fwd(p(Z), p(G), None, M * N))
    check(L.cm_gemm_bf16_gelu(M, N, K, p(A), K, p(W), N, p(bias), p(Z2), p(G2), N))
    d, dZ, dZb, dZ2, dZb2 = (new(t) for t in (torch.float32, torch.float32, torch.bfloat16, torch.float32,
                                              torch.bfloat16))
    check(L.cm_gemm_bf16(0, 1, M, N, K, p(A), K, p(Wt), K, p(d), N, None, 0.0))
    check(L.cm_gelu_bwd(p(d), p(Z), p(dZb), p(dZ), M * N))
    check(L.cm_gemm_bf16_gelu_back(M, N, K, p(A), K, p(Wt), K, p(Z), p(dZ2), p(dZb2), N))
    torch.cuda.synchronize()
    for a, b in ((Z, Z2), (G, G2), (dZ, dZ2), (dZb, dZb2)):
        assert torch.equal(a, b)


def test_many_sums_and_adam_steps_in_one_launch():
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    from cochlearmodel_amd.mlp import _ptrs
    import ctypes as C
    L = lib()
    rng = np.random.default_rng(9)
    dev = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    M, cols = 77, [1, 32, 33, 0, 512, 31, 64, 5]
    print(f"colsums M={M} N={cols}", flush=True)
    xs = [dev(M, n) for n in cols]
    one, many = ([torch.full((n,), 7.0, device="cuda") for n in cols] for _ in range(2))
    for x, o, n in zip(xs, one, cols):
        if n:
            check(L.cm_colsum(x.data_ptr(), o.data_ptr(), M, n))
    check(L.cm_colsums(8, _ptrs(xs), _ptrs(many), M, (C.c_int * 8)(*cols)))
    sizes = [1, 256, 257, 0, 70001]
    print(f"adams n={sizes}", flush=True)
    w, g, m, v = ([dev(n).abs() for n in sizes] for _ in range(4))
    wb = [torch.zeros(n, dtype=torch.bfloat16, device="cuda") if k % 2 else None for k, n in enumerate(sizes)]
    ref = [[t.clone() for t in s] for s in (w, m, v)]
    rwb = [None if t is None else t.clone() for t in wb]
    wd = [0.0, 0.1, 0.2, 0.0, 0.5]
    for k, n in enumerate(sizes):
        if n:
            check(L.cm_adam(ref[0][k].data_ptr(), None if rwb[k] is None else rwb[k].data_ptr(), g[k].data_ptr(),
                            ref[1][k].data_ptr(), ref[2][k].data_ptr(), n, 1e-2, 0.9, 0.999, 1e-8, 3, wd[k]))
    check(L.cm_adams(5, _ptrs(w), _ptrs(wb), _ptrs(g), _ptrs(m), _ptrs(v), (C.c_int64 * 5)(*sizes),
                     (C.c_float * 5)(*wd), 1e-2, 0.9, 0.999, 1e-8, 3))
    torch.cuda.synchronize()
    for a, b in [*zip(one, many), *zip(ref[0], w), *zip(ref[1], m), *zip(ref[2], v)]:
        assert torch.equal(a, b)
    for a, b in zip(rwb, wb):
        assert a is None or torch.equal(a, b)
    assert L.cm_colsums(9, _ptrs(xs), _ptrs(many), M, (C.c_int * 8)(*cols)) == -3
    assert L.cm_adams(0, None, None, None, None, None, None, None, 0.0, 0.0, 0.0, 0.0, 1) == -3


@pytest.mark.parametrize("K,dims", [(1, [(1, 1)]), (129, [(65, 33), (1, 70), (64, 64), (130, 5)]),
                                    (1024, [(769, 512), (512, 512), (512, 256)]),
                                    (40, [(1100, 1030), (3, 2), (64, 1025)])])
def test_weight_gradients_in_one_launch_equal_single_products(K, dims):
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    from cochlearmodel_amd.mlp import _ptrs
    import ctypes as C
    L = lib()
    print(f"weight grads K={K} {dims}", flush=True)
    rng = np.random.default_rng(K)
    dev = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda().bfloat16()
    A, B = [dev(K, m) for m, _ in dims], [dev(K, n) for _, n in dims]
    one, many = ([torch.full((m, n), 7.0, device="cuda") for m, n in dims] for _ in range(2))
    for a, b, c, (m, n) in zip(A, B, one, dims):
        check(L.cm_gemm_bf16(1, 0, m, n, K, a.data_ptr(), m, b.data_ptr(), n, c.data_ptr(), n, None, 0.0))
    num = C.c_int * len(dims)
    check(L.cm_weight_grads(len(dims), K, num(*(m for m, _ in dims)), num(*(n for _, n in dims)), _ptrs(A), _ptrs(B),
                            _ptrs(many)))
    torch.cuda.synchronize()
    for a, b in zip(one, many):
        assert torch.equal(a, b)
    assert L.cm_weight_grads(0, K, None, None, None, None, None) == -3
