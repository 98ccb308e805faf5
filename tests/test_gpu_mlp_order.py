"""Bias gradients add their rows in order, one after another from 0, bit for bit:
sums of one matrix at the edges of the kernels' tiles (16 columns, 512 rows; 256
columns), on either side of the line between them, and the ten first steps of a training run, whose gradients, parameters and outputs
follow from those sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _row_order(x):
    """Column sums of float32 rows, row 0 first."""
    return np.add.accumulate(x, axis=0, dtype=np.float32)[-1]


@pytest.mark.parametrize("M,N", [(1, 1), (2, 16), (3, 17), (64, 15), (65, 512), (511, 33), (512, 16), (513, 31),
                                 (240, 300), (241, 300), (300, 8193), (480, 8193), (481, 8193), (245, 65553),
                                 (1023, 5), (1024, 512), (1025, 769), (2049, 48), (8192, 256)])
def test_column_sums_add_the_rows_in_order(M, N):
    torch = _cuda()
    from cochlearmodel_amd._lib import check, lib
    print(f"colsum order M={M} N={N}", flush=True)
    rng = np.random.default_rng(M * 1000 + N)
    x = (rng.standard_normal((M, N)) * 10.0 ** rng.uniform(-3, 3, (M, 1))).astype(np.float32)
    x[:, N // 2] = -0.0
    d = torch.from_numpy(x).cuda()
    db = torch.full((N,), float("nan"), device="cuda")
    check(lib().cm_colsum(d.data_ptr(), db.data_ptr(), M, N))
    torch.cuda.synchronize()
    want = _row_order(x)
    want[N // 2] = 0.0   # the sum starts at 0
    assert db.cpu().numpy().tobytes() == want.tobytes()


@pytest.mark.parametrize("B", [33, 1024, 1500])
def test_training_follows_the_row_ordered_sums(B):
    torch = _cuda()
    from cochlearmodel_amd import mlp
    print(f"ten training steps at batch {B}", flush=True)
    rng = np.random.default_rng(B)
    X, T = (torch.from_numpy(rng.standard_normal((B, n)).astype(np.float32)).cuda() for n in (mlp.N_IN, mlp.N_OUT))
    a, b = mlp.WarmStartMLP(seed=3), mlp.WarmStartMLP(seed=3)
    for step in range(10):
        ya, yb = a.forward(X), b.forward(X)
        la, lb = a.backward(T, B), b.backward(T, B)
        assert la == float(a.rowloss[:B].sum().item()) / (B * mlp.N_OUT) and la == lb
        for g, d in zip(b.gb, b.dZ + [b.dY]):
            g.copy_(torch.from_numpy(_row_order(d[:B].cpu().numpy())))
        for u, v in zip([ya, *a.gb, *a.gW], [yb, *b.gb, *b.gW]):
            assert torch.equal(u, v), step
        a.adam_step(1e-3)
        b.adam_step(1e-3)
    for u, v in zip(a.W + a.b, b.W + b.b):
        assert torch.equal(u, v)
