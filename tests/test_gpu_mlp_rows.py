"""The error model's kernels at row counts around their tiles (16 rows, two
tiles a step, a workgroup per 256 gradient rows) and with feature rows that
are not 8-byte aligned, against the CPU fp32 reference; NaN features."""
import numpy as np
import pytest

from film_grain_amd import synth
from tests import mlp_ref

pytestmark = pytest.mark.gpu


def _case(rng, n, shift):
    import torch
    P = rng.normal(0, 0.3, mlp_ref.N_PARAMS).astype(np.float32)
    P[mlp_ref.P_W1 + 12 * 64:mlp_ref.P_B1] = 0.0
    X = np.zeros((n, 16), np.float32)
    X[:, :12] = rng.uniform(-1, 1, (n, 12))
    X = mlp_ref.bf16(X)
    bits = (np.ascontiguousarray(X).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)
    buf = torch.zeros(n * 16 + shift, dtype=torch.int16, device="cuda:0")
    buf[shift:] = torch.from_numpy(bits.reshape(-1)).to("cuda:0")
    return P, X, buf[shift:].view(n, 16)


@pytest.mark.parametrize("n,shift", [(1, 0), (15, 0), (17, 1), (32, 0), (33, 3), (255, 0), (257, 1), (4097, 0),
                                     (65537, 0), (200001, 1)])
@pytest.mark.parametrize("kind", ["squared", "nll"])
def test_rows_around_the_tiles(hip_ctx, n, shift, kind):
    import torch
    rng = np.random.default_rng(n)
    P, X, Xd = _case(rng, n, shift)
    t = rng.normal(0, 1, n).astype(np.float32)
    Pd, td = torch.from_numpy(P).to("cuda:0"), torch.from_numpy(t).to("cuda:0")
    guard = torch.full((n + 64,), 7.0, device="cuda:0")
    hip_ctx.mlp_forward(Pd, Xd, out=guard[:n])
    assert torch.all(guard[n:] == 7.0)  # rows past n are not written
    y_ref = mlp_ref.forward(P, X)[-1]
    assert np.abs(guard[:n].cpu().numpy() - y_ref).max() <= 1e-3 * (np.abs(y_ref).max() + 1e-6)
    grad = torch.zeros(mlp_ref.N_PARAMS, dtype=torch.float32, device="cuda:0")
    loss = torch.zeros(1, dtype=torch.float32, device="cuda:0")
    hip_ctx.mlp_grad(Pd, Xd, td, grad, loss, loss_kind=kind)
    g_ref, l_ref = mlp_ref.grad(P, X, t, loss=kind)
    # The reference rounds the same operands to BF16; one that falls on the
    # other side of a rounding is off by 2^-8 of one row's term, about
    # 2^-8 / sqrt(n) of the sum; the rest is the order of f32 sums (measured: at
    # most 3e-6 of a block beyond 4096 rows, 2.4e-4 at 17, and 3e-7 of the loss).
    bound = 2.0 ** -8 / np.sqrt(n) + 2e-5
    for name, d in _blocks(grad.cpu().numpy(), g_ref):
        assert d <= bound, (n, kind, name, d)
    assert abs(float(loss.item()) - l_ref) <= 4e-6 * abs(l_ref) + 1e-6


_BLOCKS = [("W1", mlp_ref.P_W1, mlp_ref.P_B1), ("b1", mlp_ref.P_B1, mlp_ref.P_W2), ("W2", mlp_ref.P_W2, mlp_ref.P_B2),
           ("b2", mlp_ref.P_B2, mlp_ref.P_W3), ("w3", mlp_ref.P_W3, mlp_ref.P_B3), ("b3", mlp_ref.P_B3, mlp_ref.N_PARAMS)]


def _blocks(got, want):
    """(name, relative distance in norm) of each parameter block."""
    return [(name, float(np.linalg.norm((got - want)[i:j])) / max(float(np.linalg.norm(want[i:j])), 1e-30))
            for name, i, j in _BLOCKS]


@pytest.mark.parametrize("n,shift", [(1, 0), (15, 0), (17, 1), (255, 0), (257, 1), (4097, 0), (65537, 0), (200001, 1),
                                     (200016, 0)])
@pytest.mark.parametrize("kind", ["squared", "nll"])
def test_no_row_is_lost_or_taken_twice(hip_ctx, n, shift, kind):
    """Targets that the model meets at all rows but those of the last tile and
    a few others: the gradient is theirs alone, so that one of them lost or
    doubled moves it by far more than the bound, at any number of rows."""
    import torch
    rng = np.random.default_rng(n + 1)
    P, X, Xd = _case(rng, n, shift)
    y = mlp_ref.forward(P, X)[-1]
    rows = np.unique(np.concatenate([np.arange((n - 1) // 16 * 16, n), rng.choice(n, min(n, 8), replace=False)]))
    if kind == "squared":  # dL/dy = 2 (y - t)
        t = y.astype(np.float32)
        t[rows] = y[rows] - rng.choice([0.7, 1.3], len(rows))
    else:  # dL/dy = 1 - t^2 e^(-2y)
        t = np.exp(y).astype(np.float32)
        t[rows] = np.exp(y[rows]) * rng.choice([1.5, 2.0], len(rows))
    grad = torch.zeros(mlp_ref.N_PARAMS, dtype=torch.float32, device="cuda:0")
    loss = torch.zeros(1, dtype=torch.float32, device="cuda:0")
    hip_ctx.mlp_grad(torch.from_numpy(P).to("cuda:0"), Xd, torch.from_numpy(t).to("cuda:0"), grad, loss,
                     loss_kind=kind)
    each = np.stack([mlp_ref.grad(P, X[r:r + 1], t[r:r + 1], n_total=n, loss=kind)[0] for r in rows])
    want = each.sum(0)
    # measured: at most 4e-3 at 200001 rows, whose own y differ from the
    # reference's in the last bits
    bound = 1e-2
    got = _blocks(grad.cpu().numpy(), want)
    print(f"[rows] n {n} {kind}: " + " ".join(f"{name} {d:.1e}" for name, d in got), flush=True)
    for name, d in got:
        assert d <= bound, (n, kind, name, d)
    for g in each:  # without the row
        assert max(d for _, d in _blocks(want - g, want)) > 4 * bound
    l_ref = mlp_ref.loss_terms(y, t.astype(np.float64), kind)[0].sum()
    assert abs(float(loss.item()) - l_ref) <= 1e-5 * abs(l_ref)


def test_nan_features_act_as_before_the_first_relu(hip_ctx):
    """A NaN feature makes its row's first layer NaN, which relu turns to 0;
    the other rows of its tile are untouched."""
    import torch
    rng = np.random.default_rng(5)
    P, X, Xd = _case(rng, 48, 0)
    Xd = Xd.clone()
    Xd[20, 3] = 0x7FC0
    y = hip_ctx.mlp_forward(torch.from_numpy(P).to("cuda:0"), Xd).cpu().numpy()
    y_ref = mlp_ref.forward(P, X)[-1]
    rows = np.arange(48) != 20
    assert np.abs(y - y_ref)[rows].max() <= 1e-3 * np.abs(y_ref).max()
    h2 = np.maximum(P[mlp_ref.P_B2:mlp_ref.P_B2 + 64], 0)
    want = float(h2 @ mlp_ref.bf16(P[mlp_ref.P_W3:mlp_ref.P_W3 + 64]) + P[mlp_ref.P_B3])
    assert abs(y[20] - want) <= 1e-4 * max(1.0, abs(want))


@pytest.mark.parametrize("bits", [0x7FC0, 0x7F80])
@pytest.mark.parametrize("n,row", [(48, 20), (1025, 1024)])
def test_a_bad_feature_stays_in_its_row_of_the_gradient(hip_ctx, bits, n, row):
    """A NaN feature, or an infinite one whose weights are negative, makes its
    row's first layer NaN or -inf, which relu turns to 0: the row acts as one of
    zero hidden values, and of the gradient only the bad feature's own row of
    dW1 (NaN or infinity times 0) is NaN."""
    import torch
    rng = np.random.default_rng(n)
    P, X, Xd = _case(rng, n, 0)
    P[3 * 64:4 * 64] = -np.abs(P[3 * 64:4 * 64]) - 0.01
    t = rng.normal(0, 1, n).astype(np.float32)
    Xd = Xd.clone()
    Xd[row, 3] = bits
    grad = torch.zeros(mlp_ref.N_PARAMS, dtype=torch.float32, device="cuda:0")
    loss = torch.zeros(1, dtype=torch.float32, device="cuda:0")
    hip_ctx.mlp_grad(torch.from_numpy(P).to("cuda:0"), Xd, torch.from_numpy(t).to("cuda:0"), grad, loss)
    got = grad.cpu().numpy()
    others = np.arange(n) != row
    want, l_ref = mlp_ref.grad(P, X[others], t[others], n_total=n)
    P0 = P.copy()  # the row's hidden values are 0
    P0[mlp_ref.P_W1:mlp_ref.P_B1] = 0.0
    P0[mlp_ref.P_B1:mlp_ref.P_W2] = -1.0
    g0, l0 = mlp_ref.grad(P0, X[:1], t[row:row + 1], n_total=n)
    want = want + g0
    bad = np.zeros(mlp_ref.N_PARAMS, bool)
    bad[3 * 64:4 * 64] = True
    assert np.array_equal(np.isnan(got), bad)
    d = np.linalg.norm((got - want)[~bad]) / np.linalg.norm(want[~bad])
    print(f"[bad feature] n {n}: {d:.2e}", flush=True)
    assert d <= 2.0 ** -8
    assert abs(float(loss.item()) - (l_ref + l0)) <= 1e-4 * (l_ref + l0)


@pytest.mark.parametrize("shift", [0, 1, 4])
def test_feature_rows_at_any_alignment(hip_ctx, shift):
    import torch
    u = torch.from_numpy(synth.sinusoid_field(37, 23, 4, n_waves=3)).to("cuda:0")
    want = hip_ctx.mlp_features(u, 55, 34, 1.5, 0.1, 0.05, 0.8, 1)
    buf = torch.full((55 * 34 * 16 + 2 * shift + 16,), 123, dtype=torch.int16, device="cuda:0")
    hip_ctx.mlp_features(u, 55, 34, 1.5, 0.1, 0.05, 0.8, 1, out=buf[shift:shift + 55 * 34 * 16])
    assert torch.equal(buf[shift:shift + 55 * 34 * 16].view(-1, 16), want)
    assert torch.all(buf[:shift] == 123) and torch.all(buf[shift + 55 * 34 * 16:] == 123)


@pytest.mark.parametrize("n", [1, 31, 513])
def test_forward_adds_in_a_fixed_order(hip_ctx, n):
    """The sample budgets are a ceiling of the predictions, so the order of the
    forward pass's additions is part of its result: the bias after the layer's
    sum, layer 3 one column after the other, products and sums rounded apart.
    Integer operands make every sum before the biases exact whatever its order
    (|z2| <= 64 * 256 * 3 < 2^24), so the prediction is known to the bit."""
    import torch
    rng = np.random.default_rng(n)
    P = np.zeros(mlp_ref.N_PARAMS, np.float32)
    P[:12 * 64] = rng.integers(-3, 4, 12 * 64)
    P[mlp_ref.P_B1:mlp_ref.P_W2] = rng.integers(-20, 21, 64)
    P[mlp_ref.P_W2:mlp_ref.P_B2] = rng.integers(-3, 4, 64 * 64)
    P[mlp_ref.P_B2:mlp_ref.P_W3] = rng.normal(0, 30, 64)
    P[mlp_ref.P_W3:mlp_ref.P_B3] = rng.normal(0, 0.3, 64)
    P[mlp_ref.P_B3] = 0.37
    X = np.zeros((n, 16), np.float32)
    X[:, :12] = rng.integers(-4, 5, (n, 12))
    W1, b1, W2, b2, w3, b3 = mlp_ref.unpack(P)
    h1 = np.maximum(X @ W1 + b1, 0)
    assert h1.max() <= 256  # exact in BF16
    h2 = np.maximum((h1 @ W2) + b2[None, :], np.float32(0))
    assert h2.dtype == np.float32
    # lane g of a row holds columns 16 cb + 4 g + i
    prod = (h2 * mlp_ref.bf16(w3)[None, :]).reshape(n, 4, 4, 4)  # row, cb, g, i
    acc = np.zeros((n, 4), np.float32)
    for cb in range(4):
        for i in range(4):
            acc = acc + prod[:, cb, :, i]
    want = ((acc[:, 0] + acc[:, 1]) + (acc[:, 2] + acc[:, 3])) + b3
    bits = (X.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)
    got = hip_ctx.mlp_forward(torch.from_numpy(P).to("cuda:0"), torch.from_numpy(bits).to("cuda:0")).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.astype(np.float32).view(np.uint32))
