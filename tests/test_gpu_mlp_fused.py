"""The fused network pass at the edges of its tiles (32 rows, 32-feature
chunks, one or several tiles a block) against the FP64 oracle with the
kernel's operands rounded to BF16."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from phylocaml_amd import device as D

    return D.Context(0)


def _bf(a):
    import torch

    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16().double().numpy()


def _rounded(p, X, t, n_in, H):
    """Outputs, loss and gradients with every MFMA operand in BF16."""
    W1, b1, W2, b2, w3, b3 = MO.unpack(p.astype(np.float64), n_in, H)
    X, W1, W2 = _bf(X), _bf(W1), _bf(W2)
    Z1 = X @ W1 + b1
    H1 = _bf(MO.gelu(Z1))
    Z2 = H1 @ W2 + b2
    H2 = MO.gelu(Z2)
    y = H2 @ w3 + b3
    d = y - t
    dy = d / len(t)
    dZ2 = np.outer(dy, w3) * MO.gelu_grad(Z2)
    dZ1 = (_bf(dZ2) @ W2.T) * MO.gelu_grad(Z1)
    g = [X.T @ _bf(dZ1), dZ1.sum(0), H1.T @ _bf(dZ2), dZ2.sum(0), _bf(H2).T @ _bf(dy), dy.sum()]
    return y, 0.5 * np.mean(d * d), g


# a last row alone in its tile, a full tile, more tiles than blocks of the
# backward (256) and of the forward (768); one and two feature chunks, rows
# readable 16 bytes at a time or not; a size that takes the GEMM path
@pytest.mark.parametrize("n_in,H,B", [(32, 128, 1), (32, 128, 32), (5, 128, 33), (33, 128, 100),
                                      (64, 128, 257), (1, 64, 31), (32, 64, 4097), (63, 64, 65),
                                      (32, 128, 8192 + 33), (32, 128, 16384 + 5), (32, 128, 65536 + 5),
                                      (32, 64, 65536 + 5), (65, 128, 40)])
def test_fused_pass_matches_rounded_oracle(ctx, n_in, H, B):
    from phylocaml_amd import device as D, mlp

    rng = np.random.default_rng(B + n_in)
    net = mlp.MLP(ctx, n_in, H, 3)
    p = net.get_params()
    sizes = [n_in * H, H, H * H, H, H, 1]
    o = n_in * H
    p[o:o + H] = 0.1 * rng.standard_normal(H)  # biases start at zero
    net.set_params(p)
    X = rng.standard_normal((B, n_in)).astype(np.float32)
    t = rng.standard_normal(B).astype(np.float32)
    y, loss, g = _rounded(p, X, t, n_in, H)
    # FP32 sums put ~1e-3 of the BF16 roundings on the other side (2^-8 each):
    # ~1.2e-4 of the norm a stage, four stages deep; the output layer's gradient
    # is two stages deep, and unrounded H2 and dy (2^-9 each) would be ~1e-3 off
    tol = 1e-3
    got = net.forward(D.to_device(X)).cpu().numpy()
    assert np.linalg.norm(got - y) <= tol * (np.linalg.norm(y) + 1e-3)
    for _ in range(2):  # the partial sums are rewritten by every call
        gg, gl = net.gradients(D.to_device(X), D.to_device(t))
    assert abs(gl - loss) <= tol * loss
    o = 0
    for s, want in zip(sizes, g):
        want = np.ravel(want)
        rel = 4e-4 if o == n_in * H + H + H * H + H else tol
        assert np.linalg.norm(gg[o:o + s] - want) <= rel * (np.linalg.norm(want) + 1e-6), (s, o)
        o += s
