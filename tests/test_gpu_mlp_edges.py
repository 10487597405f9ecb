"""Network kernels at the edges of their node blocks: forward (16 nodes a wave,
weights kept over the blocks), weight gradients (4 nodes a product) and the
reduction of their partials, against the FP64 oracle."""
import numpy as np
import pytest

import oracle.mlp_oracle as MO
from tests.test_gpu_mlp import _inputs, _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 15, 17, 63, 65, 255, 257, 1025, 32769])
def test_forward_and_gradient(cuda, n):
    import torch

    from plugin_navierstokes_amd.learned import MLP

    P, X = _params(7), _inputs(n, n)
    T = np.random.default_rng(n + 1).normal(size=(n, 4)).astype(np.float32)
    mlp = MLP(P)
    xt, tt = torch.from_numpy(X).to(cuda), torch.from_numpy(T).to(cuda)
    Y, z1, z2 = mlp.forward(xt, cache=True)
    ref, cache = MO.forward(P, X)
    # BF16 inputs, activations and weights: 2^-9 relative each, over three layers
    assert np.all(np.abs(Y.cpu().numpy() - ref) <= 2.0 ** -7 * MO.output_scale(P, X))
    assert torch.equal(Y, mlp.forward(xt))  # without the caches
    mlp.gradient(xt, tt)
    g = mlp.G.cpu().numpy().astype(np.float64)
    # the gradient in float64 from the kernel's own pre-activations (their rounding,
    # and so the set of active units, is the forward's)
    Z1, Z2 = z1.cpu().numpy().astype(np.float64), z2.cpu().numpy().astype(np.float64)
    _, _, W2, _, W3, _ = MO.unpack(P)
    W2, W3 = MO.bf16(W2), MO.bf16(W3)[:4]
    H1, H2, Xb = MO.bf16(np.maximum(Z1, 0)), MO.bf16(np.maximum(Z2, 0)), MO.bf16(X)
    dY = 2.0 / (4 * n) * (Y.cpu().numpy().astype(np.float64) - T)
    S1 = (np.abs(dY) @ np.abs(W3)) * (Z2 > 0)
    D1 = (dY @ W3) * (Z2 > 0)
    S0 = (S1 @ np.abs(W2)) * (Z1 > 0)
    D0 = (D1 @ W2) * (Z1 > 0)
    # FP32 sums of n products in any order, of factors with up to 4 and 4 + 128
    # products behind them; a few roundings of dY
    c = (n + 4 + 128 + 16) * 2.0 ** -24
    for name, a, b, D, S, R in [("W1", MO.OFF_W1, MO.OFF_B1, D0, S0, Xb), ("b1", MO.OFF_B1, MO.OFF_W2, D0, S0, None),
                                ("W2", MO.OFF_W2, MO.OFF_B2, D1, S1, H1), ("b2", MO.OFF_B2, MO.OFF_W3, D1, S1, None),
                                ("W3", MO.OFF_W3, MO.OFF_W3 + 4 * MO.H, dY, np.abs(dY), H2),
                                ("b3", MO.OFF_B3, MO.OFF_B3 + 4, dY, np.abs(dY), None)]:
        R = np.ones((n, 1)) if R is None else R
        want, scale = (D.T @ R).reshape(-1), (S.T @ np.abs(R)).reshape(-1)
        assert np.all(np.abs(g[a:b] - want) <= c * scale + 1e-30), name
