"""The network's products with their fused ends (bias, activation, loss, bias gradients) at the edges of
their tiles, against the CPU oracle (oracle/mlp_ref.py) that rounds where the device rounds.

The device's FP32 sums differ from float64 by ~1e-6, which moves a few activations or gradients across a
BF16 rounding boundary; each is then off by one step, at most 2^-7 of itself, so that the relative L2
distance stays below 2^-7.  A row or column lost from the largest case would show as 1 / sqrt(8192) = 1.1e-2."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import mlp_ref  # noqa: E402
from golden_state import rel_l2  # noqa: E402
from mithra_amd import abi  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -7


@pytest.mark.parametrize("dims,members,n", [
    ([1, 1], 1, 1),                  # one product, nothing below it
    ([5, 70, 33, 1], 3, 63),         # odd strides: element loads
    ([8, 64, 64, 65], 2, 65),        # a tile and one row or column
    ([264, 512, 128], 5, 1),         # one row
    ([16] * 18 + [8], 1, 40),        # more layers than one launch of the bias gradients takes
    ([264, 512, 512, 256], 5, 1700),  # the forward products in 128 x 128 tiles, with all members
    ([40, 512, 384], 1, 8192),       # dZ of the hidden layer in 128 x 128 tiles, dW in 64 x 64
])
def test_network_matches_oracle(dims, members, n):
    rng = np.random.default_rng(n + len(dims))
    mlp = abi.MLP(dims, members=members, seed=8)
    p = mlp.params().reshape(members, -1)
    p += rng.normal(0.0, 0.05, p.shape).astype(np.float32)  # biases that are not zero
    mlp.set_params(p)
    x = rng.normal(0.0, 1.0, (n, dims[0])).astype(np.float32)
    t = rng.normal(0.0, 1.0, (n, dims[-1])).astype(np.float32)
    y = mlp.forward(x)
    e = members - 1
    ref, _ = mlp_ref.forward(p[e], dims, x, bf16_products=True)
    assert rel_l2(y[e], ref) <= TOL
    g, loss = mlp.gradients(e, x, t)
    g_ref, l_ref = mlp_ref.gradients(p[e], dims, x, t, bf16_products=True)
    assert abs(loss - l_ref) <= TOL * l_ref
    o = 0
    for a, b in zip(dims[:-1], dims[1:]):
        for name, size in (("W", a * b), ("b", b)):
            err = rel_l2(g[o:o + size], g_ref[o:o + size])
            print(f"{name} {a}x{b}: {err:.2e}", flush=True)
            assert err <= TOL
            o += size
