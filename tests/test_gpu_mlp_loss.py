"""The loss of the networks: squares of FP32 differences summed in FP64, so that many equal terms give the term.

With all parameters zero the outputs are zero and every term is t^2 for targets t.  N terms summed in
FP64 are off by N 2^-53 at most, and the mean is rounded to float once: nearest to t^2, which the targets are
chosen not to put near the middle of two floats.  A mean over an epoch is multiplied by a float and
added in FP32 besides: two roundings more."""
import numpy as np
import pytest

from mithra_amd import abi

pytestmark = pytest.mark.gpu


def targets():
    t = np.random.default_rng(5).uniform(0.5, 2.0, 40).astype(np.float32)
    sq = t.astype(np.float64) ** 2
    ulp = np.spacing(sq.astype(np.float32)).astype(np.float64)
    off = np.abs(sq - sq.astype(np.float32)) / ulp
    return t[off < 0.45]


@pytest.mark.parametrize("dims,n", [([3, 1], 1), ([5, 70], 100), ([8, 64], 128), ([8, 512], 8192)])
def test_equal_terms(dims, n):
    mlp = abi.MLP(dims, members=1, seed=1)
    x = np.ones((n, dims[0]), np.float32)
    ts = targets()
    assert len(ts) > 20
    for t in ts:
        mlp.set_params(np.zeros(mlp.n_params, np.float32))
        want = np.float32(float(t) ** 2)
        tgt = np.full((n, dims[-1]), t, np.float32)
        assert np.float32(mlp.gradients(0, x, tgt)[1]) == want
        assert mlp.train_step(x, tgt, 1e-3)[0] == want


def test_equal_terms_over_an_epoch():
    dims, n = [8, 256], 4096
    x = np.ones((n, dims[0]), np.float32)
    for t in targets():
        mlp = abi.MLP(dims, members=1, seed=1)
        mlp.set_params(np.zeros(mlp.n_params, np.float32))
        mlp.set_data(x, np.full((n, dims[-1]), t, np.float32))
        loss = mlp.train_epochs(1, n, 1e-3)[0]
        assert abs(float(loss) / float(t) ** 2 - 1.0) <= 4 * 2.0 ** -24
        mlp.close()
