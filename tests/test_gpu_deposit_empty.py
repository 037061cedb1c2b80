"""The row-tiled deposit where most workgroups list nothing: a bunch of a few planes deposited onto a J that is
not zero, with and without a reset before, against the CPU oracle.

J is a sum of a node's shares, in another order than the oracle's; a node of the bunch takes fewer than 2000 of
them, each within the largest share, so that J agrees to 2000 roundings of the largest value in FP64 and to one
rounding of FP32 more in that storage.  A node outside the bunch keeps its value, or zero, exactly."""
import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["nsfd_o2", "nsfd_o2_sc_seeded"])
@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_FP32_BULK])
@pytest.mark.parametrize("reset", [True, False])
def test_deposit_leaves_empty_tiles(name, precision, reset):
    case = Case(name)
    g, n = case.grid, 2000
    sc = g.space_charge
    rng = np.random.default_rng(17)
    q = np.zeros((n, 11))
    for c, axis in enumerate("xyz"):
        mid = 0.5 * (getattr(g, axis + "min") + getattr(g, axis + "max"))
        d = getattr(g, "d" + axis)
        q[:, 1 + c] = mid + rng.uniform(-2.0, 2.0, n) * d
        q[:, 4 + c] = q[:, 1 + c] + rng.uniform(-0.4, 0.4, n) * d
    q[:, 0] = rng.normal(1.0, 0.1, n)
    q[:, 10] = 1.0
    kind = np.float64 if precision == abi.PRECISION_FP64 else np.float32
    j0 = (1e-3 * rng.normal(size=3 * g.nodes)).astype(kind).astype(np.float64)
    r0 = (1e-3 * rng.normal(size=g.nodes)).astype(kind).astype(np.float64)
    out = []
    for backend in ("gpu", "oracle"):
        dom = case.open(backend, precision) if backend == "gpu" else case.open(backend)
        dom.set_potentials(2, j0, r0 if sc else None)
        dom.set_particles(q)
        if reset:
            dom.current_reset()
        dom.current_update()
        j, r = dom.get_potentials(2)
        out.append(np.column_stack([j.reshape(-1, 3), r]) if sc else j.reshape(-1, 3))
    got, want = out
    before = np.column_stack([j0.reshape(-1, 3), r0]) if sc else j0.reshape(-1, 3)
    if reset:
        before = np.zeros_like(before)
    top = np.max(np.abs(want), axis=0)
    eps = 2000 * 2.0 ** -53 + (2.0 ** -24 if precision == abi.PRECISION_FP32_BULK else 0.0)
    assert np.all(np.abs(got - want) <= eps * top)
    quiet = np.all(want == before, axis=1)
    assert 0.5 < np.mean(quiet) < 1.0
    assert np.array_equal(got[quiet], before[quiet])
