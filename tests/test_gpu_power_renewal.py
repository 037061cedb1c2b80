"""The power sampler's running sums against the sampler that walks the whole ring, where they have to start
afresh: samples that never meet slot 0, and values in the ring that are infinite or far larger than those
that follow.

The fields are uniform over the mesh: A^n = 0 and A^{n+1} along x of one value a step, so that E_x is that value
over the time step, B is zero, and at a frequency whose phase hardly turns over the ring every term of
the sums, of the nodes' powers and of the planes' sum has one sign.  Each of the Nf additions of the walk then
rounds by at most 2^-53 of the sum, and P is a product of two such sums: 2 Nf 2^-53, doubled for the
frequency's small sine sums."""
import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu

NF = 8
RTOL = 4 * NF * 2.0 ** -53


def sampled(values, times, copies):
    """P of the samples `times`, E_x being values[i] at the i-th."""
    case = Case("nsfd_o2")
    dom, n = case.open("gpu"), case.grid.nodes
    z = case.power._arrays[0][:1]
    w = np.full(copies, 1e-3 / case.grid.dt)
    dom.power_setup(abi.make_power_params(z, w, NF, case.power.pc, case.gamma, case.beta, case.c0), len(times))
    dom.set_potentials(0, np.zeros(3 * n))
    a = np.zeros((n, 3))
    for row, (t, v) in enumerate(zip(times, values)):
        a[:, 0] = -v * case.grid.dt
        dom.set_potentials(2, a)
        dom.field_evaluate()
        dom.power_sample(t, row)
    P = dom.power_fetch(0, len(times), 1, copies)[:, 0, 0]
    dom.close()
    return P


def both(values, times):
    return sampled(values, times, 1), sampled(values, times, NF // 8 + 1)  # 16 copies > 2 NF: no sums are kept


def agree(running, walked):
    assert np.array_equal(np.isfinite(running), np.isfinite(walked))
    ok = np.isfinite(walked)
    assert np.all(walked[ok] != 0.0)
    assert np.max(np.abs(running[ok] / walked[ok] - 1.0)) <= RTOL


@pytest.mark.parametrize("stride", [2, 3, 7])
def test_samples_that_miss_slot_0(stride):
    """A value 1e30 times those after it leaves the ring when its slot is sampled again; from the pass after
    that on, whatever slots the samples meet, nothing of it is left."""
    times = 1 + stride * np.arange(6 * NF)
    values = np.random.default_rng(stride).uniform(1.0, 2.0, len(times))
    values[1] = 1e30
    running, walked = both(values, times)
    left = 1 + len({int(t) % NF for t in times})   # the sample that takes it out
    agree(running[:left], walked[:left])
    again = left + 1 + next(i for i, t in enumerate(times[left + 1:]) if t % NF <= times[left + i] % NF)
    agree(running[again:], walked[again:])


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_that_are_not_finite(bad):
    """P is not finite while one of them is in the ring, and as exact as ever from then on: also until slot 0
    comes round, with a value 1e14 times the others in the ring when the last one leaves it."""
    times = np.arange(4 * NF)
    values = np.random.default_rng(1).uniform(1.0, 2.0, len(times))
    values[3], values[5] = bad, 1e14
    running, walked = both(values, times)
    assert np.array_equal(np.isfinite(walked), (times < 3) | (times >= 3 + NF))
    agree(running, walked)

