"""A step's push and power sample in one launch against the two calls: the same bits, for particle counts around
a workgroup's, with and without planes to sample, and in the timed step, which keeps them apart."""
import numpy as np
import pytest

from golden_state import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["nsfd_o2", "nsfd_o2_sc_seeded", "fd_o1_array", "nsfd_o2_optical"])
@pytest.mark.parametrize("n", [0, 1, 255, 257, None])
def test_step_samples_as_the_calls_do(name, n):
    case = Case(name)
    q = case.arr("pre0_particles")
    q = q if n is None else np.resize(q, (n, 11))
    doms = [case.open("gpu") for _ in range(3)]
    for d in doms:
        d.set_particles(q)
    calls, step, timed = doms
    calls.field_update(case.time0, case.seed)
    calls.bunch_advance(case.bunch, case.undulators, case.time_bunch0, case.dtb, case.n_sub)
    calls.power_sample(0, 0)
    args = (case.time0, case.seed, case.bunch, case.undulators, case.time_bunch0, case.dtb, case.n_sub, 0, 0)
    step.step(*args)
    timed.step_timed(*args)
    rows = [d.power_fetch(0, 1, case.power_N, case.power_Nl) for d in doms]
    parts = [d.get_particles() for d in doms]
    for r, p in zip(rows[1:], parts[1:]):
        assert np.array_equal(r, rows[0])
        assert np.array_equal(p, parts[0])
