"""The push in an undulator's field on and off axis, against the CPU oracle: sinh and cosh of k_u y on both
sides of one radian, where the device changes from their series to the library's, in the undulator
and in both fringes.

Both sides round every product of the field and of the Boris step; sinh, cosh, sin, cos and exp differ by a few
units in the last place, which the field's gradient carries into the next sub-step (an input 4 units off
ends 46 off after three).  The bound is 64 units of the largest momentum for each sub-step."""
import math

import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sub", [1, 3])
@pytest.mark.parametrize("radians", [0.3, 1.0, 4.0])
def test_push_matches_oracle(radians, n_sub):
    case = Case("nsfd_o2")
    g, n = case.grid, 4099
    rng = np.random.default_rng(int(10 * radians) + n_sub)
    q = np.zeros((n, 11))
    for c, axis in enumerate("xyz"):
        lo, hi = getattr(g, axis + "min"), getattr(g, axis + "max")
        q[:, 1 + c] = rng.uniform(lo + 0.05 * (hi - lo), hi - 0.05 * (hi - lo), n)
    y = np.sort(np.abs(q[:, 2]))[-1]
    und = abi.Undulator()
    u = case.undulators[0]
    for name, _ in abi.Undulator._fields_:
        setattr(und, name, getattr(u, name))
    und.theta = math.pi / 2.0  # the field varies along y
    und.lu = 2.0 * math.pi * y / radians  # the farthest particle lies at k_u y = radians
    # the bunch spans the entrance fringe, the periods and the exit fringe
    und.length = 1
    lab = case.gamma * (q[:, 3] + case.beta * case.c0 * (case.time_bunch0 + case.dt_shift))
    und.rb = 0.5 * (lab.min() + lab.max()) - 0.5 * und.lu
    q[:, 0] = 1.0
    q[:, 4:7] = q[:, 1:4]
    q[:, 7:10] = rng.normal(0.0, 0.1, (n, 3))
    q[:, 10] = 1.0
    out = []
    for backend in ("gpu", "oracle"):
        dom = case.open(backend)
        dom.set_potentials(0, np.zeros(3 * g.nodes))
        dom.set_particles(q)
        for s in range(n_sub):
            dom.bunch_update(case.bunch, [und], case.time_bunch0 + s * case.dtb)
        out.append(dom.get_particles())
    got, want = out
    assert np.max(np.abs(want[:, 7:10] - q[:, 7:10])) > 1e-6
    for cols in (slice(1, 4), slice(7, 10)):
        assert np.max(np.abs(got[:, cols] - want[:, cols])) <= 64 * n_sub * 2.0 ** -52 * np.max(np.abs(want[:, cols]))
    assert np.array_equal(got[:, 10], want[:, 10])
