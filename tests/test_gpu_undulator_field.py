"""The push in an undulator's field on and off axis, against the CPU oracle: sinh and cosh of k_u y on both
sides of one radian, where the device changes from their series to the library's, inside the undulator
and in both fringes.

Both sides round every product of the field and of the Boris step; sinh, cosh, sin, cos and exp differ by a few
units in the last place.  The bound for a particle is 64 units of its largest momentum and of the field's
largest kick at its height (the kicks grow as cosh k_u y); positions are held to the bunch's largest.  Each
sub-step starts from the oracle's particles: what the field's gradient makes of a difference in
the sub-steps that follow is not the device's rounding (a position's last place, times gamma k_u and the
kick, is hundreds of units in a field this strong)."""
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
    for c, axis in enumerate("xy"):
        lo, hi = getattr(g, axis + "min"), getattr(g, axis + "max")
        q[:, 1 + c] = rng.uniform(lo + 0.05 * (hi - lo), hi - 0.05 * (hi - lo), n)
    y = np.max(np.abs(q[:, 2]))
    und = abi.Undulator()
    u = case.undulators[0]
    for name, _ in abi.Undulator._fields_:
        setattr(und, name, getattr(u, name))
    und.theta = math.pi / 2.0  # the field varies along y
    und.lu = 2.0 * math.pi * y / radians  # the farthest particle lies at k_u y = radians
    und.length = 1
    # the bunch spans half a period of the entrance fringe, the period and half a period of the exit fringe
    ahead = case.beta * case.c0 * (case.time_bunch0 + case.dt_shift)
    und.rb = case.gamma * (0.5 * (g.zmin + g.zmax) + ahead) - 0.5 * und.lu
    lz = rng.uniform(-0.5 * und.lu, 1.5 * und.lu, n)
    q[:, 3] = (lz + und.rb) / case.gamma - ahead
    assert q[:, 3].min() > g.zmin and q[:, 3].max() < g.zmax
    inside, kuy = (lz > 0.0) & (lz < und.lu), 2.0 * math.pi / und.lu * np.abs(q[:, 2])
    for where in (inside, lz < 0.0, lz > und.lu):
        assert np.sum(where & (kuy <= 1.0)) > 200
        assert radians <= 1.0 or np.sum(where & (kuy > 1.0)) > 200
    q[:, 0] = 1.0
    q[:, 4:7] = q[:, 1:4]
    q[:, 7:10] = rng.normal(0.0, 0.1, (n, 3))
    q[:, 10] = 1.0
    gpu, ora = case.open("gpu"), case.open("oracle")
    for dom in (gpu, ora):
        dom.set_potentials(0, np.zeros(3 * g.nodes))
    unit = 64 * 2.0 ** -52
    for s in range(n_sub):
        for dom in (gpu, ora):
            dom.set_particles(q)
            dom.bunch_update(case.bunch, [und], case.time_bunch0 + s * case.dtb)
        got, want = gpu.get_particles(), ora.get_particles()
        kick = np.max(np.abs(want[:, 7:10] - q[:, 7:10]), axis=1)
        assert s > 0 or np.sum(kick > 1e-6) > 0.9 * n    # the field is there to be seen, for nearly all of them
        height = np.cosh(2.0 * math.pi / und.lu * np.abs(q[:, 2]))
        own = np.maximum(np.max(np.abs(want[:, 7:10]), axis=1), np.max(np.abs(q[:, 7:10]), axis=1))
        bound = unit * (own + np.max(kick / height) * height)
        off = np.max(np.abs(got[:, 7:10] - want[:, 7:10]), axis=1)
        print(f"largest kick {kick.max():.2e}, momenta off by {np.max(off / bound):.3f} of the bound", flush=True)
        assert np.all(off <= bound)
        assert np.max(np.abs(got[:, 1:4] - want[:, 1:4])) <= unit * np.max(np.abs(want[:, 1:4]))
        assert np.array_equal(got[:, 10], want[:, 10])
        q = want
