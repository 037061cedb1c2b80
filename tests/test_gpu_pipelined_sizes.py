"""The pipelined step against the plain one on both sides of the 5 million nodes where the fused kernel's shape 0
changes from the flat form to 4 x 64 tiles, on a mesh whose N1 is no multiple of 64.

Particles lie at least four cells apart, so that no node receives more than two contributions and the deposit's
order of adding them does not matter; then every bit agrees (see test_gpu_pipelined.py)."""
import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu

BELOW, ABOVE = (131, 147, 259), (131, 147, 260)  # 4.99 and 5.01 million nodes


def inputs(size, sc, solver):
    case = Case("nsfd_o2_sc" if sc else "nsfd_o2")
    g = abi.Grid.from_buffer_copy(case.grid)
    g.N0, g.N1, g.N2 = size
    g.solver = solver
    for axis, n in zip("xyz", size):
        d = getattr(g, "d" + axis)
        setattr(g, axis + "min", -0.5 * (n - 1) * d)
        setattr(g, axis + "max", 0.5 * (n - 1) * d)
    g.zp0, g.zp1 = g.zmin, g.zmax
    rng = np.random.default_rng(sum(size) + sc)
    levels = [(rng.standard_normal(3 * g.nodes) * 1e-9, rng.standard_normal(g.nodes) * 1e-3 if sc else None)
              for _ in range(2)]
    # one particle in every 4 x 4 x 4 cells of a coarse lattice's corner, some next to the faces
    at = np.array([(i, j, k) for i in (1, 20, 64, 127) for j in (1, 63, 64 + 8, 140) for k in range(1, size[2] - 4, 8)])
    q = np.zeros((len(at), 11))
    for c, axis in enumerate("xyz"):
        q[:, 1 + c] = getattr(g, axis + "min") + (at[:, c] + rng.uniform(0.2, 0.8, len(at))) * getattr(g, "d" + axis)
    q[:, 0] = case.arr("pre0_particles").reshape(-1, 11)[0, 0]
    q[:, 4:7] = q[:, 1:4]
    q[:, 10] = 1.0
    return case, g, levels, q


def march(case, g, levels, q, pipelined, shape=None):
    dom = abi.Domain(g, case.coeffs)
    if shape is not None:
        dom.set_fused_tile(shape)
    for level, (a, phi) in enumerate(levels):
        dom.set_potentials(level, a, phi)
    dom.set_particles(q)
    dom.current_update()
    time, tb, steps = case.time0, case.time_bunch0, 3
    for n in range(steps):
        args = (time, None, case.bunch, case.undulators, tb, case.dtb, case.n_sub, n)
        if pipelined:
            dom.step_pipelined(*args, more=n < steps - 1)
            assert dom.pipeline_pending() == (n < steps - 1)
        else:
            dom.step(*args)
        time += case.dt
        tb += case.n_sub * case.dtb
    out = [dom.get_particles(), *dom.get_fields()]
    for level in (0, 1, 2):
        out += [a for a in dom.get_potentials(level) if a is not None]
    dom.close()
    return out


@pytest.mark.parametrize("size,sc,solver", [(BELOW, 0, abi.SOLVER_NSFD), (BELOW, 1, abi.SOLVER_NSFD),
                                            (ABOVE, 0, abi.SOLVER_NSFD), (ABOVE, 1, abi.SOLVER_NSFD),
                                            (ABOVE, 0, abi.SOLVER_FD)])
def test_pipelined_is_the_plain_step(size, sc, solver):
    made = inputs(size, sc, solver)
    plain = march(*made, False)
    assert all(np.all(np.isfinite(a)) and np.any(a) for a in plain)
    shapes = (None, 0, 1, 2, 3) if size == ABOVE and solver == abi.SOLVER_NSFD else (None,)
    for shape in shapes:
        for i, (a, b) in enumerate(zip(march(*made, True, shape), plain)):
            assert np.array_equal(a, b), (shape, i)
