"""The counting order's row starts and the lazy evaluation's bunch extent.

Row starts: meshes whose row counts end inside, at and past a workgroup's chunk of the scan (4096 rows,
up to 2^17) and one row count above it, deposited and compared with the oracle, which needs every
particle in its row.  Extent: a lazy march gives the same particles and power as one that evaluates
E/B everywhere, whichever of the deposit and the evaluation comes first after a push."""
import numpy as np
import pytest

from golden_state import Case, rel_l2
from test_gpu_deposit import deposit, grid, particles

pytestmark = pytest.mark.gpu


# (N2 - 1) N0 rows: 4095, 4096, 4097, 8192, 12288, 131070, 131072
@pytest.mark.parametrize("shape", [(39, 6, 106), (64, 5, 65), (17, 6, 242), (4, 6, 2049), (96, 5, 129),
                                   (255, 5, 515), (256, 5, 513)])
def test_rows_match_oracle(shape):
    nx, ny, nz = shape
    g = grid(nx, ny, nz)
    rec = particles(g, 20000, seed=nx)
    jg, _ = deposit(g, rec, "gpu")
    jo, _ = deposit(g, rec, "oracle")
    assert np.any(jo)
    assert rel_l2(jg, jo) < 1e-13


@pytest.mark.parametrize("order", ["deposit", "no_deposit", "two_pushes"])
@pytest.mark.parametrize("fixed", [False, True])
def test_lazy_extent(order, fixed):
    case = Case("nsfd_o2")
    out = []
    for lazy in (0, 1):
        dom = case.open("gpu")
        dom.set_lazy_fields(lazy)
        if fixed:
            dom.set_deterministic(True)
        time, tb = case.time0, case.time_bunch0
        for step in range(12):
            dom.field_update(time, case.seed)
            for _ in range(2 if order == "two_pushes" else 1):
                dom.bunch_advance(case.bunch, case.undulators, tb, case.dtb, 1)
                tb += case.dtb
            dom.power_sample(step, step)
            dom.field_shift()
            dom.current_reset()
            if order != "no_deposit" or step % 3 == 0:
                dom.current_update()
            time += case.dt
        out.append((dom.get_particles(), dom.power_fetch(0, 12, case.power_N, case.power_Nl)))
        dom.close()
    for a, b in zip(*out):
        # fixed order: the same sums; else the deposit's summation order, carried through 12 steps
        assert np.array_equal(a, b) if fixed else rel_l2(b, a) < 1e-12
