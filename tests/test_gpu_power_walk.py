"""The cost of a power sample with many frequencies, whose running sums would take more than half the ring's
memory, so that each sample walks the ring: the loads of a walk have to be in flight together.

The bound is four times what the card's copy rate gives for the ring's bytes, once for each frequency.  Waiting
for each load in turn costs eleven times; the walk as it should be is within two."""
import time

import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu


def test_walk_streams():
    case, nl, nf, n = Case("nsfd_o2"), 40, 140, 128
    g = abi.Grid.from_buffer_copy(case.grid)
    g.N0, g.N1, g.N2 = n, n, 16
    for axis, m in zip("xyz", (n, n, 16)):
        d = getattr(g, "d" + axis)
        setattr(g, axis + "min", -0.5 * (m - 1) * d)
        setattr(g, axis + "max", 0.5 * (m - 1) * d)
    g.zp0, g.zp1 = g.zmin, g.zmax
    dom = abi.Domain(g, case.coeffs)
    w = np.linspace(0.9, 1.1, nl) * case.power._arrays[1][0]
    dom.power_setup(abi.make_power_params([0.0], w, nf, case.power.pc, case.gamma, case.beta, case.c0), 1)
    took = []
    for step in range(12):
        dom.synchronize()
        t = time.perf_counter()
        dom.power_sample(step, 0)
        dom.synchronize()
        took.append(time.perf_counter() - t)
    floor = nl * nf * 4 * 8 * (n - 4) ** 2 / (abi.copy_bandwidth(256 << 20, 5) * 1e9)
    print(f"median {np.median(took) * 1e6:.0f} us, ring's bytes {floor * 1e6:.0f} us", flush=True)
    assert np.median(took) <= 4.0 * floor
    dom.close()
