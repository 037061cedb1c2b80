"""Reads of a domain's state in chunks: what was written comes back bit for bit, in the caller's layout and
load order, for sizes of one chunk and of many with a ragged last one."""
import ctypes as C

import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu


def _domain(shape, precision, space_charge):
    case = Case("nsfd_o2_sc_seeded" if space_charge else "nsfd_o2")
    g = abi.Grid()
    C.memmove(C.byref(g), C.byref(case.grid), C.sizeof(g))
    g.N0, g.N1, g.N2 = shape
    g.space_charge = space_charge
    for axis, n in zip("xyz", shape):
        d = getattr(g, "d" + axis)
        setattr(g, axis + "min", -0.5 * (n - 1) * d)
        setattr(g, axis + "max", 0.5 * (n - 1) * d)
    g.zp0, g.zp1 = g.zmin, g.zmax
    return abi.Domain(g, case.coeffs, precision=precision)


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_FP32_BULK])
@pytest.mark.parametrize("space_charge", [0, 1])
@pytest.mark.parametrize("shape", [(7, 9, 11), (61, 67, 97)])
def test_fields_come_back(shape, space_charge, precision):
    rng = np.random.default_rng(sum(shape))
    dom = _domain(shape, precision, space_charge)
    n = dom.grid.nodes
    want = []
    for level in (0, 1, 2):
        a, phi = rng.normal(size=3 * n), rng.normal(size=n)
        dom.set_potentials(level, a, phi if space_charge else None)
        want.append((a, phi))
    kind = np.float64 if precision == abi.PRECISION_FP64 else np.float32
    for level in (0, 1, 2):
        a, phi = dom.get_potentials(level)
        assert np.array_equal(a, want[level][0].astype(kind).astype(np.float64))
        if space_charge:
            assert np.array_equal(phi, want[level][1].astype(kind).astype(np.float64))
    dom.field_evaluate()
    e, b = dom.get_fields()
    assert np.any(e) and np.any(b)
    fp = C.POINTER(C.c_float)
    for which in (0, 1):  # one of the two alone
        out = np.empty(3 * n, np.float32)
        ptr = out.ctypes.data_as(fp)
        assert dom.f["get_fields"](dom.h, ptr if which == 0 else None, ptr if which == 1 else None) == 0
        assert np.array_equal(out, (e, b)[which])
    a0, phi0 = dom.get_potentials(0)
    for count in (1, 257, 70001):
        at = rng.integers(0, n, count)
        se, sb, sa, sphi = dom.sample_nodes(at)
        assert np.array_equal(se, e.reshape(n, 3)[at]) and np.array_equal(sb, b.reshape(n, 3)[at])
        assert np.array_equal(sa, a0.reshape(n, 3)[at])
        assert np.array_equal(sphi, phi0[at] if space_charge else np.zeros(count))


@pytest.mark.parametrize("n", [1, 63, 2978, 2979, 5957, 5958, 40001])  # 5957 records: the last that fit one slot
def test_particles_come_back_in_load_order(n):
    rng = np.random.default_rng(n)
    dom = _domain((32, 32, 64), abi.PRECISION_FP64, 0)
    g = dom.grid
    q = rng.normal(size=(n, 11))
    for c, axis in enumerate("xyz"):
        lo, hi = getattr(g, axis + "min"), getattr(g, axis + "max")
        q[:, 1 + c] = rng.uniform(lo + 0.2 * (hi - lo), hi - 0.2 * (hi - lo), n)
    q[:, 4:7] = q[:, 1:4]
    q[:, 10] = 0.0
    dom.set_particles(q)
    assert np.array_equal(dom.get_particles(), q)
    dom.set_reorder_interval(1)
    for _ in range(3):  # the arrays are put into the order of the cells
        dom.current_reset()
        dom.current_update()
    assert np.array_equal(dom.get_particles(), q)
