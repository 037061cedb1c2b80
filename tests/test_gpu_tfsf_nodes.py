"""The one-launch TF/SF injection against the oracle: meshes whose axes have five nodes (planes coincide),
six (the inner planes are neighbours) and more, so that every kind of crossing of the planes occurs, in FP64
and FP32-bulk, single and batched."""
import numpy as np
import pytest

from golden_state import Case, load_oracle, rel_l2
from mithra_amd import abi

pytestmark = pytest.mark.gpu

SIZES = [(5, 5, 5), (6, 6, 6), (7, 6, 5), (5, 9, 70), (6, 13, 40), (13, 7, 66), (20, 70, 33)]


def setup(size):
    case = Case("nsfd_o2_sc_seeded")
    g = abi.Grid.from_buffer_copy(case.grid)
    g.N0, g.N1, g.N2 = size
    rng = np.random.default_rng(sum(size))
    levels = [rng.standard_normal(3 * g.nodes) * 1e-9 for _ in range(3)]
    phis = [rng.standard_normal(g.nodes) for _ in range(3)]
    return case, g, levels, phis


def update(case, dom, levels, phis, seed):
    for lvl, (a, f) in enumerate(zip(levels, phis)):
        dom.set_potentials(lvl, a, f)
    dom.field_update(case.time0 + 3.0 * case.dt, seed)
    return dom.get_potentials(2)[0]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kind", [0, 1, 2])   # plane wave, truncated plane wave, Gaussian beam
def test_injection_matches_oracle(size, kind):
    case, g, levels, phis = setup(size)
    seed = abi.Seed.from_buffer_copy(case.seed)
    seed.seed_type = kind
    seed.amplitude *= 1e6                      # as large as the potentials it is added to
    seed.radius[:] = [3.0 * r for r in seed.radius]
    ora = update(case, abi.Domain(g, case.coeffs, lib=load_oracle(), prefix="oracle_"), levels, phis, seed)
    gpu = update(case, abi.Domain(g, case.coeffs), levels, phis, seed)
    f32 = update(case, abi.Domain(g, case.coeffs, precision=abi.PRECISION_FP32_BULK), levels, phis, seed)
    off = update(case, abi.Domain(g, case.coeffs), levels, phis, None)
    assert rel_l2(off, ora) > 1e-2             # the injection is there to be seen
    # the device's cos, exp and atan are within a few ulp of the host's
    assert rel_l2(gpu, ora) < 1e-13
    assert rel_l2(f32, ora) < 1e-6
