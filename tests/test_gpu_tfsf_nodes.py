"""The one-launch TF/SF injection against the oracle: meshes whose axes have five nodes (planes coincide),
six (the inner planes are neighbours) and more, so that every kind of crossing of the planes occurs, in FP64
and FP32-bulk; and a batch of them against the single domains."""
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


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_FP32_BULK])
def test_batched_injection_is_the_single_one(precision):
    """A batch of all the meshes, with a seed each, against each mesh stepped by itself: the same
    injections from the same expressions.  One particle, so that the deposit adds in one order."""
    seeds, single, batch, bare = [], [], [], []
    for i, size in enumerate(SIZES):
        case, g, levels, phis = setup(size)
        seed = abi.Seed.from_buffer_copy(case.seed)
        seed.seed_type = i % 3
        seed.amplitude *= 1e6
        seed.radius[:] = [3.0 * r for r in seed.radius]
        seeds.append(seed)
        q = np.zeros((1, 11))
        q[0, 0], q[0, 10] = 1.0, 1.0
        for c, axis in enumerate("xyz"):
            lo, d = getattr(g, axis + "min"), getattr(g, "d" + axis)
            q[0, 1 + c] = q[0, 4 + c] = lo + 2.4 * d
        for doms in (single, batch, bare):
            doms.append(abi.Domain(g, case.coeffs, precision=precision))
            for lvl, (a, f) in enumerate(zip(levels, phis)):
                doms[-1].set_potentials(lvl, a, f)
            doms[-1].set_particles(q)
    steps, time = 2, case.time0 + 3.0 * case.dt
    b = abi.Batch(batch)
    for i, seed in enumerate(seeds):
        b.instance(i, time, case.time_bunch0, case.dtb, case.n_sub, steps, case.bunch, case.undulators)
        b.seed(i, seed)
    assert b.run(steps) == steps
    for doms, with_seed in ((single, True), (bare, False)):
        for dom, seed in zip(doms, seeds):
            for n in range(steps):
                dom.step(time + n * case.dt, seed if with_seed else None, case.bunch, case.undulators,
                         case.time_bunch0 + n * case.n_sub * case.dtb, case.dtb, case.n_sub, n)
    for size, one, many, off in zip(SIZES, single, batch, bare):
        a, ref = many.get_potentials(0)[0], one.get_potentials(0)[0]
        assert rel_l2(off.get_potentials(0)[0], ref) > 1e-2, size
        assert np.array_equal(a, ref), size
    b.close()
