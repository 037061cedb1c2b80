"""The power sampler's running DFT sums against the sampler that walks the whole ring.

The running sums are kept up to 16 doubles a node per frequency in half the ring's memory; a set-up
with more frequencies walks the ring at every sample.  Both run on one march of a golden job for more
than two passes over the ring (the sums start afresh each pass), sampled at every step, with gaps in
n_time, and with a time that is sampled twice."""
import numpy as np
import pytest

from golden_state import Case
from mithra_amd import abi

pytestmark = pytest.mark.gpu

# The walk over the ring rounds each of its Nf additions: Nf 2^-53 < 5e-15 of the terms' sum of magnitudes for
# the 40 slots here.  P is a difference of products of such sums, added over nodes of both signs; 1e-11 of the
# largest P leaves room for what these cancel, a factor of 2000.  (Where nothing cancels, the samplers are held
# to their roundings in test_gpu_power_renewal.py.)
RTOL = 1e-11


def sampled(case, nf, copies, times):
    z, w = case.power._arrays
    dom = case.open("gpu")
    dom.power_setup(abi.make_power_params(z, np.repeat(w, copies), nf, case.power.pc, case.gamma, case.beta, case.c0),
                    len(times))
    time, tb = case.time0, case.time_bunch0
    for row, n in enumerate(times):
        dom.field_update(time, case.seed)
        dom.bunch_advance(case.bunch, case.undulators, tb, case.dtb, case.n_sub)
        dom.power_sample(n, row)
        dom.field_shift()
        dom.current_reset()
        dom.current_update()
        tb += case.dtb * case.n_sub
        time += case.dt
    P = dom.power_fetch(0, len(times), len(z), copies * len(w))
    dom.close()
    return P


@pytest.mark.parametrize("nf", [8, 17, 40])
def test_running_sums_match_the_ring(nf):
    case = Case("nsfd_o2_sc_seeded")
    times = list(range(2 * nf + 5)) + [2 * nf + 5, 2 * nf + 5, 3 * nf + 9, 7 * nf]
    running = sampled(case, nf, 1, times)
    walked = sampled(case, nf, nf // 8 + 1, times)     # 16 copies > 2 nf: no sums are kept
    assert np.abs(walked).max() > 0.0
    scale = np.abs(walked).max()
    for c in range(walked.shape[2]):
        assert np.abs(running[:, :, 0] - walked[:, :, c]).max() <= RTOL * scale


def test_planes_and_frequencies():
    """Several planes, one of them outside the domain (its rows stay zero), and frequencies that
    repeat give each (plane, frequency) the single set-up's power."""
    case = Case("nsfd_o2_sc_seeded")
    z, w = (np.asarray(a) for a in case.power._arrays)
    many_z = np.array([z[0], case.grid.zmax + 10.0 * case.grid.dz, z[0] - 3.0 * case.grid.dz])
    many_w = np.array([w[0], 1.1 * w[0], w[0]])
    steps = 30
    out = []
    for zz, ww in ((many_z, many_w), (z[:1], w[:1])):
        dom = case.open("gpu")
        dom.power_setup(abi.make_power_params(zz, ww, 40, case.power.pc, case.gamma, case.beta, case.c0), steps)
        time, tb = case.time0, case.time_bunch0
        for n in range(steps):
            dom.step(time, case.seed, case.bunch, case.undulators, tb, case.dtb, case.n_sub, n, n)
            tb += case.dtb * case.n_sub
            time += case.dt
        out.append(dom.power_fetch(0, steps, len(zz), len(ww)))
        dom.close()
    many, one = out
    assert np.all(many[:, 1] == 0.0)
    scale = np.abs(one).max()
    assert np.abs(many[:, 0, 0] - one[:, 0, 0]).max() <= RTOL * scale
    assert np.array_equal(many[:, 0, 0], many[:, 0, 2])
    assert np.abs(many[:, 0, 1]).max() > 0.0 and not np.array_equal(many[:, 0, 0], many[:, 2, 0])
