"""The batch's row orders: instances whose row counts lie around the scan's blocks of 1024, marched together and
one by one, and a batch with more rows than one launch of the scan takes.  Both ways differ only in
the order of the deposit's additions, as in the batch's own test (1e-12 over some 90 steps; the long mesh marches
90 of its 2100, over which the bunching would grow from that rounding as it grows from noise)."""
import tempfile

import numpy as np
import pytest

from golden_state import rel_l2
from mithra_amd import abi, scan

pytestmark = pytest.mark.gpu


class Short(scan.Instance):
    n_steps = 90


@pytest.mark.parametrize("shapes", [
    [(16, 63, 400), (16, 64, 4096), (16, 65, 4100), (32, 97, 2000), (31, 100, 257)],
    [(64, 2100, 3000), (16, 65, 500)],
], ids=["blocks", "long"])
def test_orders_match_single_runs(shapes):
    tol = 1e-12
    insts = scan.generate(len(shapes), seed=23, n_perp=(16, 16), n_z=(64, 64), n_particles=(500, 500))
    for i, (perp, z, n) in zip(insts, shapes):
        i.n_perp, i.n_z, i.n_particles = perp, z, n
        if z > 90:
            i.__class__ = Short
    with tempfile.TemporaryDirectory() as w1, tempfile.TemporaryDirectory() as w2:
        single = scan.prepare(insts, w1, abi.PRECISION_FP64)
        batch = scan.prepare(insts, w2, abi.PRECISION_FP64)
        rows = [(p.dom.grid.N2 - 1) * p.dom.grid.N0 for p in batch]
        print("rows", rows, flush=True)
        assert (max(rows) >= 1 << 17) == (shapes[0][1] == 2100)
        res_s, _ = scan.run_single(single)
        res_b, _, _ = scan.run_batch(batch, autotune=False)
        for p, q, (ps, bs), (pb, bb) in zip(single, batch, res_s, res_b):
            assert rel_l2(pb, ps) <= tol
            assert np.max(np.abs(bb - bs)) <= tol * max(1e-3, np.max(np.abs(bs)))
            assert rel_l2(q.dom.get_particles(), p.dom.get_particles()) <= tol
