"""The row-tiled deposit at the edges of its tiles and of the rule that sizes them: the last chunk of node
planes a single plane, the last tile a single row, one row per tile, the widest rows that fit, both
workgroup sizes (under and over 200 halves a workgroup), with and without rho."""
import numpy as np
import pytest

from golden_state import rel_l2
from mithra_amd import abi
from test_gpu_deposit import deposit, grid, particles

pytestmark = pytest.mark.gpu

# (N0, N1, N2), space charge, particles
CASES = [
    ((3, 3, 3), 0, 500),              # the smallest mesh: a full chunk and a plane, one interior node row
    ((4, 5, 4), 1, 2000),
    ((17, 45, 31), 0, 40000),         # 16-row tiles shrunk to fill the GPU; odd planes; few halves
    ((17, 45, 31), 1, 400),
    ((9, 70, 12), 0, 200000),         # many halves a workgroup (512 threads)
    ((34, 257, 515), 0, 60000),       # tiles not shrunk: the last one a single row
    ((5, 853, 7), 0, 20000),          # 853 nodes: the widest row of J that fits
    ((5, 640, 7), 1, 20000),          # and of J with rho
    ((5, 854, 6), 0, 20000),          # one too many: atomic adds
]


@pytest.mark.parametrize("shape,sc,n", CASES)
def test_tiles_match_oracle(shape, sc, n):
    """J and rho to the rounding of the summation order: each node sums at most some 10^4 weights, so
    1e-13 of the norm bounds it (2^-53 times the root of that count, and a margin of ten)."""
    g = grid(*shape, sc=sc)
    rec = particles(g, n, seed=sum(shape) + sc)
    for twice in (False, True):
        jg, rg = deposit(g, rec, "gpu", twice=twice)
        jo, ro = deposit(g, rec, "oracle", twice=twice)
        assert np.any(jg) == np.any(jo)     # three nodes to an axis leave no cell inside: no current
        assert np.any(jo) or min(shape) == 3
        assert rel_l2(jg, jo) < 1e-13
        if sc:
            assert rel_l2(rg, ro) < 1e-13


def test_fp32_tiles():
    g = grid(9, 70, 12, sc=1)
    rec = particles(g, 100000, seed=3)
    jg, rg = deposit(g, rec, "gpu", precision=abi.PRECISION_FP32_BULK)
    jo, ro = deposit(g, rec, "oracle")
    # one rounding of the double sum to float
    assert rel_l2(jg, jo) < 1e-7 and rel_l2(rg, ro) < 1e-7
