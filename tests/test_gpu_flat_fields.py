"""The flat form of the field kernels (tile shape 0) at the sizes where its plane index, its boundary
lanes and its planes per workgroup can go wrong: N1 around the wavefront and at its smallest, meshes of
three planes, and meshes large enough for each number of planes per workgroup."""
import numpy as np
import pytest

from mithra_amd import abi
from golden_state import load_oracle
from test_gpu_fields import grid

pytestmark = pytest.mark.gpu

# (N0, N1, N2): N1 = 3 leaves the y faces to the boundary pass, 4 is the first that takes them
SIZES = [(5, 3, 7), (6, 4, 9), (3, 5, 3), (9, 63, 11), (9, 64, 12), (7, 66, 5), (20, 257, 6), (61, 131, 91)]


def coeffs(rng):
    c = abi.Coeffs()
    for name, n in (("a", 6), ("bB", 5), ("cB", 5), ("dB", 5), ("eE", 5), ("fE", 5), ("gE", 5), ("hC", 17)):
        getattr(c, name)[:] = rng.uniform(-1.0, 1.0, n)
    c.hC[0] = 2.5
    c.alpha, c.beta = 1.1, 0.07
    return c


def update(dom, levels, phis):
    for lvl, a in enumerate(levels):
        dom.set_potentials(lvl, a, phis[lvl])
    dom.field_update(0.0, None)
    a, phi = dom.get_potentials(2)
    return [a, *dom.get_fields()] + ([] if phi is None else [phi])


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("sc", [0, 1])
@pytest.mark.parametrize("solver", [abi.SOLVER_NSFD, abi.SOLVER_FD])
def test_flat_field_update_bit_exact(size, sc, solver):
    """One unseeded field update in FP64 against the oracle, bit for bit (the same operations in the
    same order), and in FP32-bulk against the LDS-staged shape, which computes the same expressions."""
    g = grid(*size, sc)
    g.solver = solver
    rng = np.random.default_rng(sum(size) + sc)
    c, n = coeffs(rng), g.nodes
    levels = [rng.standard_normal(3 * n) * 1e-6 for _ in range(3)]
    phis = [rng.standard_normal(n) if sc else None for _ in range(3)]
    flat = abi.Domain(g, c)
    flat.set_tiles(0, 0)
    ref = update(abi.Domain(g, c, lib=load_oracle(), prefix="oracle_"), levels, phis)
    for a, b in zip(update(flat, levels, phis), ref):
        assert np.array_equal(a, b)
    out = []
    for shape in (0, 7):
        d = abi.Domain(g, c, precision=abi.PRECISION_FP32_BULK)
        d.set_tiles(shape, shape)
        out.append(update(d, levels, phis))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nodes,precision,shapes", [((20, 20, 20), abi.PRECISION_FP64, (0, 0)),
                                                    ((200, 180, 150), abi.PRECISION_FP64, (7, 0)),
                                                    ((200, 128, 320), abi.PRECISION_FP64, (7, 8)),
                                                    ((200, 180, 150), abi.PRECISION_FP32_BULK, (0, 0))])
def test_default_shapes_match_flat(nodes, precision, shapes):
    """A domain's starting shapes on both sides of sizes in the rule are the ones it names and compute what
    the flat form computes."""
    g = grid(*nodes, 0)
    rng = np.random.default_rng(3)
    c, n = coeffs(rng), g.nodes
    levels = [rng.standard_normal(3 * n) * 1e-6 for _ in range(3)]
    out = []
    for tiles in (None, (0, 0), shapes):
        d = abi.Domain(g, c, precision=precision)
        assert d.tiles()[:2] == shapes
        if tiles:
            d.set_tiles(*tiles)
        out.append(update(d, levels, [None] * 3))
    for got in out[1:]:
        for a, b in zip(got, out[0]):
            assert np.array_equal(a, b)
