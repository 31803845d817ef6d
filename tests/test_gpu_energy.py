"""The energy audit against the oracle's on meshes at the edges of its
chunks and blocks: one partial block, one more plane than a chunk, planes
of several blocks, graded spacings, and more than one material row."""
import numpy as np
import pytest

from helpers import random_start, spec_from
from oracle import reference_math as rm
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,h", [((4, 4, 4), 1.0), ((5, 16, 16), 0.3), ((37, 11, 9), 1.0), ((33, 40, 23), 0.7)])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
def test_energy_equals_the_oracle_on_chunk_edges(nodes, h, precision):
    rng = np.random.default_rng(3)
    x, y, z = (np.concatenate([[0.0], np.cumsum(h * rng.uniform(0.8, 1.2, n - 1))]) for n in nodes)
    tables = []
    for _ in range(3):
        c = np.zeros((6, 6))
        c[:3, :3] = rng.uniform(0.5, 1.0, (3, 3)) + 2 * np.eye(3)
        c[[3, 4, 5], [3, 4, 5]] = rng.uniform(0.3, 0.9, 3)
        tables.append(c)
    rho = rng.uniform(0.5, 2.0, 3)
    ids = rng.integers(0, 3, nodes).astype(np.uint8)
    rows = np.array([np.concatenate([c[:3, :3].ravel(), np.diag(c)[3:], [r]]) for c, r in zip(tables, rho)])
    dt = np.float64(0.1 * h)
    wave = rng.standard_normal(3)
    spec = spec_from(x, y, z, ids, rows, dt, wave)
    start = random_start(nodes, 5)
    C, P = rm.dense_material(ids, tables, rho)
    pb = rm.Problem(x, y, z, C, P, dt, wave)
    ctx = fdtd.Context(spec, precision=precision)
    try:
        for f in ("ux", "uy", "uz"):
            ctx.set(f, start[f])
            ctx.set(f + "_old", 0.5 * start[f])
        s = rm.State(*nodes)
        for f in ("ux", "uy", "uz"):
            getattr(s, f)[...] = start[f]
            getattr(s, f + "_new")[...] = start[f]
            getattr(s, f + "_old")[...] = 0.5 * start[f]
        for tt in range(3):
            ctx.step(1)
            rm.step(s, pb, tt)
            # FP64: a few ulp a term and the order of the sum; FP32: the
            # fields' rounding, 2^-24 a value and step in a quadratic form
            tol = 1e-13 if precision == "fp64" else 2e-6
            e, ref = ctx.energy(), rm.energy(s, pb)
            assert abs(e - ref) <= tol * abs(ref)
    finally:
        ctx.close()
