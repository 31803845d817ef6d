"""The boundary-face launch at the sizes where its rows, row segments and box
edges end: the smallest mesh, rows one cell shorter and longer than a segment
of 64, several segments.  Faces, edges and probe points on faces must be the
oracle's bits in FP64, and a batch of such members what each gives alone."""
import numpy as np
import pytest

from helpers import random_start, run_from, spec_from, uniform_crystal
from phonomena_amd import fdtd, problem

pytestmark = pytest.mark.gpu
FIELDS = ["ux", "uy", "uz", "ux_old", "uy_old", "uz_old"]
NODES = [(4, 4, 4), (4, 6, 5), (6, 9, 65), (7, 5, 66), (5, 12, 67), (9, 7, 131), (30, 4, 20), (19, 40, 9)]


def _problem(nodes, steps=24):
    return uniform_crystal([n - 1 for n in nodes], 0.3, incl=(19300.0, 2.0e11, 1.6e11, 8, 3), steps=steps, seed=3)


def _spec(nodes, every, **kw):
    return spec_from(*_problem(nodes, **kw), probe=(0, 1, nodes[0], 0, 1, nodes[1]), every=every)


@pytest.mark.parametrize("nodes", NODES)
def test_faces_bitwise_vs_oracle(nodes):
    from oracle import brute
    steps = 3 * max(nodes)  # the front (half a cell a step) reaches every face
    x, y, z, ids, rows, dt, wave = _problem(nodes, steps)
    fd = [np.diff(a) for a in (x, y, z)]
    sd = [np.mean([f[1:], f[:-1]], axis=0) for f in fd]
    mur = problem.mur_coefficients(rows[int(ids[0, 0, 0])], np.float64(dt), fd, sd)
    probe = (0, 1, nodes[0], 0, 1, nodes[1])
    st, frames = brute.run(x, y, z, ids, rows, dt, mur, wave, steps, probe=probe, every=3)
    ctx = fdtd.Context(spec_from(x, y, z, ids, rows, dt, wave, probe=probe, every=3), precision="fp64", kernel="tiled")
    ctx.step(steps)
    for f in ("ux", "uy", "uz"):
        assert np.array_equal(ctx.get(f), st[f]), f
    assert np.array_equal(ctx.probes(), frames)
    ctx.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
def test_batch_of_edge_sizes_equals_alone(precision):
    steps = 21  # a group of captured steps, then loose ones, whose frames go on counting
    specs = [_spec(n, every=2 + i % 3) for i, n in enumerate(NODES)]
    starts = [random_start(n, i) for i, n in enumerate(NODES)]
    ref = [run_from(s, st, precision, "tiled", steps) for s, st in zip(specs, starts)]
    b = fdtd.Batch(precision)
    ctxs = [fdtd.Context(s, precision=precision) for s in specs]
    for c, st in zip(ctxs, starts):
        for f in ("ux", "uy", "uz"):
            c.set(f, st[f])
            c.set(f + "_old", 0.5 * st[f])
        b.add(c)
    b.step(16)
    b.step(steps - 16)
    b.sync()
    for i, c in enumerate(ctxs):
        for f in FIELDS:
            assert np.array_equal(c.get(f), ref[i][f]), (NODES[i], f)
        assert np.array_equal(c.probes(), ref[i]["probes"]), NODES[i]
    b.close()
    # the counters the batch left are those of stepping alone
    for c, s, st in zip(ctxs, specs, starts):
        c.step(3)
        c.sync()
        more = run_from(s, st, precision, "tiled", steps + 3)
        assert np.array_equal(c.get("uz"), more["uz"]) and np.array_equal(c.probes(), more["probes"])
        c.close()
