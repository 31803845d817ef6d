"""Block steps of small meshes (several whole steps a launch) against the
per-node sweep with its face and probe kernels: the same bits in every
field of both levels and every probe frame, whatever the step counts of the
calls, on meshes of one and of many blocks per axis."""
import numpy as np
import pytest

from helpers import FIELDS, random_start, spec_from
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu


def _spec(nodes, h, graded, sponge, surface, every, steps):
    """A mesh of random materials (asymmetric normal block), a random source and a probe grid on the faces' cells too."""
    rng = np.random.default_rng(sum(nodes))
    ax = []
    for n in nodes:
        f = np.full(n - 1, h)
        if graded:
            f = h * rng.uniform(0.7, 1.4, n - 1)
        ax.append(np.concatenate([[0.0], np.cumsum(f)]))
    rows = []
    for _ in range(5):
        c = rng.uniform(0.5, 1.0, (3, 3)) + np.eye(3) * 2.0
        rows.append(np.concatenate([c.ravel(), rng.uniform(0.3, 0.9, 3), [rng.uniform(0.5, 2.0)]]))
    rows = np.array(rows)
    ids = rng.integers(0, 5, nodes).astype(np.uint8)
    layers = [rng.uniform(0.0, 0.1, n) for n in nodes] if sponge else None
    spec = spec_from(*ax, ids, rows, 0.2 * h * 0.7, rng.standard_normal(steps), probe=(0, 1, nodes[0], 0, 1, nodes[1]),
                     every=every, sponge=layers)
    spec.surface = surface
    return spec


def _run(spec, start, precision, kernel, calls):
    ctx = fdtd.Context(spec, precision=precision, kernel=kernel)
    try:
        for c in ("ux", "uy", "uz"):
            ctx.set(c, start[c])
            ctx.set(c + "_old", 0.5 * start[c])
        for n in calls:
            ctx.step(n)
        out = {f: ctx.get(f) for f in FIELDS}
        out["probes"] = ctx.probes()
    finally:
        ctx.close()
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("nodes,h,graded,sponge,surface,every", [
    ((4, 4, 4), 1.0, False, False, 0, 1),      # the smallest mesh: one block
    ((5, 6, 7), 0.3, False, True, 1, 2),
    ((31, 21, 6), 1.0, False, False, 0, 3),    # whole columns, halo in x and y
    ((12, 9, 40), 0.5, False, True, 0, 1),     # boxes cut along z
    ((58, 39, 13), 0.3, True, True, 1, 4),     # graded, cut along every axis
    ((41, 64, 23), 0.7, True, False, 0, 5),    # the largest boxes
])
def test_block_steps_equal_the_per_node_sweep(precision, nodes, h, graded, sponge, surface, every):
    calls = (1, 2, 3, 4, 5, 8)  # single, remainders of every launch size
    spec = _spec(nodes, h, graded, sponge, surface, every, sum(calls))
    start = random_start(nodes, 7)
    got = _run(spec, start, precision, "auto", calls)
    want = _run(spec, start, precision, "naive", calls)
    for f in want:
        assert np.all(np.isfinite(want[f])), f
        assert np.array_equal(got[f], want[f]), f
