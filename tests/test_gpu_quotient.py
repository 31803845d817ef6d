"""FP64 on spacings that are not powers of two against the per-node sweep,
which divides: the same bits over the displacements' whole range.  The tiled
sweep takes quotients from reciprocals where stiffnesses are within their
range, and a tile falls back to divisions for tiny and huge values, zeros
among them (the mesh with a layer here; interior tiles without one in
test_gpu_quotient_tiles.py); block steps, and the tiled sweep at stiffnesses
out of the range, divide."""
import numpy as np
import pytest

from helpers import FIELDS, spec_from
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu


def _spec(nodes, h, stiffness, steps, sponge=False):
    rng = np.random.default_rng(nodes[0])
    x, y, z = (np.concatenate([[0.0], np.cumsum(h * rng.uniform(0.7, 1.5, n - 1))]) for n in nodes)
    rows = []
    for _ in range(4):
        c = rng.uniform(0.5, 1.0, (3, 3)) + 2 * np.eye(3)
        rows.append(np.concatenate([c.ravel() * stiffness, rng.uniform(0.3, 0.9, 3) * stiffness, [rng.uniform(0.5, 2.0)]]))
    rows = np.array(rows)
    rows[1, 1] = 0.0  # an entry that is 0
    ids = rng.integers(0, 4, nodes).astype(np.uint8)
    dt = 0.1 * h / np.sqrt(stiffness)
    layers = [rng.uniform(0.0, 0.1, n) for n in nodes] if sponge else None
    return spec_from(x, y, z, ids, rows, dt, rng.standard_normal(steps) * 1e-3, sponge=layers)


def _start(nodes, kind, seed=3):
    rng = np.random.default_rng(seed)
    shapes = {"ux": (nodes[0] - 1,) + nodes[1:], "uy": (nodes[0], nodes[1] - 1, nodes[2]),
              "uz": nodes[:2] + (nodes[2] - 1,)}
    out = {}
    for c, s in shapes.items():
        a = rng.standard_normal(s)
        if kind == "decay":  # a front whose values run through the whole range to 0 along x
            a = a * np.exp2(-np.linspace(0.0, 1200.0, s[0]))[:, None, None]
        elif kind == "spots":  # values at and beyond the range's ends in a few places, subnormal and huge ones
            a[rng.random(s) < 0.3] = 0.0
            for v in (5e-324, 2.0 ** -1040, 2.0 ** -900, 2.0 ** -753, 2.0 ** -752, 2.0 ** -700, 2.0 ** 410):
                a[tuple(rng.integers(0, n) for n in s)] = v
        if c != "ux":
            a[0] = 0.0
        out[c] = a
    return out


@pytest.mark.parametrize("nodes,h,stiffness,sponge", [
    ((24, 17, 9), 0.3, 1.0, False),         # block steps
    ((24, 17, 9), 1e-4, 5e10, True),
    ((70, 66, 70), 0.7, 1e-9, False),       # the march, dividing: stiffnesses below the quotients' range
    ((70, 66, 70), 1e-4, 1e11, True),
])
@pytest.mark.parametrize("kind", ["full", "decay", "spots"])
def test_quotients_equal_divisions(nodes, h, stiffness, sponge, kind):
    steps = 7
    spec = _spec(nodes, h, stiffness, steps, sponge)
    start = _start(nodes, kind)
    got = {}
    for kernel in ("auto", "tiled", "naive"):
        ctx = fdtd.Context(spec, precision="fp64", kernel=kernel)
        try:
            for c in ("ux", "uy", "uz"):
                ctx.set(c, start[c])
                ctx.set(c + "_old", 0.5 * start[c])
            ctx.step(steps)
            got[kernel] = {f: ctx.get(f) for f in FIELDS}
        finally:
            ctx.close()
    for kernel in ("auto", "tiled"):
        for f in FIELDS:
            assert np.array_equal(got[kernel][f], got["naive"][f], equal_nan=True), (kernel, f)
