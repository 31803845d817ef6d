"""Marched FP64 quotients from reciprocals against the per-node sweep, which
divides: the same bits on tiles clear of every y and z face as well as at
them, in x chunks at and off the x faces, with and without the absorbing
layer, for every tile shape.  The stiffnesses are within the quotients' range
(CASES; test_host_calls.py checks that quotients are what runs)."""
import numpy as np
import pytest

from helpers import FIELDS
from phonomena_amd import fdtd
from test_gpu_quotient import _spec, _start

pytestmark = pytest.mark.gpu
STEPS = 5
# nodes, spacing, stiffness, absorbing layer, tile (0, 0: AUTO's): a tile owns 2 rows and lanes less than it has
CASES = [
    ((70, 66, 70), 0.7, 1.0, False, (0, 0)),
    ((70, 66, 70), 0.7, 4e-6, False, (8, 32)),  # entries from 1.2e-6, the least allowed is 2^-20
    ((70, 66, 70), 1e-4, 1e11, False, (16, 32)),
    ((70, 66, 70), 0.3, 1.0, True, (8, 32)),
    ((9, 50, 70), 0.7, 1.0, False, (8, 32)),    # every plane near an x face
    ((40, 50, 140), 0.3, 1.0, False, (8, 64)),
    ((40, 50, 140), 1e-4, 5e10, True, (8, 64)),
]


@pytest.mark.parametrize("nodes,h,stiffness,sponge,tile", CASES)
@pytest.mark.parametrize("kind", ["full", "decay", "spots"])
def test_marched_quotients_equal_divisions(nodes, h, stiffness, sponge, tile, kind):
    spec = _spec(nodes, h, stiffness, STEPS, sponge)
    start = _start(nodes, kind, seed=8)
    got = {}
    for kernel, shape in (("tiled" if tile[0] else "auto", tile), ("naive", (0, 0))):
        ctx = fdtd.Context(spec, precision="fp64", kernel=kernel, tile_j=shape[0], tile_z=shape[1])
        try:
            for c in ("ux", "uy", "uz"):
                ctx.set(c, start[c])
                ctx.set(c + "_old", 0.5 * start[c])
            ctx.step(STEPS)
            got[kernel == "naive"] = {f: ctx.get(f) for f in FIELDS}
        finally:
            ctx.close()
    for f in FIELDS:
        assert np.array_equal(got[False][f], got[True][f], equal_nan=True), f
    assert kind != "full" or all(np.all(np.isfinite(v)) for v in got[True].values())
