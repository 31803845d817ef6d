"""FP64 displacements near the largest double: where the reference's
2 u - u_old overflows, so do the kernels (the same infinities and NaN in the
same cells), in every FP64 kernel and flavour, damped or not."""
import numpy as np
import pytest

from helpers import FIELDS, spec_from
from oracle import reference_math as rm
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu
NODES = (14, 11, 9)


@pytest.mark.parametrize("h", [1.0, 3.0])  # reciprocal products; divisions (out of the quotients' range)
@pytest.mark.parametrize("damped", [False, True])
def test_overflow_as_in_the_reference(h, damped):
    x, y, z = (np.arange(n) * h for n in NODES)
    c = np.zeros((6, 6))
    c[:3, :3] = 0.5e-3 + 2e-3 * np.eye(3)
    c[[3, 4, 5], [3, 4, 5]] = 0.7e-3
    row = np.concatenate([c[:3, :3].ravel(), np.diag(c)[3:], [1.0]])
    ids = np.zeros(NODES, np.uint8)
    dt = np.float64(0.2 * h)
    wave = np.zeros(2)
    layers = [np.full(n, 0.01) for n in NODES] if damped else None
    C, P = rm.dense_material(ids, [c], np.array([1.0]))
    pb = rm.Problem(x, y, z, C, P, dt, wave, sponge=layers)
    s = rm.State(*NODES)
    start = {}
    rng = np.random.default_rng(1)
    for f in ("ux", "uy", "uz"):
        a = 1.2e308 * (1.0 - 1e-3 * rng.random(getattr(s, f).shape))
        a[rng.random(a.shape) < 0.3] *= 0.5  # 2 u - u_old stays finite there
        if f != "ux":
            a[0] = 0.0
        start[f] = a
        getattr(s, f)[...] = a
        getattr(s, f + "_new")[...] = a
        getattr(s, f + "_old")[...] = 0.8 * a
    spec = spec_from(x, y, z, ids, np.array([row]), dt, wave, sponge=layers)
    ctxs = {k: fdtd.Context(spec, precision="fp64", kernel=k) for k in ("auto", "naive", "tiled", "strip")}
    try:
        for ctx in ctxs.values():
            for f in ("ux", "uy", "uz"):
                ctx.set(f, start[f])
                ctx.set(f + "_old", 0.8 * start[f])
        with np.errstate(all="ignore"):
            for tt in range(2):
                rm.step(s, pb, tt)
                want = {f: getattr(s, f) for f in FIELDS}
                assert tt > 0 or (np.isinf(want["ux"]).any() and np.isfinite(want["ux"]).any())
                for k, ctx in ctxs.items():
                    ctx.step(1)
                    for f in FIELDS:
                        assert np.array_equal(ctx.get(f), want[f], equal_nan=True), (k, tt, f)
    finally:
        for ctx in ctxs.values():
            ctx.close()
