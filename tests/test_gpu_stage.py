"""Staged transfers at their edges: fields of less than a chunk, of exactly
some chunks and an element more, of more chunks than lanes; probe rings that
wrap; two host threads at once on one device; after pf_trim."""
import threading

import numpy as np
import pytest

from helpers import spec_from, uniform_crystal
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu
CHUNK = 512 << 10  # bytes


def _context(cells, precision="fp64", **kw):
    x, y, z, ids, rows, dt, wave = uniform_crystal(cells, 1.0, steps=40)
    return fdtd.Context(spec_from(x, y, z, ids, rows, dt, wave, **kw), precision=precision, tune=False)


def _round_trip(ctx, seed):
    rng = np.random.default_rng(seed)
    for f in ("ux", "uy_old", "uz"):
        a = rng.standard_normal(ctx._shapes[f.replace("_old", "")])
        if ctx.precision == "fp32":
            a = a.astype(np.float32).astype(np.float64)
        ctx.set(f, a)
        assert np.array_equal(ctx.get(f), a), f


# ux of (nx-1) x ny x nz nodes: 8 KiB a row of planes of 32 x 32
@pytest.mark.parametrize("nx", [5, 65, 66, 130, 600])  # < 1 chunk, 1, 1 and a plane, 2 and a plane, 9 and more
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_fields_round_trip_over_chunk_edges(nx, precision):
    ctx = _context((nx - 1, 31, 31), precision)
    try:
        assert (nx - 1) * 32 * 32 * 8 % CHUNK == 0 or nx not in (65,)
        _round_trip(ctx, nx)
        fdtd.check(fdtd.load().pf_trim())
        _round_trip(ctx, nx + 1)
    finally:
        ctx.close()


def test_probe_frames_of_a_wrapped_ring():
    full = _context((40, 36, 20), probe=(0, 1, 41, 0, 1, 37), every=1)
    short = _context((40, 36, 20), probe=(0, 1, 41, 0, 1, 37), every=1, cap=7)
    try:
        for n in (3, 4, 6, 20):
            full.step(n)
            short.step(n)
            a, b = full.probes(), short.probes()
            assert b.shape[0] == min(7, a.shape[0])
            assert np.array_equal(a[-b.shape[0]:], b)
    finally:
        full.close()
        short.close()


def test_two_threads_share_the_lanes():
    ctxs = [_context((200, 40, 40)) for _ in range(2)]
    errors = []

    def work(i):
        try:
            for k in range(6):
                _round_trip(ctxs[i], 10 * i + k)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
        assert not errors
    finally:
        for c in ctxs:
            c.close()
