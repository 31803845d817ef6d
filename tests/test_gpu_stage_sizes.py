"""Staged transfers over the sizes at which their chunks change (512 KiB up
to 16 MiB, 1 MiB up to 64 MiB, 2 MiB beyond; 2 MiB towards the device) and
at which the first of them are issued in one more group, and
with the pinned memory made larger and given back between them."""
import threading

import numpy as np
import pytest

from helpers import spec_from
from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu


def _context(nx):
    """ux of nx - 1 planes of 32 x 32 nodes: 8 KiB a plane."""
    x, y, z = (np.arange(n, dtype=np.float64) for n in (nx, 32, 32))
    rows = np.array([[3.0, 1, 1, 1, 3, 1, 1, 1, 3, 1, 1, 1, 1.0]])
    return fdtd.Context(spec_from(x, y, z, np.zeros((nx, 32, 32), np.uint8), rows, 0.2, np.zeros(4)),
                        precision="fp64", tune=False)


@pytest.mark.parametrize("planes", [(255, 2048, 8193), (8192,), (2049, 256), (4097, 64),
                                    (128, 130, 192, 300, 576, 1024, 1025, 1088)])  # 2, 3, 5, 9, 16, 17 chunks
def test_round_trips_where_the_chunks_change(planes):
    for n in planes:
        ctx = _context(n + 1)
        try:
            for f in ("ux", "uz_old"):
                a = np.random.default_rng(n).standard_normal(ctx._shapes[f[:2]])
                ctx.set(f, a)
                assert np.array_equal(ctx.get(f), a), (n, f)
        finally:
            ctx.close()


def test_the_chunks_of_a_transfer_follow_the_steps_before_it():
    """A fetch is ordered after the steps on the context's stream, a set
    before the next ones."""
    ctx = _context(2050)
    try:
        a = np.random.default_rng(5).standard_normal(ctx._shapes["uz"])
        for _ in range(3):
            ctx.set("uz", a)
            ctx.step(1)
            assert np.array_equal(ctx.get("uz_old")[1:], a[1:])  # the level before the step (its wall has the source)
            assert np.any(ctx.get("uz")[1:] != a[1:])
    finally:
        ctx.close()


def test_threads_of_one_device_all_finish():
    """Four host threads' transfers and audits over the one pinned piece: each
    ends, within a minute, with its own values."""
    ctxs = [_context(700 + 300 * i) for i in range(4)]
    left = list(range(4))

    def work(i):
        rng = np.random.default_rng(i)
        for _ in range(6):
            a = rng.standard_normal(ctxs[i]._shapes["uy"])
            ctxs[i].set("uy", a)
            assert np.isfinite(ctxs[i].energy())
            assert np.array_equal(ctxs[i].get("uy"), a)
        left.remove(i)

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads)
    assert not left
    for c in ctxs:
        c.close()
