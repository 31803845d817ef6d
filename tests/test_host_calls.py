"""The library's host code over a stand-in HIP runtime (host_runtime.cpp: two
devices, kernels that do nothing), without a GPU: which device its objects
are made on, what it allocates and when, what it launches.  Every case runs
in a process of its own, whose HIP calls all come to the stand-in."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
sys.path[:0] = [%r, %r]
hip = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
hip.host_count.restype = ctypes.c_longlong
hip.host_launch.restype = ctypes.c_char_p
import numpy as np
from helpers import spec_from, uniform_crystal
from phonomena_amd import fdtd

def count(what):
    return hip.host_count(what.encode())

def launches():
    return [hip.host_launch(i).decode() for i in range(hip.host_launches())]

def grid(i):
    v = (ctypes.c_int * 5)()
    hip.host_grid(i, v)
    return list(v)

def device():
    d = ctypes.c_int()
    hip.hipGetDevice(ctypes.byref(d))
    return d.value

def context(cells, precision="fp64", kernel="auto", tune=False, steps=40, spacing=1.0, **kw):
    x, y, z, ids, rows, dt, wave = uniform_crystal(cells, spacing, steps=steps)
    return fdtd.Context(spec_from(x, y, z, ids, rows, dt, wave, **kw), precision=precision, kernel=kernel, tune=tune)
"""


@pytest.fixture(scope="session")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host_runtime.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", so, os.path.join(HERE, "host_runtime.cpp")],
                   check=True)
    return so


def run(runtime, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, HERE, runtime) + body], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("current", [0, 1])
@pytest.mark.parametrize("pinned", [True, False])  # without pinned memory a transfer goes through device scratch
def test_transfers_of_a_context_stay_on_its_device(runtime, current, pinned):
    run(runtime, """
hip.host_fail_host_malloc(%d)
hip.hipSetDevice(1)
c = context((70, 40, 40), probe=(0, 1, 70, 0, 1, 40), every=1)
hip.hipSetDevice(%d)
c.step(2)
for f in ("ux", "uy_old"):
    c.get(f)
    c.set(f, np.zeros(c._shapes[f[:2]]))
c.probes()
assert device() == %d
for what in ("malloc", "host_malloc", "stream", "event"):
    assert count(what + "@0") == 0, what
assert (count("host_malloc@1") > 0) == %s
""" % (not pinned, current, current, pinned))


def test_the_largest_blocks_get_their_lds_on_every_device(runtime):
    run(runtime, """
for dev in (0, 1):
    hip.hipSetDevice(dev)
    for cells in ((49, 94, 23), (74, 98, 17)):
        c = context(cells, tune=True, spacing=0.3)
        c.step(4)
        c.close()
    assert count("large_lds@%d" % dev) > 0
""")


def test_transfers_make_no_streams_and_keep_their_pinned_memory(runtime):
    run(runtime, """
def plugin_run(cells):
    c = context(cells)
    made = count("stream")
    c.step(2)
    for f in ("ux", "uy", "uz", "ux_old"):
        c.get(f)
    fdtd.dft(np.ones((700, 1000)), nf=500)
    assert count("stream") == made  # a stream's hardware queue takes milliseconds to make
    c.close()

plugin_run((90, 60, 40))
before = count("host_malloc"), count("event")
assert before[0] <= 3  # one piece: with the context, larger for a 1.8 MB field, for 5.6 MB of traces
for k in range(5):
    plugin_run((90, 60, 40))
assert (count("host_malloc"), count("event")) == before
plugin_run((230, 90, 60))  # 10 MB a field
fdtd.check(fdtd.load().pf_trim())
assert count("host_free") == count("host_malloc")
""")


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
def test_an_audit_allocates_nothing(runtime, precision, pinned):
    run(runtime, """
hip.host_fail_host_malloc(%d)
def allocations():
    return [count(w) for w in ("malloc", "host_malloc", "event", "stream")]

for cells in ((40, 30, 20), (70, 80, 30)):
    c = context(cells, precision=%r)
    c.step(1)
    made = allocations()
    c.energy()
    c.step(1)
    c.energy()
    assert allocations() == made
    c.close()
""" % (not pinned, precision))


@pytest.mark.parametrize("pinned", [True, False])
def test_transfers_and_audits_without_host_memory_do_not_throw(runtime, pinned):
    """No C++ exception may leave a C entry: without memory for a thread or a
    function object a transfer runs on the caller's thread."""
    run(runtime, """
hip.host_fail_host_malloc(%d)
c = context((120, 40, 40), probe=(0, 1, 120, 0, 1, 40), every=1)
a = np.zeros(c._shapes["ux"])
x = np.ones((900, 1000))
c.get("ux")
hip.host_fail_new(1)
for f in ("ux", "uz_old"):
    c.get(f)
c.set("ux", a)
c.step(20)
c.probes()
c.energy()
fdtd.dft(x, nf=500)
hip.host_fail_new(0)
c.close()
""" % (not pinned))


@pytest.mark.parametrize("precision,shapes,default", [("fp32c", 5, (16, 32)), ("fp32", 5, (16, 32)),
                                                      ("fp64", 3, (8, 32))])
@pytest.mark.parametrize("cells,chunk", [((60, 50, 24), 8), ((170, 170, 80), 32)])
def test_the_autotuner_tries_the_default(runtime, precision, shapes, default, cells, chunk):
    """The candidates, one by one: the stand-in's clock makes each the
    fastest in turn.  Their number is the steps a caller has to leave for them."""
    run(runtime, """
FASTEST = ctypes.CFUNCTYPE(ctypes.c_float, ctypes.c_int, ctypes.c_int)
found = set()
ctxs = [context(%r, precision=%r, steps=2000) for _ in range(3)]
b = fdtd.Batch(%r)
for c in ctxs:
    b.add(c)
n = 4 * %d
for k in range(n):
    calls = [0]
    def clock(_a, _b):
        calls[0] += 1
        return 1.0 if calls[0] == k + 1 else 2.0
    f = FASTEST(clock)
    hip.host_elapsed(f)
    before = ctxs[0].steps_done
    best = b.autotune(trial_steps=1)
    assert calls[0] == n and ctxs[0].steps_done - before == 2 * n
    found.add((best["tile_j"], best["tile_z"], best["tile_x"]))
assert len(found) == n
assert %r in found, sorted(found)
""" % (cells, precision, precision, shapes, default + (chunk,)))


def test_reciprocals_are_made_for_the_kernels_that_read_them(runtime):
    run(runtime, """
def made(cells, kernel, spacing, tune=True):
    before = count("malloc")
    c = context(cells, kernel=kernel, spacing=spacing, tune=tune)
    return c, count("malloc") - before

small, large = (30, 24, 12), (90, 70, 60)
plain = made(large, "naive", 0.3)[1]
assert made(large, "strip", 0.3)[1] == plain
assert made(large, "tiled", 0.3)[1] == plain + 6     # exact quotients
assert made(large, "tiled", 0.5)[1] == plain + 6     # reciprocal products
c, n = made(small, "auto", 0.3)                      # block steps with divisions: two more levels
assert n == plain + 2
c.step(4)
assert "k_block_stepsIdLi0E" in launches()[-1]
# a batch marches its members, with quotients
d, _ = made(large, "auto", 0.7, tune=False)
b = fdtd.Batch("fp64")
for m in (c, d):
    b.add(m)
b.step(1)
assert count("malloc") > 0 and any("k_batch_sweepIdLi4E" in k for k in launches())
b.remove(c)
c.step(4)
assert "k_block_stepsIdLi0E" in launches()[-1]
""")


def test_the_quotient_cases_run_quotients(runtime):
    """test_gpu_quotient_tiles.py's meshes march with quotients; in
    test_gpu_quotient.py the small ones step in blocks (with divisions), and
    the one with stiffnesses near 1e-9 is out of the quotients' range and
    divides."""
    run(runtime, """
import test_gpu_quotient_tiles as q

def routed(nodes, h, stiffness, sponge, tile):
    c = fdtd.Context(q._spec(nodes, h, stiffness, 3, sponge), precision="fp64", kernel="tiled" if tile[0] else "auto",
                     tile_j=tile[0], tile_z=tile[1])
    n = len(launches())
    c.step(3)
    c.close()
    return launches()[n]

for nodes, h, stiffness, sponge, tile in q.CASES:
    k = routed(nodes, h, stiffness, sponge, tile)
    assert "k_sweep_tiledIdLi4ELb%dE" % sponge in k, (nodes, k)
    assert tile == (0, 0) or k.count("ELi%dELi%dEE" % tile) == 1, k
assert "k_block_stepsIdLi0ELb0E" in routed((24, 17, 9), 0.3, 1.0, False, (0, 0))
assert "k_block_stepsIdLi0ELb1E" in routed((24, 17, 9), 1e-4, 5e10, True, (0, 0))
assert "k_sweep_tiledIdLi0ELb0E" in routed((70, 66, 70), 0.7, 1e-9, False, (0, 0))
assert "k_sweep_tiledIdLi4ELb1E" in routed((70, 66, 70), 1e-4, 1e11, True, (0, 0))
""")


def test_the_block_step_cases_step_in_blocks(runtime):
    """test_gpu_block.py's meshes step in blocks in every precision, between
    them in launches of 1 to 4 steps and cut along every axis; a mesh beyond
    the dispatch's line marches."""
    run(runtime, """
import test_gpu_block as t

cases = next(m for m in t.test_block_steps_equal_the_per_node_sweep.pytestmark if m.args[0].startswith("nodes")).args[1]
steps, cut, threads = set(), [0, 0, 0], 0
for precision in ("fp64", "fp32", "fp32c"):
    for nodes, h, graded, sponge, surface, every in cases:
        c = fdtd.Context(t._spec(nodes, h, graded, sponge, surface, every, 23), precision=precision)
        n = len(launches())
        for calls in (1, 2, 3, 4, 5, 8):
            c.step(calls)
        c.close()
        done = 0
        for i in range(n, len(launches())):
            assert "k_block_steps" in launches()[i], (precision, nodes, launches()[i])
            b = grid(i)
            done += b[3]
            steps.add(b[3])
            cut = [max(a, v) for a, v in zip(cut, b)]
            threads = max(threads, b[4])
        assert done == 23
assert steps == {1, 2, 3, 4} and min(cut) > 1 and threads > 512, (steps, cut, threads)
for precision in ("fp64", "fp32", "fp32c"):
    c = context((64, 64, 40), precision=precision, tune=True)
    c.step(1)
    assert not any("k_block_steps" in k for k in launches()[-2:])
""")


@pytest.mark.parametrize("cells,tile,rounds", [
    ((60, 60, 60), (16, 64), 1), ((60, 60, 60), (8, 32), 1), ((128, 128, 28), (8, 32), 1),
    ((257, 795, 11), (16, 64), 2), ((136, 614, 11), (8, 32), 2), ((166, 515, 11), (8, 32), 2)])
def test_x_chunks_by_the_rounds_of_a_launch(runtime, cells, tile, rounds):
    """A launch of several rounds takes the chunk of at least 16 planes with the
    most useful planes per plane time; one that is a single round with such
    chunks may take shorter ones."""
    run(runtime, """
cells, tile = %r, %r
slots = 2 * 256  # the stand-in's resident blocks
c = context(cells, precision="fp32", kernel="tiled", steps=2)
c = fdtd.Context(c.spec, precision="fp32", kernel="tiled", tile_j=tile[0], tile_z=tile[1])
c.step(1)
i = max(i for i, k in enumerate(launches()) if "k_sweep_tiled" in k)
nz, ny, nx, planes = grid(i)[:4]
n = cells[0] + 1
assert nx == -(-n // planes)
useful = {}
for k in range(1, n + 1):
    p = -(-n // k)
    if 16 <= p <= 253 and -(-n // p) == k:
        useful[p] = n / (-(-(ny * nz * k) // slots) * (p + 1))
best = max(useful.values())
long = min(p for p in useful if useful[p] == best)  # ties: more chunks
if ny * nz * -(-n // long) > slots:
    assert %d > 1 and planes == long, (planes, long)
else:
    assert %d == 1 and ny * nz * nx <= slots and planes <= long, (planes, long)
""" % (cells, tile, rounds, rounds))
