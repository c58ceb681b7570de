"""The engine's host side on the CPU: what it allocates, waits for and
launches, over a HIP runtime that runs nothing (tests/hip_stub.cpp).  Every
test runs its program in a process of its own, where the stand-in's entry
points come before the runtime's."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

PRELUDE = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_log.restype = ctypes.c_char_p
stub.stub_live.restype = ctypes.c_long
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
import numpy as np
from cgenie_amd import engine as E
from cgenie_amd import grid as G
from cases import make_case

def log():
    t = stub.stub_log().decode().splitlines()
    stub.stub_clear()
    return t

def fail(what, n):
    stub.stub_fail(what.encode(), ctypes.c_long(n))

def member(eng, c, prec=E.FP64, bgc=False, diso=True):
    m = eng.add_member(eng.add_grid(c.g, c.k1), c.tset.L, prec, c.diff, diso=diso)
    eng.set_velocity(m, c.u)
    eng.upload(m, c.ts)
    if bgc:
        eng.bgc_init(m, E.default_bgc_params(1.0 / 96, c.tset), c.light, c.mld)
    return m
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "hip_stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", str(so)],
                   check=True)
    return str(so)


def run(stub, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, stub, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    return r.stdout


def test_downloads_follow_the_fills_of_a_new_member(stub):
    """A member's arrays are cleared by fills that the host does not wait for.
    A download packs on a stream of its own and comes after them: until then
    the state's buffer index holds anything."""
    run(stub, """
c = make_case(8, 6, 4, kind="config2", seed=3)
eng = E.Engine(0)

def ordered(t):
    packs = [i for i, s in enumerate(t) if s.startswith("launch k_pack")]
    fills = [i for i, s in enumerate(t) if s == "memset null"]
    assert packs and fills, t
    waits = [i for i, s in enumerate(t) if s == "sync null" and fills[-1] < i < packs[0]]
    assert waits or t[packs[0]].endswith("null"), t

gid = eng.add_grid(c.g, c.k1)
for prec in (E.FP64, E.FP32C):
    log()
    m = eng.add_member(gid, c.tset.L, prec, c.diff)
    eng.download(m, c.ts.shape)
    ordered(log())
eng.upload(m, c.ts)
eng.bgc_init(m, E.default_bgc_params(1.0 / 96, c.tset), c.light, c.mld)
eng.bgc_download(m, 3, c.ts.shape)
ordered(log())
eng.close()
""")

FLUX = """
def flux(eng, ids):
    log()
    eng.tstepo(ids, 1)
    return [s.split()[1] for s in log() if s.startswith("launch k_flux")]
"""


@pytest.mark.parametrize("prec,shape", [("FP64", "(8, 256, 2, 1)"), ("FP32C", "(6, 256, 2, 1)")])
def test_the_starting_shape_set_again_is_the_automatic_one(stub, prec, shape):
    """A small batch takes the split by levels with the shape an engine starts
    with, also when that was changed and set again, and whole columns with any
    other; the tuner times the split among its shapes and leaves it on where it
    is the fastest."""
    run(stub, FLUX + f"""
from cgenie_amd import autotune
prec, shape = E.{prec}, {shape}
c = make_case(36, 36, 16, kind="ts", L=24, seed=5)
eng = E.Engine(0)
ids = [member(eng, c, prec)]
split = ["k_flux<%s,2,256,2,3>" % ("double" if prec == E.FP64 else "float")]
assert autotune.AUTOMATIC[prec] == shape
assert flux(eng, ids) == split
for other in ((2,) + shape[1:], shape[:1] + (128,) + shape[2:], shape[:2] + (3, 1), shape[:3] + (0,)):
    eng.set_tile(prec, *other)
    got = flux(eng, ids)
    assert split[0] not in got and len(got) == 1 + other[3], (other, got)
    eng.set_tile(prec, *shape)
    assert flux(eng, ids) == split, other
eng.set_tile(prec, 4, 128, 3, 0)
best = autotune.tune(eng, ids, (36, 36, 16), 24, prec, reps=2, use_cache=False, write_cache=False)
assert (best["tracer_block"], best["cols"], best["ring"], best["iso_prepass"]) == shape
assert flux(eng, ids) == split
many = [member(eng, c, prec) for _ in range(40)]
assert split[0] not in flux(eng, many)
eng.close()
""")


def test_batches_without_isoneutral_mixing(stub):
    """Where no member mixes along isoneutrals the flux has no pre-pass, and
    whole columns take over from the split by levels at smaller batches; one
    member that mixes brings both back."""
    run(stub, """
c = make_case(36, 36, 16, kind="ts", L=24, seed=5)

def flux(n, mixing, prec=E.FP64):
    eng = E.Engine(0)
    ids = [member(eng, c, prec, diso=q < mixing) for q in range(n)]
    log()
    eng.tstepo(ids, 1)
    names = [s.split()[1] for s in log() if s.startswith("launch k_flux")]
    eng.close()
    return names

split, whole, pre = "k_flux<double,2,256,2,3>", "k_flux<double,8,256,2,2>", "k_flux<double,2,256,2,1>"
assert flux(12, 12) == [split] and flux(32, 32) == [pre, whole]
assert flux(10, 0) == [split] and flux(12, 0) == [whole] and flux(32, 0) == [whole]
assert flux(12, 1) == [split] and flux(32, 1) == [pre, whole]
split, whole, pre = "k_flux<float,2,256,2,3>", "k_flux<float,6,256,2,2>", "k_flux<float,2,256,2,1>"
assert flux(16, 16, E.FP32C) == [split] and flux(20, 20, E.FP32C) == [pre, whole]
assert flux(8, 0, E.FP32C) == [split] and flux(10, 0, E.FP32C) == [whole]
""")


def test_a_capture_that_fails_leaves_nothing(stub):
    """Each allocation and each step of a capture fails once: what it had
    allocated is given back, and the workspace of the flux split by levels,
    where it is what cannot be had, is done without."""
    run(stub, """
c = make_case(18, 18, 8, kind="config2", L=8, seed=5)
eng = E.Engine(0)
m = member(eng, c, E.FP32C, bgc=True)
eng.step([m], 1)
before = stub.stub_live()
refused = 0
for what in ("malloc", "capture"):
    for n in range(3):
        fail(what, n)
        try:
            g = eng.capture([m], 2)
        except E.CgoError:
            refused += 1
        else:
            eng.drop_graph(g)
        fail(what, -1)
        assert stub.stub_live() == before, (what, n, log())
assert refused == 4, refused        # the lists, and the capture's three steps; not the workspace
assert "bad" not in " ".join(log())
eng.close()
""")


def test_engines_leave_nothing(stub):
    """An engine that cannot be created, and one that is closed with members,
    a graph, surface fluxes and downloads behind it, gives everything back."""
    run(stub, """
import ctypes as C
from cgenie_amd import surface as SF
L = E.load()
for what, k in (("malloc", 2), ("event", 8)):
    for n in range(k):
        fail(what, n)
        h = C.c_void_p()
        assert L.cgo_create(0, C.byref(h)) == -2 and not h.value
        fail(what, -1)
        assert stub.stub_live() == 0, (what, n, log())
g = G.make_grid(36, 36, 8, nyear=96)
w = G.read_world(sys.argv[2] + "/tests/golden/worbe2", 36, 36)
su = SF.surflux_setup(g, w.k1)
eng = E.Engine(0)
gid = eng.add_grid(g, w.k1)
eng.set_momentum(gid, g, w)
eng.set_surflux(gid, su)
m = eng.add_member(gid, 2, E.FP64, G.diffusivities(2000.0, 1e-5))
eng.set_wind(m, np.load(sys.argv[2] + "/tests/golden/worbe2_wind.npz")["stress"])
eng.set_surface(m, *SF.atmosphere(g, w.k1, 64, ice=True))
gr = eng.capture([m], 2)
eng.sync()
eng.download(m, (8, 36, 36, 2))
eng.close()
assert stub.stub_live() == 0, log()
assert "bad" not in " ".join(log())
""")


def test_member_bytes_cover_the_allocation(stub):
    """cgo_member_bytes, by which runs are admitted, is what a member takes."""
    run(stub, """
for dims, L in (((8, 6, 4), 2), ((18, 18, 8), 9), ((36, 36, 16), 24)):
    for prec in (E.FP64, E.FP32C):
        c = make_case(*dims, kind="config2" if L > 7 else "ts", L=L, seed=5)
        eng = E.Engine(0)
        gid = eng.add_grid(c.g, c.k1)
        for bgc in (False, True)[:1 + (L > 7)]:
            log()
            m = eng.add_member(gid, L, prec, c.diff)
            if bgc:
                log()
                eng.bgc_init(m, E.default_bgc_params(1.0 / 96, c.tset), c.light, c.mld)
            got = [int(s.split()[1]) for s in log() if s.startswith("malloc")]
            assert got == [eng.member_bytes(gid, L, prec, bgc)], (dims, L, prec, bgc, got)
        eng.close()
""")


def test_the_eager_workspace_gives_way_to_a_member(stub):
    """Where no memory is left for a member, the eager steps' workspace is
    freed for it; the next small step takes one again, or whole columns."""
    run(stub, FLUX + """
c = make_case(18, 18, 8, kind="config2", L=8, seed=5)
eng = E.Engine(0)
m = member(eng, c, E.FP32C, bgc=True)
eng.step([m], 1)
gid = eng.add_grid(c.g, c.k1)
log()
fail("malloc", 0)
q = eng.add_member(gid, 8, E.FP32C, c.diff)
t = log()
assert t.index("free") < [i for i, s in enumerate(t) if s.startswith("malloc")][0] and "sync s1" in t[:t.index("free")], t
eng.remove_member(q)
fail("malloc", 0)
assert flux(eng, [m]) == ["k_flux<float,2,256,2,1>", "k_flux<float,6,256,2,2>"]
assert flux(eng, [m]) == ["k_flux<float,2,256,2,3>"]
for given_up in (True, False):
    fail("malloc", 0)
    try:
        eng.add_member(gid, 8, E.FP32C, c.diff)
        assert given_up
    except E.CgoError:
        assert not given_up
eng.close()
assert stub.stub_live() == 0
""")


def test_captured_lists_hold_what_the_kernels_read(stub):
    """A captured step's lists name a member once per kernel family that it
    takes part in: transport, and BIOGEM."""
    run(stub, """
eng = E.Engine(0)
for kind, L, n in (("ts", 3, 1), ("config2", 8, 2)):
    m = member(eng, make_case(18, 18, 8, kind=kind, L=L, seed=5), bgc=kind != "ts")
    eng.step([m], 1)
    log()
    eng.capture([m], 1)
    assert "malloc %d" % (4 * n) in log()
eng.close()
""")


def test_many_columns_take_whole_columns(stub):
    """Batches of many wet columns take whole columns, FP32C ones where they
    have BIOGEM; fewer, or transport alone, the split by levels."""
    run(stub, FLUX + """
c, t = (make_case(18, 18, 8, kind=k, L=8, seed=5) for k in ("config2", "ts"))

def form(n, prec, case):
    eng = E.Engine(0)
    got = flux(eng, [member(eng, case, prec, bgc=case is c) for _ in range(n)])
    eng.close()
    return "split" if got[-1].endswith(",3>") else "whole"

assert [form(n, E.FP32C, c) for n in (32, 80, 120)] == ["split", "whole", "whole"]
assert [form(n, E.FP32C, t) for n in (80, 120)] == ["split", "split"]
assert [form(n, E.FP64, c) for n in (120, 144)] == ["split", "whole"]
""")
