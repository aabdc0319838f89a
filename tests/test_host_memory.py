"""What the library's host code does with device memory, on a HIP runtime that
has none (fake_hip.cpp, built with g++): each script runs in a process of its
own, with the fake loaded first (no GPU)."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = r"""
import ctypes as ct, os, sys
fake = ct.CDLL(sys.argv[1], mode=os.RTLD_NOW | ct.RTLD_GLOBAL)
fake.fake_live.restype = fake.fake_launches.restype = fake.fake_bad_frees.restype = fake.fake_lost.restype = fake.fake_news.restype = ct.c_uint64
fake.fake_limit.argtypes = [ct.c_uint64]
sys.path[:0] = [sys.argv[2], os.path.join(sys.argv[2], "tests")]
import numpy as np
from grudon_amd import api
live, limit, UNLIMITED = fake.fake_live, fake.fake_limit, 2 ** 64 - 1


def ring(n, k=8):
    rp = np.arange(n + 1) * k
    col = (np.repeat(np.arange(n), k) + np.tile(np.arange(1, k + 1), n)) % n
    return rp.astype(np.uint32), col.astype(np.uint32)


def context():
    ctx = api.Context(0)
    ctx.set_layout(False)  # (kernels do nothing here)
    return ctx


def needs_new():
    # (where another allocator, a sanitizer's, has taken operator new)
    if fake.fake_news() == 0:
        print("done")
        sys.exit(0)


def refused(f, what):
    try:
        f()
    except api.GrdError as e:
        assert what in str(e), e
        return True
    return False
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("no g++ or HIP headers on this machine")
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run([gxx, "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROCM, "include"), os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", out], check=True)
    return out


def _run(fake, body):
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, fake, ROOT], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and p.stdout.split()[-1:] == ["done"], (p.returncode, p.stdout, p.stderr)


def test_freed_memory_is_given_back(fake):
    """What a context keeps goes back when it is asked to trim, and when it ends."""
    _run(fake, r"""
ctx = context()
base = live()
G = api.Graph.from_csr(ctx, *ring(5000))
S = api.State(G, api.CC)
assert live() > base
S.free()
G.free()
assert live() > base  # kept for the next allocations
ctx.trim()
assert live() == base
G = api.Graph.from_csr(ctx, *ring(5000))
G.free()
ctx.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""")


@pytest.mark.parametrize("call", ["graph", "weights"])
def test_kept_memory_serves_every_context(fake, call):
    """No allocation fails while another context of the device only keeps blocks:
    neither one through a context's own blocks nor a plain one."""
    _run(fake, r"""
A, B = context(), context()
G = api.Graph.from_csr(A, *ring(5000))
used = live()
G.free()
assert live() == used  # A keeps all of it
limit(used)
if "%s" == "graph":
    G = api.Graph.from_csr(B, *ring(5000))
    G.free()
else:
    B.selector_load(np.zeros(api.MLP_PARAMS, dtype=np.uint16))
limit(UNLIMITED)
A.close()
G = api.Graph.from_csr(B, *ring(5000))  # (a context that is gone is not asked)
G.free()
B.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""" % call)


def test_device_of_another_context_is_left_alone(fake):
    """A context on another device keeps its blocks."""
    _run(fake, r"""
A, B = context(), api.Context(1)
G = api.Graph.from_csr(A, *ring(5000))
used = live()
G.free()
limit(used)
assert refused(lambda: B.selector_load(np.zeros(api.MLP_PARAMS, dtype=np.uint16)), "failed")
assert live() == used
limit(UNLIMITED)
A.close()
B.close()
print("done")
""")


def test_freeing_needs_no_memory(fake):
    """Objects can be freed while the host has no memory left: the blocks that
    cannot be noted for later use go back to the device."""
    _run(fake, r"""
ctx = context()
needs_new()
base = live()
L = api.lib()
G = api.Graph.from_csr(ctx, *ring(5000))
states = [api.State(G, api.CC) for _ in range(3)]
B = api.Batch(ctx, [ring(100)])
calls = [(L.grd_batch_free, B.h)] + [(L.grd_state_free, S.h) for S in states] + [(L.grd_graph_free, G.h)]
ctx._live.clear()
B.h = G.h = None
for S in states:
    S.h = None
fake.fake_new_fails(1)
rc = 0
for f, h in calls:
    rc |= f(h)
fake.fake_new_fails(0)
assert rc == 0 and live() == base and fake.fake_bad_frees() == 0
ctx.close()
assert live() == 0
print("done")
""")


def test_state_creation_without_host_memory_fails_cleanly(fake):
    """Whichever host allocation of a state's creation fails, the call returns an
    error (no exception through the C interface) and no device block is lost."""
    _run(fake, r"""
fake.fake_new_fails_in.argtypes, fake.fake_new_left.restype = [ct.c_long], ct.c_long
ctx = context()
needs_new()
ctx.set_pull_tiling(3, 4)
G = api.Graph.from_csr(ctx, *ring(5000))
L = api.lib()
base = live()
failures = 0
for algo in (api.CC, api.PR_PULL):
    for k in range(1, 10000):
        h = ct.c_void_p()
        fake.fake_new_fails_in(k)
        rc = L.grd_state_create(G.h, algo, ct.byref(h))
        left = fake.fake_new_left()
        fake.fake_new_fails_in(0)
        if rc == 0:
            assert L.grd_state_free(h) == 0
        if left:
            break
        failures += rc != 0
        assert rc in (0, 3)  # (the state is created all the same, or GRD_ERR_OOM)
    assert rc == 0
assert failures > 20
G.free()
ctx.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""")


@pytest.mark.parametrize("algo,weighted", [("CC", False), ("SSSP", True), ("PR_PULL", False)])
@pytest.mark.parametrize("mode", [1, 2, 3])
def test_a_failed_state_leaves_its_graph_as_it_was(fake, algo, weighted, mode):
    """With too little device memory for a state and the regrouping it asks for,
    however far it gets, nothing half made stays behind: after all the failures
    the graph and its state hold what they hold without one."""
    _run(fake, r"""
algo, weighted, mode = api.%s, %s, %d
ctx = context()
rp, col = ring(5000)
w = np.arange(len(col), dtype=np.uint32) if weighted else None


def graph():
    ctx.set_pull_tiling(0)
    G = api.Graph.from_csr(ctx, rp, col, w)
    for a in (api.CC, api.PR_PULL):  # (what a graph computes once for every state)
        api.State(G, a).free()
    ctx.set_pull_tiling(mode, 4)
    ctx.trim()
    return G, live()


G, base = graph()
S = api.State(G, algo)
ctx.trim()
want = live() - base
S.free()
G.free()
G, base = graph()
failures, made = 0, []
for extra in range(0, 1 << 22, 5000):
    limit(base + extra)
    if not refused(lambda: made.append(api.State(G, algo)), "failed"):
        break
    failures += 1
ctx.trim()
assert failures > 3 and live() - base == want, (failures, live() - base, want)
made.pop().free()
G.free()
limit(UNLIMITED)
ctx.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""" % (algo, weighted, mode))


def test_batch_blocks_are_cut_when_they_change(fake):
    """Tiles that give a batch the same blocks cost nothing; without memory for
    other blocks the tuning fails and the batch has none to run over until there
    is memory again."""
    _run(fake, r"""
ctx = context()
launches = fake.fake_launches
large = api.Batch(ctx, [ring(300000)])  # 2.4 M arcs: blocks of 4096 for every tile
small = api.Batch(ctx, [ring(3000)])
for tile in (1024, 2048, 4096):
    at = launches()
    large.tune(tile=tile)
    assert launches() == at
    small.tune(tile=tile)
    assert launches() > at
small.tune(tile=1024)
ctx.trim()
limit(0)
assert refused(lambda: small.tune(tile=4096), "failed")
at = launches()
assert refused(lambda: small.pagerank(), "failed") and launches() == at
assert refused(lambda: small.autotune(), "failed")
limit(UNLIMITED)
at = launches()
small.tune(tile=4096)
assert launches() > at
small.free()
large.free()
ctx.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""")


@pytest.mark.parametrize("what", ["graph", "mode 1", "mode 2", "mode 3", "batch"])
def test_host_arrays_outlive_their_copies(fake, what):
    """Copies run at the next synchronisation at the latest, and device memory
    runs out at every allocation in turn: whatever a failing call copies from is
    there until the copy has run."""
    _run(fake, r"""
what = "%s"
fake.fake_defer(1)
ctx = context()
rp, col = ring(5000)
w = np.arange(len(col), dtype=np.uint32)
G = api.Graph.from_csr(ctx, rp, col, w)
for a in (api.CC, api.PR_PULL):
    api.State(G, a).free()
if what.startswith("mode"):
    ctx.set_pull_tiling(int(what[-1]), 4)


def make():
    if what == "graph":
        return api.Graph.from_csr(ctx, rp, col, w)
    if what == "batch":
        return api.Batch(ctx, [(rp, col)])
    return api.State(api.Graph.from_csr(ctx, rp, col, w), api.PR_PULL)


failures, made = 0, []
fake.fake_mallocs_left.argtypes = [ct.c_uint64]
for n in range(1000):
    ctx.trim()
    fake.fake_mallocs_left(n)
    if not refused(lambda: made.append(make()), "failed"):
        break
    failures += 1
fake.fake_mallocs_left(UNLIMITED)
assert failures > 10 and fake.fake_lost() == 0, (failures, fake.fake_lost())
ctx.close()
assert live() == 0 and fake.fake_bad_frees() == 0
print("done")
""" % what)
