"""The builder's host side under several builds at once: what it holds while it
waits, and what its staged copies share. Each test runs in a process of its
own, with some of the runtime's entry points looked at (cpp/hip_shim.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

TESTS = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys, threading
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)  # before the runtime
sys.path.insert(0, sys.argv[2])
import numpy as np
import conftest, oracle_py as orc
svo = conftest.load_package()

def mesh(faces, seed, scale=0.01):
    rng = np.random.default_rng(seed)
    centre = rng.uniform(0.1, 0.9, (faces, 1, 3))
    tab = np.zeros((4 * faces, 9), np.float32)  # the fourth vertex is unused
    tab[:, :3] = (centre + rng.normal(scale=scale, size=(faces, 4, 3))).reshape(-1, 3)
    tab[:, 6:] = 255.0
    idx = (4 * np.arange(faces)[:, None] + np.arange(3)).astype(np.int32).reshape(-1)
    return tab, np.full(faces, 3, np.int32), idx

def build(m, res=64):
    return svo.VoxelOctree.build_from_mesh(m[0], False, m[1], m[2], res, threads=8, memory_budget=1 << 30).words()

def expect(m, res=64):
    return orc.Mesh(m[0], False, m[1], m[2]).build(res, 8, 1 << 30)[1]

def at_once(meshes, times=1):
    got = [[] for _ in meshes]
    start = threading.Barrier(len(meshes))
    def work(k):
        start.wait()
        for _ in range(times):
            got[k].append(build(meshes[k]))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(meshes))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    return got
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("shim") / "hip_shim.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(TESTS, "cpp", "hip_shim.cpp"), "-ldl", "-o", out], check=True)
    return out


def _run(shim, code):
    r = subprocess.run([sys.executable, "-u", "-c", PRELUDE + code, shim, TESTS], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


def test_staged_copies_record_events_of_their_own_workspace(shim):
    """An event can only be recorded in streams of its device, so each
    workspace has its own: none is recorded in the streams of two."""
    print("[gpu] two builds at once, arrays of more than a staging chunk", flush=True)
    _run(shim, """
meshes = [mesh(60000, 1), mesh(60001, 2)]
want = [expect(m) for m in meshes]
distinct = ctypes.c_int(0)
for _ in range(20):
    for got, words in zip(at_once(meshes, 2), want):
        assert all(np.array_equal(g, words) for g in got)
    most = shim.shim_streams_per_event(ctypes.byref(distinct))
    if distinct.value > 1:
        break
assert distinct.value > 1 and most == 1, (distinct.value, most)
""")


def test_the_upload_chunk_goes_with_the_copies(shim):
    """Two builds whose arrays fit the shared chunk together: each reaches its
    first stream synchronisation while the other stands in its own, so neither
    waits there with the chunk."""
    print("[gpu] two builds at once, arrays of less than a staging chunk", flush=True)
    _run(shim, """
meshes = [mesh(20000, 1), mesh(20001, 2)]
want = [expect(m) for m in meshes]
assert all(m[0].nbytes + m[1].nbytes + m[2].nbytes < 1 << 23 and len(m[0]) + len(m[1]) >= 1 << 16 for m in meshes)
at_once(meshes, 3)
shim.shim_meet(2)
got = at_once(meshes)
assert shim.shim_met() == 1
assert all(np.array_equal(g[0], words) for g, words in zip(got, want))
""")


def test_builds_at_once_on_every_upload_path(shim):
    """Six threads, each its own mesh: host loops and pageable copies, the
    device's checks with the shared chunk, and arrays of several chunks."""
    print("[gpu] six builds at once", flush=True)
    _run(shim, """
meshes = [mesh(n, k) for k, n in enumerate((300, 9000, 16400, 30000, 60000, 70000))]
want = [expect(m) for m in meshes]
for got, words in zip(at_once(meshes, 5), want):
    assert all(np.array_equal(g, words) for g in got)
""")


def test_builds_without_memory_to_pin(shim):
    """Every copy path of a mesh build where no pinned memory is to be had: host
    loops, the shared checks with one chunk's arrays, arrays of several chunks,
    and a result of several."""
    print("[gpu] builds without pinned memory", flush=True)
    _run(shim, """
cases = [(mesh(300, 1), 64), (mesh(20000, 2), 64), (mesh(60000, 3), 64), (mesh(9000, 4, 0.05), 256)]
want = [expect(*c) for c in cases]
assert want[-1].nbytes > 1 << 23
shim.shim_pinning(0)
for c, words in zip(cases, want):
    assert np.array_equal(build(*c), words)
""")
