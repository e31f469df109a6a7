"""The library's host code over a HIP runtime on the host (tests/host/hip_stub.cpp:
two devices, memory is host memory, kernels do nothing), each case in a process
of its own: what a caller's current device, missing pinned memory or missing
threads may not change.  No GPU needed."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "host", "hip_stub.cpp")

PRELUDE = """
import ctypes as C, sys, threading
import numpy as np
stub = C.CDLL({stub!r}, mode=C.RTLD_GLOBAL)
stub.stub_limits.argtypes = [C.c_int, C.c_int, C.c_long]
stub.stub_device_max.argtypes = [C.c_long]
sys.path.insert(0, {root!r})
from femorph_amd import femx, meshgen
from femorph_amd.mesh import BoundaryConditions, Mesh
assert femx.device_count() == 2

def log():
    b = C.create_string_buffer(1 << 20)
    stub.stub_log(b, len(b))
    return [l.split() for l in b.value.decode().splitlines()]

def vms(n_nodes):
    # 6 tets and nodes that no element uses: a state of any size
    m = meshgen.tet_cube(1)
    m = Mesh(np.vstack([m.coords, np.full((n_nodes - 8, 3), 2.0)]), m.conn)
    dm = femx.DeviceMesh(m)
    g = femx.VMSSolver(dm, BoundaryConditions(), rho=1.0, mu=0.01, inv_eps=1.0, c1=4.0, c2=2.0, dt=0.01)
    sol = np.random.default_rng(n_nodes).normal(size=(n_nodes, 4))
    g.set_state(sol)
    return g, sol

def check(g, sol):
    np.testing.assert_array_equal(g.get_state()[0], sol)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("no host compiler or HIP headers")
    out = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", STUB, "-o", out], check=True)
    return out


def _run(stub, code):
    script = PRELUDE.format(stub=stub, root=ROOT) + textwrap.dedent(code) + "\nprint('ok')\n"
    r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), (r.returncode, r.stdout + r.stderr)


# one chunk of 2 MiB holds 65,516 nodes' states, 6 tets' subgrid velocities
# and the error flag, each rounded up to 64 bytes
@pytest.mark.parametrize("n_nodes", [100, 65516, 65517, 400000])
def test_read_back_with_another_current_device(stub, n_nodes):
    """A state is read by a thread whose current device is not the handle's;
    that device stays the thread's."""
    _run(stub, f"""
    g, sol = vms({n_nodes})
    assert stub.hipSetDevice(1) == 0
    check(g, sol)
    assert stub.stub_device() == 1
    assert stub.hipSetDevice(1) == 0
    h, hsol = vms({n_nodes})
    err = []
    def reader():  # a new thread's current device is 0
        try:
            check(h, hsol)
            assert stub.stub_device() == 0
        except BaseException as e:
            err.append(e)
    t = threading.Thread(target=reader)
    t.start()
    t.join()
    assert not err, err
    """)


# no pinned memory at all, one chunk only, an odd number; no threads, one; pool given back
@pytest.mark.parametrize("pinned,threads", [(0, 99), (1, 99), (3, 99), (99, 0), (99, 1), (0, 0)])
@pytest.mark.parametrize("n_nodes", [100, 65516, 65517, 400000])
def test_read_back_without_pinned_memory_or_threads(stub, n_nodes, pinned, threads):
    _run(stub, f"""
    g, sol = vms({n_nodes})
    stub.stub_limits({pinned}, {threads}, -1)
    for _ in range(3):
        check(g, sol)
    stub.stub_limits(99, 99, -1)
    femx.set_device_cache(0)
    check(g, sol)
    """)


def test_log_of_a_union_member_waits_for_the_union(stub):
    """The log row of a handle in a union is written on the union's stream:
    the read (and what the exit condition adds) on the handle's own stream
    comes after it."""
    _run(stub, """
    m = meshgen.hex_cube(7, 0.0)
    g = femx.SUPGSolver(femx.DeviceMesh(m), BoundaryConditions(), rho=1.0, mu=0.01, alpha=1.0, cI=4.0, dt=0.01,
                        precision=femx.FEMX_MIXED)
    g.set_state(np.zeros((m.n_nodes, 3)))
    g.step(1)
    log()
    g.get_log()
    own = {l[1] for l in log() if l[0] == "read"}
    assert len(own) == 1
    own = own.pop()
    u = femx.SUPGUnion()
    u.add(g, 3)
    u.step(2)
    union = {l[1] for l in log() if l[0] == "launch"}
    assert len(union) == 1 and own not in union
    g.get_log()
    calls = [l for l in log() if l[1] == own]
    assert calls[0] == ["wait", own, union.pop()], calls
    assert calls[1][0] == "read", calls
    u.remove(g)
    """)


@pytest.mark.parametrize("n_nodes", [100, 65516, 65517, 400000])
def test_read_back_without_host_memory(stub, n_nodes):
    """No exception for want of host memory leaves a C entry or ends a helper
    thread: the state comes back all the same."""
    _run(stub, f"""
    g, sol = vms({n_nodes})
    out = np.zeros_like(sol)
    read = lambda: femx.load().femx_vms_get_state(g._h, out.ctypes.data_as(C.POINTER(C.c_double)), None, None)
    for _ in range(3):
        stub.stub_limits(99, 99, 0)
        status = read()
        stub.stub_limits(99, 99, -1)
        assert status == 0
        np.testing.assert_array_equal(out, sol)
        out[:] = 0.0
    """)


@pytest.mark.parametrize("n", [7, 44])
def test_supg_state_without_room_for_its_staging(stub, n):
    """A SUPG state is read where the device has no room left for the array
    that all of it would pass through, and its fields where there is room for
    one of them; without any, the fields are refused."""
    _run(stub, f"""
    m = meshgen.hex_cube({n}, 0.0)
    g = femx.SUPGSolver(femx.DeviceMesh(m), BoundaryConditions(), rho=1.0, mu=0.01, alpha=1.0, cI=4.0, dt=0.01)
    sol = np.random.default_rng(1).normal(size=(m.n_nodes, 3))
    g.set_state(sol)
    out = np.zeros_like(sol)
    p = out.ctypes.data_as(C.POINTER(C.c_double))
    stub.stub_device_max(0)
    assert femx.load().femx_supg_get_state(g._h, p, None, None, None, None) == 0
    np.testing.assert_array_equal(out, sol)
    try:
        g.get_state()
        assert False
    except femx.FemxError as e:
        assert "hipMalloc" in str(e)
    stub.stub_device_max(2 * 8 * m.n_elems)
    np.testing.assert_array_equal(g.get_state()["sol"], sol)
    stub.stub_device_max(-1)
    assert femx.load().femx_supg_get_state(g._h, p, None, None, None, None) == 0
    """)
