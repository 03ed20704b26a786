"""Host code of the library under a HIP runtime without a device (hip_stub.c, preloaded
in a child process): which calls are made, in which order, and what follows when one
of them fails. Each test is a program of its own; kernels do not run."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
import numpy as np
sys.path.insert(0, {here!r})
from conftest import load_vespa
V = load_vespa()
L = V.load_library()
S = C.CDLL({stub!r})
S.stub_log.restype = C.c_char_p
S.stub_pinned.restype = C.c_void_p
S.stub_pinned.argtypes = [C.c_size_t]
def log(): return [l.split() for l in S.stub_log().decode().splitlines()]
MIB = 1 << 20
def addr(a): return C.c_void_p(a.ctypes.data)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", so,
                    os.path.join(HERE, "hip_stub.c"), "-ldl", "-lpthread"], check=True)
    return so


def run(stub, program):
    env = dict(os.environ, LD_PRELOAD=stub, VESPAHIP_HOST_THREADS="4", OPENBLAS_NUM_THREADS="1")
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(here=HERE, stub=stub) + textwrap.dedent(program)],
                       env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_device_memory_as_the_host_side_is_not_touched_by_the_cpu(stub):
    """A large copy whose host side is device (or pinned) memory is one copy of the runtime
    on those two pointers, as a small one is; pageable memory goes through the slots."""
    run(stub, """
        from vespa_jl_amd._lib import DeviceBuffer
        a, b = DeviceBuffer(8 * MIB), DeviceBuffer(8 * MIB)
        for f in (L.vh_buffer_upload, L.vh_buffer_download):
            S.stub_clear()
            assert f(a.ptr, b.ptr, 8 * MIB) == 0
            copies = [l for l in log() if l[0] == "copy"]
            assert [[int(x, 16) for x in c[1:3]] + [int(c[3])] for c in copies] == [[a.ptr, b.ptr, 8 * MIB]]
        h = np.arange(8 * MIB, dtype=np.uint8)
        S.stub_clear()
        assert L.vh_buffer_upload(a.ptr, addr(h), 8 * MIB) == 0
        assert len([l for l in log() if l[0] == "copy"]) == 4
        assert C.string_at(a.ptr, 8 * MIB) == h.tobytes()
        """)


def test_copies_without_threads(stub):
    """Where no thread can be made (a process at its limit) large copies still work, in
    the calling thread, and no exception reaches the C entry."""
    run(stub, """
        from vespa_jl_amd._lib import DeviceBuffer
        S.stub_no_threads(1)
        a = DeviceBuffer(9 * MIB + 5)
        h = np.random.default_rng(1).integers(0, 256, 9 * MIB + 5, dtype=np.uint8)
        o = np.zeros(h.size - 1, np.uint8)
        a.upload(h)
        assert L.vh_buffer_download(addr(o), a.ptr + 1, o.size) == 0   # odd source: no kernel
        assert np.array_equal(h[1:], o)
        """)


def test_small_host_batches_wait_once(stub):
    """The flux backend queues its three uploads, the kernel and the download, and waits
    for the last only; a small copy without a stream is the runtime's synchronous one."""
    run(stub, """
        from vespa_jl_amd._lib import DeviceBuffer
        WL = np.ones((100, 5)); F = np.empty_like(WL); ax = np.ones(100, np.int32)
        V.compute_face_fluxes(V.HIPFlux(), V.IdealHydro(1.4), F, WL, WL, ax)
        S.stub_clear()
        V.compute_face_fluxes(V.HIPFlux(), V.IdealHydro(1.4), F, WL, WL, ax)
        assert [l[0] for l in log()] == ["copy", "copy", "copy", "launch", "copy", "sync"]
        a = DeviceBuffer(800).upload(WL[:20])
        S.stub_clear()
        a.download(F[:20])
        a.upload(F[:20])
        assert [l[0] for l in log()] == ["copy", "copy"]
        """)
