"""Host copies around the size where they change from the runtime's path to the pinned
slots (4 MiB), at whole and partial chunks (2 MiB), alone and from several threads."""
import threading

import numpy as np
import pytest

from conftest import load_vespa

V = load_vespa()
from vespa_jl_amd._lib import DeviceBuffer  # noqa: E402

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _round_trip(nbytes, seed):
    a = np.random.default_rng(seed).integers(0, 256, size=nbytes, dtype=np.uint8)
    b = np.zeros_like(a)
    buf = DeviceBuffer(nbytes)
    buf.upload(a)
    buf.download(b)
    buf.free()
    return bool(np.array_equal(a, b))


@pytest.mark.parametrize("nbytes", [1, 4 * MIB - 1, 4 * MIB, 4 * MIB + 1, 6 * MIB, 8 * MIB + 12345, 40 * MIB + 8])
def test_round_trip_is_bytewise(nbytes):
    print(f"round trip {nbytes}", flush=True)
    assert _round_trip(nbytes, nbytes % 97)


def test_round_trips_from_several_threads():
    print("round trips from 6 threads", flush=True)
    ok = [False] * 6

    def work(i):
        ok[i] = all(_round_trip(5 * MIB + 4099 * i + j, 10 * i + j) for j in range(3))
    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(ok)


@pytest.mark.parametrize("nbytes", [4 * MIB + 1, 4 * MIB + 16, 6 * MIB + 15, 9 * MIB + 12345])
@pytest.mark.parametrize("offset", [0, 1, 8, 16, 2 * MIB + 48])
def test_copies_inside_an_allocation(nbytes, offset):
    """Chunks moved by the kernel (16-byte aligned device addresses) and by the runtime (others),
    with partial 16-byte groups at the end, up to the allocation's last byte."""
    print(f"copies of {nbytes} at {offset}", flush=True)
    a = np.random.default_rng(nbytes + offset).integers(0, 256, size=nbytes + offset, dtype=np.uint8)
    buf = DeviceBuffer(a.nbytes)
    V.check(V.load_library().vh_buffer_upload(buf.ptr + offset, a.ctypes.data + offset, nbytes))
    out = np.zeros(nbytes + 2, dtype=np.uint8)
    V.check(V.load_library().vh_buffer_download(out.ctypes.data + 1, buf.ptr + offset, nbytes))
    assert np.array_equal(out[1:-1], a[offset:]) and out[0] == 0 and out[-1] == 0
    buf.free()


def test_device_memory_as_the_host_side():
    """What the runtime copies stays accepted at every size."""
    for n in (MIB, 8 * MIB):
        x = np.random.default_rng(n).integers(0, 256, size=n, dtype=np.uint8)
        a, b = DeviceBuffer(n), DeviceBuffer(n).upload(x)
        V.check(V.load_library().vh_buffer_upload(a.ptr, b.ptr, n))
        assert np.array_equal(a.download(np.zeros_like(x)), x)
        a.upload(np.zeros_like(x))
        V.check(V.load_library().vh_buffer_download(a.ptr, b.ptr, n))
        assert np.array_equal(a.download(np.zeros_like(x)), x)
