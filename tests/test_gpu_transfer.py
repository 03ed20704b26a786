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
