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
        h = np.arange(8 * MIB - 1, dtype=np.uint8)
        S.stub_clear()
        assert L.vh_buffer_upload(a.ptr + 1, addr(h), h.size) == 0   # odd target: no kernel
        assert len([l for l in log() if l[0] == "copy"]) == 4
        assert C.string_at(a.ptr + 1, h.size) == h.tobytes()
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
        assert L.vh_buffer_upload(a.ptr + 1, addr(h), o.size) == 0     # odd addresses: no kernel
        assert L.vh_buffer_download(addr(o), a.ptr + 1, o.size) == 0
        assert np.array_equal(h[:-1], o)
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


LOOP = """
        clk = (C.c_double * 8).from_address(S.stub_pinned(64))
        looks = []
        @C.CFUNCTYPE(None, C.c_char_p)
        def on_sync(kind):
            if kind == b"event" and not looks:   # the loop's first reduction: dt = cfl
                clk[2] = 1.0
            elif kind == b"stream":              # the clock after what was queued
                looks.append(steps() - sum(looks))
                clk[0], clk[1], clk[3], clk[5] = t0 + 0.3 * sum(looks), 0.3, sum(looks), tfinal
                if not clk[0] < tfinal * (1 - 1e-12): clk[7] = 1.0
        S.stub_on_sync(on_sync)
"""


@pytest.mark.parametrize("legs,queued", [(1, [1]), (2, [2]), (3, [3]), (8, [8]), (12, [8, 4])])
def test_steps_queued_for_a_leg(stub, legs, queued):
    """A loop with a final time queues one step, learns dt from the first reduction
    and queues what the leg holds (at most 8 before the first look at the clock): a leg of
    one step is one step, not eight of which seven do nothing."""
    run(stub, f"""
        prob = V.Problem("l", (24, 20), ((0.0, 1.0),) * 2, 1.4, "periodic", lambda x, y, z: (1.0, 0.0, 0.0, 0.0, 1.0), 1.0, 0.3)
        sim = V.Simulation(V.UniformMesh((24, 20), prob.domain), prob)
        t0, tfinal = 0.0, {legs} * 0.3 - 0.1
        prob.tfinal = tfinal
        def steps(): return (len([l for l in log() if l[0] == "launch"]) - 2) // 3   # cfl and begin, then 3 per step
        S.stub_clear()
        {LOOP}
        V.evolve(sim)
        assert looks == {queued}, looks
        """)


@pytest.mark.parametrize("legs,queued", [(1, [1]), (2, [2]), (8, [8]), (12, [8, 4])])
def test_block_steps_queued_for_a_leg(stub, legs, queued):
    run(stub, f"""
        from vespa_jl_amd import blockmesh as BM
        m = BM.BlockMesh(2, 0, (1.0 / 8, 1.0 / 8), 1.4, [0], [[8, 8, 1]], [[0, 0, 0]], [[0] * 4 + [1, 1]])
        s = BM.BlockSimulation(m, np.float64, cfl=0.3)
        s.set_launch(use_graph=False)
        t0, tfinal = 0.0, {legs} * 0.3 - 0.1
        per = None
        def launches(): return len([l for l in log() if l[0] == "launch"])
        S.stub_clear()
        s.step(0.1)
        per = launches()   # the dt, then a step's launches; in a loop a tail follows them
        def steps(): return (launches() - 2) // per
        S.stub_clear()
        {LOOP}
        s.evolve(tfinal)
        assert looks == {queued}, looks
        """)


@pytest.mark.parametrize("call", ["hipStreamCreateWithFlags", "hipEventCreateWithFlags", "hipEventRecord",
                                  "hipStreamWaitEvent"])
def test_block_stages_stay_ordered_when_a_fork_or_join_fails(stub, call):
    """The shape classes of a stage run side by side on forked streams. Whatever call of the
    fork or the join fails, every launch of a stage still follows all of the one before it
    (the happens-before order of the log), and the context's stream ends behind them all."""
    run(stub, f"""
        from vespa_jl_amd import blockmesh as BM
        m = BM.random_block_pairs(12, seed=3, rank=3)
        def known(ops):
            hb, ev, host, seen, n = {{}}, {{}}, set(), [], 0
            for o in ops:
                h = hb.setdefault(o[1], set()) if o[0] != "event" else None
                if o[0] == "launch":
                    h |= host
                    seen.append((o[1], set(h)))
                    h.add(len(seen) - 1)
                elif o[0] == "record": ev[o[2]] = set(h)
                elif o[0] == "wait": h |= ev.get(o[2], set())
                elif o[0] == "sync": host |= h
            return seen, hb, host
        most = 0
        for fail_at in [-1] + list(range(16)):
            s = BM.BlockSimulation(m, np.float64, cfl=0.3)
            S.stub_clear()
            S.stub_fail({call!r}.encode(), fail_at)
            s.step(0.1)
            S.stub_fail(b"", -1)
            seen, hb, host = known([l for l in log() if l[0] in ("launch", "record", "wait", "sync")])
            k = (len(seen) - 3) // 2   # the dt, then twice: link fluxes and k classes
            assert k >= 3 and len(seen) == 2 * k + 3
            stage = [0, 1] + [2] * k + [3] + [4] * k
            most = max(most, len(set(st for st, _ in seen)))
            for i, (_, h) in enumerate(seen):
                missing = [j for j in range(i) if stage[j] != stage[i] and j not in h]
                assert not missing, ({call!r}, fail_at, i, missing)
            assert hb[seen[0][0]] | host == set(range(len(seen))), ({call!r}, fail_at)
            s.close()
        assert most >= 3   # without a failure they do run side by side
        """)


def test_automatic_z_planes_follow_the_mesh(stub):
    """The automatic number of planes per tile stays automatic when only graphs are
    switched off, and is chosen anew by a regrid and by another tile width; an explicit one
    stays, and -1 goes back to the rule."""
    run(stub, """
        from vespa_jl_amd import blockmesh as BM
        from test_gpu_blocks import three_boxes
        small, large, src = three_boxes()
        want = BM.BlockSimulation(large, np.float64).info()["zchunk"]
        wide = BM.BlockSimulation(large, np.float64)
        wide.set_tiling(4)
        assert BM.BlockSimulation(small, np.float64).info()["zchunk"] == 1 and want == 2
        for set_up in (lambda s: None, lambda s: s.set_launch(use_graph=False),
                       lambda s: (s.set_launch(zchunk=5), s.set_launch(zchunk=-1))):
            s = BM.BlockSimulation(small, np.float64)
            set_up(s)
            s.regrid(large, src)
            assert s.info()["zchunk"] == want
            s.set_tiling(4)
            assert s.info()["zchunk"] == wide.info()["zchunk"] == 4
        s = BM.BlockSimulation(small, np.float64)
        s.set_launch(zchunk=1)
        s.regrid(large, src)
        assert s.info()["zchunk"] == 1
        assert L.vh_blocks_set_launch(s._h, -2, 0, 0) != 0
        """)


def test_launch_defaults_of_a_grid(stub):
    """zchunk 0 is the library's march for the variant (the default variant's is the one a new
    grid has), and the tuners try the defaults and marches shorter than them."""
    run(stub, """
        from vespa_jl_amd import autotune as AT, blockmesh as BM
        def sim(dims, T=np.float64):
            prob = V.Problem("l", dims, ((0.0, 1.0),) * len(dims), 1.4, "periodic", lambda x, y, z: (1.0, 0.0, 0.0, 0.0, 1.0), 1.0, 0.3)
            return V.Simulation(V.UniformMesh(dims, prob.domain), prob, eltype=T)
        for dims in ((60, 52, 44), (96, 96, 96), (171, 130, 97), (256, 256, 128), (33, 20), (50,)):
            for T in (np.float64, np.float32):
                s = sim(dims, T)
                d = s.launch()
                for v in range(s.tile_count()):
                    s.set_launch(v, 0)
                    if s.launch()["tile"] == d["tile"]: assert s.launch() == d, (dims, d, s.launch())
                s.set_launch(0, 7)
                assert s.launch()["zchunk"] == (7 if len(dims) == 3 else 1)
        s = sim((60, 52, 44))
        d = s.launch()
        r = AT.tune_grid(s, steps=1, use_cache=False)
        tried = [(t["tile"], t["zchunk"]) for t in r["trials"]]
        assert (d["tile"], d["zchunk"]) in tried and d["zchunk"] == 1
        assert {1, 2, 4, 8, 16, 32} <= {z for _, z in tried}
        m = BM.random_block_pairs(12, seed=3, rank=3)
        b = BM.BlockSimulation(m, np.float64, cfl=0.3)
        z = b.info()["zchunk"]
        r = AT.tune_blocks(b, steps=1, use_cache=False)
        assert {-1, 0, 1, 2, 4, 8, 16} <= {t["zchunk"] for t in r["trials"]}
        assert {t["max_tile_x"] for t in r["trials"] if t["zchunk"] == -1 and t["max_workgroups"] == 0} == {16, 32}
        """)


def test_sizes_of_the_fused_reverse_form(stub):
    """The tiled kernel runs (one launch per evaluation, the passes take three) on periodic
    sizes of 10 to 16 and above 17, and not where its output is the state it reads."""
    run(stub, """
        from vespa_jl_amd import adjoint as AD
        from vespa_jl_amd._lib import DeviceBuffer
        for n in range(2, 70):
            assert AD.fused_covers(n, 32) == AD.fused_covers(32, n) == (10 <= n <= 16 or n > 17)
        def launches(dims, bc="periodic", fused=True, alias=False):
            prob = V.Problem("l", dims, ((0.0, 1.0),) * len(dims), 1.4, bc, lambda x, y, z: (1.0, 0.0, 0.0, 0.0, 1.0), 1.0, 0.3)
            sim = V.Simulation(V.UniformMesh(dims, prob.domain), prob)
            AD.set_form(sim, fused)
            U, w, o = (DeviceBuffer(40 * sim.ncell) for _ in range(3))
            S.stub_clear()
            V.check(L.vh_grid_step_vjp(sim._h, U.ptr, 0.1, w.ptr, U.ptr if alias else o.ptr))
            return len([l for l in log() if l[0] == "launch"]) - 2   # the dt and stage 1
        for dims in ((10, 10), (16, 48), (18, 33), (50, 37), (32, 32), (64, 16)):
            assert launches(dims) == 2 and launches(dims, fused=False) == 6
            assert launches(dims, alias=True) == 4
        for dims in ((17, 40), (40, 17), (9, 40), (40, 9), (12,), (16, 16, 16)):
            assert launches(dims) == 6
        assert launches((32, 32), "outflow") == 6
        """)


def test_gravity_keeps_no_vector_it_does_not_use(stub):
    """Work vectors of the Poisson solve: r and two p on a uniform grid, whose operator is
    applied again instead of stored, and Ap on a block mesh."""
    run(stub, """
        from vespa_jl_amd import blockmesh as BM
        def allocated(f):
            S.stub_clear()
            f()
            return [int(l[1]) for l in log() if l[0] == "malloc"]
        dims = (16, 12, 10)
        prob = V.Problem("l", dims, ((0.0, 1.0),) * 3, 1.4, "periodic", lambda x, y, z: (1.0, 0.0, 0.0, 0.0, 1.0), 1.0, 0.3)
        sim = V.Simulation(V.UniformMesh(dims, prob.domain), prob)
        a = allocated(lambda: V.enable_gravity(sim))
        assert 3 * 8 * sim.ncell in a and max(a) == 3 * 8 * sim.ncell and 8 in a
        m = BM.random_block_pairs(4, seed=3, rank=3)
        s = BM.BlockSimulation(m, np.float64)
        assert 4 * 8 * s.ncell in allocated(lambda: s.enable_gravity())
        """)


def test_side_streams_are_made_once(stub):
    """Streams for the shape classes of a stage: none for a mesh of one class, for others as
    many as its stages fork, taken over from meshes that are gone (a bounded number is kept),
    never shared by two that live."""
    run(stub, """
        from vespa_jl_amd import amr, blockmesh as BM
        def made(): return [l[1] for l in log() if l[0] == "stream"]
        def launched(): return {l[1] for l in log() if l[0] == "launch"}
        def stepped(m, **kw):
            s = BM.BlockSimulation(m, np.float64, cfl=0.3)
            s.set_launch(**kw)
            S.stub_clear()
            s.evolve(max_steps=1)
            return s
        flat = amr.QuadBlocks(3, 8, 1).mesh()
        m = BM.random_block_pairs(12, seed=3, rank=3)
        for graph in (True, False):
            stepped(flat, use_graph=graph).close()
            assert made() == []
        a = stepped(m)
        first = made()
        assert 2 <= len(first) <= 4 and launched() >= set(first)
        b = stepped(m, use_graph=False)
        second = made()
        assert len(second) == len(first) and not launched() & set(first)
        a.close()
        c = stepped(m, use_graph=False)
        assert made() == [] and launched() >= set(first) and not launched() & set(second)
        b.close()
        c.close()
        S.stub_clear()
        many = [BM.BlockSimulation(m, np.float64, cfl=0.3) for _ in range(8)]
        for s in many: s.step(0.1)
        total = len(made()) - len(many) + len(first) + len(second)   # without the contexts' own
        S.stub_clear()
        for s in many: s.close()
        gone = len([l for l in log() if l[0] == "destroy"]) - len(many)
        assert total == 8 * len(first) and gone == total - 16
        """)
