"""GPU parity of the fused unsplit RK2 MUSCL step (PPMKernels muscl_step_3d!,
lib/PPMKernels/src/muscl_grid.jl:314-370) against the oracle, through the C ABI:
bit-identical states and recorded fluxes in Float64 and Float32 on grids whose
sizes are not tile multiples, both tile shapes, ng 2..4; fill_periodic! and
max_wavespeed; and the published benchmark workload (256³ active cells + 4 ghost
zones, Float32) stepped once against the oracle."""
import numpy as np
import pytest

from conftest import load_vespa

V = load_vespa()
from vespa_jl_amd import muscl as M  # noqa: E402
from vespa_jl_amd._lib import VespaHIPError  # noqa: E402

pytestmark = pytest.mark.gpu
G14 = 1.4


def smooth_state(dims, seed, dtype, mach=0.5):
    """Smooth seeded state: ρ ∈ [0.6, 1.4], p ∈ [0.5, 0.9], |v| ~ mach·c."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = dims
    Z, Y, X = np.meshgrid(np.arange(nz) / nz, np.arange(ny) / ny, np.arange(nx) / nx, indexing="ij")

    def field(a):
        k = rng.integers(1, 4, 3)
        ph = rng.uniform(0, 2 * np.pi, 2)
        return a * (np.sin(2 * np.pi * (k[0] * X + k[1] * Y) + ph[0]) * np.cos(2 * np.pi * k[2] * Z + ph[1]))
    rho = 1.0 + field(0.4)
    p = 0.7 + field(0.2)
    vx, vy, vz = field(mach), field(mach), field(mach)
    etot = p / ((G14 - 1) * rho) + 0.5 * (vx * vx + vy * vy + vz * vz)
    return M.prim_to_cons(rho, vx, vy, vz, etot).reshape(5, -1).astype(dtype)


CASES = [((22, 19, 13), 3), ((26, 26, 26), 3), ((9, 12, 40), 2), ((21, 21, 21), 4), ((40, 7, 9), 3)]


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,ng", CASES)
def test_step_bitwise(O, dims, ng, dtype, variant):
    print(f"muscl step {dims} ng={ng} {np.dtype(dtype).name} variant {variant}", flush=True)
    U = smooth_state(dims, seed=sum(dims), dtype=dtype)
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype)
    try:
        g.set_tiles(variant, 8 if variant else 16)
        g.upload(U)
        for s in range(2):
            rec = s == 1
            frec_o = O.muscl_step_3d(U, dims, ng, 0.004, G14, 1.5, 0.05, 1e-10, record=rec)
            g.step(0.004, fluxrec=rec)
            np.testing.assert_array_equal(g.state(), U, err_msg=f"step {s}")
        np.testing.assert_array_equal(g.fluxrec(), frec_o)
    finally:
        g.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_extreme_operands_bitwise(O, dtype):
    """Quotients by a shared denominator and the limiter where they could go wrong:
    subnormal quotients and their ties (odd multiples of the least subnormal over even
    densities), zeros, huge values, and cells holding infinities and NaN."""
    dims, ng = (20, 18, 17), 3
    rng = np.random.default_rng(5)
    n = int(np.prod(dims))
    least = np.finfo(dtype).smallest_subnormal
    U = np.empty((5, n), dtype=dtype)
    U[0] = rng.integers(1, 9, n)
    for q in (1, 2, 3):
        kind = rng.integers(0, 4, n)
        U[q] = np.where(kind == 0, 0.0, np.where(kind == 1, rng.integers(-40, 40, n) * least, np.where(
            kind == 2, rng.normal(size=n).astype(dtype) * np.finfo(dtype).tiny, rng.normal(size=n))))
    U[4] = rng.uniform(2.0, 30.0, n)
    for i, v in enumerate((np.inf, -np.inf, np.nan, np.finfo(dtype).max)):
        U[i + 1, rng.integers(0, n, 2)] = v
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype)
    g.upload(U)
    with np.errstate(all="ignore"):
        O.muscl_step_3d(U, dims, ng, 0.004, G14, 1.5, 0.05, 1e-10)
    g.step(0.004)
    np.testing.assert_array_equal(g.state(), U)
    assert np.isfinite(U).mean() > 0.5
    g.close()


def test_reference_driver_cases_bitwise(O):
    """The reference's conservation case (26³ blob, dt 0.02, dx 1, 3 steps) and a
    cold supersonic line (eint floor, zero-sign paths)."""
    from test_muscl_oracle import _blob
    for dtype in (np.float64, np.float32):
        U = _blob(26, 13.5, 2.2).astype(dtype)
        g = M.MusclGrid((26, 26, 26), 3, G14, 1.5, 1.0, eltype=dtype)
        g.upload(U)
        for _ in range(3):
            O.muscl_step_3d(U, (26, 26, 26), 3, 0.02, G14, 1.5, 1.0)
            g.step(0.02)
        np.testing.assert_array_equal(g.state(), U)
        g.close()
    n, ng = 16, 3
    dims = (n, 2 * ng + 1, 2 * ng + 1)
    x = np.arange(n)
    rho = np.broadcast_to(1.0 + 0.5 * (x > 5), dims[::-1]).ravel()
    U = np.zeros((5, rho.size))
    U[0] = rho
    U[1] = rho * 2.0
    U[3] = -0.0
    U[4] = rho * (0.5 * 4.0 - 1e-3)
    g = M.MusclGrid(dims, ng, G14)
    g.upload(U)
    O.muscl_step_3d(U, dims, ng, 1e-3, G14)
    g.step(1e-3)
    got = g.state()
    np.testing.assert_array_equal(got, U)
    assert np.array_equal(np.signbit(got), np.signbit(U))
    g.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_fill_periodic_and_wavespeed(O, dtype):
    dims, ng = (20, 17, 23), 3
    U = smooth_state(dims, seed=4, dtype=dtype, mach=2.0)
    U[4, ::7] *= -1.0                                      # negative eint in some cells
    g = M.MusclGrid(dims, ng, G14, eltype=dtype)
    try:
        g.upload(U)
        assert g.max_wavespeed() == O.muscl_max_wavespeed(U, G14)
        g.fill_periodic()
        for f in range(5):
            O.muscl_fill_periodic(U[f], dims, ng)
        np.testing.assert_array_equal(g.state(), U)
    finally:
        g.close()


def test_array_form_and_errors(O):
    dims, ng = (12, 11, 10), 2
    U = smooth_state(dims, seed=9, dtype=np.float64)
    fields = [U[f].copy() for f in range(5)]
    fr = np.empty((3, 5, U.shape[1]))
    M.muscl_step_3d(*fields, dims, ng, dt=0.01, gamma=G14, dx=0.1, fluxrec=fr)
    fo = O.muscl_step_3d(U, dims, ng, 0.01, G14, 1.5, 0.1, record=True)
    np.testing.assert_array_equal(np.stack(fields), U)
    np.testing.assert_array_equal(fr, fo)
    with pytest.raises(VespaHIPError, match="ghost"):
        M.MusclGrid(dims, 1, G14)
    with pytest.raises(VespaHIPError, match="2\\*ng\\+1"):
        M.MusclGrid((4, 12, 12), 2, G14)
    g = M.MusclGrid(dims, ng, G14)
    with pytest.raises(VespaHIPError, match="recorded"):
        g.fluxrec()
    g.close()


def test_benchmark_workload_one_step_bitwise(O):
    """256³ active + 4 ghost zones per side, Float32, dt = 0.2·dx, dx = 1/256."""
    print("muscl 264^3 f32 vs oracle", flush=True)
    dims, ng = (264, 264, 264), 4
    U = smooth_state(dims, seed=1234, dtype=np.float32, mach=0.3)
    g = M.MusclGrid(dims, ng, G14, 1.5, 1.0 / 256, eltype=np.float32)
    try:
        g.upload(U)
        g.step(0.2 / 256)
        O.muscl_step_3d(U, dims, ng, 0.2 / 256, G14, 1.5, 1.0 / 256)
        got = g.state()
        assert np.array_equal(got, U)
    finally:
        g.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_flux_register_gather(O, dtype):
    """boundary_flux_register on the device equals the host-loop reference over the
    same recorded fluxes, key for key and value for value (the reference's index-
    mapping lock, test/test_reflux_capture.jl:36-51)."""
    from test_muscl_oracle import register_ref, _rec_state
    n, ng, dt = 12, 3, 0.008
    dx = 1.0 / n
    U, dims = _rec_state(n, ng)
    g = M.MusclGrid(dims, ng, G14, 1.5, dx, eltype=dtype)
    try:
        g.upload(U.astype(dtype))
        g.step(dt, fluxrec=True)
        frec = g.fluxrec()
        reg = M.boundary_flux_register(g, dt)
        flux, interior, act = register_ref(frec, dims, ng, dt, dx)
        assert reg.act == act
        assert reg.flux == flux
        assert reg.interior == interior
    finally:
        g.close()
    # an anisotropic grid with one active cell along z (no interior z faces)
    dims2 = (14, 11, 7)
    U2 = smooth_state(dims2, seed=3, dtype=dtype)
    g = M.MusclGrid(dims2, 3, G14, 1.5, 0.1, eltype=dtype)
    try:
        g.upload(U2)
        g.step(0.004, fluxrec=True)
        reg = M.boundary_flux_register(g, 0.004)
        flux, interior, act = register_ref(g.fluxrec(), dims2, 3, 0.004, 0.1)
        assert reg.flux == flux and reg.interior == interior and act[2] == 1
    finally:
        g.close()


def with_ge(U, cold=False):
    rho = U[0]
    u, v, w = U[1] / rho, U[2] / rho, U[3] / rho
    eint = U[4] / rho - rho.dtype.type(0.5) * (u * u + v * v + w * w)
    if cold:
        eint = np.full_like(rho, 1e-5)
        U = U.copy()
        U[4] = rho * (eint + rho.dtype.type(0.5) * (u * u + v * v + w * w))
    return np.vstack([U, rho * eint]).copy()


@pytest.mark.parametrize("cold", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,ng", [((22, 19, 13), 3), ((21, 21, 21), 4)])
def test_dual_energy_bitwise(O, dims, ng, dtype, cold):
    """muscl_step_3d!(…; ge, eta1): six fields, the η₁ selection (warm and cold
    flows take different branches), ρe advection and the end-of-step sync, recorded
    fluxes with six fields and the flux register read through their stride."""
    print(f"muscl dual {dims} ng={ng} {np.dtype(dtype).name} cold={cold}", flush=True)
    U = with_ge(smooth_state(dims, seed=sum(dims) + 1, dtype=dtype, mach=1.5), cold=cold)
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype, dual=True, eta1=1e-3)
    try:
        g.upload(U)
        for s in range(2):
            rec = s == 1
            frec_o = O.muscl_step_3d(U, dims, ng, 0.004, G14, 1.5, 0.05, 1e-10, record=rec)
            g.step(0.004, fluxrec=rec)
            np.testing.assert_array_equal(g.state(), U, err_msg=f"step {s}")
        fr = g.fluxrec()
        np.testing.assert_array_equal(fr, frec_o)
        from test_muscl_oracle import register_ref
        reg = M.boundary_flux_register(g, 0.004)
        flux, interior, act = register_ref(np.ascontiguousarray(fr[:, :5]), dims, ng, 0.004, 0.05)
        assert reg.flux == flux and reg.interior == interior
    finally:
        g.close()


def test_dual_energy_array_form(O):
    dims, ng = (12, 11, 10), 2
    U = with_ge(smooth_state(dims, seed=5, dtype=np.float64))
    fields = [U[f].copy() for f in range(6)]
    fr = np.empty((3, 6, U.shape[1]))
    M.muscl_step_3d(*fields[:5], dims, ng, dt=0.01, gamma=G14, dx=0.1, ge=fields[5], eta1=1e-3, fluxrec=fr)
    fo = O.muscl_step_3d(U, dims, ng, 0.01, G14, 1.5, 0.1, record=True)
    np.testing.assert_array_equal(np.stack(fields), U)
    np.testing.assert_array_equal(fr, fo)


def test_dual_energy_refused_after_device_pointer_is_shared():
    """Enabling dual energy reallocates the state; once the device address has
    been handed out the call is refused and the context stays usable."""
    import ctypes as C
    dims, ng = (10, 9, 8), 2
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10)
    try:
        L = V.load_library()
        p = C.c_void_p()
        assert L.vh_muscl_state_device_ptr(g._h, C.byref(p)) == 0 and p.value
        assert L.vh_muscl_enable_dual_energy(g._h, 1e-3) == -1
        assert b"state_device_ptr" in L.vh_last_error()
        p2 = C.c_void_p()
        assert L.vh_muscl_state_device_ptr(g._h, C.byref(p2)) == 0 and p2.value == p.value
        U = smooth_state(dims, seed=2, dtype=np.float64)
        g.upload(U)
        g.step(0.002)
        assert np.isfinite(g.state()).all()
    finally:
        g.close()
    # enabling first, then taking the pointer, is the supported order
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, dual=True, eta1=1e-3)
    try:
        p = C.c_void_p()
        assert V.load_library().vh_muscl_state_device_ptr(g._h, C.byref(p)) == 0
        assert V.load_library().vh_muscl_enable_dual_energy(g._h, 2e-3) == 0     # already on: eta1 only
    finally:
        g.close()


# Fast profile: per field, max |fast − oracle| / max |oracle| after three steps.
FAST_TOL = {np.float64: 1e-12, np.float32: 1e-5}


def _rel_err(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return (np.abs(a - b).max(axis=-1) / np.maximum(np.abs(b).max(axis=-1), 1e-300)).max()


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_fast_profile_within_tolerance(O, dtype, dual):
    """The fast arithmetic profile (contracted a*b+c, refined reciprocals, rsqrt sound
    speeds) against the oracle: states and recorded fluxes within FAST_TOL after
    three steps, and not bit-identical to them (the fast kernels ran)."""
    print(f"muscl fast {np.dtype(dtype).name} dual={dual}", flush=True)
    dims, ng = (26, 23, 19), 3
    U = smooth_state(dims, seed=77, dtype=dtype, mach=0.8)
    if dual:
        U = with_ge(U)
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype, dual=dual, eta1=1e-3)
    try:
        with pytest.raises(ValueError):
            g.set_mode("approximate")
        g.set_mode("fast")
        g.upload(U)
        for s in range(3):
            rec = s == 2
            frec_o = O.muscl_step_3d(U, dims, ng, 0.004, G14, 1.5, 0.05, 1e-10, record=rec)
            g.step(0.004, fluxrec=rec)
        got = g.state()
        assert np.isfinite(got).all()
        assert _rel_err(got, U) <= FAST_TOL[dtype]
        assert not np.array_equal(got, U)
        fr = g.fluxrec()
        assert _rel_err(fr.reshape(3 * g.nf, -1), frec_o.reshape(3 * g.nf, -1)) <= FAST_TOL[dtype]
        g.set_mode("exact")                      # back to the bit-identical kernels
        g.upload(U)
        frec_o = O.muscl_step_3d(U, dims, ng, 0.004, G14, 1.5, 0.05, 1e-10, record=True)
        g.step(0.004, fluxrec=True)
        np.testing.assert_array_equal(g.state(), U)
        np.testing.assert_array_equal(g.fluxrec(), frec_o)
    finally:
        g.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_fast_profile_benchmark_workload(dtype):
    """256³ active + 4 ghost zones: the fast profile within FAST_TOL of the exact
    profile (bit-identical to the oracle at this size) after two steps."""
    print(f"muscl 264^3 fast vs exact {np.dtype(dtype).name}", flush=True)
    dims, ng = (264, 264, 264), 4
    U = smooth_state(dims, seed=99, dtype=dtype, mach=0.3)
    res = {}
    for mode in ("exact", "fast"):
        g = M.MusclGrid(dims, ng, G14, 1.5, 1.0 / 256, eltype=dtype)
        try:
            g.set_mode(mode)
            g.upload(U)
            for _ in range(2):
                g.step(0.2 / 256)
            res[mode] = g.state()
        finally:
            g.close()
    assert np.isfinite(res["fast"]).all()
    assert _rel_err(res["fast"], res["exact"]) <= FAST_TOL[dtype]


# ---------------- bc! (ghost refill before each RK stage) ----------------

def _outflow_fill(V, dims, ng):
    """Zero-gradient ghost zones: every ghost cell copies the nearest active
    cell (a host bc!; V is (nf, N) or (nf, nz, ny, nx))."""
    nx, ny, nz = dims
    A = V.reshape((V.shape[0], nz, ny, nx))
    ix = np.clip(np.arange(nx), ng, nx - ng - 1)
    iy = np.clip(np.arange(ny), ng, ny - ng - 1)
    iz = np.clip(np.arange(nz), ng, nz - ng - 1)
    A[...] = A[:, iz][:, :, iy][:, :, :, ix].copy()


def _periodic_fill(O, V, dims, ng):
    for q in range(V.shape[0]):
        O.muscl_fill_periodic(V[q].reshape(-1), dims, ng)


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_bc_periodic_on_device_bitwise(O, dtype, dual):
    """bc! = fill_periodic! before each stage, filled by the library on the device,
    against the oracle's step with the same refill hook: every cell bit for bit
    over two steps (ghost cells combine the unfilled input, as the reference)."""
    dims, ng = (22, 19, 13), 3
    print(f"muscl bc periodic {np.dtype(dtype).name} dual={dual}", flush=True)
    U = smooth_state(dims, seed=7, dtype=dtype)
    if dual:
        U = with_ge(U)
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype, dual=dual)
    try:
        g.set_bc("periodic")
        g.upload(U)
        Uo = np.ascontiguousarray(U.copy())
        for _ in range(2):
            g.step(0.02)
            O.muscl_step_3d_bc(Uo, dims, ng, 0.02, lambda V, s: _periodic_fill(O, V, dims, ng), G14, 1.5, 0.05)
        assert np.array_equal(g.state(), Uo)
    finally:
        g.close()


@pytest.mark.parametrize("mode", ["exact", "fast"])
@pytest.mark.parametrize("dims,ng,dual,dtype", [((21, 12, 40), 4, False, np.float32), ((9, 12, 33), 2, True, np.float64),
                                                ((10, 40, 9), 3, False, np.float64), ((37, 9, 18), 3, True, np.float32)])
def test_bc_periodic_images_equal_the_filled_copy(O, V, dims, ng, dual, dtype, mode):
    """Stages that read ghost cells from their periodic images against the general path,
    which refills a copy (here by a host hook): states and recorded fluxes of three steps,
    down to as many active cells as ghosts along an axis."""
    U = smooth_state(dims, seed=3, dtype=dtype)
    if dual:
        U = with_ge(U)
    gs = [M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype, dual=dual) for _ in range(2)]
    gs[0].set_bc("periodic")
    gs[1].set_bc(lambda W, stage: _periodic_fill(O, W.reshape(len(U), -1), dims, ng))
    for g in gs:
        g.set_mode(mode)
        g.upload(U)
        for k in range(3):
            g.step(0.01, fluxrec=k == 2)
    np.testing.assert_array_equal(gs[0].state(), gs[1].state())
    np.testing.assert_array_equal(gs[0].fluxrec(), gs[1].fluxrec())
    for g in gs:
        g.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_bc_host_callback_outflow_bitwise(O, dtype):
    """A host bc! (zero-gradient ghosts) through the C ABI's callback: the library
    hands the stage's device state to the caller before each stage; against the
    oracle's step with the same hook, every cell bit for bit. A no-op callback is
    bc! = nothing; a failing one is an error and leaves the state as it was."""
    dims, ng = (21, 21, 21), 4
    print(f"muscl bc host outflow {np.dtype(dtype).name}", flush=True)
    U = smooth_state(dims, seed=9, dtype=dtype)
    g = M.MusclGrid(dims, ng, G14, 1.5, 0.05, 1e-10, eltype=dtype)
    stages = []
    try:
        g.set_bc(lambda V, s: (stages.append(s), _outflow_fill(V, dims, ng)))
        g.upload(U)
        g.step(0.02, fluxrec=True)
        Uo = np.ascontiguousarray(U.copy())
        fo = O.muscl_step_3d_bc(Uo, dims, ng, 0.02, lambda V, s: _outflow_fill(V, dims, ng), G14, 1.5, 0.05,
                                record=True)
        assert stages == [0, 1]
        assert np.array_equal(g.state(), Uo)
        assert np.array_equal(g.fluxrec(), fo)
        # no-op callback == no bc!
        g.upload(U)
        g.set_bc(lambda V, s: None)
        g.step(0.02)
        a = g.state()
        g.set_bc(None)
        g.upload(U)
        g.step(0.02)
        assert np.array_equal(a, g.state())
        # a failing callback
        g.upload(U)

        def bad(V, s):
            if s == 1:
                raise RuntimeError("no ghost data")
        g.set_bc(bad)
        with pytest.raises(VespaHIPError, match="bc! callback"):
            g.step(0.02)
        assert np.array_equal(g.state(), U)
    finally:
        g.close()


def test_bc_array_form(O):
    """muscl_step_3d(...; bc=...) on host arrays: bc!(D, S1, S2, S3, Tau)."""
    dims, ng = (12, 11, 10), 3
    U = smooth_state(dims, seed=3, dtype=np.float64)
    f = [u.copy() for u in U]
    calls = []

    def bc(*fs):
        calls.append(len(fs))
        for q in fs:
            O.muscl_fill_periodic(q, dims, ng)
    M.muscl_step_3d(*f, dims, ng, dt=0.02, gamma=G14, dx=0.05, bc=bc)
    Uo = np.ascontiguousarray(U.copy())
    O.muscl_step_3d_bc(Uo, dims, ng, 0.02, lambda V, s: _periodic_fill(O, V, dims, ng), G14, 1.5, 0.05)
    assert calls == [5, 5]
    assert np.array_equal(np.stack(f), Uo)
