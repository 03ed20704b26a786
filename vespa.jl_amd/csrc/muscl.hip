// Host side of PPMKernels' unsplit SSP-RK2 MUSCL step (lib/PPMKernels/src/muscl_grid.jl:212-370,
// lib/PPMKernels/src/muscl.jl) on a ghosted 3D grid: the vh_muscl_* entry points, and the
// profile-independent kernels (fill_periodic!, max_wavespeed, the flux-register gathers).
//
// The reference runs, per stage, a cons→prim kernel, then per axis a transpose, the
// PLM+HLL flux line over every pencil, a divergence kernel into a slab and an
// untranspose-add into dU, then the RK combine: ~20 kernels and ~60 full-grid
// passes per step. Here one launch per stage (muscl.h, compiled in the exact and the
// fast arithmetic profile by muscl_kernels.hip) does it all for a tile of 16×16 (or
// 32×8) cells marching along z: the plane's primitives (plus a two-deep halo in x
// and y) are staged in LDS, each cell reconstructs its hi- and lo-face states per
// axis, each face's HLL flux is evaluated once, and each cell sums its divergence
// in the reference's order and writes the combined state; z faces are pipelined
// in registers down the column. Optional flux recording (½F per stage at the lo
// face of each cell, grid-order momenta) is written in the same pass.
#include <float.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/vespahip.h"
#include "host.h"
#include "muscl_common.h"

namespace vh {
namespace {

// fill_periodic! (lib/PPMKernels/src/muscl_grid.jl:644-670) for the five fields:
// every ghost cell copies the periodic image inside the interior.
template <typename T>
__global__ void __launch_bounds__(256) fill_periodic_kernel(T* __restrict__ U, MusclDev G) {
  const int nx = G.n[0], ny = G.n[1], nz = G.n[2], ng = G.ng;
  const long long n = G.ncell;
  const int nix = nx - 2 * ng, niy = ny - 2 * ng, niz = nz - 2 * ng;
  for (long long c = (long long)blockIdx.x * 256 + threadIdx.x; c < n; c += (long long)gridDim.x * 256) {
    const int i = (int)(c % nx);
    const long long t = c / nx;
    const int j = (int)(t % ny), k = (int)(t / ny);
    const bool gh = i < ng || i >= nx - ng || j < ng || j >= ny - ng || k < ng || k >= nz - ng;
    if (!gh) continue;
    const int si = i < ng ? i + nix : (i >= nx - ng ? i - nix : i);
    const int sj = j < ng ? j + niy : (j >= ny - ng ? j - niy : j);
    const int sk = k < ng ? k + niz : (k >= nz - ng ? k - niz : k);
    const long long s = ((long long)sk * ny + sj) * nx + si;
    for (int q = 0; q < G.nf; ++q) U[q * n + c] = U[q * n + s];
  }
}

// max_wavespeed (lib/PPMKernels/src/muscl_grid.jl:672-695): per-workgroup maxima.
template <typename T>
__global__ void __launch_bounds__(256) wavespeed_kernel(const T* __restrict__ U, MusclDev G,
                                                        double* __restrict__ partials) {
  __shared__ double red[4];
  const T g = T(G.gamma);
  const long long n = G.ncell;
  bool any = false;
  T m = T(0);
  for (long long c = (long long)blockIdx.x * 256 + threadIdx.x; c < n; c += (long long)gridDim.x * 256) {
    const T d = U[c], u = U[n + c] / d, v = U[2 * n + c] / d, w = U[3 * n + c] / d;
    const T eint = U[4 * n + c] / d - T(0.5) * (u * u + v * v + w * w);
    const T cs = sqrtT(jmax(g * (g - T(1)) * eint, T(0)));
    const T s = cs + jmax(absT(u), jmax(absT(v), absT(w)));
    m = any ? jmax(m, s) : s;
    any = true;
  }
  double md = any ? (double)m : -HUGE_VAL;
  for (int o = 32; o > 0; o >>= 1) md = jmax(md, __shfl_xor(md, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = md;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = jmax(jmax(red[0], red[1]), jmax(red[2], red[3]));
}

// boundary_flux_register's gathers (lib/PPMKernels/src/reflux_capture.jl:52-77,86-131) for
// one axis a: the lo and hi boundary planes ([side][field][u2][u1]) and the interior
// hi faces of active cells 1..act-1 ([field][u2][u1][c]), each value Float64(F)·sc.
// b1 < b2 are the other two axes; u1, u2 run over their active cells.
template <typename T>
__global__ void __launch_bounds__(256) flux_register_kernel(const T* __restrict__ frec, MusclDev G, int a, double sc,
                                                            double* __restrict__ planes, double* __restrict__ inner) {
  const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
  const int ng = G.ng;
  const int act[3] = {G.n[0] - 2 * ng, G.n[1] - 2 * ng, G.n[2] - 2 * ng};
  const long long n = G.ncell;
  const long long str[3] = {1, G.n[0], (long long)G.n[0] * G.n[1]};
  const long long m1 = act[b1], m2 = act[b2];
  const long long nplane = 2 * 5 * m1 * m2;
  const long long ninner = inner && act[a] > 1 ? 5 * (long long)(act[a] - 1) * m1 * m2 : 0;
  for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < nplane + ninner; t += (long long)gridDim.x * 256) {
    long long q = t < nplane ? t : t - nplane;
    int p, comp;
    long long u1, u2;
    if (t < nplane) {
      u1 = q % m1;
      q /= m1;
      u2 = q % m2;
      q /= m2;
      comp = (int)(q % 5);
      p = q / 5 ? ng + act[a] : ng;
    } else {
      const long long c = q % (act[a] - 1);
      q /= act[a] - 1;
      u1 = q % m1;
      q /= m1;
      u2 = q % m2;
      comp = (int)(q / m2);
      p = ng + (int)c + 1;
    }
    const long long cell = p * str[a] + (ng + u1) * str[b1] + (ng + u2) * str[b2];
    const double v = (double)frec[((long long)a * G.nf + comp) * n + cell] * sc;
    if (t < nplane) planes[t] = v;
    else inner[t - nplane] = v;
  }
}

constexpr int kWsWgs = 1024;

}  // namespace
}  // namespace vh

using namespace vh;

struct vh_muscl {
  MusclDev G{};
  int dtype = VH_F64, device = 0;
  int mode = VH_EXACT;
  size_t esize = 8;
  double dx = 1.0;
  int variant = 0;   // 0: 16×16 tiles, 1: 32×8
  void* U = nullptr;
  void* U1 = nullptr;
  void* frec = nullptr;
  double* partials = nullptr;
  hipStream_t stream = nullptr;
  bool state_ptr_shared = false;   // vh_muscl_state_device_ptr has handed out U
  // bc! (vh_muscl_set_bc): the refill kind, the caller's hook, and the buffer
  // holding the refilled copy of a step's input
  int bc_kind = VH_MUSCL_BC_NONE;
  vh_muscl_bc_fn bc_fn = nullptr;
  void* bc_user = nullptr;
  void* Ub = nullptr;
  size_t ub_bytes = 0;
};

namespace {

int tile_x(int variant) { return variant == 1 ? 32 : 16; }
int tile_y(int variant) { return variant == 1 ? 8 : 16; }

void set_tiles(vh_muscl* m) {
  const int TX = tile_x(m->variant), TY = tile_y(m->variant);
  m->G.tiles_x = (m->G.n[0] + TX - 1) / TX;
  m->G.tiles_y = (m->G.n[1] + TY - 1) / TY;
  m->G.chunks_z = (m->G.n[2] + m->G.zchunk - 1) / m->G.zchunk;
}

void launch_stage(vh_muscl* m, bool stage2, bool rec, const void* Us, const void* U0, void* Uout) {
  if (!U0) U0 = Us;   // both stages read U0 (stage 1: its base)
  if (m->mode == VH_FAST)
    fast::muscl_launch_stage(m->dtype, m->variant, m->G.nf, stage2, rec, m->G, m->stream, Us, U0, Uout, m->frec);
  else
    exact::muscl_launch_stage(m->dtype, m->variant, m->G.nf, stage2, rec, m->G, m->stream, Us, U0, Uout, m->frec);
}

void launch_fill_periodic(vh_muscl* m, void* state) {
  const unsigned nb = (unsigned)std::min<long long>(4096, (m->G.ncell + 255) / 256);
  if (m->dtype == VH_F64) fill_periodic_kernel<double><<<nb, 256, 0, m->stream>>>((double*)state, m->G);
  else fill_periodic_kernel<float><<<nb, 256, 0, m->stream>>>((float*)state, m->G);
}

// bc! before a stage (lib/PPMKernels/src/muscl_grid.jl:316-322, 339, 350).
int apply_bc(vh_muscl* m, void* state, int stage) {
  if (m->bc_kind == VH_MUSCL_BC_PERIODIC) {
    launch_fill_periodic(m, state);
    VH_HIP(hipGetLastError());
  } else if (m->bc_kind == VH_MUSCL_BC_CALLBACK) {
    const int rc = m->bc_fn(m->bc_user, state, (void*)m->stream, stage);
    if (rc) return fail(-3, "the bc! callback returned %s%lld", "", (long long)rc);
  }
  return 0;
}

// One step: U1 = U + dU(U), then U = ½((U + U1) + dU(U1)) written over U.
// With a periodic bc! the stages read ghost cells from their images. With a callback
// the input is copied to Ub and refilled there (U keeps the unfilled input, the
// reference's D0), stage 1 writes U1 = U + dU(Ub), and U1 is refilled in place
// before stage 2. A failing callback leaves U as it was.
int enqueue_step(vh_muscl* m, double dt, bool rec) {
  const double dtdx = m->dtype == VH_F64 ? dt / m->dx : (double)((float)dt / (float)m->dx);
  m->G.dtdx = dtdx;
  if (m->bc_kind == VH_MUSCL_BC_NONE) {
    launch_stage(m, false, rec, m->U, m->U, m->U1);
    launch_stage(m, true, rec, m->U1, m->U, m->U);
    return 0;
  }
  // fill_periodic! as the stages' reading rule: no copy of the input and no fill passes
  // (264³ f32: 132 + 2·61 µs per step of 1.5 ms). Where an axis has fewer active cells than
  // ghosts the image of a ghost cell is itself one, and the fill runs as such.
  bool images = m->bc_kind == VH_MUSCL_BC_PERIODIC;
  for (int d = 0; d < 3; ++d) images = images && m->G.n[d] - 2 * m->G.ng >= m->G.ng;
  if (images) {
    m->G.wrap = 1;
    launch_stage(m, false, rec, m->U, m->U, m->U1);
    launch_stage(m, true, rec, m->U1, m->U, m->U);
    m->G.wrap = 0;
    return 0;
  }
  const size_t bytes = (size_t)m->G.nf * m->G.ncell * m->esize;
  if (m->ub_bytes < bytes) {
    VH_HIP(hipStreamSynchronize(m->stream));
    if (m->Ub) VH_HIP(hipFree(m->Ub));
    m->Ub = nullptr;
    m->ub_bytes = 0;
    VH_HIP(hipMalloc(&m->Ub, bytes));
    m->ub_bytes = bytes;
  }
  VH_HIP(hipMemcpyAsync(m->Ub, m->U, bytes, hipMemcpyDeviceToDevice, m->stream));
  if (int rc = apply_bc(m, m->Ub, 0)) return rc;
  launch_stage(m, false, rec, m->Ub, m->U, m->U1);
  if (int rc = apply_bc(m, m->U1, 1)) return rc;
  launch_stage(m, true, rec, m->U1, m->U, m->U);
  return 0;
}

}  // namespace

extern "C" {

int vh_muscl_create(vh_muscl** out, const int32_t* dims, int32_t ng, double gamma, double theta, double small_rho,
                    double dx, int32_t dtype) {
  if (!out || !dims) return fail(-1, "null argument%s", "");
  *out = nullptr;
  if (dtype != VH_F64 && dtype != VH_F32) return fail(-1, "dtype must be VH_F64 or VH_F32%s (got %lld)", "", dtype);
  if (ng < 2) return fail(-1, "the MUSCL stencil needs at least 2 ghost zones%s (got %lld)", "", ng);
  for (int d = 0; d < 3; ++d)
    if (dims[d] < 2 * ng + 1 || dims[d] > (1 << 20))
      return fail(-1, "each axis needs 2*ng+1 .. 2^20 cells%s (axis %lld)", "", d);
  if (!(gamma > 1.0) || !(dx > 0.0)) return fail(-1, "gamma must exceed 1 and dx be positive%s", "");
  const long long n = (long long)dims[0] * dims[1] * dims[2];
  if (n > 0x7fffffffLL) return fail(-1, "grid too large%s (%lld cells)", "", n);
  vh_muscl* m = new vh_muscl();
  for (int d = 0; d < 3; ++d) m->G.n[d] = dims[d];
  m->G.ng = ng;
  m->G.xcd_remap = 1;
  m->G.ncell = n;
  m->G.gamma = gamma;
  m->G.theta = theta;
  m->G.small = small_rho;
  m->G.nf = 5;
  m->G.eta1 = 1e-3;
  m->dx = dx;
  m->dtype = dtype;
  m->esize = dtype == VH_F64 ? 8 : 4;
  m->variant = 0;
  if (hipGetDevice(&m->device) != hipSuccess) {
    delete m;
    return fail(-2, "no HIP device%s", "");
  }
  // 16×16 tiles; planes per workgroup from the grid's size (at most 8; Float64 runs three
  // workgroups per compute unit, Float32 four). Step times at the pick against 8
  // planes (µs): 48×42×36 f64 dual, recording 42 (1) for 185; 72³ f64 fast 71 (4) for 98;
  // 108×100×90 f32 113 (6) for 139; 136³ f64 and 264³ keep 8 ± 5%.
  const long long columns = (long long)((dims[0] + 15) / 16) * ((dims[1] + 15) / 16);
  m->G.zchunk = march_planes(columns, dims[2], 8, dtype == VH_F64 ? 3 : 4, cu_count(m->device));
  set_tiles(m);
  const size_t bytes = (size_t)5 * n * m->esize;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess || hipMalloc(&m->U, bytes) != hipSuccess ||
      hipMalloc(&m->U1, bytes) != hipSuccess || hipMalloc(&m->partials, sizeof(double) * kWsWgs) != hipSuccess) {
    vh_muscl_destroy(m);
    return fail(-2, "device allocation of %s%lld bytes failed", "", (long long)(2 * bytes));
  }
  if (hipMemsetAsync(m->U, 0, bytes, m->stream) != hipSuccess || hipStreamSynchronize(m->stream) != hipSuccess) {
    vh_muscl_destroy(m);
    return fail(-2, "device initialisation failed%s", "");
  }
  *out = m;
  return 0;
}

int vh_muscl_destroy(vh_muscl* m) {
  if (!m) return 0;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  (void)hipFree(m->U);
  (void)hipFree(m->U1);
  (void)hipFree(m->frec);
  (void)hipFree(m->partials);
  (void)hipFree(m->Ub);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return 0;
}

int64_t vh_muscl_ncell(const vh_muscl* m) { return m ? m->G.ncell : -1; }

int vh_muscl_upload(vh_muscl* m, const void* U) {
  if (!m || !U) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  VH_HIP(copy_up(m->U, U, (size_t)m->G.nf * m->G.ncell * m->esize, m->stream));
  return 0;
}

int vh_muscl_download(vh_muscl* m, void* U) {
  if (!m || !U) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  VH_HIP(copy_down(U, m->U, (size_t)m->G.nf * m->G.ncell * m->esize, m->stream));
  return 0;
}

int vh_muscl_state_device_ptr(vh_muscl* m, void** ptr) {
  if (!m || !ptr) return fail(-1, "null argument%s", "");
  *ptr = m->U;
  m->state_ptr_shared = true;
  return 0;
}

int vh_muscl_enable_dual_energy(vh_muscl* m, double eta1) {
  if (!m) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  VH_HIP(hipStreamSynchronize(m->stream));
  if (m->G.nf == 6) {
    m->G.eta1 = eta1;
    return 0;
  }
  // Adding the sixth field moves the state to a new allocation: refuse once a
  // caller holds the old address (it would point at freed memory).
  if (m->state_ptr_shared)
    return fail(-1, "vh_muscl_enable_dual_energy after vh_muscl_state_device_ptr: the state would move%s; "
                "enable dual energy before taking the device pointer", "");
  m->G.eta1 = eta1;
  const size_t b5 = (size_t)5 * m->G.ncell * m->esize, b6 = (size_t)6 * m->G.ncell * m->esize;
  void *U = nullptr, *U1 = nullptr;
  if (hipMalloc(&U, b6) != hipSuccess || hipMalloc(&U1, b6) != hipSuccess) {
    (void)hipFree(U);
    return fail(-2, "device allocation of %s%lld bytes failed", "", (long long)(2 * b6));
  }
  VH_HIP(hipMemcpyAsync(U, m->U, b5, hipMemcpyDeviceToDevice, m->stream));
  VH_HIP(hipMemsetAsync((char*)U + b5, 0, b6 - b5, m->stream));
  VH_HIP(hipStreamSynchronize(m->stream));
  (void)hipFree(m->U);
  (void)hipFree(m->U1);
  (void)hipFree(m->frec);
  m->U = U;
  m->U1 = U1;
  m->frec = nullptr;
  m->G.nf = 6;
  return 0;
}

int vh_muscl_set_mode(vh_muscl* m, int32_t mode) {
  if (!m) return fail(-1, "null argument%s", "");
  if (mode != VH_EXACT && mode != VH_FAST) return fail(-1, "mode must be VH_EXACT or VH_FAST%s (got %lld)", "", mode);
  VH_HIP(hipStreamSynchronize(m->stream));
  m->mode = mode;
  return 0;
}

int vh_muscl_set_tiles(vh_muscl* m, int32_t variant, int32_t zchunk) {
  if (!m) return fail(-1, "null argument%s", "");
  if (variant < 0 || variant > 1) return fail(-1, "tile variant must be 0 (16x16) or 1 (32x8)%s", "");
  if (zchunk < 1 || zchunk > 1024) return fail(-1, "zchunk out of range%s (%lld)", "", zchunk);
  VH_HIP(hipStreamSynchronize(m->stream));
  m->variant = variant;
  m->G.zchunk = zchunk;
  set_tiles(m);
  return 0;
}

int vh_muscl_step(vh_muscl* m, double dt, int32_t record) {
  if (!m) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  if (record && !m->frec) VH_HIP(hipMalloc(&m->frec, (size_t)3 * m->G.nf * m->G.ncell * m->esize));
  if (int rc = enqueue_step(m, dt, record != 0)) return rc;
  VH_HIP(hipGetLastError());
  return 0;
}

int vh_muscl_set_bc(vh_muscl* m, int32_t kind, vh_muscl_bc_fn fn, void* user) {
  if (!m) return fail(-1, "null argument%s", "");
  if (kind != VH_MUSCL_BC_NONE && kind != VH_MUSCL_BC_PERIODIC && kind != VH_MUSCL_BC_CALLBACK)
    return fail(-1, "unknown bc kind%s %lld", "", kind);
  if (kind == VH_MUSCL_BC_CALLBACK && !fn) return fail(-1, "VH_MUSCL_BC_CALLBACK needs a function%s", "");
  VH_HIP(hipSetDevice(m->device));
  VH_HIP(hipStreamSynchronize(m->stream));
  m->bc_kind = kind;
  m->bc_fn = kind == VH_MUSCL_BC_CALLBACK ? fn : nullptr;
  m->bc_user = kind == VH_MUSCL_BC_CALLBACK ? user : nullptr;
  return 0;
}

int vh_muscl_fluxrec_download(vh_muscl* m, void* frec) {
  if (!m || !frec) return fail(-1, "null argument%s", "");
  if (!m->frec) return fail(-1, "no step has recorded fluxes yet%s", "");
  VH_HIP(copy_down(frec, m->frec, (size_t)3 * m->G.nf * m->G.ncell * m->esize, m->stream));
  return 0;
}

int vh_muscl_fill_periodic(vh_muscl* m) {
  if (!m) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  launch_fill_periodic(m, m->U);
  VH_HIP(hipGetLastError());
  return 0;
}

int vh_muscl_max_wavespeed(vh_muscl* m, double* out) {
  if (!m || !out) return fail(-1, "null argument%s", "");
  VH_HIP(hipSetDevice(m->device));
  const int nb = (int)std::min<long long>(kWsWgs, (m->G.ncell + 255) / 256);
  if (m->dtype == VH_F64) wavespeed_kernel<double><<<nb, 256, 0, m->stream>>>((const double*)m->U, m->G, m->partials);
  else wavespeed_kernel<float><<<nb, 256, 0, m->stream>>>((const float*)m->U, m->G, m->partials);
  VH_HIP(hipGetLastError());
  std::vector<double> p(nb);
  VH_HIP(copy_down(p.data(), m->partials, sizeof(double) * nb, m->stream));
  double r = p[0];
  for (int i = 1; i < nb; ++i) r = std::isnan(r) ? r : (std::isnan(p[i]) || p[i] > r ? p[i] : r);
  *out = r;
  return 0;
}

int vh_muscl_flux_register(vh_muscl* m, double dt, double* planes, double* interior) {
  if (!m || !planes) return fail(-1, "null argument%s", "");
  if (!m->frec) return fail(-1, "no step has recorded fluxes yet%s", "");
  VH_HIP(hipSetDevice(m->device));
  const int ng = m->G.ng;
  const long long act[3] = {m->G.n[0] - 2LL * ng, m->G.n[1] - 2LL * ng, m->G.n[2] - 2LL * ng};
  long long np = 0, ni = 0;
  for (int a = 0; a < 3; ++a) {
    const long long t = act[(a + 1) % 3] * act[(a + 2) % 3];
    np += 10 * t;
    ni += 5 * (act[a] - 1) * t;
  }
  double* d = nullptr;
  VH_HIP(hipMalloc(&d, sizeof(double) * (np + (interior ? ni : 0))));
  const double sc = dt * (m->dx * m->dx);   // ∫F·area·dt = F·dt·dx²
  long long op = 0, oi = 0;
  hipError_t e = hipSuccess;
  for (int a = 0; a < 3 && e == hipSuccess; ++a) {
    const long long t = act[(a + 1) % 3] * act[(a + 2) % 3];
    const long long work = 10 * t + (interior ? 5 * (act[a] - 1) * t : 0);
    const unsigned nb = (unsigned)std::min<long long>(4096, (work + 255) / 256);
    double* pl = d + op;
    double* in = interior ? d + np + oi : nullptr;
    if (m->dtype == VH_F64)
      flux_register_kernel<double><<<nb, 256, 0, m->stream>>>((const double*)m->frec, m->G, a, sc, pl, in);
    else
      flux_register_kernel<float><<<nb, 256, 0, m->stream>>>((const float*)m->frec, m->G, a, sc, pl, in);
    e = hipGetLastError();
    op += 10 * t;
    oi += 5 * (act[a] - 1) * t;
  }
  if (e == hipSuccess) e = copy_down(planes, d, sizeof(double) * np, m->stream);
  if (e == hipSuccess && interior) e = copy_down(interior, d + np, sizeof(double) * ni, m->stream);
  (void)hipFree(d);
  if (e != hipSuccess) return fail(-2, "HIP error %s in the flux register gather%s", hipGetErrorString(e));
  return 0;
}

int vh_muscl_sync(vh_muscl* m) {
  if (!m) return fail(-1, "null argument%s", "");
  VH_HIP(hipStreamSynchronize(m->stream));
  return 0;
}

int vh_muscl_time_steps(vh_muscl* m, double dt, int64_t nsteps, int32_t record, double* ms_step, double* ms_stage2) {
  if (!m || nsteps <= 0 || nsteps > 100000) return fail(-1, "bad argument%s (nsteps %lld)", "", nsteps);
  VH_HIP(hipSetDevice(m->device));
  if (record && !m->frec) VH_HIP(hipMalloc(&m->frec, (size_t)3 * m->G.nf * m->G.ncell * m->esize));
  if (int rc = enqueue_step(m, dt, record != 0)) return rc;   // untimed warm-up
  hipEvent_t e0, e1, s0, s1;
  VH_HIP(hipEventCreate(&e0));
  VH_HIP(hipEventCreate(&e1));
  VH_HIP(hipEventCreate(&s0));
  VH_HIP(hipEventCreate(&s1));
  VH_HIP(hipEventRecord(e0, m->stream));
  int rc = 0;
  for (int64_t k = 0; k < nsteps && !rc; ++k) rc = enqueue_step(m, dt, record != 0);
  VH_HIP(hipEventRecord(e1, m->stream));
  if (rc) {
    (void)hipStreamSynchronize(m->stream);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipEventDestroy(s0);
    (void)hipEventDestroy(s1);
    return rc;
  }
  VH_HIP(hipStreamSynchronize(m->stream));
  float tot = 0;
  VH_HIP(hipEventElapsedTime(&tot, e0, e1));
  // stage-2 launches timed one by one
  double st2 = 0;
  const int k2 = (int)std::min<int64_t>(nsteps, 20);
  for (int k = 0; k < k2; ++k) {
    launch_stage(m, false, record != 0, m->U, m->U, m->U1);
    VH_HIP(hipEventRecord(s0, m->stream));
    launch_stage(m, true, record != 0, m->U1, m->U, m->U);
    VH_HIP(hipEventRecord(s1, m->stream));
    VH_HIP(hipStreamSynchronize(m->stream));
    float a = 0;
    VH_HIP(hipEventElapsedTime(&a, s0, s1));
    st2 += a;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipEventDestroy(s0);
  (void)hipEventDestroy(s1);
  VH_HIP(hipGetLastError());
  if (ms_step) *ms_step = (double)tot / nsteps;
  if (ms_stage2) *ms_stage2 = st2 / k2;
  return 0;
}

}  // extern "C"
