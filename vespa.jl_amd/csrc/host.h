// Host-side error plumbing shared by the translation units of the library.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "common.h"

namespace vh {

// Records a formatted message for vh_last_error() and returns code.
int fail(int code, const char* fmt, const char* a = "", long long b = 0);

}  // namespace vh

#define VH_HIP(call)                                                                     \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess) return ::vh::fail(-2, "HIP error %s (code %lld) at " #call,    \
                                            hipGetErrorString(e_), (long long)e_);       \
  } while (0)

namespace vh {

// Estimated time (in units of a few µs) of a z-marching stage launch: `wgs` workgroups
// of `planes` planes each. A plane of a workgroup costs 2 + r when r workgroups
// share a compute unit (measured at 32³-200³: 5.5, 7.4 and 9.3 µs for r = 1, 2, 3 in
// the exact Float64 form; the fixed part is the latency of its loads and barriers),
// and the prologue 0.7 planes. per_cu: resident workgroups of the kernel per unit.
inline double march_cost(long long wgs, int planes, int per_cu, int cus) {
  const long long slots = (long long)per_cu * cus;
  const long long rem = wgs % slots;
  const long long r = (rem + cus - 1) / cus;
  return (planes + 0.7) * ((double)(wgs / slots) * (2 + per_cu) + (rem ? 2 + r : 0));
}

// Planes per workgroup for `columns` tiles of an nz-plane grid: `most` (the fastest on
// grids that fill the chip) unless a shorter march is estimated 5% faster, because
// the grid would leave compute units idle. Stage 1 / stage 2 measured at the pick
// against `most` = 16 (µs): 60×52×44 f64 exact 21/23 (1 plane) for 97/102; 96³ f64 exact 60/64
// (5) for 96/102; 171×130×97 f32 exact 97/107 (10) for 117/129; 128³ and 256³ keep 16 ± 5%.
inline int march_planes(long long columns, int nz, int most, int per_cu, int cus, double* cost = nullptr) {
  int best = most < nz ? most : nz;
  double c = march_cost(columns * ((nz + best - 1) / best), best, per_cu, cus);
  const double limit = 0.95 * c;
  for (int z = best - 1; z >= 1; --z) {
    const double cz = march_cost(columns * ((nz + z - 1) / z), z, per_cu, cus);
    if (cz < limit && cz < c) {
      c = cz;
      best = z;
    }
  }
  if (cost) *cost = c;
  return best;
}

// Compute units of `device` (256 on MI355X; also if the query fails).
inline int cu_count(int device) {
  int n = 0;
  return hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && n > 0 ? n : 256;
}

// Copy between the device (the current one) and a host array, ordered after the work on s and
// complete on return (transfer.hip).
hipError_t copy_up(void* dev, const void* host, size_t bytes, hipStream_t s);
hipError_t copy_down(void* host, const void* dev, size_t bytes, hipStream_t s);
// copy_up that may still be under way on return: host stays as it is until s is waited for.
hipError_t enqueue_up(void* dev, const void* host, size_t bytes, hipStream_t s);

// Clock kernels of the uniform-grid context, shared with the block context.
// clock (kClockDoubles): [0] t, [1] dt, [2] max CFL term, [3] steps; of a step loop also
// [4] cfl, [5] tfinal (0: none; infinite is a final time as any other), [6] the time at which
// the loop ends, [7] non-zero once it has ended. `host` is pinned memory that receives a copy (null: none).
constexpr int kClockDoubles = 8;
void enqueue_dt_finalize(hipStream_t s, const double* partials, int np, double cfl, double* clock, double* host);
void enqueue_set_dt(hipStream_t s, double* clock, double dt);
// A step loop: begin sets the clock from the CFL partials of the current state; a
// tail after each step's stage 2 advances the clock and sets the next dt from the
// partials of the new state (and stores it to *dt_log unless null).
void enqueue_loop_begin(hipStream_t s, const double* partials, int np, double t, double cfl, double tfinal, bool clip,
                        double* clock, double* host, double* dt_log = nullptr);
void enqueue_step_tail(hipStream_t s, const double* partials, int np, double* clock, double* host,
                       double* dt_log = nullptr);
// Steps of dt until time_left has passed: 1 to most (1 also for a NaN).
long long steps_within(double time_left, double dt, long long most);

// The host side of a step loop on s: queue(n) queues n steps with their tails, clk is the clock's
// pinned copy. Without a final time (clip false) all steps are queued at once. With one, the host
// looks at the clock before it queues more than the remaining time holds at the current dt, at
// most 64 steps; steps queued beyond the end do nothing, but their launches take time
// (eight queued for a leg of one step made it 100 µs where a look per step took 64, at
// 64²). So one step is queued first, which is always taken, and the host waits for
// begin's reduction while it runs (`look` is recorded behind begin), and reads the largest CFL
// term alone: the rest of the clock may be on its way from that step's tail. one_by_one:
// queue() needs the step before it to have ended.
template <typename Queue>
int run_step_loop(hipStream_t s, hipEvent_t look, const volatile double* clk, double t, double cfl, double tfinal,
                  bool clip, long long limit, bool one_by_one, Queue queue) {
  if (clip && !one_by_one && limit > 1) VH_HIP(hipEventRecord(look, s));
  for (long long queued = 0; queued < limit && clk[7] == 0.0;) {
    const bool first = queued == 0;
    long long n = limit - queued;
    if (one_by_one || (clip && first)) n = 1;
    else if (clip) n = steps_within(clk[5] - clk[0], clk[1], n < 64 ? n : 64);
    if (int rc = queue(n)) return rc;
    queued += n;
    if (clip && first && !one_by_one && queued < limit) {
      VH_HIP(hipEventSynchronize(look));
      const double m = clk[2];
      n = steps_within(tfinal - t, m == 0.0 ? HUGE_VAL : cfl / m, limit < 8 ? limit : 8) - 1;
      if (int rc = n > 0 ? queue(n) : 0) return rc;
      queued += n;
    }
    if (clip || queued >= limit) VH_HIP(hipStreamSynchronize(s));
  }
  return 0;
}

}  // namespace vh

namespace vh {

// Reverse-mode launchers (adjoint.hip), Float64 uniform grids. Face buffers
// gL/gR per axis hold 5 SoA fields over adj_face_slots(G, axis) face slots.
long long adj_face_slots(const GridDev& G, int axis);
void adj_launch_prim(hipStream_t s, const double* U, double* W, const GridDev& G);
void adj_launch_faces(hipStream_t s, const double* W, const double* lam, const GridDev& G, double* const gL[3],
                      double* const gR[3]);
void adj_launch_cells(hipStream_t s, const double* U, const double* W, double* const gL[3], double* const gR[3],
                      const double* base1, double a1, const double* base2, double a2, double beta,
                      const double* dtp, const GridDev& G, double* out);
// Fused single-kernel form for 2D grids periodic on both axes with 10 to 16 or
// more than 17 cells along each; returns false (nothing launched) otherwise.
bool adj_fused_covers(long long nx, long long ny);
bool adj_launch_jat_fused(hipStream_t s, const double* U, const double* lam, const double* base1, double a1,
                          const double* base2, double a2, double beta, const double* dtp, const GridDev& G,
                          double* out);

}  // namespace vh

namespace vh {

// Self-gravity on uniform grids (gravity.hip). φ and the CG vectors are stored
// at the state's precision; dot products and the matrix-vector sums in Float64.
struct GravParams {
  double G = 1.0;
  int gper = 0;            // bit d: φ periodic along axis d
  int project_mean = 1;
  long long maxiter = 500;
  double tol = 1e-8;
};
struct GravBuffers {
  void* phi = nullptr;     // ncell values
  void* work = nullptr;    // r and two p; block meshes also Ap (kGravWork, kGravWorkCsr values per cell)
  const void* rho = nullptr;
  void* state = nullptr;   // CG state block (device)
  double* sumv = nullptr;  // Σ V (device), summed cell by cell on the host as the reference does
  double* partials = nullptr;  // kGravPartials per-workgroup partial sums (device)
  void* host_state = nullptr;  // pinned; the kernels write done, iters, relres here
};
constexpr int kGravStateBytes = 64;
constexpr int kGravPartials = 4096;
constexpr int kGravWork = 3, kGravWorkCsr = 4;
void grav_apply(hipStream_t s, int dtype, const GridDev& G, int gper, const void* x, void* out);
void grav_accel(hipStream_t s, int dtype, const GridDev& G, int gper, const void* phi, void* g);
int grav_solve(hipStream_t s, int dtype, const GridDev& G, const GravParams& P, GravBuffers& B, long long* iters,
               double* relres);

// The composite operator of a block mesh in CSR form (the reference's
// PoissonKAStruct, src/gravity.jl:455-600), built on the host per mesh: row c
// lists its face neighbours in the face walk's order with coef = area/d, and
// the gravity stencil gives per cell and axis the lo/hi neighbour (the cell
// itself at a Neumann side) and d_lo + d_hi. Device pointers.
struct GravCsr {
  long long n = 0;
  const int* rowptr = nullptr;      // n + 1
  const int* colidx = nullptr;
  const double* coef = nullptr;
  const double* vol = nullptr;      // per-cell volume
  const int* glo = nullptr;         // 3·n, [axis][cell]
  const int* ghi = nullptr;
  const double* gsum = nullptr;     // 3·n, [axis][cell]
  int rank = 1;
};
void grav_csr_apply(hipStream_t s, int dtype, const GravCsr& A, const void* x, void* out);
void grav_csr_accel(hipStream_t s, int dtype, const GravCsr& A, const void* phi, void* g);
int grav_csr_solve(hipStream_t s, int dtype, const GravCsr& A, const GravParams& P, GravBuffers& B, long long* iters,
                   double* relres);

}  // namespace vh

namespace vh {

// Block-mesh regrid (regrid.hip). RemapDev: per destination block, the source
// block that contains it, the level difference and the position of its first
// cell in the source block's cells.
struct RemapDev {
  int src, shift;
  int o[3];
};
void regrid_indicator(hipStream_t s, int dtype, int nblocks, const BlockDev* blocks, const int* repmap, int rank,
                      const void* rho, double* cell_g, double* block_max);
void regrid_remap(hipStream_t s, int dtype, int ndst, const BlockDev* dst_blocks, const BlockDev* src_blocks,
                  const RemapDev* map, const void* Us, long long ns, void* Ud, long long nd, int nf);

}  // namespace vh
