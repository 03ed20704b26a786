// Launchers of the reverse-mode kernels (adjoint.h), Float64 uniform grids.
// Built once, in the fast arithmetic profile (FMA contraction, refined hardware
// reciprocals): the reverse mode needs no bit parity with the reference.
#include <algorithm>

#include "adjoint.h"
#include "host.h"

namespace vh {

static unsigned grid_for(long long n) { return (unsigned)((n + 255) / 256); }

long long adj_face_slots(const GridDev& G, int axis) {
  long long s = 1;
  for (int d = 0; d < 3; ++d) s *= (d == axis ? G.n[d] + 1 : G.n[d]);
  return s;
}

void adj_launch_prim(hipStream_t s, const double* U, double* W, const GridDev& G) {
  hipLaunchKernelGGL(VH_PROFILE_NS::adj_prim_kernel, dim3(grid_for(G.ncell)), dim3(256), 0, s, U, W, G);
}

static VH_PROFILE_NS::AdjFaces faces_of(double* const gL[3], double* const gR[3], int rank) {
  VH_PROFILE_NS::AdjFaces F{};
  for (int d = 0; d < rank; ++d) {
    F.gL[d] = gL[d];
    F.gR[d] = gR[d];
  }
  return F;
}

template <int RANK>
static void launch_faces(hipStream_t s, const double* W, const double* lam, const GridDev& G,
                         const VH_PROFILE_NS::AdjFaces& F) {
  long long slots = 0;
  for (int d = 0; d < RANK; ++d) slots = std::max(slots, adj_face_slots(G, d));
  hipLaunchKernelGGL(VH_PROFILE_NS::adj_face_kernel<RANK>, dim3(grid_for(slots), RANK), dim3(256), 0, s, W, lam, G, F);
}

void adj_launch_faces(hipStream_t s, const double* W, const double* lam, const GridDev& G, double* const gL[3],
                      double* const gR[3]) {
  const VH_PROFILE_NS::AdjFaces F = faces_of(gL, gR, G.rank);
  if (G.rank == 3) launch_faces<3>(s, W, lam, G, F);
  else if (G.rank == 2) launch_faces<2>(s, W, lam, G, F);
  else launch_faces<1>(s, W, lam, G, F);
}

template <int RANK>
static void launch_cells(hipStream_t s, const double* U, const double* W, const VH_PROFILE_NS::AdjFaces& F,
                         const double* base1, double a1, const double* base2, double a2, double beta,
                         const double* dtp, const GridDev& G, double* out) {
  hipLaunchKernelGGL(VH_PROFILE_NS::adj_cell_kernel<RANK>, dim3((unsigned)((G.ncell + 63) / 64)), dim3(64 * RANK), 0, s,
                     U, W, F, base1, a1, base2, a2, beta, dtp, G, out);
}

void adj_launch_cells(hipStream_t s, const double* U, const double* W, double* const gL[3], double* const gR[3],
                      const double* base1, double a1, const double* base2, double a2, double beta,
                      const double* dtp, const GridDev& G, double* out) {
  const VH_PROFILE_NS::AdjFaces F = faces_of(gL, gR, G.rank);
  if (G.rank == 3) launch_cells<3>(s, U, W, F, base1, a1, base2, a2, beta, dtp, G, out);
  else if (G.rank == 2) launch_cells<2>(s, U, W, F, base1, a1, base2, a2, beta, dtp, G, out);
  else launch_cells<1>(s, U, W, F, base1, a1, base2, a2, beta, dtp, G, out);
}

// The last tile's halo (two cells past the tile) has to wrap around once only:
// every size but 1..9 and 17. The fused form is the faster one at all the others:
// 10² 10.8 µs in passes, 7.7 fused; 50×37 14 and 11; 100² 15 and 10; 512² 47 and 23;
// 1500×1100 319 and 134; 2048² 749 and 352.
bool adj_fused_covers(long long nx, long long ny) {
  auto covers = [](long long n, int tile) { return n > 0 && (n + tile - 1) / tile * tile + 2 < 2 * n; };
  return covers(nx, VH_PROFILE_NS::JTX) && covers(ny, VH_PROFILE_NS::JTY);
}

bool adj_launch_jat_fused(hipStream_t s, const double* U, const double* lam, const double* base1, double a1,
                          const double* base2, double a2, double beta, const double* dtp, const GridDev& G,
                          double* out) {
  using VH_PROFILE_NS::JTX;
  using VH_PROFILE_NS::JTY;
  const bool periodic = G.bc[0] == BC_PERIODIC && G.bc[2] == BC_PERIODIC;
  if (G.rank != 2 || !periodic) return false;
  if (out == U || out == lam) return false;   // other tiles read these cells; the passes read them before out is written
  if (!adj_fused_covers(G.n[0], G.n[1])) return false;
  const dim3 grid((G.n[0] + JTX - 1) / JTX, (G.n[1] + JTY - 1) / JTY);
  hipLaunchKernelGGL(VH_PROFILE_NS::adj_jat2d_periodic_kernel, grid, dim3(VH_PROFILE_NS::JNT), 0, s, U, lam, base1, a1,
                     base2, a2, beta, dtp, G, out);
  return true;
}

}  // namespace vh
