// Step loop of a 1D grid that fits one workgroup (gfx950): the whole run of SSP-RK2
// steps with its CFL reductions in one launch, the state in registers and LDS.
//
// A 1D run is a serial chain: at 400 cells a step of three launches takes 16 µs, of
// which the arithmetic is under 2. Here a lane owns item f: cell f and the face
// between cells f − 1 and f (n + 1 items; kLineLanes lanes take more than one each on
// the larger grids). Per stage:
//   1  publish the cell's primitive state to LDS (and the ghosts or wrapped copies next to
//      the ends); barrier;
//   2  reconstruct both sides of the item's face from four states, evaluate its flux and
//      publish it; barrier;
//   3  update the cell from its two faces.
// The slope of cell f − 1 is formed twice (by items f − 1 and f): 30 operations against a
// third exchange and barrier. The CFL maximum of the new state goes through one LDS
// slot per wave that every lane reads after the next barrier 1, so the reduction needs no
// barrier of its own, and every lane forms the same dt.
//
// Bound: latency (barriers, divisions and square roots in sequence) with one wave per SIMD,
// VALU issue with four. Measured per step, exact Float64 / fast Float32, against three launches
// per step over many workgroups (16.6 / 14.9 µs at any of these sizes): 64 cells 3.5 / 2.2 µs,
// 400 cells 5.0 / 2.7, 1023 cells 8.4 / 4.0, 2040 cells 16.1 / 6.5. The limit is the LDS of a
// Float64 grid, about where the Float64 times meet; Float32 grids have the same limit, though their
// LDS would hold twice the cells.
#pragma once

#include "stencil.h"

namespace vh {
namespace VH_PROFILE_NS {

template <typename T>
struct LineLDS {
  T w[5][kLineMax + 4];      // cell i at i + 2
  T f[5][kLineMax + 1];      // flux of the face below cell i at i
  double red[kLineLanes / 64];
};

// At most max_steps steps from U in place and time t, to tstop and no further than tfinal
// (0: no final time). host: the clock (host.h) at the end. PL: items per lane.
template <typename T, bool FLOOR64, int PL>
__global__ void __launch_bounds__(kLineLanes, 1) rk_line_kernel(T* __restrict__ U, GridDev G, double t, double cflnum,
                                                                double tfinal, double tstop, long long max_steps,
                                                                double* host) {
  __shared__ LineLDS<T> S;
  const T g = T(G.gamma), igm1 = T(G.igm1), a0 = T(G.area[0]);
  const int n = G.n[0], nt = blockDim.x, tid = threadIdx.x;
  const long long nn = n;
  const int blo = G.bc[0], bhi = G.bc[1];
  const bool per = blo == BC_PERIODIC;
  const bool clip = tfinal > 0.0;
  double dt = 0.0, m = 0.0;
  long long k = 0;
  T* wf = &S.w[0][0];
  T* ff = &S.f[0][0];
  constexpr int WP = kLineMax + 4, FP = kLineMax + 1;

  Cons<T> u[PL], u0[PL];
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int c = tid + j * nt;
    if (c < n) u[j] = load_cons(U, nn, c);
  }
  // Primitive state of every cell to LDS, with the states beyond the ends.
  auto publish = [&](bool with_cfl) {
    CflMax<T, 1> cfl;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int c = tid + j * nt;
      if (c < n) {
        const Prim<T> w = cons2prim<T, FLOOR64>(u[j], g, G.gamma);
        lds_put5(wf, WP, c + 2, w);
        if (per) {
          if (c < 2) lds_put5(wf, WP, c + n + 2, w);
          if (c >= n - 2) lds_put5(wf, WP, c - n + 2, w);
        } else {
          if (c == 0) lds_put5(wf, WP, 1, ghost(w, blo, 1));
          if (c == n - 1) lds_put5(wf, WP, n + 2, ghost(w, bhi, 1));
        }
        if (with_cfl) cfl.add(w, g);
      }
    }
    if (with_cfl) {
      double v = cfl.a0;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v = vmax(v, __shfl_xor(v, o, 64));
      if ((tid & 63) == 0) S.red[tid >> 6] = v;
    }
    __syncthreads();
  };
  auto fluxes = [&]() {
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int f = tid + j * nt;
      if (f <= n) {
        // states of cells f − 2 .. f + 1; an end face of a walled grid uses one side only
        const Prim<T> w1 = lds_get5(wf, WP, f + 1), w2 = lds_get5(wf, WP, f + 2);
        Prim<T> L, R;
        if (per || f > 0) L = face_value(w1, slope(lds_get5(wf, WP, f), w1, w2), T(0.5));
        if (per || f < n) R = face_value(w2, slope(w1, w2, lds_get5(wf, WP, f + 3)), T(-0.5));
        lds_putf(ff, FP, f, axis_face<false>(f, n, blo, bhi, L, R, g, igm1, 1));
      }
    }
    __syncthreads();
  };
  // Flux sum of cell c in the face walk's order (see stencil.h).
  auto gather = [&](int c) {
    const Cons<T> lo = lds_getf(ff, FP, c), hi = lds_getf(ff, FP, c + 1);
    Cons<T> acc;
    acc.d = acc.mx = acc.my = acc.mz = acc.e = T(0);
    if (c > 0) acc_add(acc, lo, -a0);
    acc_add(acc, hi, a0);
    if (c == 0) acc_add(acc, lo, -a0);
    return acc;
  };

  publish(true);
  for (;;) {
    double mm = S.red[0];
    for (int i = 1; i < nt / 64; ++i) mm = vmax(mm, S.red[i]);
    m = mm / G.w[0];
    dt = m == 0.0 ? HUGE_VAL : cflnum / m;
    if (clip) dt = vmin(dt, tfinal - t);
    if (k >= max_steps || (clip && !(t < tstop))) break;
    const T invV = T(dt) / (T(1.0) * T(G.V));
    fluxes();
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int c = tid + j * nt;
      u0[j] = u[j];
      if (c < n) {
        const Cons<T> acc = gather(c);
        u[j].d = u[j].d - invV * acc.d;
        u[j].mx = u[j].mx - invV * acc.mx;
        u[j].my = u[j].my - invV * acc.my;
        u[j].mz = u[j].mz - invV * acc.mz;
        u[j].e = u[j].e - invV * acc.e;
      }
    }
    publish(false);
    fluxes();
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int c = tid + j * nt;
      if (c < n) {
        const Cons<T> acc = gather(c);
        const T h = T(0.5);
        u[j].d = h * u0[j].d + h * (u[j].d - invV * acc.d);
        u[j].mx = h * u0[j].mx + h * (u[j].mx - invV * acc.mx);
        u[j].my = h * u0[j].my + h * (u[j].my - invV * acc.my);
        u[j].mz = h * u0[j].mz + h * (u[j].mz - invV * acc.mz);
        u[j].e = h * u0[j].e + h * (u[j].e - invV * acc.e);
      }
    }
    t += dt;
    ++k;
    publish(true);
  }
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int c = tid + j * nt;
    if (c < n) store_cons(U, nn, c, u[j]);
  }
  if (tid == 0) {
    host[0] = t;
    host[1] = dt;
    host[2] = m;
    host[3] = (double)k;
    host[7] = clip && !(t < tstop) ? 1.0 : 0.0;
  }
}

}  // namespace VH_PROFILE_NS
}  // namespace vh
