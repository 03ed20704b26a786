// Self-gravity on a uniform grid (gfx950): the Poisson solve ∇²φ = 4πGρ by
// conjugate gradients on A = −∇²·V, and g = −∇φ.
//
// The reference solves on the composite leaf mesh with a CSR adjacency built on
// the host (src/gravity.jl:248-336, ext/VespaKAGravityExt.jl:21-63). On a uniform
// grid that adjacency is the 2·rank-point stencil, so the matrix-vector product
// here is a stencil gather (one lane per cell, no index arrays), summed in
// Float64 in the row order the CSR build produces — lo neighbours that precede
// the cell (z, y, x), the cell's hi neighbours (x, y, z), then lo neighbours
// wrapped by a periodic φ boundary (x, y, z) — so each product matches the
// reference's bit for bit. Non-periodic φ faces contribute nothing (homogeneous
// Neumann, src/gravity.jl:124-128).
//
// One CG iteration is two launches on a uniform grid. The direction kernel reads
// r and the previous p, writes the new p (into the other of two buffers, since its
// neighbours still read the old one) and forms p·Ap from values of the new p recomputed
// at the stencil's points; the update kernel applies the stencil to p once more
// instead of storing Ap, and updates φ, r and r·r. That moves 64 bytes per Float64 cell and
// iteration (88 with separate matrix-vector, update and direction passes). On a
// block mesh, whose rows cost 12 bytes per entry, the direction kernel stores Ap.
// Scalars need no launch of their own: every workgroup sums the at most 1024 partials
// of the launch before it, in the same order, so all take the same α, β and stopping
// decision, and workgroup 0 records them. Once the solve is done later launches return
// at once; the host queues kCgChunk iterations ahead of the chunk whose end it waits for.
// Dot products are Float64 (src/gravity.jl:338-343).
//
// Bound: memory traffic (the vectors of 128³ Float64, 17 MB each, stay in the 256 MB cache)
// and, below about 64³, the latency of two dependent launches, each a chain of partial
// sums, row loads and a reduction (4-5 µs). Measured per iteration, Float64 periodic, against
// five launches (matrix-vector product with 64-bit index divisions, α, update, β, direction):
// 24³ 20.3 → 12.0 µs, 64³ 20.5 → 13.0, 128³ 59.4 → 32.8, 256³ 387 → 293 (3.7 TB/s).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gravity.h"
#include "host.h"

namespace vh {

constexpr int GNT = 256;
// Workgroups (= partials) of the CG kernels, four per compute unit: 2048 ran 128³ in 37.6 µs
// per iteration (each workgroup sums twice the partials), 512 in 35.3.
constexpr int kCgWgs = 1024;
static_assert(4 * kCgWgs <= kGravPartials, "four partial arrays");
constexpr int kCgChunk = 8;
constexpr double kFourPi = 4.0 * 3.141592653589793;

__device__ __forceinline__ double gsum_block(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double r = red[0];
#pragma unroll
  for (int i = 1; i < GNT / 64; ++i) r += red[i];
  return r;
}

__device__ __forceinline__ void gcoords(const GridDev& G, long long c, int* co) {
  co[0] = (int)(c % G.n[0]);
  const long long q = c / G.n[0];
  co[1] = (int)(q % G.n[1]);
  co[2] = (int)(q / G.n[1]);
}

// State of a solve. rs[k & 1] is r·r before iteration k: iteration k + 1 records its
// own while other workgroups still read the one before.
struct CgState {
  double rs[2], relres, bnorm;
  double iters;      // iterations taken (as double)
  int done;          // 1: converged, stalled or out of iterations
  int pad;
};
static_assert(sizeof(CgState) <= kGravStateBytes, "CG state block");

// Sum of np partials by one workgroup, the same order in every workgroup.
__device__ __forceinline__ double psum(const double* __restrict__ partials, int np, double* red) {
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += GNT) s += partials[i];
  return gsum_block(s, red);
}

// V consecutive values, loaded and stored at once (V·sizeof(T)-byte aligned).
template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
  T v[V];
};
template <int V, typename T>
__device__ __forceinline__ Pack<T, V> ldp(const T* p, long long i) {
  return *reinterpret_cast<const Pack<T, V>*>(p + i);
}
template <int V, typename T>
__device__ __forceinline__ void stp(T* p, long long i, const Pack<T, V>& x) {
  *reinterpret_cast<Pack<T, V>*>(p + i) = x;
}

// f(c) for the workgroup's share of n cells, c the first of a lane's V consecutive cells
// (n a multiple of V). 256 lanes take consecutive cells; the workgroups of one XCD (round
// robin by index) walk one contiguous eighth of the cells side by side, so that a
// plane's neighbours are in their L2.
template <int V, typename F>
__device__ __forceinline__ void for_cells(long long n, F f) {
  const long long nch = (n / V + GNT - 1) / GNT;
  const int parts = gridDim.x % 8 == 0 ? 8 : 1;
  const int part = blockIdx.x % parts;
  const long long end = nch * (part + 1) / parts;
  for (long long ch = nch * part / parts + blockIdx.x / parts; ch < end; ch += gridDim.x / parts) {
    const long long c = (ch * GNT + threadIdx.x) * V;
    if (c < n) f(c);
  }
}

// x / d for x < 2^31 as a multiplication (Granlund and Montgomery, Division by invariant integers
// using multiplication, 1994): m = ceil(2^(31+l)/d) with 2^l >= d exceeds
// 2^(31+l)/d by less than 2^l/d, so the product is off by less than 1/d.
struct FastDiv {
  unsigned m;
  int shift;   // l − 1, or −1 for d = 1
};
static FastDiv fast_div_by(int d) {
  int l = 0;
  while ((1LL << l) < d) ++l;
  return {(unsigned)(((1ULL << (31 + l)) + d - 1) / (unsigned)d), l - 1};
}
__device__ __forceinline__ unsigned fdiv(unsigned x, FastDiv f) {
  return f.shift < 0 ? x : __umulhi(x, f.m) >> f.shift;
}

// Rows c .. c + V − 1 of the uniform operator on the values x(i) (packs x.pack(i)): per
// cell Σ coef·(x_c − x_nb) in Float64 in the CSR build's order (see the top of the file).
// V > 1 needs rows of a multiple of V cells: the lane's cells lie in one row, and
// one load per side serves all of them along y and z.
template <int RANK, int VN>
struct UniformRow {
  static constexpr bool kStoreAp = false;
  static constexpr int V = VN;
  int n[3];
  int gper;
  int wide;        // 1: 2^31 cells or more (64-bit divisions)
  FastDiv dx, dy;
  double coef[3];
  template <typename T, typename X>
  __device__ __forceinline__ void operator()(long long c, Pack<T, V>& own, Pack<T, V>& out, X x) const {
    int co[3];
    if (wide) {
      const long long q = c / n[0];
      co[0] = (int)(c - q * n[0]);
      co[2] = (int)(q / n[1]);
      co[1] = (int)(q - (long long)co[2] * n[1]);
    } else {
      const unsigned q = fdiv((unsigned)c, dx), z = RANK > 1 ? fdiv(q, dy) : 0;
      co[0] = (int)((unsigned)c - q * (unsigned)n[0]);
      co[1] = (int)(q - z * (unsigned)n[1]);
      co[2] = (int)z;
    }
    own = x.pack(c);
    // a side without a neighbour reads the cell itself and adds 0
    Pack<T, V> lo[RANK], hi[RANK];
    bool has_lo[RANK], has_hi[RANK];
    {
      const bool per = gper & 1;
      const int last = co[0] + V - 1;
      const long long cl = co[0] > 0 ? c - 1 : (per ? c + (n[0] - 1) : c);
      const long long ch = last + 1 < n[0] ? c + V : (per ? c + (V - n[0]) : c);
      has_lo[0] = co[0] > 0 || per;
      has_hi[0] = last + 1 < n[0] || per;
      lo[0].v[0] = x.one(cl);
      hi[0].v[V - 1] = x.one(ch);
#pragma unroll
      for (int j = 1; j < V; ++j) {
        lo[0].v[j] = own.v[j - 1];
        hi[0].v[j - 1] = own.v[j];
      }
    }
    long long st = n[0];
#pragma unroll
    for (int d = 1; d < RANK; ++d) {
      const bool per = gper >> d & 1;
      const long long wrap = (long long)(n[d] - 1) * st;
      const long long cl = co[d] > 0 ? c - st : (per ? c + wrap : c);
      const long long ch = co[d] + 1 < n[d] ? c + st : (per ? c - wrap : c);
      has_lo[d] = co[d] > 0 || per;
      has_hi[d] = co[d] + 1 < n[d] || per;
      lo[d] = x.pack(cl);
      hi[d] = x.pack(ch);
      st *= n[d];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const double xc = (double)own.v[j];
      double l[RANK];
      double s = 0.0;
#pragma unroll
      for (int d = RANK - 1; d >= 0; --d) {
        const bool has = has_lo[d] || (d == 0 && j > 0);
        l[d] = has ? coef[d] * (xc - (double)lo[d].v[j]) : 0.0;
        s += co[d] > 0 || (d == 0 && j > 0) ? l[d] : 0.0;
      }
#pragma unroll
      for (int d = 0; d < RANK; ++d) {
        const bool has = has_hi[d] || (d == 0 && j < V - 1);
        s += has ? coef[d] * (xc - (double)hi[d].v[j]) : 0.0;
      }
#pragma unroll
      for (int d = 0; d < RANK; ++d) s += co[d] > 0 || (d == 0 && j > 0) ? 0.0 : l[d];
      out.v[j] = (T)s;
    }
  }
};

// Row c of the CSR operator (_lap_csr_cpu!, src/gravity.jl:326-336).
struct CsrRow {
  static constexpr bool kStoreAp = true;
  static constexpr int V = 1;
  const int* rowptr;
  const int* colidx;
  const double* coef;
  template <typename T, typename X>
  __device__ __forceinline__ void operator()(long long c, Pack<T, 1>& own, Pack<T, 1>& out, X x) const {
    own = x.pack(c);
    const double xc = (double)own.v[0];
    double s = 0.0;
    for (int k = rowptr[c]; k < rowptr[c + 1]; ++k) s += coef[k] * (xc - (double)x.one(colidx[k]));
    out.v[0] = (T)s;
  }
};

// The values an operator is applied to: an array, or r + βp.
template <typename T, int V>
struct ArrayX {
  const T* x;
  __device__ __forceinline__ T one(long long i) const { return x[i]; }
  __device__ __forceinline__ Pack<T, V> pack(long long i) const { return ldp<V>(x, i); }
};
template <typename T, int V>
struct DirX {
  const T* r;
  const T* p;
  T b;
  __device__ __forceinline__ T one(long long i) const { return r[i] + b * p[i]; }
  __device__ __forceinline__ Pack<T, V> pack(long long i) const {
    const Pack<T, V> a = ldp<V>(r, i), q = ldp<V>(p, i);
    Pack<T, V> o;
#pragma unroll
    for (int j = 0; j < V; ++j) o.v[j] = a.v[j] + b * q.v[j];
    return o;
  }
};

// out = A·x, stored at T.
template <typename T, typename Row>
__global__ void __launch_bounds__(GNT) lap_kernel(const T* __restrict__ x, T* __restrict__ out, long long n, Row row) {
  constexpr int V = Row::V;
  for_cells<V>(n, [&](long long c) {
    Pack<T, V> own, a;
    row(c, own, a, ArrayX<T, V>{x});
    stp<V>(out, c, a);
  });
}

// Partials of Σ V·a (vols null: the constant volume vol).
template <typename T>
__global__ void __launch_bounds__(GNT) vsum_kernel(const T* __restrict__ a, const double* __restrict__ vols, double vol,
                                                   long long n, double* __restrict__ partials) {
  __shared__ double red[GNT / 64];
  double s = 0.0;
  for_cells<1>(n, [&](long long i) { s += (vols ? vols[i] : vol) * (double)a[i]; });
  s = gsum_block(s, red);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// r = b − A·φ with b = T(−4πG(ρ − ρ̄)·V), ρ̄ = Σ ρV / Σ V from the partials psv (null: 0);
// partials of r·r and b·b (src/gravity.jl:230-246, 280-289).
template <typename T, typename Row>
__global__ void __launch_bounds__(GNT) cg_init_kernel(const T* __restrict__ rho, const T* __restrict__ phi,
                                                      T* __restrict__ r, long long n, Row row, double G, double vol,
                                                      const double* __restrict__ vols, const double* psv,
                                                      const double* __restrict__ sumv, double* rr, double* bb) {
  __shared__ double red[GNT / 64];
  const double rb = psv ? psum(psv, gridDim.x, red) / *sumv : 0.0;
  double srr = 0.0, sbb = 0.0;
  constexpr int V = Row::V;
  for_cells<V>(n, [&](long long c) {
    const Pack<T, V> rh = ldp<V>(rho, c);
    Pack<T, V> own, Ap, res;
    row(c, own, Ap, ArrayX<T, V>{phi});
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const T b = (T)(-kFourPi * G * ((double)rh.v[j] - rb) * (vols ? vols[c + j] : vol) * 1.0);
      const T v = b - Ap.v[j];
      res.v[j] = v;
      srr += (double)v * (double)v;
      sbb += (double)b * (double)b;
    }
    stp<V>(r, c, res);
  });
  srr = gsum_block(srr, red);
  sbb = gsum_block(sbb, red);
  __syncthreads();
  if (threadIdx.x == 0) {
    rr[blockIdx.x] = srr;
    bb[blockIdx.x] = sbb;
  }
}

// Start of iteration k (1-based): relres = √(r·r)/‖b‖, stop at the tolerance (not before
// the first iteration) or after maxiter; else p ← r + βp with β = r·r over the last
// one (k = 1: p ← r) and the partials of p·Ap. Also run after the last iteration for
// its stopping test.
template <typename T, typename Row>
__global__ void __launch_bounds__(GNT) cg_dir_kernel(const T* __restrict__ r, const T* __restrict__ p0,
                                                     T* __restrict__ p1, T* __restrict__ Ap, long long n, Row row,
                                                     long long k, double tol, long long maxiter,
                                                     const double* __restrict__ rr, const double* __restrict__ bb,
                                                     double* __restrict__ pap, CgState* st, CgState* host) {
  __shared__ double red[GNT / 64];
  const int ended = st->done;   // the loads of the state and the partials overlap
  const double rs0 = st->rs[(k - 1) & 1];
  double bnorm = st->bnorm;
  const double rs = psum(rr, gridDim.x, red);
  if (ended) return;
  if (k == 1) {
    bnorm = sqrt(psum(bb, gridDim.x, red));
    if (bnorm == 0.0) bnorm = 1.0;
  }
  const double relres = sqrt(rs) / bnorm;
  const bool done = (k > 1 && relres <= tol) || k > maxiter;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->rs[k & 1] = rs;
    st->bnorm = bnorm;
    st->relres = relres;
    st->iters = (double)(k - 1);
    host->relres = relres;
    host->iters = (double)(k - 1);
    if (done) {
      st->done = 1;
      host->done = 1;
    }
  }
  if (done) return;
  const T b = k == 1 ? T(0) : (T)(rs / rs0);
  double dot = 0.0;
  constexpr int V = Row::V;
  auto cells = [&](auto x) {
    for_cells<V>(n, [&](long long c) {
      Pack<T, V> pc, a;
      row(c, pc, a, x);
      stp<V>(p1, c, pc);
      if constexpr (Row::kStoreAp) stp<V>(Ap, c, a);
#pragma unroll
      for (int j = 0; j < V; ++j) dot += (double)pc.v[j] * (double)a.v[j];
    });
  };
  if (k == 1) cells(ArrayX<T, V>{r});
  else cells(DirX<T, V>{r, p0, b});
  dot = gsum_block(dot, red);
  if (threadIdx.x == 0) pap[blockIdx.x] = dot;
}

// End of iteration k: α = r·r / p·Ap (stop when p·Ap <= 0), φ += αp, r −= αAp (at T),
// partials of r·r.
template <typename T, typename Row>
__global__ void __launch_bounds__(GNT) cg_update_kernel(T* __restrict__ phi, T* __restrict__ r, const T* __restrict__ p,
                                                        const T* __restrict__ Ap, long long n, Row row, long long k,
                                                        const double* __restrict__ pap, double* __restrict__ rr,
                                                        CgState* st, CgState* host) {
  __shared__ double red[GNT / 64];
  const int ended = st->done;
  const double rs = st->rs[k & 1];
  const double pAp = psum(pap, gridDim.x, red);
  if (ended) return;
  if (pAp <= 0.0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->done = 1;
      host->iters = (double)k;
      host->done = 1;
    }
    return;
  }
  const T a = (T)(rs / pAp);
  double s = 0.0;
  constexpr int V = Row::V;
  for_cells<V>(n, [&](long long c) {
    Pack<T, V> ph = ldp<V>(phi, c), ri = ldp<V>(r, c);
    Pack<T, V> pc, ap;
    if constexpr (Row::kStoreAp) {
      pc = ldp<V>(p, c);
      ap = ldp<V>(Ap, c);
    } else {
      row(c, pc, ap, ArrayX<T, V>{p});
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      ph.v[j] += a * pc.v[j];
      ri.v[j] -= a * ap.v[j];
      s += (double)ri.v[j] * (double)ri.v[j];
    }
    stp<V>(phi, c, ph);
    stp<V>(r, c, ri);
  });
  s = gsum_block(s, red);
  if (threadIdx.x == 0) rr[blockIdx.x] = s;
}

__global__ void cg_clear_kernel(CgState* st) { *st = CgState{}; }

// φ −= T(Σ V·φ / Σ V) from the partials of Σ V·φ.
template <typename T>
__global__ void __launch_bounds__(GNT) sub_mean_kernel(T* __restrict__ phi, long long n, const double* __restrict__ psv,
                                                       const double* __restrict__ sumv) {
  __shared__ double red[GNT / 64];
  const T mu = (T)(psum(psv, gridDim.x, red) / *sumv);
  for_cells<1>(n, [&](long long i) { phi[i] -= mu; });
}

// g_d = −(φ_hi − φ_lo)/T(d_lo + d_hi) per cell from the CSR stencil (_gax,
// src/gravity.jl:403-410), 3 SoA fields; axes beyond the rank are 0.
template <typename T>
__global__ void __launch_bounds__(GNT) csr_accel_kernel(const T* __restrict__ phi, T* __restrict__ g,
                                                        const int* __restrict__ glo, const int* __restrict__ ghi,
                                                        const double* __restrict__ gsum, long long n, int rank) {
  for (long long c = (long long)blockIdx.x * GNT + threadIdx.x; c < n; c += (long long)gridDim.x * GNT)
    for (int d = 0; d < 3; ++d) {
      if (d >= rank) {
        g[d * n + c] = T(0);
        continue;
      }
      const T wlo = phi[glo[d * n + c]], whi = phi[ghi[d * n + c]];
      g[d * n + c] = -(whi - wlo) / T(gsum[d * n + c]);
    }
}

// g_d = −(φ_hi − φ_lo)/T(d_lo + d_hi) per cell (src/gravity.jl:403-410), 3 SoA fields.
template <typename T>
__global__ void __launch_bounds__(GNT) accel_kernel(const T* __restrict__ phi, T* __restrict__ g, GridDev G, int gper) {
  for (long long c = (long long)blockIdx.x * GNT + threadIdx.x; c < G.ncell; c += (long long)gridDim.x * GNT) {
    int co[3];
    gcoords(G, c, co);
    for (int d = 0; d < 3; ++d)
      g[d * G.ncell + c] = d < G.rank ? VH_PROFILE_NS::grav_axis<T>(phi, G, gper, c, co, d) : T(0);
  }
}

// ---- host side ----

static int grid_blocks(long long n) {
  long long b = (n + GNT - 1) / GNT;
  if (b > 4096) b = 4096;
  return (int)(b < 1 ? 1 : b);
}

static int cg_blocks(long long n) {
  const long long b = (n + GNT - 1) / GNT;
  return (int)std::min<long long>(b, kCgWgs);
}

template <int RANK, int V>
static UniformRow<RANK, V> uniform_row(const GridDev& G, int gper) {
  UniformRow<RANK, V> R{};
  for (int d = 0; d < 3; ++d) {
    R.n[d] = G.n[d];
    R.coef[d] = d < RANK ? G.area[d] / (0.5 * (G.w[d] + G.w[d])) : 0.0;
  }
  R.gper = gper;
  R.wide = G.ncell >= (1LL << 31);
  R.dx = fast_div_by(G.n[0]);
  R.dy = fast_div_by(G.n[1]);
  return R;
}
// f(row) with the uniform operator of the grid's rank for values of type T: 16-byte packs
// where rows divide into them and `aligned` says the arrays start on 16 bytes.
template <typename T, typename F>
static auto with_uniform(const GridDev& G, int gper, bool aligned, F f) {
  auto rank = [&](auto v) {
    constexpr int V = decltype(v)::value;
    if (G.rank == 3) return f(uniform_row<3, V>(G, gper));
    if (G.rank == 2) return f(uniform_row<2, V>(G, gper));
    return f(uniform_row<1, V>(G, gper));
  };
  constexpr int P = 16 / sizeof(T);
  if (aligned && G.n[0] % P == 0) return rank(std::integral_constant<int, P>());
  return rank(std::integral_constant<int, 1>());
}

template <typename T, typename Row>
static void apply_row(hipStream_t s, long long n, const Row& row, const void* x, void* out) {
  hipLaunchKernelGGL((lap_kernel<T, Row>), dim3(cg_blocks(n / Row::V)), dim3(GNT), 0, s, (const T*)x, (T*)out, n, row);
}

void grav_apply(hipStream_t s, int dtype, const GridDev& G, int gper, const void* x, void* out) {
  const bool aligned = (((uintptr_t)x | (uintptr_t)out) & 15) == 0;   // the caller's arrays
  if (dtype == 0)
    with_uniform<double>(G, gper, aligned, [&](const auto& row) { apply_row<double>(s, G.ncell, row, x, out); });
  else
    with_uniform<float>(G, gper, aligned, [&](const auto& row) { apply_row<float>(s, G.ncell, row, x, out); });
}

void grav_accel(hipStream_t s, int dtype, const GridDev& G, int gper, const void* phi, void* g) {
  const int nb = grid_blocks(G.ncell);
  if (dtype == 0)
    hipLaunchKernelGGL(accel_kernel<double>, dim3(nb), dim3(GNT), 0, s, (const double*)phi, (double*)g, G, gper);
  else
    hipLaunchKernelGGL(accel_kernel<float>, dim3(nb), dim3(GNT), 0, s, (const float*)phi, (float*)g, G, gper);
}

// Plain CG (_cg_csr_run!, src/gravity.jl:248-322) on the operator `row` over n cells;
// vols: per-cell volumes, or null and the constant volume vol.
template <typename T, typename Row>
static int solve_t(hipStream_t s, const Row& row, long long n, const double* vols, double vol, const GravParams& P,
                   GravBuffers& B, long long* iters, double* relres) {
  const dim3 nb(cg_blocks(n / Row::V)), nt(GNT);
  T* phi = (T*)B.phi;
  T* r = (T*)B.work;
  T* p[2] = {r + n, r + 2 * n};
  T* Ap = Row::kStoreAp ? r + 3 * n : nullptr;
  const T* rho = (const T*)B.rho;
  CgState* st = (CgState*)B.state;
  CgState* host = (CgState*)B.host_state;
  double* rr = B.partials;
  double* pap = rr + kCgWgs;
  double* aux = pap + kCgWgs;
  double* bb = aux + kCgWgs;
  const double* sumv = B.sumv;
  *host = CgState{};
  hipLaunchKernelGGL(cg_clear_kernel, dim3(1), dim3(1), 0, s, st);
  if (P.project_mean) hipLaunchKernelGGL(vsum_kernel<T>, nb, nt, 0, s, rho, vols, vol, n, aux);
  hipLaunchKernelGGL((cg_init_kernel<T, Row>), nb, nt, 0, s, rho, (const T*)phi, r, n, row, P.G, vol, vols,
                     P.project_mean ? (const double*)aux : (const double*)nullptr, sumv, rr, bb);
  auto direction = [&](long long k) {
    hipLaunchKernelGGL((cg_dir_kernel<T, Row>), nb, nt, 0, s, (const T*)r, (const T*)p[k & 1], p[(k + 1) & 1], Ap, n,
                       row, k, P.tol, P.maxiter, (const double*)rr, (const double*)bb, pap, st, host);
  };
  direction(1);
  // Chunks of iterations; while the host waits for the end of one the next is queued.
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipError_t e = hipEventCreateWithFlags(&ev[0], hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&ev[1], hipEventDisableTiming);
  const volatile int* done = &host->done;
  long long k = 1;
  for (int j = 0; e == hipSuccess && k <= P.maxiter && !*done; ++j) {
    for (int i = 0; i < kCgChunk && k <= P.maxiter; ++i, ++k) {
      hipLaunchKernelGGL((cg_update_kernel<T, Row>), nb, nt, 0, s, phi, r, (const T*)p[(k + 1) & 1], (const T*)Ap, n,
                         row, k, (const double*)pap, rr, st, host);
      direction(k + 1);
    }
    e = hipEventRecord(ev[j & 1], s);
    if (e == hipSuccess && j > 0) e = hipEventSynchronize(ev[(j - 1) & 1]);
  }
  // volume-weighted mean projection (src/gravity.jl:310-320)
  if (e == hipSuccess && P.project_mean) {
    hipLaunchKernelGGL(vsum_kernel<T>, nb, nt, 0, s, (const T*)phi, vols, vol, n, aux);
    hipLaunchKernelGGL(sub_mean_kernel<T>, nb, nt, 0, s, phi, n, (const double*)aux, sumv);
  }
  if (e == hipSuccess) e = hipGetLastError();
  const hipError_t es = hipStreamSynchronize(s);
  if (e == hipSuccess) e = es;
  for (hipEvent_t v : ev)
    if (v) (void)hipEventDestroy(v);
  VH_HIP(e);
  *iters = (long long)host->iters;
  *relres = host->relres;
  return 0;
}

int grav_solve(hipStream_t s, int dtype, const GridDev& G, const GravParams& P, GravBuffers& B, long long* iters,
               double* relres) {
  if (dtype == 0)
    return with_uniform<double>(G, P.gper, true, [&](const auto& row) {
      return solve_t<double>(s, row, G.ncell, nullptr, G.V, P, B, iters, relres);
    });
  return with_uniform<float>(G, P.gper, true, [&](const auto& row) {
    return solve_t<float>(s, row, G.ncell, nullptr, G.V, P, B, iters, relres);
  });
}

void grav_csr_apply(hipStream_t s, int dtype, const GravCsr& A, const void* x, void* out) {
  const CsrRow row{A.rowptr, A.colidx, A.coef};
  if (dtype == 0) apply_row<double>(s, A.n, row, x, out);
  else apply_row<float>(s, A.n, row, x, out);
}

void grav_csr_accel(hipStream_t s, int dtype, const GravCsr& A, const void* phi, void* g) {
  const int nb = grid_blocks(A.n);
  if (dtype == 0)
    hipLaunchKernelGGL(csr_accel_kernel<double>, dim3(nb), dim3(GNT), 0, s, (const double*)phi, (double*)g, A.glo,
                       A.ghi, A.gsum, A.n, A.rank);
  else
    hipLaunchKernelGGL(csr_accel_kernel<float>, dim3(nb), dim3(GNT), 0, s, (const float*)phi, (float*)g, A.glo,
                       A.ghi, A.gsum, A.n, A.rank);
}

int grav_csr_solve(hipStream_t s, int dtype, const GravCsr& A, const GravParams& P, GravBuffers& B, long long* iters,
                   double* relres) {
  const CsrRow row{A.rowptr, A.colidx, A.coef};
  if (dtype == 0) return solve_t<double>(s, row, A.n, A.vol, 0.0, P, B, iters, relres);
  return solve_t<float>(s, row, A.n, A.vol, 0.0, P, B, iters, relres);
}

}  // namespace vh
