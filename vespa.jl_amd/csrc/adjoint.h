// Reverse mode of one SSP-RK2 step on a uniform grid (Float64, dt fixed).
//
// Forward (invV = dt/V): U1 = U − invV·A(U),  U2 = ½U + ½(U1 − invV·A(U1)).
// Reverse with w = ∂L/∂U2:
//   λ1 = ½w − ½·invV·A'(U1)ᵀw,   ∂L/∂U = ½w + λ1 − invV·A'(U)ᵀλ1.
// A'(U)ᵀλ is evaluated in three passes:
//   adj_prim_kernel   W = cons2prim(U) per cell;
//   adj_face_kernel   one lane per face: the face states (PLM-minmod), the
//                     flux VJP applied to area·(λ_left − λ_right) (one side at a
//                     domain boundary, with the ghost folded back), giving the
//                     adjoints of the two face states;
//   adj_cell_kernel   one lane per cell and axis: gathers the face-state adjoints of its
//                     own faces and the slope adjoints of itself and its two
//                     neighbours per axis (minmod active branch), maps the
//                     primitive adjoint to conserved variables and writes
//                     a1·base1 + a2·base2 + beta·invV·A'ᵀλ.
// Non-smooth points take the active branch: minmod's selected argument (zero
// when the signs differ), the Davis min/max active argument, the upwind HLLC
// branch, the pressure floor when it is the larger argument.
#pragma once

#include "hydro.h"

namespace vh {
namespace VH_PROFILE_NS {

using D5 = Prim<double>;

// Division and the sound speed: correctly rounded in the exact profile, refined
// hardware reciprocal / rsqrt in the fast profile (the reverse mode needs no bit
// parity; it is tested to 1e-12 against a scatter-form CPU restatement).
__device__ __forceinline__ double adiv(double a, double b) {
#if VH_FAST_PROFILE
  return fast_div(a, b);
#else
  return a / b;
#endif
}
__device__ __forceinline__ double asound(double g, double p, double r) { return sound(g, p, r); }

template <int A>
__device__ __forceinline__ double& ncomp(D5& w) {
  if constexpr (A == 0) return w.vx;
  else if constexpr (A == 1) return w.vy;
  else return w.vz;
}
template <int A>
__device__ __forceinline__ double ncomp(const D5& w) {
  if constexpr (A == 0) return w.vx;
  else if constexpr (A == 1) return w.vy;
  else return w.vz;
}

__device__ __forceinline__ void d5_add(D5& a, const D5& b) {
  a.r += b.r; a.vx += b.vx; a.vy += b.vy; a.vz += b.vz; a.p += b.p;
}
__device__ __forceinline__ D5 d5_zero() {
  D5 z;
  z.r = z.vx = z.vy = z.vz = z.p = 0.0;
  return z;
}

// Transpose of the ghost map (outflow: identity; reflecting: flip the normal velocity).
template <int A>
__device__ __forceinline__ D5 ghostT(const D5& b, int bc) {
  D5 o = b;
  if (bc == BC_REFLECTING) ncomp<A>(o) = -ncomp<A>(b);
  return o;
}

// cons2prim adjoint at U: Wb → Ub (src/eos.jl:8-25).
__device__ __forceinline__ Cons<double> c2p_vjp(const Cons<double>& U, double g, const D5& Wb) {
  const double rho = U.d;
  const double inv = recip(rho);
  const double vx = U.mx * inv, vy = U.my * inv, vz = U.mz * inv;
  const double v2 = (vx * vx + vy * vy) + vz * vz;
  const double kin = (0.5 * rho) * v2;
  const double pc = (g - 1.0) * (U.e - kin);
  const double pf = 1e-12 * kin;
  double kinb, Eb;
  if (pf > pc) {
    kinb = Wb.p * 1e-12;
    Eb = 0.0;
  } else {
    kinb = -Wb.p * (g - 1.0);
    Eb = Wb.p * (g - 1.0);
  }
  const double vbx = Wb.vx + kinb * rho * vx, vby = Wb.vy + kinb * rho * vy, vbz = Wb.vz + kinb * rho * vz;
  const double invb = vbx * U.mx + vby * U.my + vbz * U.mz;
  Cons<double> o;
  o.d = Wb.r + kinb * 0.5 * v2 - invb * inv * inv;
  o.mx = vbx * inv;
  o.my = vby * inv;
  o.mz = vbz * inv;
  o.e = Eb;
  return o;
}

__device__ __forceinline__ double energy64(const D5& W, double g) {
  return adiv(W.p, g - 1.0) + (0.5 * W.r) * ((W.vx * W.vx + W.vy * W.vy) + W.vz * W.vz);
}

__device__ __forceinline__ void energy_vjp(const D5& W, double g, double Eb, D5& Wb) {
  Wb.r += Eb * 0.5 * ((W.vx * W.vx + W.vy * W.vy) + W.vz * W.vz);
  Wb.vx += Eb * W.r * W.vx;
  Wb.vy += Eb * W.r * W.vy;
  Wb.vz += Eb * W.r * W.vz;
  Wb.p += adiv(Eb, g - 1.0);
}

// euler_flux adjoint (src/riemann.jl:9-20) along axis A (0-based).
template <int A>
__device__ __forceinline__ void eflux_vjp(const D5& W, double g, const Cons<double>& Fb, D5& Wb) {
  const double r = W.r, p = W.p, un = ncomp<A>(W);
  const double E = energy64(W, g);
  double rb = Fb.d * un, unb = Fb.d * r, pb = 0.0;
  const double mbx = Fb.mx * un, mby = Fb.my * un, mbz = Fb.mz * un;
  unb += Fb.mx * (r * W.vx) + Fb.my * (r * W.vy) + Fb.mz * (r * W.vz);
  pb += A == 0 ? Fb.mx : (A == 1 ? Fb.my : Fb.mz);
  rb += mbx * W.vx + mby * W.vy + mbz * W.vz;
  Wb.vx += mbx * r;
  Wb.vy += mby * r;
  Wb.vz += mbz * r;
  const double Eb = Fb.e * un;
  pb += Fb.e * un;
  unb += Fb.e * (E + p);
  energy_vjp(W, g, Eb, Wb);
  Wb.r += rb;
  Wb.p += pb;
  ncomp<A>(Wb) += unb;
}

// hllc_flux adjoint (src/riemann.jl:33-88) along axis A: accumulates WLb, WRb.
template <int A>
__device__ void hllc_vjp(const D5& WL, const D5& WR, double g, const Cons<double>& ob, D5& WLb, D5& WRb) {
  const double rL = WL.r, rR = WR.r, pL = WL.p, pR = WR.p;
  const double unL = ncomp<A>(WL), unR = ncomp<A>(WR);
  const double cL = asound(g, pL, rL), cR = asound(g, pR, rR);
  const double xL = cL * cL, xR = cR * cR;
  const double aL = unL - cL, aR = unR - cR, bL = unL + cL, bR = unR + cR;
  const double SL = vmin(aL, aR), SR = vmax(bL, bR);
  if (SL >= 0.0) {
    eflux_vjp<A>(WL, g, ob, WLb);
    return;
  }
  if (SR <= 0.0) {
    eflux_vjp<A>(WR, g, ob, WRb);
    return;
  }
  const double tL = rL * unL, tR = rR * unR;
  const double num = pR - pL + tL * (SL - unL) - tR * (SR - unR);
  const double den = rL * (SL - unL) - rR * (SR - unR);
#if VH_FAST_PROFILE
  // one refined reciprocal per denominator, shared by the value and its adjoint
  const double deninv = recip(den);
  const double Ss = num * deninv;
#else
  const double Ss = adiv(num, den);
#endif
  const bool useL = Ss >= 0.0;
  const D5 W = useL ? WL : WR;
  D5 Wb = d5_zero();
  const double SK = useL ? SL : SR;
  const double r = W.r, un = ncomp<A>(W), p = W.p;
  const double E = energy64(W, g);
  const double q = r * (SK - un);
  const double d3 = SK - Ss;
  const double rinv = recip(r);
  const double qinv = recip(q);
  const double d3inv = recip(d3);
#if VH_FAST_PROFILE
  const double factor = q * d3inv;
  const double vs0 = A == 0 ? Ss : W.vx, vs1 = A == 1 ? Ss : W.vy, vs2 = A == 2 ? Ss : W.vz;
  const double Aa = Ss - un, Bb = Ss + p * qinv;
  const double Es = E * rinv + Aa * Bb;
#else
  const double factor = adiv(q, d3);
  const double vs0 = A == 0 ? Ss : W.vx, vs1 = A == 1 ? Ss : W.vy, vs2 = A == 2 ? Ss : W.vz;
  const double Aa = Ss - un, Bb = Ss + adiv(p, q);
  const double Es = adiv(E, r) + Aa * Bb;
#endif
  // out = F(W) + SK·(Us − Uk), Us = factor·(1, vs, Es), Uk = (r, r·v, E)
  const double SKb0 = ob.d * (factor - r) + ob.mx * (factor * vs0 - r * W.vx) + ob.my * (factor * vs1 - r * W.vy) +
                      ob.mz * (factor * vs2 - r * W.vz) + ob.e * (factor * Es - E);
  double SKb = SKb0;
  eflux_vjp<A>(W, g, ob, Wb);
  const double u0 = SK * ob.d, u1 = SK * ob.mx, u2 = SK * ob.my, u3 = SK * ob.mz, u4 = SK * ob.e;
  const double factorb = u0 + u1 * vs0 + u2 * vs1 + u3 * vs2 + u4 * Es;
  const double vsb0 = u1 * factor, vsb1 = u2 * factor, vsb2 = u3 * factor;
  const double Esb = u4 * factor;
  double rb = 0.0, unb = 0.0, pb = 0.0, Eb = 0.0, Ssb = 0.0, qb = 0.0;
  // Uk = prim2cons(W) with adjoint −SK·ob
  rb -= u0;
  rb -= u1 * W.vx + u2 * W.vy + u3 * W.vz;
  Wb.vx -= u1 * r;
  Wb.vy -= u2 * r;
  Wb.vz -= u3 * r;
  Eb -= u4;
  // Es = E/r + Aa·Bb
  Eb += Esb * rinv;
  rb -= Esb * E * rinv * rinv;
  const double Ab = Esb * Bb, Bbb = Esb * Aa;
  Ssb += Ab;
  unb -= Ab;
  Ssb += Bbb;
  pb += Bbb * qinv;
  qb -= Bbb * p * qinv * qinv;
  if (A == 0) { Ssb += vsb0; } else { Wb.vx += vsb0; }
  if (A == 1) { Ssb += vsb1; } else { Wb.vy += vsb1; }
  if (A == 2) { Ssb += vsb2; } else { Wb.vz += vsb2; }
  // factor = q/(SK − Ss)
  qb += factorb * d3inv;
  const double d3b = -factorb * factor * d3inv;
  SKb += d3b;
  Ssb -= d3b;
  // q = r·(SK − un)
  rb += qb * (SK - un);
  SKb += qb * r;
  unb -= qb * r;
  energy_vjp(W, g, Eb, Wb);
  Wb.r += rb;
  Wb.p += pb;
  ncomp<A>(Wb) += unb;
  if (useL) d5_add(WLb, Wb);
  else d5_add(WRb, Wb);
  double SLb = useL ? SKb : 0.0, SRb = useL ? 0.0 : SKb;
  // Ss = num/den
#if !VH_FAST_PROFILE
  const double deninv = recip(den);
#endif
  const double numb = Ssb * deninv, denb = -Ssb * Ss * deninv;
  double rLb = 0, rRb = 0, pLb = 0, pRb = 0, unLb = 0, unRb = 0, cLb = 0, cRb = 0;
  pRb += numb;
  pLb -= numb;
  const double tLb = numb * (SL - unL);
  rLb += tLb * unL;
  unLb += tLb * rL;
  SLb += numb * tL;
  unLb -= numb * tL;
  const double tRb = -numb * (SR - unR);
  rRb += tRb * unR;
  unRb += tRb * rR;
  SRb -= numb * tR;
  unRb += numb * tR;
  rLb += denb * (SL - unL);
  SLb += denb * rL;
  unLb -= denb * rL;
  rRb -= denb * (SR - unR);
  SRb -= denb * rR;
  unRb += denb * rR;
  if (aL <= aR) { unLb += SLb; cLb -= SLb; } else { unRb += SLb; cRb -= SLb; }
  if (bL >= bR) { unLb += SRb; cLb += SRb; } else { unRb += SRb; cRb += SRb; }
  const double xLb = adiv(cLb, 2.0 * cL), xRb = adiv(cRb, 2.0 * cR);
  const double rLi = recip(rL), rRi = recip(rR);
  pLb += xLb * g * rLi;
  rLb -= xLb * xL * rLi;
  pRb += xRb * g * rRi;
  rRb -= xRb * xR * rRi;
  WLb.r += rLb;
  WLb.p += pLb;
  ncomp<A>(WLb) += unLb;
  WRb.r += rRb;
  WRb.p += pRb;
  ncomp<A>(WRb) += unRb;
}

// minmod(c − l, r − c) adjoint per component: sb → (lb, cb, rb) contributions.
__device__ __forceinline__ void minmod_vjp1(double l, double c, double r, double sb, double& lb, double& cb,
                                            double& rb) {
  const double a = c - l, b = r - c;
  if (a * b <= 0.0) return;
  if (vabs(a) < vabs(b)) {
    cb += sb;
    lb -= sb;
  } else {
    rb += sb;
    cb -= sb;
  }
}

__device__ __forceinline__ D5 load_w(const double* __restrict__ W, long long n, long long c) {
  D5 w;
  w.r = W[c]; w.vx = W[n + c]; w.vy = W[2 * n + c]; w.vz = W[3 * n + c]; w.p = W[4 * n + c];
  return w;
}
__device__ __forceinline__ void store_w(double* __restrict__ W, long long n, long long c, const D5& w) {
  W[c] = w.r; W[n + c] = w.vx; W[2 * n + c] = w.vy; W[3 * n + c] = w.vz; W[4 * n + c] = w.p;
}

__global__ void __launch_bounds__(256) adj_prim_kernel(const double* __restrict__ U, double* __restrict__ W,
                                                       GridDev G) {
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= G.ncell) return;
  store_w(W, G.ncell, c, cons2prim<double, false>(load_cons(U, G.ncell, c), G.gamma, G.gamma));
}

// Strides and face-slot geometry along axis A.
struct AxisGeo {
  long long stride;   // cell index stride along A
  int n;              // cells along A
};
template <int A>
__device__ __forceinline__ AxisGeo axis_geo(const GridDev& G) {
  AxisGeo a;
  a.n = G.n[A];
  a.stride = A == 0 ? 1 : (A == 1 ? (long long)G.n[0] : (long long)G.n[0] * G.n[1]);
  return a;
}

// The three coordinates of slot or cell s in a box of m0 × m1 × any; in 32 bits where all
// of the box's `total` items fit (a 64-bit quotient is some 100 instructions).
__device__ __forceinline__ void split3(long long s, long long total, int m0, int m1, int& i, int& j, int& k) {
  if (total <= 0xffffffffLL) {
    const unsigned u = (unsigned)s, r = u / (unsigned)m0;
    i = (int)(u - r * (unsigned)m0);
    k = (int)(r / (unsigned)m1);
    j = (int)(r - (unsigned)k * (unsigned)m1);
  } else {
    i = (int)(s % m0);
    j = (int)((s / m0) % m1);
    k = (int)(s / ((long long)m0 * m1));
  }
}
__device__ __forceinline__ D5 d5_select(bool on, const D5& a, const D5& b) {
  D5 o;
  o.r = on ? a.r : b.r; o.vx = on ? a.vx : b.vx; o.vy = on ? a.vy : b.vy; o.vz = on ? a.vz : b.vz; o.p = on ? a.p : b.p;
  return o;
}

struct AdjFaces {
  double* gL[3];
  double* gR[3];
};

// Face slots along A: (n_A + 1) per line, slot coordinate q ∈ [0, n_A] is the
// face between cells q−1 and q (periodic axes use q ∈ [0, n_A) with q = 0 the
// wrapped face). Output gL/gR: 5 SoA fields over the slots. A domain boundary's face
// has one side in the grid: the other is its ghost, and the ghost's adjoint folds back.
template <int A>
__device__ __forceinline__ void adj_face(const double* __restrict__ W, const double* __restrict__ lam, const GridDev& G,
                                         long long s, double* __restrict__ gL, double* __restrict__ gR) {
  const int m0 = A == 0 ? G.n[0] + 1 : G.n[0];
  const int m1 = A == 1 ? G.n[1] + 1 : G.n[1];
  const int m2 = A == 2 ? G.n[2] + 1 : G.n[2];
  const long long ns = (long long)m0 * m1 * m2;
  if (s >= ns) return;
  int i, j, k;
  split3(s, ns, m0, m1, i, j, k);
  const int q = A == 0 ? i : (A == 1 ? j : k);
  const AxisGeo ax = axis_geo<A>(G);
  const int blo = G.bc[2 * A], bhi = G.bc[2 * A + 1];
  const bool per = blo == BC_PERIODIC;
  const long long n = G.ncell;
  D5 bL = d5_zero(), bR = d5_zero();
  if (per && q == ax.n) {   // unused slot of a periodic axis
    store_w(gL, ns, s, bL);
    store_w(gR, ns, s, bR);
    return;
  }
  const bool isL = per || q > 0, isR = q < ax.n;   // is there a cell on this side
  const int qr = isR ? q : ax.n - 1;
  const int ql = q > 0 ? q - 1 : (per ? ax.n - 1 : 0);
  const int ci = A == 0 ? qr : i, cj = A == 1 ? qr : j, ck = A == 2 ? qr : k;
  const long long cr = ((long long)ck * G.n[1] + cj) * G.n[0] + ci;   // cell q (or the last cell at q = n)
  const long long cl = cr + (long long)(ql - qr) * ax.stride;         // cell q−1 (or the first at q = 0)
  const bool hll = ql > 0 || per, hrr = qr < ax.n - 1 || per;
  const long long cll = ql > 0 ? cl - ax.stride : (per ? cl + (long long)(ax.n - 1) * ax.stride : cl);
  const long long crr = qr < ax.n - 1 ? cr + ax.stride : (per ? cr - (long long)(ax.n - 1) * ax.stride : cr);
  // All four cells of the face's line are read at once; ghosts replace by selection.
  D5 w0 = load_w(W, n, cll), w1 = load_w(W, n, cl), w2 = load_w(W, n, cr), w3 = load_w(W, n, crr);
  Cons<double> ll = load_cons(lam, n, cl), lr = load_cons(lam, n, cr);
  const D5 c1 = w1;
  w1 = d5_select(isL, w1, ghost(w2, blo, A + 1));
  w2 = d5_select(isR, w2, ghost(c1, bhi, A + 1));
  w0 = d5_select(hll, w0, ghost(c1, blo, A + 1));
  w3 = d5_select(hrr, w3, ghost(w2, bhi, A + 1));
  D5 WL = face_value(w1, slope(w0, w1, w2), 0.5);
  D5 WR = face_value(w2, slope(w1, w2, w3), -0.5);
  if (!isL) WL = ghost(WR, blo, A + 1);
  if (!isR) WR = ghost(WL, bhi, A + 1);
  const double a = G.area[A];
  const double z = 0.0;
  Cons<double> mu;
  mu.d = (isL ? a * ll.d : z) - (isR ? a * lr.d : z);
  mu.mx = (isL ? a * ll.mx : z) - (isR ? a * lr.mx : z);
  mu.my = (isL ? a * ll.my : z) - (isR ? a * lr.my : z);
  mu.mz = (isL ? a * ll.mz : z) - (isR ? a * lr.mz : z);
  mu.e = (isL ? a * ll.e : z) - (isR ? a * lr.e : z);
  hllc_vjp<A>(WL, WR, G.gamma, mu, bL, bR);
  if (!isL) {
    d5_add(bR, ghostT<A>(bL, blo));
    bL = d5_zero();
  }
  if (!isR) {
    d5_add(bL, ghostT<A>(bR, bhi));
    bR = d5_zero();
  }
  store_w(gL, ns, s, bL);
  store_w(gR, ns, s, bR);
}

// The axes' faces in one launch (blockIdx.y = axis): a small grid leaves the chip part
// idle in a launch of each. Bound: latency of the dependent loads, then hllc_vjp's arithmetic
// (112 registers, 4 waves per SIMD); one hllc_vjp serves inner and boundary faces, where a
// wave that held both went through it three times. 60×52×44: three launches of 15.0, 10.7 and
// 10.6 µs → 16.4 µs.
template <int RANK>
__global__ void __launch_bounds__(256) adj_face_kernel(const double* __restrict__ W, const double* __restrict__ lam,
                                                       GridDev G, AdjFaces F) {
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;
  if (RANK == 1 || blockIdx.y == 0) adj_face<0>(W, lam, G, s, F.gL[0], F.gR[0]);
  else if (RANK == 2 || blockIdx.y == 1) adj_face<RANK == 1 ? 0 : 1>(W, lam, G, s, F.gL[1], F.gR[1]);
  else adj_face<RANK == 3 ? 2 : 0>(W, lam, G, s, F.gL[2], F.gR[2]);
}

// Primitive adjoint gathered by cell c (coordinate p along A) from axis A, added to Wb. The line's
// cells p−2..p+2 and faces are read at once, at the cell's own place where there is none.
template <int A>
__device__ __forceinline__ void gather_axis(const double* __restrict__ W, const double* __restrict__ gL,
                                            const double* __restrict__ gR, const GridDev& G, long long c, int i, int j,
                                            int k, D5& Wb) {
  const AxisGeo ax = axis_geo<A>(G);
  const int m0 = A == 0 ? G.n[0] + 1 : G.n[0];
  const int m1 = A == 1 ? G.n[1] + 1 : G.n[1];
  const int m2 = A == 2 ? G.n[2] + 1 : G.n[2];
  const long long ns = (long long)m0 * m1 * m2;
  const int p = A == 0 ? i : (A == 1 ? j : k);
  const int nA = ax.n;
  const int blo = G.bc[2 * A], bhi = G.bc[2 * A + 1];
  const bool per = blo == BC_PERIODIC;
  const long long n = G.ncell;
  const long long fstride = A == 0 ? 1 : (A == 1 ? (long long)m0 : (long long)m0 * m1);
  const long long f0 = ((long long)k * m1 + j) * m0 + i;   // slot of the lo face
  // slot of face coordinate p + d and cell at p + d (wrapped on periodic axes, also those of
  // one cell; clamped else)
  auto slot = [&](int d) -> long long {
    int x = p + d;
    if (per) x = x < 0 ? max(x + nA, 0) : (x >= nA ? min(x - nA, nA - 1) : x);
    else x = x < 0 ? 0 : (x > nA ? nA : x);
    return f0 + (long long)(x - p) * fstride;
  };
  auto cell_at = [&](int d) -> long long {
    int x = p + d;
    if (per) x = x < 0 ? max(x + nA, 0) : (x >= nA ? min(x - nA, nA - 1) : x);
    else x = x < 0 ? 0 : (x >= nA ? nA - 1 : x);
    return c + (long long)(x - p) * ax.stride;
  };
  const bool hl = p > 0 || per, hr = p < nA - 1 || per;
  const bool hl2 = p > 1 || per, hr2 = p < nA - 2 || per;
  const long long cc[5] = {cell_at(-2), cell_at(-1), c, cell_at(1), cell_at(2)};
  const long long sl[3] = {slot(0), slot(1), slot(2)}, sr[3] = {slot(-1), slot(0), slot(1)};
  double* out[5] = {&Wb.r, &Wb.vx, &Wb.vy, &Wb.vz, &Wb.p};
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    const double* Wf = W + f * n;
    const double* gl = gL + f * ns;
    const double* gr = gR + f * ns;
    double w[5], l[3], r[3];
#pragma unroll
    for (int d = 0; d < 5; ++d) w[d] = Wf[cc[d]];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      l[d] = gl[sl[d]];
      r[d] = gr[sr[d]];
    }
    const bool flipl = f == A + 1 && blo == BC_REFLECTING, fliph = f == A + 1 && bhi == BC_REFLECTING;
    if (!hl) w[1] = flipl ? -w[2] : w[2];
    if (!hr) w[3] = fliph ? -w[2] : w[2];
    if (!hl2) w[0] = flipl ? -w[1] : w[1];
    if (!hr2) w[4] = fliph ? -w[3] : w[3];
    double v = *out[f];
    v += l[1];   // own hi face
    v += r[1];   // own lo face
    double lb = 0.0, cb = 0.0, rb = 0.0;
    minmod_vjp1(w[1], w[2], w[3], 0.5 * l[1] - 0.5 * r[1], lb, cb, rb);
    v += cb;
    if (!hl) v += flipl ? -lb : lb;
    if (!hr) v += fliph ? -rb : rb;
    double lb2 = 0.0, cb2 = 0.0, rb2 = 0.0;
    minmod_vjp1(w[2], w[3], w[4], 0.5 * l[2] - 0.5 * r[2], lb2, cb2, rb2);   // hi neighbour: c is its lo
    if (hr) v += lb2;
    double lb3 = 0.0, cb3 = 0.0, rb3 = 0.0;
    minmod_vjp1(w[0], w[1], w[2], 0.5 * l[0] - 0.5 * r[0], lb3, cb3, rb3);   // lo neighbour: c is its hi
    if (hl) v += rb3;
    asm volatile("" : "+v"(v)::"memory");   // complete here: keeps the next field's loads out of this one's registers
    *out[f] = v;
  }
}

// out = a1·base1 + a2·base2 + (beta·dt/V)·A'(U)ᵀλ (base2 may be null). out may
// alias base1 or base2 (each lane reads and writes its own cell only).
// One wave per axis of 64 cells, the sums joined through LDS: a lane that walked the axes one
// after the other left 2 waves per SIMD at 60×52×44 and its loads in a chain. Field by field
// the gather needs 68 registers; with all fields' loads in flight it needs 186 and is slower.
// 60×52×44: 26.7 → 21.1 µs (25.0 with 186 registers). Whole A'ᵀλ in passes, before and now (µs):
// 200 cells 12.0, 11.9; 60² 25.9, 13.7; 400² 51, 39; 1200×1000 279, 236; 24×20×16 31.5, 14.9;
// 60×52×44 64.6, 42.7; 128×128×96 488, 418.
template <int RANK>
__global__ void __launch_bounds__(64 * RANK) adj_cell_kernel(const double* __restrict__ U, const double* __restrict__ W,
                                                       AdjFaces F, const double* base1, double a1,
                                                       const double* base2, double a2, double beta,
                                                       const double* __restrict__ dtp, GridDev G, double* out) {
  __shared__ double part[RANK > 1 ? RANK - 1 : 1][5][64];
  const long long n = G.ncell;
  const int lane = threadIdx.x & 63, axis = threadIdx.x >> 6;
  const long long c = (long long)blockIdx.x * 64 + lane;
  const bool on = c < n;
  D5 Wb = d5_zero();
  if (on) {
    int i, j, k;
    split3(c, n, G.n[0], G.n[1], i, j, k);
    if (RANK == 1 || axis == 0) gather_axis<0>(W, F.gL[0], F.gR[0], G, c, i, j, k, Wb);
    else if (RANK == 2 || axis == 1) gather_axis<RANK == 1 ? 0 : 1>(W, F.gL[1], F.gR[1], G, c, i, j, k, Wb);
    else gather_axis<RANK == 3 ? 2 : 0>(W, F.gL[2], F.gR[2], G, c, i, j, k, Wb);
  }
  if constexpr (RANK > 1) {
    if (axis > 0) {
      double(*o)[64] = part[axis - 1];
      o[0][lane] = Wb.r; o[1][lane] = Wb.vx; o[2][lane] = Wb.vy; o[3][lane] = Wb.vz; o[4][lane] = Wb.p;
    }
    __syncthreads();
    if (axis > 0) return;
#pragma unroll
    for (int x = 0; x < RANK - 1; ++x) {
      Wb.r += part[x][0][lane]; Wb.vx += part[x][1][lane]; Wb.vy += part[x][2][lane]; Wb.vz += part[x][3][lane];
      Wb.p += part[x][4][lane];
    }
  }
  if (!on) return;
  const Cons<double> Ub = c2p_vjp(load_cons(U, n, c), G.gamma, Wb);
  const double s = beta * (*dtp / (1.0 * G.V));
  const double ub[5] = {Ub.d, Ub.mx, Ub.my, Ub.mz, Ub.e};
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    double v = a1 * base1[f * n + c];
    if (base2) v += a2 * base2[f * n + c];
    out[f * n + c] = v + s * ub[f];
  }
}

// ---------------------------------------------------------------------------
// Fused A'(U)ᵀλ for 2D grids periodic on both axes: one workgroup per 16×16 tile
// computes W for the tile and a cross-shaped halo of three cells, every face
// adjoint its cells need (the tile's faces plus one more on each side), and the
// gather, in LDS; one launch instead of four, no face buffers in HBM.
// Bound: the phases wait for each other (loads, faces, gather, stores), so what
// counts is that a second workgroup fills a compute unit meanwhile. 81,440 B of LDS
// and 128 registers let two of 512 lanes share it; 608 faces over 512 lanes leave the
// second pass to two waves. Per launch at 512²: one 32×16 tile per compute unit 29.0 µs
// (at 512, 640, 768 and 1024 lanes alike, 26.5 with the cell's state kept in registers),
// 16×16 with 320 lanes 33.0, with 512 25.8, with the XCD ranges below 23.1. At 256² 13.9 →
// 9.9 µs, at 2048² 443 → 353 µs; sizes that the 32×16 tile did not divide went through
// the passes: 500×400 60 → 23 µs, 10² 15 → 7.7 µs.
constexpr int JTX = 16, JTY = 16, JNT = 512;
constexpr int JNXF = JTY * (JTX + 3);   // x faces of a tile (one extra on the lo side, two on the hi)
constexpr int JNYF = (JTY + 3) * JTX;   // y faces of a tile

struct JatLDS {
  double W[5][JTY + 6][JTX + 6];   // rows y0-3..y0+JTY+2, cols x0-3..x0+JTX+2 (the corners stay unused)
  double L[5][JTY + 4][JTX + 4];   // λ, rows y0-2..y0+JTY+1, cols x0-2..x0+JTX+1
  double Gx[2][5][JTY][JTX + 2];   // x-face state adjoints: [0] left state of faces 1.., [1] right state of faces 0..
  double Gy[2][5][JTY + 2][JTX];   // y-face state adjoints, the same
};

// W and λ of one cell, (row, col) in tile coordinates.
__device__ __forceinline__ D5 jat_w(const JatLDS& S, int row, int col) {
  D5 w;
  w.r = S.W[0][row + 3][col + 3]; w.vx = S.W[1][row + 3][col + 3]; w.vy = S.W[2][row + 3][col + 3];
  w.vz = S.W[3][row + 3][col + 3]; w.p = S.W[4][row + 3][col + 3];
  return w;
}
__device__ __forceinline__ Cons<double> jat_l(const JatLDS& S, int row, int col) {
  Cons<double> l;
  l.d = S.L[0][row + 2][col + 2]; l.mx = S.L[1][row + 2][col + 2]; l.my = S.L[2][row + 2][col + 2];
  l.mz = S.L[3][row + 2][col + 2]; l.e = S.L[4][row + 2][col + 2];
  return l;
}
__device__ __forceinline__ void jat_put_w(JatLDS& S, int row, int col, const D5& w) {
  S.W[0][row + 3][col + 3] = w.r; S.W[1][row + 3][col + 3] = w.vx; S.W[2][row + 3][col + 3] = w.vy;
  S.W[3][row + 3][col + 3] = w.vz; S.W[4][row + 3][col + 3] = w.p;
}
__device__ __forceinline__ void jat_put_l(JatLDS& S, int row, int col, const Cons<double>& l) {
  S.L[0][row + 2][col + 2] = l.d; S.L[1][row + 2][col + 2] = l.mx; S.L[2][row + 2][col + 2] = l.my;
  S.L[3][row + 2][col + 2] = l.mz; S.L[4][row + 2][col + 2] = l.e;
}
__device__ __forceinline__ Cons<double> mu_of(double a, const Cons<double>& l, const Cons<double>& r) {
  Cons<double> m;
  m.d = a * l.d - a * r.d;
  m.mx = a * l.mx - a * r.mx;
  m.my = a * l.my - a * r.my;
  m.mz = a * l.mz - a * r.mz;
  m.e = a * l.e - a * r.e;
  return m;
}
__device__ __forceinline__ D5 d5_swap_xy(const D5& w, bool on) {
  D5 o = w;
  o.vx = on ? w.vy : w.vx;
  o.vy = on ? w.vx : w.vy;
  return o;
}
__device__ __forceinline__ Cons<double> c_swap_xy(const Cons<double>& f, bool on) {
  Cons<double> o = f;
  o.mx = on ? f.my : f.mx;
  o.my = on ? f.mx : f.my;
  return o;
}

// Slope adjoint terms of one component gathered by a cell from its own slope and
// its two neighbours' slopes along one axis, added to Wb. w[0..4] = W at offsets
// −2..+2; gl[0..2] = left-state adjoints of the faces at offsets −1/2, 1/2, 3/2;
// gr[0..2] = right-state adjoints of the faces at −3/2, −1/2, 1/2.
__device__ __forceinline__ double gather_line(const double w[5], const double gl[3], const double gr[3], double Wb) {
  Wb += gl[1];   // the cell's hi face
  Wb += gr[1];   // and its lo face
  double lb = 0.0, cb = 0.0, rb = 0.0;
  minmod_vjp1(w[1], w[2], w[3], 0.5 * gl[1] - 0.5 * gr[1], lb, cb, rb);
  Wb += cb;
  double lb2 = 0.0, cb2 = 0.0, rb2 = 0.0;
  minmod_vjp1(w[2], w[3], w[4], 0.5 * gl[2] - 0.5 * gr[2], lb2, cb2, rb2);   // hi neighbour: this cell is its lo
  Wb += lb2;
  double lb3 = 0.0, cb3 = 0.0, rb3 = 0.0;
  minmod_vjp1(w[0], w[1], w[2], 0.5 * gl[0] - 0.5 * gr[0], lb3, cb3, rb3);   // lo neighbour: this cell is its hi
  Wb += rb3;
  return Wb;
}

// out = a1·base1 + a2·base2 + beta·(dt/V)·A'(U)ᵀλ for a 2D grid periodic on both
// axes, one launch. Phases (two barriers): load the tile's W (halo 3) and λ (halo
// 2) in a cross shape; evaluate every x and y face VJP of the tile plus the faces
// its cells' slope adjoints reach (304 + 304 faces, two passes over the 512
// lanes; a y face runs in the frame of an x face, x and y exchanged); gather
// both axes per cell and map the primitive adjoint to conserved variables.
__global__ void __launch_bounds__(JNT, 4) adj_jat2d_periodic_kernel(const double* __restrict__ U,
                                                                 const double* __restrict__ lam,
                                                                 const double* base1, double a1,
                                                                 const double* base2, double a2, double beta,
                                                                 const double* __restrict__ dtp, GridDev G,
                                                                 double* out) {
  __shared__ JatLDS S;
  const int nx = G.n[0], ny = G.n[1];
  const long long n = G.ncell;
  const int tid = threadIdx.x;
  const int tx = tid % JTX, ty = tid / JTX;
  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous range of tiles, so that
  // its L2 serves the halo columns (25.8 → 23.1 µs at 512²).
  const int nt = gridDim.x * gridDim.y, id = blockIdx.y * gridDim.x + blockIdx.x;
  const int xcd = id & 7, q8 = nt >> 3, r8 = nt & 7;
  const int tile = xcd * q8 + (xcd < r8 ? xcd : r8) + (id >> 3);
  const int x0 = tile % gridDim.x * JTX, y0 = tile / gridDim.x * JTY;
  const double g = G.gamma;
  auto wrapx = [&](int x) { return x < 0 ? x + nx : (x >= nx ? x - nx : x); };
  auto wrapy = [&](int y) { return y < 0 ? y + ny : (y >= ny ? y - ny : y); };
  auto cidx = [&](int x, int y) { return (long long)wrapy(y) * nx + wrapx(x); };
  // ---- load: own cell, then the cross-shaped halos of W (3) and λ (2) ----
  const long long c = cidx(x0 + tx, y0 + ty);
  constexpr int NWX = 6 * JTY, NLX = 4 * JTY, NWY = 6 * JTX, NLY = 4 * JTX;
  static_assert(NWX + NLX + NWY + NLY <= JNT && JTX * JTY <= JNT, "one halo item and one cell per lane");
  Cons<double> Uc;
  if (tid < JTX * JTY) {
    Uc = load_cons(U, n, c);
    jat_put_w(S, ty, tx, cons2prim<double, false>(Uc, g, g));
    jat_put_l(S, ty, tx, load_cons(lam, n, c));
  }
  const int h = tid < JTX * JTY ? tid + (JNT - JTX * JTY) : tid - JTX * JTY;   // halo items start on the idle lanes
  if (h < NWX + NWY) {
    int row, col;
    if (h < NWX) {
      const int q = h % 6;
      row = h / 6;
      col = q < 3 ? q - 3 : JTX + q - 3;   // −3, −2, −1 | JTX .. JTX+2
    } else {
      const int i = (h - NWX) / JTX;
      row = i < 3 ? i - 3 : JTY + i - 3;
      col = (h - NWX) % JTX;
    }
    jat_put_w(S, row, col, cons2prim<double, false>(load_cons(U, n, cidx(x0 + col, y0 + row)), g, g));
  } else if (h < NWX + NWY + NLX + NLY) {
    const int hl = h - (NWX + NWY);
    int row, col;
    if (hl < NLX) {
      const int q = hl % 4;
      row = hl / 4;
      col = q < 2 ? q - 2 : JTX + q - 2;   // −2, −1 | JTX, JTX+1
    } else {
      const int i = (hl - NLX) / JTX;
      row = i < 2 ? i - 2 : JTY + i - 2;
      col = (hl - NLX) % JTX;
    }
    jat_put_l(S, row, col, load_cons(lam, n, cidx(x0 + col, y0 + row)));
  }
  __syncthreads();

  // ---- face VJPs, x faces then y faces in one item list ----
  //   x face (r, ql), ql = 0..JTX+2: between columns ql−2 and ql−1 of row r;
  //   y face (ql, cc), ql = 0..JTY+2: between rows ql−2 and ql−1 of column cc.
#pragma unroll 1
  for (int h = tid; h < JNXF + JNYF; h += JNT) {
    const bool isy = h >= JNXF;
    const int q = isy ? h - JNXF : h;
    int row, col, dr, dc;
    if (!isy) {
      row = q / (JTX + 3);
      col = q % (JTX + 3) - 3;   // cell ql−3 (the face's w0)
      dr = 0;
      dc = 1;
    } else {
      row = q / JTX - 3;
      col = q % JTX;
      dr = 1;
      dc = 0;
    }
    const D5 w0 = jat_w(S, row, col), w1 = jat_w(S, row + dr, col + dc), w2 = jat_w(S, row + 2 * dr, col + 2 * dc),
             w3 = jat_w(S, row + 3 * dr, col + 3 * dc);
    const D5 WL = d5_swap_xy(face_value(w1, slope(w0, w1, w2), 0.5), isy);
    const D5 WR = d5_swap_xy(face_value(w2, slope(w1, w2, w3), -0.5), isy);
    const Cons<double> mu =
        c_swap_xy(mu_of(isy ? G.area[1] : G.area[0], jat_l(S, row + dr, col + dc), jat_l(S, row + 2 * dr, col + 2 * dc)),
                  isy);
    D5 bL = d5_zero(), bR = d5_zero();
    hllc_vjp<0>(WL, WR, g, mu, bL, bR);
    bL = d5_swap_xy(bL, isy);
    bR = d5_swap_xy(bR, isy);
    // No cell gathers the left adjoint of a line's first face or the right one of its last.
    const int f = isy ? q / JTX : q % (JTX + 3);
    const int last = isy ? JTY + 2 : JTX + 2;
    const int gp = isy ? (JTY + 2) * JTX : JTY * (JTX + 2);
    const int o = isy ? q : row * (JTX + 2) + f;
    double* gb = (isy ? &S.Gy[0][0][0][0] : &S.Gx[0][0][0][0]) + o;
    if (f > 0) {
      double* l = gb - (isy ? JTX : 1);
      l[0] = bL.r; l[gp] = bL.vx; l[2 * gp] = bL.vy; l[3 * gp] = bL.vz; l[4 * gp] = bL.p;
    }
    if (f < last) {
      double* r = gb + 5 * gp;
      r[0] = bR.r; r[gp] = bR.vx; r[2 * gp] = bR.vy; r[3 * gp] = bR.vz; r[4 * gp] = bR.p;
    }
  }
  __syncthreads();

  // ---- gather both axes per cell, one component at a time ----
  if (tid >= JTX * JTY || x0 + tx >= nx || y0 + ty >= ny) return;
  D5 Wb = d5_zero();
  double* comp[5] = {&Wb.r, &Wb.vx, &Wb.vy, &Wb.vz, &Wb.p};
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    double w[5], gl[3], gr[3];
#pragma unroll
    for (int k = 0; k < 5; ++k) w[k] = S.W[f][ty + 3][tx + 1 + k];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      gl[k] = S.Gx[0][f][ty][tx + k];
      gr[k] = S.Gx[1][f][ty][tx + k];
    }
    const double vx = gather_line(w, gl, gr, 0.0);
#pragma unroll
    for (int k = 0; k < 5; ++k) w[k] = S.W[f][ty + 1 + k][tx + 3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      gl[k] = S.Gy[0][f][ty + k][tx];
      gr[k] = S.Gy[1][f][ty + k][tx];
    }
    double wb = gather_line(w, gl, gr, vx);
    // The value is complete here: without this the compiler sinks all ten gathers
    // below the last of their loads and holds 130 loaded values in registers.
    asm volatile("" : "+v"(wb)::"memory");
    *comp[f] = wb;
  }
  const Cons<double> Ub = c2p_vjp(Uc, g, Wb);
  const double sc = beta * (*dtp / (1.0 * G.V));
  const double ub[5] = {Ub.d, Ub.mx, Ub.my, Ub.mz, Ub.e};
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    double v = a1 * base1[f * n + c];
    if (base2) v += a2 * base2[f * n + c];
    out[f * n + c] = v + sc * ub[f];
  }
}

}  // namespace VH_PROFILE_NS
}  // namespace vh
