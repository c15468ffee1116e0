// hm_adjoint.hip -- discrete adjoint of the WENO5 + RK4 step (gfx950, FP64).
//
// The reference has no adjoint; this differentiates this library's own
// discretisation of the NavierStokes3D right-hand side by hand, in reverse
// mode: component-wise and characteristic-wise WENO5 (JS, mapped, Z and YC
// weights) with Roe or Rusanov upwinding (the operator of
// src/HyParFunctions/HyperbolicFunction.c:31-222, NavierStokes3DUpwind.c:40-124,
// 349-420), and the viscous term (NavierStokes3DParabolicFunction.c:50-325).
//
// rhs_i = -sum_d dxinv_i (F_{i+1/2} - F_{i-1/2}) along each direction, so the
// adjoint of interface flux F_{i-1/2} is  g = dxinv_i lam_i - dxinv_{i-1} lam_{i-1}.
// The interface-flux VJP spreads g over the 6 stencil cells as a flux-adjoint
// part (later multiplied by the flux Jacobian transpose of the cell, once per
// cell) and a direct solution-adjoint part (WENO of the solution, Rusanov
// speed).  One workgroup owns one or several whole grid lines along the
// direction: the lines' states and fluxes live in LDS (sized to the lines),
// each thread is one interface, and each thread writes its six stencil
// contributions to an LDS record that the owning cells then sum in a fixed
// order, so the result is deterministic.
//
// Within an RK4 step the stage adjoint mu_s = dt b_s lam + dt a_{s+1,s}
// nu_{s+1} is formed on the fly from lam and the previous stage's nu, and
// the last direction adds the finished nu_s into the step adjoint.
//
// Non-smooth points (the max of the Rusanov speeds, |v|) take the derivative
// of the branch the forward evaluation selects.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "hm_device.h"
#include "hm_internal.h"

namespace hm {

constexpr int VJP_LINE_MAX = 512;  // longest grid line an adjoint workgroup holds
constexpr int VJP_CS = 11;         // doubles per cell record of a line VJP: state [5], flux [5], pad
constexpr int VJP_ES = 13;         // doubles per exchange record of the component-wise line VJP: [12], pad
constexpr int VJP_LDS = VJP_CS + VJP_ES;  // doubles of LDS per cell of the component-wise line VJP

__device__ __forceinline__ int wrapn(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// Lines per workgroup of the line VJPs: a block of `threads` threads (a
// multiple of 64, at least n) takes threads / n consecutive lines of length n.
__host__ __device__ __forceinline__ int vjp_lines_per_block(int threads, int n) { return threads / n; }

// Threads of a block for lines of length n: of the blocks of at most 256
// threads the one whose lanes are busiest, the larger of equals.  More lines
// per block leave fewer lanes idle (a 66-cell line alone fills half of two
// wavefronts) and make the y and z lines' accesses of neighbouring lanes
// neighbours in x.  Lines over 256 cells take a block each.  At 256 threads
// the characteristic kernel's LDS (240 B per thread) leaves two blocks per CU,
// the two wavefronts per SIMD its registers allow.
inline int vjp_threads(int n) {
  if (n > 256) return (n + 63) / 64 * 64;
  int best = 0;
  double eff = 0.0;
  for (int t = (n + 63) / 64 * 64; t <= 256; t += 64) {
    const double e = (double)(t / n * n) / t;
    if (e >= eff) {
      eff = e;
      best = t;
    }
  }
  return best;
}

// This thread's place in work item `item` (a group of lines = threads / n
// consecutive lines) of a direction with nlines lines of length n.  Threads
// run through the lines of the group first and along the line second, and so
// do their LDS records: thread r holds cell and interface t of line
// item * lines + r % lines in record r, and the record k places further along
// the line is r + k lines, wrapped at size = lines * n.  live is false for
// threads past the group's last line.
struct LineSlot {
  size_t line;
  int t, r, lines, size;
  bool live;
  __device__ __forceinline__ int at(int k) const {
    const int i = r + k * lines;
    return i < 0 ? i + size : (i >= size ? i - size : i);
  }
};
__device__ __forceinline__ LineSlot line_slot(size_t item, int n, size_t nlines) {
  LineSlot s;
  s.lines = vjp_lines_per_block((int)blockDim.x, n);
  s.size = s.lines * n;
  const int r = (int)threadIdx.x, t = r / s.lines;
  s.line = item * s.lines + (r - t * s.lines);
  s.live = r < s.size && s.line < nlines;
  s.t = s.live ? t : 0;
  s.r = s.live ? r : 0;
  if (!s.live) s.line = 0;
  return s;
}

// One side of WENO5 in the form of hm_pass.hip: from l_k = 3/4 (beta_k + eps)
// and the candidates' differences p_k from the upwind cell's value (times 2,
// 12, 6), c = twice the difference of the interpolated value from that cell's
// value, and the reverse of it: ob times the derivative of c with respect to
// p_k (w1..w3), l_k (g1..g3) and, for the YC weights, the stencil's 4th
// difference d4 (gt).  W selects the weights
// (include/interpolation.h:265-285, 314-341, 426-447, 479-500).  With
// q_k = the product of the other two l, h_k = p_k - kappa_k c,
// kappa = 1, 6, 3, and N, A the sums of a_k p_k and kappa_k a_k:
//  * JS:     a_k = q_k^2;              d c/d l_k = -2 a_k h_k/(l_k A)
//  * Z, YC:  a_k = q_k^2 (l_k^2 + t^2), t = l_3 - l_1 (Z) or 3/4 d4^2 (YC);
//            d c/d l_k = -2 t^2 q_k^2 h_k/(l_k A), and t's own derivative
//            2 t sum(q_k^2 h_k)/A goes into g1, g3 (Z) or gt (YC)
//  * mapped: the JS weights u_k mapped by u (c + c^2 - 3 c u + u^2)/
//            (c^2 + u (1 - 2c)) and renormalised; the adjoint goes back
//            through the mapping and the JS normalisation
//  * optimal (no_limiting): the constant weights 0.1, 0.6, 0.3
// (sum a_k h_k = 0 takes the cross terms out.)  One reciprocal of
// A l_1 l_2 l_3 gives 1/A and 1/(l_1 l_2 l_3); the mapped weights take a second
// one for the mapping.  The reciprocal itself, l^-7 or l^-9, is as large as
// 1e280 for an epsilon of 1e-40 in a uniform region: ob multiplies 1/A alone.
struct W5Side {
  double c, w1, w2, w3, g1, g2, g3, gt;
};

template <int W>
__device__ __forceinline__ W5Side w5_side(double l1, double l2, double l3, double p1, double p2, double p3, double d4,
                                          double ob) {
  W5Side r;
  r.gt = 0.0;
  if (W == WENO_OPTIMAL) {
    r.c = 0.1 * (p1 + p2 + p3);
    r.w1 = r.w2 = r.w3 = 0.1 * ob;
    r.g1 = r.g2 = r.g3 = 0.0;
    return r;
  }
  const double q1 = l2 * l3, q2 = l1 * l3, q3 = l1 * l2, P = l1 * q1;
  const double s1 = q1 * q1, s2 = q2 * q2, s3 = q3 * q3;
  if (W == WENO_MAPPED) {
    const double c1 = 0.1, c2 = 0.6, c3 = 0.3;
    const double A = s1 + 3.0 * (2.0 * s2 + s3);
    const double q = nr_rcp(A * P);
    const double it = q * P;
    const double u1 = s1 * it, u2 = s2 * (6.0 * it), u3 = s3 * (3.0 * it);  // JS weights
    const double N1 = c1 + c1 * c1 - 3 * c1 * u1 + u1 * u1, D1 = c1 * c1 + u1 * (1.0 - 2.0 * c1);
    const double N2 = c2 + c2 * c2 - 3 * c2 * u2 + u2 * u2, D2 = c2 * c2 + u2 * (1.0 - 2.0 * c2);
    const double N3 = c3 + c3 * c3 - 3 * c3 * u3 + u3 * u3, D3 = c3 * c3 + u3 * (1.0 - 2.0 * c3);
    const double o1 = D2 * D3, o2 = D1 * D3, o3 = D1 * D2, DD = D1 * o1;
    const double B1 = u1 * N1 * o1, B2 = u2 * N2 * o2, B3 = u3 * N3 * o3, B = B1 + B2 + B3;
    const double qm = nr_rcp(B * DD);
    const double im = qm * DD;
    const double f1 = p1, f2 = (1.0 / 6.0) * p2, f3 = (1.0 / 3.0) * p3;
    const double w1 = B1 * im, w2 = B2 * im, w3 = B3 * im;
    r.c = w1 * f1 + w2 * f2 + w3 * f3;
    r.w1 = ob * w1;
    r.w2 = ob * w2 * (1.0 / 6.0);
    r.w3 = ob * w3 * (1.0 / 3.0);
    // d c/d a_k = DD (f_k - c)/B with a_k = u_k N_k/D_k, whose derivative
    // is ((N_k + u_k N_k') D_k - u_k N_k D_k')/D_k^2; DD/(B D_k^2) = o_k^2 qm
    const double h1 = ob * (f1 - r.c), h2 = ob * (f2 - r.c), h3 = ob * (f3 - r.c);
    const double du1 = h1 * ((N1 + u1 * (2 * u1 - 3 * c1)) * D1 - u1 * N1 * (1.0 - 2.0 * c1)) * (o1 * o1) * qm;
    const double du2 = h2 * ((N2 + u2 * (2 * u2 - 3 * c2)) * D2 - u2 * N2 * (1.0 - 2.0 * c2)) * (o2 * o2) * qm;
    const double du3 = h3 * ((N3 + u3 * (2 * u3 - 3 * c3)) * D3 - u3 * N3 * (1.0 - 2.0 * c3)) * (o3 * o3) * qm;
    // through u_k = at_k/sum at, at_k = c_k/l_k^2
    const double U = du1 * u1 + du2 * u2 + du3 * u3, iP = -2.0 * (q * A);
    r.g1 = (du1 - U) * u1 * q1 * iP;
    r.g2 = (du2 - U) * u2 * q2 * iP;
    r.g3 = (du3 - U) * u3 * q3 * iP;
    return r;
  }
  double a1 = s1, a2 = s2, a3 = s3, t = 0.0, t2 = 1.0;
  if (W != WENO_JS) {
    t = W == WENO_Z ? l3 - l1 : 0.75 * (d4 * d4);
    t2 = t * t;
    a1 *= l1 * l1 + t2;
    a2 *= l2 * l2 + t2;
    a3 *= l3 * l3 + t2;
  }
  const double A = a1 + scalar(3.0) * (2.0 * a2 + a3);
  const double q = nr_rcp(A * P);
  const double inv = q * P;
  r.c = (a1 * p1 + a2 * p2 + a3 * p3) * inv;
  const double oi = ob * inv, k = -2.0 * (W == WENO_JS ? q * A : t2 * (q * A));
  r.w1 = a1 * oi;
  r.w2 = a2 * oi;
  r.w3 = a3 * oi;
  const double h1 = (W == WENO_JS ? r.w1 : s1 * oi) * (p1 - r.c);
  const double h2 = (W == WENO_JS ? r.w2 : s2 * oi) * (p2 - 6.0 * r.c);
  const double h3 = (W == WENO_JS ? r.w3 : s3 * oi) * (p3 - 3.0 * r.c);
  r.g1 = k * (q1 * h1);
  r.g2 = k * (q2 * h2);
  r.g3 = k * (q3 * h3);
  if (W != WENO_JS) {
    const double gt = 2.0 * t * (h1 + h2 + h3);
    if (W == WENO_Z) {
      r.g3 += gt;
      r.g1 -= gt;
    } else {
      r.gt = 1.5 * d4 * gt;
    }
  }
  return r;
}

// reverse of the left- and right-biased WENO5 of one interface, as functions
// of the five first differences D of cells I-3..I+2 (the values themselves
// enter only as b[2] and b[3], which the caller takes back): sets G to
// obL d vl/d D + obR d vr/d D and returns jump = (vr - b[3]) - (vl - b[2]) +
// D[2] = vr - vl and corr = (vl - b[2]) + (vr - b[3]).  e are the second
// differences; the indicators are those of hm_pass.hip
// (l = e^2 + 3/4 x (x + e) and e^2 + 3/4 x y).  G may be D.
template <int W>
__device__ __forceinline__ void weno5_lr_vjp(const double (&D)[5], double eps34, double obL, double obR,
                                             double (&G)[5], double &jump, double &corr) {
  const double D1 = D[1], D2 = D[2], D3 = D[3];
  const double e0 = D1 - D[0], e1 = D2 - D1, e2 = D3 - D2, e3 = D[4] - D3;
  const double s0 = e0 * e0 + eps34, s1 = e1 * e1 + eps34, s2 = e2 * e2 + eps34, s3 = e3 * e3 + eps34;
  const double k34 = scalar(0.75), k23 = scalar(2.0 / 3.0);
  const double x1 = k34 * D1, x2 = k34 * D2, x3 = k34 * D3, F = 4.0 * D2;
  const W5Side L = w5_side<W>(x1 * (D1 + e0) + s0, x1 * D2 + s1, x2 * (D2 - e2) + s2, k23 * e0 + D1, 2.0 * D1 + F,
                              F - D3, (e0 + e2) - 2.0 * e1, 0.5 * obL);
  const W5Side R = w5_side<W>(x3 * (D3 - e3) + s3, x3 * D2 + s2, x2 * (D2 + e1) + s1, D3 - k23 * e3, 2.0 * D3 + F,
                              F - D1, (e1 + e3) - 2.0 * e2, -0.5 * obR);
  jump = D2 - 0.5 * (R.c + L.c);
  corr = 0.5 * (L.c - R.c);
  // onto the e and, beside them, the D
  double E0 = L.g1 * (2.0 * e0 + x1) + k23 * L.w1;
  double E1 = 2.0 * e1 * (L.g2 + R.g3) + x2 * R.g3;
  double E2 = 2.0 * e2 * (L.g3 + R.g2) - x2 * L.g3;
  double E3 = R.g1 * (2.0 * e3 - x3) - k23 * R.w1;
  const double B1 = L.g1 * (k34 * e0 + 2.0 * x1) + L.g2 * x2 + (L.w1 + 2.0 * L.w2 - R.w3);
  const double B2 = L.g2 * x1 + L.g3 * (2.0 * x2 - k34 * e2) + R.g3 * (k34 * e1 + 2.0 * x2) + R.g2 * x3 +
                    4.0 * ((L.w2 + L.w3) + (R.w2 + R.w3));
  const double B3 = R.g1 * (2.0 * x3 - k34 * e3) + R.g2 * x2 + (R.w1 + 2.0 * R.w2 - L.w3);
  if (W == WENO_YC) {
    E0 += L.gt;
    E1 += R.gt - 2.0 * L.gt;
    E2 += L.gt - 2.0 * R.gt;
    E3 += R.gt;
  }
  G[0] = -E0;
  G[1] = B1 + E0 - E1;
  G[2] = B2 + E1 - E2;
  G[3] = B3 + E2 - E3;
  G[4] = E3;
}

// gradient of c + |v_d| of one state with respect to its conserved variables
template <int DIR>
__device__ __forceinline__ void speed_vjp(const double *u, double gamma, double ab, double ub[NV]) {
  const double gm1 = gamma - 1.0;
  const double rho = u[0], ir = nr_rcp(rho);
  const double v[3] = {u[1] * ir, u[2] * ir, u[3] * ir};
  const double q2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  const double Por = gm1 * (u[4] * ir - 0.5 * q2);  // P / rho
  const double k = (0.5 * ab * gamma) * nr_rsq(gamma * Por);  // d a / d(P/rho)
  ub[0] += k * gm1 * (-u[4] * ir * ir + q2 * ir);
  for (int j = 0; j < 3; j++) ub[1 + j] += k * gm1 * (-v[j] * ir);
  ub[4] += k * gm1 * ir;
  const double vn = v[DIR];
  const double sg = vn > 0 ? 1.0 : (vn < 0 ? -1.0 : 0.0);
  ub[0] += ab * (-sg * vn * ir);
  ub[1 + DIR] += ab * (sg * ir);
}

// adjoint of the Roe-averaged velocity (gv) and total enthalpy (gH) of
// (uL, uR) onto the two states (navierstokes3d.h:144-169)
__device__ __forceinline__ void roe_avg_vjp(const double *uL, const double *uR, double gamma, const double gv[3],
                                            double gH, double ubL[NV], double ubR[NV]) {
  const double gm1 = gamma - 1.0;
  const double *U[2] = {uL, uR};
  double t[2], v[2][3], H[2], rho[2], q2[2], ird[2], rt[2];
  for (int s = 0; s < 2; s++) {
    rho[s] = U[s][0];
    const double ir = nr_rcp(rho[s]);
    ird[s] = ir;
    for (int j = 0; j < 3; j++) v[s][j] = U[s][1 + j] * ir;
    q2[s] = v[s][0] * v[s][0] + v[s][1] * v[s][1] + v[s][2] * v[s][2];
    H[s] = gamma * U[s][4] * ir - gm1 * 0.5 * q2[s];
    rt[s] = nr_rsq(rho[s]);
    t[s] = sqrt_of(rho[s], rt[s]);
  }
  const double den = nr_rcp(t[0] + t[1]);
  double va[3];
  for (int j = 0; j < 3; j++) va[j] = (t[0] * v[0][j] + t[1] * v[1][j]) * den;
  const double Ha = (t[0] * H[0] + t[1] * H[1]) * den;
  double *UB[2] = {ubL, ubR};
  for (int s = 0; s < 2; s++) {
    const double w = t[s] * den, ir = ird[s];
    double gt = gH * (H[s] - Ha) * den;
    for (int j = 0; j < 3; j++) gt += gv[j] * (v[s][j] - va[j]) * den;
    const double gHs = gH * w;
    double gvs[3];
    for (int j = 0; j < 3; j++) gvs[j] = gv[j] * w;
    UB[s][0] += 0.5 * gt * rt[s] + gHs * (-gamma * U[s][4] * ir * ir + gm1 * q2[s] * ir);
    for (int j = 0; j < 3; j++) {
      UB[s][0] += gvs[j] * (-v[s][j] * ir);
      UB[s][1 + j] += gvs[j] * ir + gHs * (-gm1 * v[s][j] * ir);
    }
    UB[s][4] += gHs * gamma * ir;
  }
}

// gradient of c + |v_d| of the Roe average of (uL, uR)
template <int DIR>
__device__ __forceinline__ void roe_speed_vjp(const double *uL, const double *uR, double gamma, double ab,
                                              double ubL[NV], double ubR[NV]) {
  const double gm1 = gamma - 1.0;
  double va[3], Ha;
  {
    double t[2], v[2][3], H[2];
    const double *U[2] = {uL, uR};
    for (int s = 0; s < 2; s++) {
      const double ir = nr_rcp(U[s][0]);
      for (int j = 0; j < 3; j++) v[s][j] = U[s][1 + j] * ir;
      H[s] = gamma * U[s][4] * ir - gm1 * 0.5 * (v[s][0] * v[s][0] + v[s][1] * v[s][1] + v[s][2] * v[s][2]);
      t[s] = nr_sqrt(U[s][0]);
    }
    const double den = nr_rcp(t[0] + t[1]);
    for (int j = 0; j < 3; j++) va[j] = (t[0] * v[0][j] + t[1] * v[1][j]) * den;
    Ha = (t[0] * H[0] + t[1] * H[1]) * den;
  }
  const double gH = 0.5 * ab * gm1 * nr_rsq(gm1 * (Ha - 0.5 * (va[0] * va[0] + va[1] * va[1] + va[2] * va[2])));
  double gv[3];
  for (int j = 0; j < 3; j++) gv[j] = -gH * va[j];
  const double sg = va[DIR] > 0 ? 1.0 : (va[DIR] < 0 ? -1.0 : 0.0);
  gv[DIR] += ab * sg;
  roe_avg_vjp(uL, uR, gamma, gv, gH, ubL, ubR);
}

// Euler flux along DIR of a cell's state (navierstokes3d.h:118-139).  As in
// the forward passes a cell without mass has no velocity: its flux enters the
// stencils of the interfaces around it and has to be finite.
template <int DIR>
__device__ __forceinline__ void vjp_flux(const double *u, double gamma, double f[NV]) {
  const double ir = u[0] == 0.0 ? 0.0 : nr_rcp(u[0]);
  const double v[3] = {u[1] * ir, u[2] * ir, u[3] * ir};
  const double P = (gamma - 1.0) * (u[4] - 0.5 * u[0] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
  f[0] = u[1 + DIR];
  for (int j = 0; j < 3; j++) f[1 + j] = u[1 + DIR] * v[j];
  f[1 + DIR] += P;
  f[4] = (u[4] + P) * v[DIR];
}

// c + |v_d| of one state
template <int DIR>
__device__ __forceinline__ double vjp_speed(const double *u, double gamma) {
  const double ir = nr_rcp(u[0]);
  const double v[3] = {u[1] * ir, u[2] * ir, u[3] * ir};
  const double q2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  return nr_sqrt(gamma * (gamma - 1.0) * (u[4] * ir - 0.5 * q2)) + fabs(v[DIR]);
}

// ub += A(u)^T fb, A = d(Euler flux along DIR)/d(conserved variables)
template <int DIR>
__device__ __forceinline__ void flux_jac_T(const double *u, double gamma, const double fb[NV], double ub[NV]) {
  const double gm1 = gamma - 1.0;
  const double rho = u[0], ir = nr_rcp(rho);
  const double v[3] = {u[1] * ir, u[2] * ir, u[3] * ir};
  const double q2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  const double P = gm1 * (u[4] - 0.5 * rho * q2);
  const double H = (u[4] + P) * ir;
  const double vn = v[DIR];
  double fm = 0.0;  // sum_i fb_{1+i} v_i
  for (int i = 0; i < 3; i++) fm += fb[1 + i] * v[i];
  ub[0] += -vn * fm + fb[1 + DIR] * gm1 * 0.5 * q2 + fb[4] * vn * (gm1 * 0.5 * q2 - H);
  for (int j = 0; j < 3; j++)
    ub[1 + j] += fb[1 + j] * vn - fb[1 + DIR] * gm1 * v[j] - fb[4] * gm1 * v[j] * vn;
  ub[1 + DIR] += fb[0] + fm + fb[4] * H;
  ub[4] += fb[1 + DIR] * gm1 + fb[4] * gamma * vn;
}

// Roe state of an interface for the adjoints of Roe upwinding and of the
// characteristic scheme, and the rows of L with their derivatives
struct RoeAdj {
  double v[3], vn, a, a2, ia, ia2, ek, h0;  // h0 = a^2/(gamma-1) + ek = the averaged enthalpy
};

template <int DIR>
__device__ __forceinline__ RoeAdj roe_adj_state(const double uL[NV], const double uR[NV], double gamma) {
  const double gm1 = gamma - 1.0;
  RoeAdj s;
  const double iL = nr_rcp(uL[0]), iR = nr_rcp(uR[0]);
  double vL[3], vR[3];
  for (int j = 0; j < 3; j++) { vL[j] = uL[1 + j] * iL; vR[j] = uR[1 + j] * iR; }
  const double qL = vL[0] * vL[0] + vL[1] * vL[1] + vL[2] * vL[2];
  const double qR = vR[0] * vR[0] + vR[1] * vR[1] + vR[2] * vR[2];
  const double HL = gamma * uL[4] * iL - gm1 * 0.5 * qL, HR = gamma * uR[4] * iR - gm1 * 0.5 * qR;
  const double tL = nr_sqrt(uL[0]), tR = nr_sqrt(uR[0]), den = nr_rcp(tL + tR);
  for (int j = 0; j < 3; j++) s.v[j] = (tL * vL[j] + tR * vR[j]) * den;
  const double H = (tL * HL + tR * HR) * den;
  s.ek = 0.5 * (s.v[0] * s.v[0] + s.v[1] * s.v[1] + s.v[2] * s.v[2]);
  s.a2 = (H - s.ek) * gm1;
  s.ia = nr_rsq(s.a2);
  s.a = sqrt_of(s.a2, s.ia);
  s.ia2 = s.ia * s.ia;
  s.vn = s.v[DIR];
  s.h0 = H;
  return s;
}

// row k of L at the Roe state: k = 0 entropy, 1 u-a, 2 u+a, 3 and 4 the two
// shear rows in row order (navierstokes3d.h:288-374)
template <int DIR>
__device__ __forceinline__ void l_row(const RoeAdj &s, double gm1, int k, double r[NV]) {
  if (k <= 2) {
    const double ia2 = s.ia2;
    if (k == 0) {
      r[0] = (s.a2 - gm1 * s.ek) * ia2;
      for (int j = 0; j < 3; j++) r[1 + j] = gm1 * s.v[j] * ia2;
      r[4] = -gm1 * ia2;
    } else {
      const double h = 0.5 * ia2, sg = k == 1 ? 1.0 : -1.0;
      r[0] = (gm1 * s.ek + sg * s.a * s.vn) * h;
      for (int j = 0; j < 3; j++) r[1 + j] = -gm1 * s.v[j] * h;
      r[1 + DIR] -= sg * s.a * h;
      r[4] = gm1 * h;
    }
    return;
  }
  for (int j = 0; j < NV; j++) r[j] = 0.0;
  if (DIR == 0) {
    if (k == 3) { r[0] = s.v[1]; r[2] = -1.0; } else { r[0] = -s.v[2]; r[3] = 1.0; }
  } else if (DIR == 1) {
    if (k == 3) { r[0] = -s.v[0]; r[1] = 1.0; } else { r[0] = s.v[2]; r[3] = -1.0; }
  } else {
    if (k == 3) { r[0] = s.v[0]; r[1] = -1.0; } else { r[0] = -s.v[1]; r[2] = 1.0; }
  }
}

// adds (d row_k / d(v, a))^T X to (gv, ab): the Roe-state derivative of
// sum_p (adjoint of the projection at p) * (row_k . x_p), X = the adjoint-
// weighted sum of the projected vectors
template <int DIR>
__device__ __forceinline__ void l_row_vjp(const RoeAdj &s, double gm1, int k, const double X[NV], double gv[3],
                                          double &ab) {
  const double a = s.a, ia2 = s.ia2, ia = s.ia, ia3 = ia2 * ia;
  const double vX = s.v[0] * X[1] + s.v[1] * X[2] + s.v[2] * X[3];
  if (k == 0) {
    for (int j = 0; j < 3; j++) gv[j] += gm1 * ia2 * (X[1 + j] - X[0] * s.v[j]);
    ab += 2.0 * gm1 * ia3 * (X[0] * s.ek - vX + X[4]);
  } else if (k <= 2) {
    const double sg = k == 1 ? 1.0 : -1.0, h = 0.5 * ia2;
    for (int j = 0; j < 3; j++) gv[j] += gm1 * h * (X[0] * s.v[j] - X[1 + j]);
    gv[DIR] += sg * a * h * X[0];
    ab += -X[0] * (2.0 * gm1 * s.ek + sg * a * s.vn) * h * ia + gm1 * ia3 * (vX - X[4]) + sg * h * X[1 + DIR];
  } else if (DIR == 0) {
    if (k == 3) gv[1] += X[0]; else gv[2] -= X[0];
  } else if (DIR == 1) {
    if (k == 3) gv[0] -= X[0]; else gv[2] += X[0];
  } else {
    if (k == 3) gv[0] += X[0]; else gv[1] -= X[0];
  }
}

// derivative of harten
__device__ __forceinline__ double harten_d(double l) {
  const double delta = 0.000001;
  return fmin(fmax(l * (1.0 / delta), -1.0), 1.0);
}

// nu (+)= (d rhs_DIR / d u)^T mu along one direction, one workgroup per group
// of lines (LineSlot), with mu = cb*lam + ca*nu_in (nu_in may be null).  mode
// VJP_WRITE stores, VJP_ADD accumulates into nu, VJP_ADD_L accumulates into nu
// and adds the finished nu into L, VJP_ADD_LSET sets L = lam + the finished nu.
// LDS (dynamic, VJP_LDS = 24 doubles per cell of the lines): a record per cell
// of its state [5] and flux [5], and one per interface of the stencil
// contributions of the flux and solution adjoints [6] each, both of odd length
// so that neighbouring records start in other banks.
enum { VJP_WRITE = 0, VJP_ADD = 1, VJP_ADD_L = 2, VJP_ADD_LSET = 3 };

// state, lam and (when given) nu_in of cell c, every load issued before any
// is used: a null check inside the variable loop would put a wait in each
// iteration
__device__ __forceinline__ void vjp_load_cell(const double *__restrict__ u, const double *__restrict__ lam,
                                              const double *__restrict__ nu_in, size_t ncell, size_t c,
                                              double (&us)[NV], double (&lm)[NV], double (&ni)[NV]) {
#pragma unroll
  for (int v = 0; v < NV; v++) {
    us[v] = u[(size_t)v * ncell + c];
    lm[v] = lam[(size_t)v * ncell + c];
    ni[v] = 0.0;
  }
  if (nu_in)
#pragma unroll
    for (int v = 0; v < NV; v++) ni[v] = nu_in[(size_t)v * ncell + c];
}

// weight of F(r+s) in D at reader r, s = -2, -1, +1, +2
__device__ __forceinline__ double d4w(int s) {
  return s == -2 ? 1.0 / 12.0 : (s == -1 ? -8.0 / 12.0 : (s == 1 ? 8.0 / 12.0 : -1.0 / 12.0));
}

// The viscous term's share of the adjoint of cell idx, (d par/d u)^T mu: QB
// plus the transposed gradient stencils over GB, then back through
// (u, v, w, T)(u) at the cell's state us (NavierStokes3DParabolicFunction.c:
// 85-108).  QB and GB are complete once the tile and ghost-layer kernels of
// the viscous adjoint have run; the x line VJP, which runs after them, adds
// this share into nu together with its own.
__device__ __forceinline__ void visc_gather_cell(const double (&us)[NV], const double *__restrict__ QB,
                                                 const double *__restrict__ GB, int nx, int ny, int nz,
                                                 double gamma, size_t idx, double (&ub)[NV]) {
  const size_t ncell = (size_t)nx * ny * nz;
  const int n[3] = {nx, ny, nz};
  const int pos[3] = {(int)(idx % nx), (int)((idx / nx) % ny), (int)(idx / ((size_t)nx * ny))};
  const size_t st[3] = {1, (size_t)nx, (size_t)nx * ny};
  double qb[4];
#pragma unroll
  for (int c = 0; c < 4; c++) qb[c] = QB[(size_t)c * ncell + idx];
  const int offs[4] = {-2, -1, 1, 2};
#pragma unroll
  for (int e = 0; e < 3; e++) {
    const size_t line0 = idx - (size_t)pos[e] * st[e];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      // reader j = m - s reads this cell with weight d4w(s) (periodic)
      const size_t j = line0 + (size_t)wrapn(pos[e] - offs[s], n[e]) * st[e];
      const double w = d4w(offs[s]);
#pragma unroll
      for (int c = 0; c < 4; c++) qb[c] += w * GB[(size_t)(c * 3 + e) * ncell + j];
    }
  }
  const double gm1 = gamma - 1.0;
  const double ir = nr_rcp(us[0]);
  const double vx = us[1] * ir, vy = us[2] * ir, vz = us[3] * ir;
  const double q2 = vx * vx + vy * vy + vz * vz;
  const double k = gamma * gm1 * qb[3];  // T = gamma (gamma-1) (e/rho - |m|^2/(2 rho^2))
  ub[0] = -(qb[0] * vx + qb[1] * vy + qb[2] * vz) * ir + k * (-us[4] * ir * ir + q2 * ir);
  ub[1] = qb[0] * ir - k * vx * ir;
  ub[2] = qb[1] * ir - k * vy * ir;
  ub[3] = qb[2] * ir - k * vz * ir;
  ub[4] = k * ir;
}

// the finished adjoint acc of cell c into nu (and L) by mode, after the
// viscous share vb when has_vb: nu = (nu + vb) + acc, the order of a
// separate viscous pass that adds vb before this one.  Every load issues
// before the first store, so that the stores (nu, L and lam may alias as
// far as the compiler knows) do not serialise the loads
__device__ __forceinline__ void vjp_store(double *__restrict__ nu, double *__restrict__ L,
                                          const double *__restrict__ lam, int mode, size_t ncell, size_t c,
                                          const double (&acc)[NV], bool has_vb, const double (&vb)[NV]) {
  if (mode == VJP_WRITE) {
#pragma unroll
    for (int v = 0; v < NV; v++) nu[(size_t)v * ncell + c] = has_vb ? vb[v] + acc[v] : acc[v];
    return;
  }
  double r[NV], l[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < NV; v++) r[v] = nu[(size_t)v * ncell + c];
  if (mode == VJP_ADD_L) {
#pragma unroll
    for (int v = 0; v < NV; v++) l[v] = L[(size_t)v * ncell + c];
  } else if (mode == VJP_ADD_LSET) {
#pragma unroll
    for (int v = 0; v < NV; v++) l[v] = lam[(size_t)v * ncell + c];
  }
  if (has_vb)
#pragma unroll
    for (int v = 0; v < NV; v++) r[v] = r[v] + vb[v];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    r[v] = r[v] + acc[v];
    nu[(size_t)v * ncell + c] = r[v];
  }
  if (mode == VJP_ADD_L || mode == VJP_ADD_LSET)
#pragma unroll
    for (int v = 0; v < NV; v++) L[(size_t)v * ncell + c] = l[v] + r[v];
}

template <int DIR, int UPW, int W, bool VG = false>
__device__ __forceinline__ void rhs_vjp_line(const double *__restrict__ u, const double *__restrict__ lam,
                                             const double *__restrict__ nu_in, double ca, double cb,
                                             double *__restrict__ nu, double *__restrict__ L, int mode, int nx,
                                             int ny, int nz, const double *__restrict__ dxg, double gamma,
                                             double eps, const double *__restrict__ QB,
                                             const double *__restrict__ GB, const LineSlot &sl, double *smem) {
  const size_t line = sl.line;
  const int t = sl.t, r0 = sl.r;
  const bool active = sl.live;
  const size_t ncell = (size_t)nx * ny * nz;
  size_t base, stride;
  if (DIR == 0) { base = line * nx; stride = 1; }
  else if (DIR == 1) { base = (line % nx) + (line / nx) * (size_t)nx * ny; stride = nx; }
  else { base = line; stride = (size_t)nx * ny; }
  const double *dxd = dxg + 3 + (DIR >= 1 ? nx + 6 : 0) + (DIR == 2 ? ny + 6 : 0);
  constexpr int CS = VJP_CS, ES = VJP_ES;
  double *sC = smem;        // [sl.size][CS]: state [5], flux [5]
  double *E = sC + CS * sl.size;  // [sl.size][ES]
  const double eps34 = 0.75 * eps;
  double g[NV] = {0, 0, 0, 0, 0};
  if (active) {
    const size_t c = base + (size_t)t * stride;
    double us[NV], lm[NV], ni[NV];
    vjp_load_cell(u, lam, nu_in, ncell, c, us, lm, ni);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      sC[r0 * CS + v] = us[v];
      // dxinv mu of this cell, staged in the (not yet used) exchange buffer
      E[r0 * ES + v] = dxd[t] * (cb * lm[v] + (nu_in ? ca * ni[v] : 0.0));
    }
    double fl[NV];
    vjp_flux<DIR>(us, gamma, fl);
#pragma unroll
    for (int v = 0; v < NV; v++) sC[r0 * CS + NV + v] = fl[v];
  }
  __syncthreads();
  if (active)
#pragma unroll
    for (int v = 0; v < NV; v++) g[v] = E[r0 * ES + v] - E[sl.at(-1) * ES + v];
  __syncthreads();
  const double *cs[6];  // records of the stencil's cells
  const double *ei[6];  // exchange records that touch this cell: slot s of interface t+3-s
#pragma unroll
  for (int s = 0; s < 6; s++) {
    cs[s] = sC + sl.at(s - 3) * CS;
    ei[s] = E + sl.at(3 - s) * ES + s;
  }
  double alpha = 0.0, abar = 0.0;
  int sel = 0;
  // Roe: d = R |Lambda| L du with du = (uR - uL)/2 and fI = fh - d
  // (NavierStokes3DUpwind.c:40-124); wR = A^T lambda_F, A = R |Lambda| L,
  // so that the solution WENO adjoints are -/+ wR/2
  double wR[NV] = {0, 0, 0, 0, 0}, du[NV] = {0, 0, 0, 0, 0};
  if (active && UPW == UPWIND_ROE) {
    double u2[NV], u3[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) { u2[v] = cs[2][v]; u3[v] = cs[3][v]; }
    const RoeAdj s = roe_adj_state<DIR>(u2, u3, gamma);
    const double gm1 = gamma - 1.0;
    const double eb = g[4];
    const double sumb = g[0] + s.v[0] * g[1] + s.v[1] * g[2] + s.v[2] * g[3];
    const double difb = g[1 + DIR] + s.vn * eb;
    double lg[5];  // (R^T lambda_F)_k |lambda_k|
    lg[0] = (sumb + s.ek * eb) * harten(s.vn);
    lg[1] = (sumb + s.h0 * eb - s.a * difb) * harten(s.vn - s.a);
    lg[2] = (sumb + s.h0 * eb + s.a * difb) * harten(s.vn + s.a);
    if (DIR == 0) { lg[3] = -g[2] - s.v[1] * eb; lg[4] = g[3] + s.v[2] * eb; }
    else if (DIR == 1) { lg[3] = g[1] + s.v[0] * eb; lg[4] = -g[3] - s.v[2] * eb; }
    else { lg[3] = -g[1] - s.v[0] * eb; lg[4] = g[2] + s.v[1] * eb; }
    lg[3] *= harten(s.vn);
    lg[4] *= harten(s.vn);
#pragma unroll 1
    for (int k = 0; k < 5; k++) {
      double row[NV];
      l_row<DIR>(s, gm1, k, row);
      const double c = k == 0 ? lg[0] : (k == 1 ? lg[1] : (k == 2 ? lg[2] : (k == 3 ? lg[3] : lg[4])));
#pragma unroll
      for (int v = 0; v < NV; v++) wR[v] += c * row[v];
    }
  }
  if (active && UPW == UPWIND_RUSANOV) {
    double u2[NV], u3[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) { u2[v] = cs[2][v]; u3[v] = cs[3][v]; }
    const double aL = vjp_speed<DIR>(u2, gamma), aR = vjp_speed<DIR>(u3, gamma);
    const RoeAdj a = roe_adj_state<DIR>(u2, u3, gamma);
    const double aA = a.a + fabs(a.vn);
    const double m01 = fmax(aL, aR), m12 = fmax(aR, aA);
    alpha = fmax(m01, m12);
    // alpha = max(max(aL,aR), max(aR,aA)): derivative of the selected term
    sel = m01 >= m12 ? (aL >= aR ? 0 : 1) : (aR >= aA ? 1 : 2);
  }
  double accF[NV], accU[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    if (active) {
      double D[5], G[5], jump, corr;
      double *e = E + r0 * ES;
#pragma unroll
      for (int part = 0; part < 2; part++) {
        // the flux, then the solution; slot s of interface t belongs to cell
        // t-3+s and takes the adjoints of the two differences next to it
#pragma unroll
        for (int s = 0; s < 5; s++) D[s] = cs[s + 1][part == 0 ? NV + v : v] - cs[s][part == 0 ? NV + v : v];
        if (part == 0) {
          weno5_lr_vjp<W>(D, eps34, 0.5 * g[v], 0.5 * g[v], G, jump, corr);
        } else {
          const double ob = UPW == UPWIND_ROE ? 0.5 * wR[v] : 0.5 * alpha * g[v];
          weno5_lr_vjp<W>(D, eps34, ob, -ob, G, jump, corr);
          G[2] -= ob;
          if (UPW == UPWIND_ROE) du[v] = 0.5 * jump;
          else abar += -0.5 * jump * g[v];
        }
        const double mean = part == 0 ? 0.5 * g[v] : 0.0;  // the mean of the two cells' fluxes
#pragma unroll
        for (int s = 0; s < 6; s++)
          e[6 * part + s] = (s > 0 ? G[s - 1] : 0.0) - (s < 5 ? G[s] : 0.0) + (s == 2 || s == 3 ? mean : 0.0);
      }
    }
    __syncthreads();
    // cell t sums slot s of interface t+3-s, s = 0..5, in that order
    accF[v] = accU[v] = 0.0;
    if (active) {
#pragma unroll
      for (int s = 0; s < 6; s++) {
        accF[v] += ei[s][0];
        accU[v] += ei[s][6];
      }
    }
    __syncthreads();
  }
  // adjoint of the upwinding's dependence on the two cells next to interface
  // t, cell t-1 (entries 0..4) and cell t (5..9): the Rusanov speed, or
  // the Roe state inside R |Lambda| L
  if (active) {
    double u2[NV], u3[NV], ub2[NV] = {0, 0, 0, 0, 0}, ub3[NV] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int v = 0; v < NV; v++) { u2[v] = cs[2][v]; u3[v] = cs[3][v]; }
    if (UPW == UPWIND_ROE) {
      const RoeAdj s = roe_adj_state<DIR>(u2, u3, gamma);
      const double gm1 = gamma - 1.0, igm1 = nr_rcp(gm1);
      // adjoint of d is -lambda_F; lambda_g = R^T (-lambda_F)
      double ld[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) ld[v] = -g[v];
      const double eb = ld[4];
      const double sumb = ld[0] + s.v[0] * ld[1] + s.v[1] * ld[2] + s.v[2] * ld[3];
      const double difb = ld[1 + DIR] + s.vn * eb;
      double lgk[5], lam_k[5], gk[5], pk[5];
      lgk[0] = sumb + s.ek * eb;
      lgk[1] = sumb + s.h0 * eb - s.a * difb;
      lgk[2] = sumb + s.h0 * eb + s.a * difb;
      if (DIR == 0) { lgk[3] = -ld[2] - s.v[1] * eb; lgk[4] = ld[3] + s.v[2] * eb; }
      else if (DIR == 1) { lgk[3] = ld[1] + s.v[0] * eb; lgk[4] = -ld[3] - s.v[2] * eb; }
      else { lgk[3] = -ld[1] - s.v[0] * eb; lgk[4] = ld[2] + s.v[1] * eb; }
      lam_k[0] = lam_k[3] = lam_k[4] = harten(s.vn);
      lam_k[1] = harten(s.vn - s.a);
      lam_k[2] = harten(s.vn + s.a);
      double gv[3] = {0, 0, 0}, ab = 0.0;
      // rows of L: p_k = l_k . du, g_k = |lambda_k| p_k
#pragma unroll
      for (int k = 0; k < 5; k++) {
        double row[NV];
        l_row<DIR>(s, gm1, k, row);
        pk[k] = row[0] * du[0] + row[1] * du[1] + row[2] * du[2] + row[3] * du[3] + row[4] * du[4];
        gk[k] = lam_k[k] * pk[k];
        double X[NV];
        const double c = lgk[k] * lam_k[k];
#pragma unroll
        for (int v = 0; v < NV; v++) X[v] = c * du[v];
        l_row_vjp<DIR>(s, gm1, k, X, gv, ab);
      }
      // R at the Roe state, with g = |Lambda| L du
      const double sum = gk[0] + gk[1] + gk[2];
      for (int j = 0; j < 3; j++) gv[j] += ld[1 + j] * sum;
      const double h0b = eb * (gk[1] + gk[2]);
      const double ekb = eb * gk[0] + h0b;
      gv[DIR] += eb * s.a * (gk[2] - gk[1]);
      ab += difb * (gk[2] - gk[1]) + h0b * 2.0 * s.a * igm1;
      if (DIR == 0) { gv[1] -= eb * gk[3]; gv[2] += eb * gk[4]; }
      else if (DIR == 1) { gv[0] += eb * gk[3]; gv[2] -= eb * gk[4]; }
      else { gv[1] += eb * gk[4]; gv[0] -= eb * gk[3]; }
      for (int j = 0; j < 3; j++) gv[j] += ekb * s.v[j];
      // |lambda_k| with Harten's fix
      const double hm = harten_d(s.vn - s.a), hp = harten_d(s.vn + s.a);
      gv[DIR] += harten_d(s.vn) * (lgk[0] * pk[0] + lgk[3] * pk[3] + lgk[4] * pk[4]) + hm * lgk[1] * pk[1] +
                 hp * lgk[2] * pk[2];
      ab += hp * lgk[2] * pk[2] - hm * lgk[1] * pk[1];
      const double ka = 0.5 * ab * gm1 * s.ia;
      for (int j = 0; j < 3; j++) gv[j] -= ka * s.v[j];
      roe_avg_vjp(u2, u3, gamma, gv, ka, ub2, ub3);
    } else {
      if (sel == 0) speed_vjp<DIR>(u2, gamma, abar, ub2);
      else if (sel == 1) speed_vjp<DIR>(u3, gamma, abar, ub3);
      else roe_speed_vjp<DIR>(u2, u3, gamma, abar, ub2, ub3);
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      E[r0 * ES + v] = ub2[v];
      E[r0 * ES + NV + v] = ub3[v];
    }
  }
  __syncthreads();
  if (active) {
    const int tp = sl.at(1);
    double uc[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      uc[v] = sC[r0 * CS + v];
      accU[v] += E[tp * ES + v] + E[r0 * ES + NV + v];
    }
    flux_jac_T<DIR>(uc, gamma, accF, accU);
    const size_t c = base + (size_t)t * stride;
    double vb[NV] = {0, 0, 0, 0, 0};
    if (VG) visc_gather_cell(uc, QB, GB, nx, ny, nz, gamma, c, vb);
    vjp_store(nu, L, lam, mode, ncell, c, accU, VG, vb);
  }
}

// ---------------------------------------------------------------------------
// characteristic-wise WENO5-JS with Roe or Rusanov upwinding
// ---------------------------------------------------------------------------
// The forward flux at an interface is F = R g with, for every characteristic
// field k (rows of L at the Roe average of the two cells next to it),
//   g_k = (fL_k + fR_k)/2 - l_k (uR_k - uL_k)/2,
// fL/fR (uL/uR) the WENO5 values of L f (L u) over the stencil and l_k = |lambda_k|
// with Harten's fix (Roe) or the Rusanov speed; this is the reference's
// R (WENO of L f) - R |Lambda| L R (WENO of L u) with L R = I
// (Interp1PrimFifthOrderWENOChar.c:86-198, NavierStokes3DUpwind.c:40-124).
// As in hm_pass.hip only first differences are projected: the mean of the two
// cells' fluxes passes L and R unchanged, so neither it nor its adjoint
// depends on the Roe state.  The reverse pass takes the five projected fields
// of the fluxes, then those of the states: the WENO adjoint of each field in
// place of its differences, then point by point back through the rows of L,
// while the derivatives of L, R and l_k with respect to the Roe state (v, a)
// are summed and finally taken back through the Roe average onto cells I-1
// and I.
// longest grid line a characteristic adjoint workgroup holds: at 512 cells
// the block is 8 wavefronts, two per SIMD (the register budget the
// two-wave hint sets for every block size) and 120 KiB of LDS
constexpr int VJP_CHAR_LINE_MAX = 512;
constexpr int VJP_CHAR_CS = VJP_CS;
constexpr int VJP_CHAR_EV = 3;                    // variables exchanged at once
constexpr int VJP_CHAR_ES = 6 * VJP_CHAR_EV + 1;  // doubles per exchange record, odd
constexpr int VJP_CHAR_LDS = VJP_CHAR_CS + VJP_CHAR_ES;  // doubles of LDS per cell of the line

// nu (+)= (d hyp_DIR-part of rhs / d u)^T mu along one direction for the
// characteristic scheme; one workgroup per group of lines, one thread per interface,
// modes as k_rhs_vjp.  LDS (dynamic, VJP_CHAR_LDS doubles per cell of the
// line), laid out as for the component-wise scheme: a record per cell of its
// state and flux and one per interface of its adjoints on the six stencil
// cells, three variables at a time.  Every cell sums the six posts that touch
// it in a fixed order, so the result is deterministic.
template <int DIR, int UPW, int W, bool VG = false>
__device__ __forceinline__ void rhs_vjp_char_line(
    const double *__restrict__ u, const double *__restrict__ lam, const double *__restrict__ nu_in, double ca,
    double cb, double *__restrict__ nu, double *__restrict__ L, int mode, int nx, int ny, int nz,
    const double *__restrict__ dxg, double gamma, double eps, const double *__restrict__ QB,
    const double *__restrict__ GB, const LineSlot &sl, double *smem) {
  const size_t line = sl.line;
  const int t = sl.t, r0 = sl.r;
  const bool active = sl.live;
  const size_t ncell = (size_t)nx * ny * nz;
  size_t base, stride;
  if (DIR == 0) { base = line * nx; stride = 1; }
  else if (DIR == 1) { base = (line % nx) + (line / nx) * (size_t)nx * ny; stride = nx; }
  else { base = line; stride = (size_t)nx * ny; }
  const double *dxd = dxg + 3 + (DIR >= 1 ? nx + 6 : 0) + (DIR == 2 ? ny + 6 : 0);
  constexpr int CS = VJP_CHAR_CS, ES = VJP_CHAR_ES;
  double *sC = smem;        // [sl.size][CS]: state [5], flux [5]
  double *E = sC + CS * sl.size;  // [sl.size][ES]
  const double gm1 = gamma - 1.0, igm1 = nr_rcp(gm1), eps34 = 0.75 * eps;
  double lF[NV] = {0, 0, 0, 0, 0};  // adjoint of the interface flux
  if (active) {
    const size_t c = base + (size_t)t * stride;
    double us[NV], lm[NV], ni[NV];
    vjp_load_cell(u, lam, nu_in, ncell, c, us, lm, ni);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      sC[r0 * CS + v] = us[v];
      // dxinv mu of this cell, staged in the (not yet used) exchange buffer
      E[r0 * ES + v] = dxd[t] * (cb * lm[v] + (nu_in ? ca * ni[v] : 0.0));
    }
    double fl[NV];
    vjp_flux<DIR>(us, gamma, fl);
#pragma unroll
    for (int v = 0; v < NV; v++) sC[r0 * CS + NV + v] = fl[v];
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int v = 0; v < NV; v++) lF[v] = E[r0 * ES + v] - E[sl.at(-1) * ES + v];
  }
  __syncthreads();
  const double *cs[6];  // records of the stencil's cells
  const double *ei[6];  // exchange records that touch this cell: slot p of interface t+3-p
#pragma unroll
  for (int p = 0; p < 6; p++) {
    cs[p] = sC + sl.at(p - 3) * CS;
    ei[p] = E + sl.at(3 - p) * ES + p * VJP_CHAR_EV;
  }
  RoeAdj s = {};
  double lk[3] = {0, 0, 0};  // |lambda| of the entropy and shear, the u-a and the u+a fields
  int sel = 0;
  if (active) {
    double u2[NV], u3[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) { u2[v] = cs[2][v]; u3[v] = cs[3][v]; }
    s = roe_adj_state<DIR>(u2, u3, gamma);
    if (UPW == UPWIND_RUSANOV) {
      // max(max(aL, aR), max(aR, aA)), the branch the forward selects
      const double aL = vjp_speed<DIR>(u2, gamma), aR = vjp_speed<DIR>(u3, gamma);
      const double aA = s.a + fabs(s.vn);
      const double m01 = fmax(aL, aR), m12 = fmax(aR, aA);
      lk[0] = lk[1] = lk[2] = fmax(m01, m12);
      sel = m01 >= m12 ? (aL >= aR ? 0 : 1) : (aR >= aA ? 1 : 2);
    } else {
      lk[0] = harten(s.vn);
      lk[1] = harten(s.vn - s.a);
      lk[2] = harten(s.vn + s.a);
    }
  }
  // the two shear fields (one row of L each: CA or CB times (x_J - v_J x_0))
  constexpr int JA = DIR == 0 ? 1 : 0, JB = DIR == 2 ? 1 : 2;  // velocity components
  constexpr double CA = DIR == 1 ? 1.0 : -1.0, CB = -CA;
  double gv[3] = {0, 0, 0}, ab = 0.0, alb = 0.0;
  // part 0 takes the WENO5 of L f back onto the cell fluxes, part 1 the WENO5
  // of L u onto the cell states; in between, the flux adjoint of every cell
  // goes through its flux Jacobian
  double acc[NV] = {0, 0, 0, 0, 0};
  auto take_back = [&](auto tag) {
    constexpr int part = decltype(tag)::value;
    constexpr int S = part == 0 ? NV : 0;  // flux or state within the cell record
    double xb[5][NV];                  // adjoints of the five differences
    if (active) {
      const double kh = 0.5 * gm1 * s.ia2, aih = 0.5 * s.ia;
      const double gek = kh * s.ek, avn = aih * s.vn;
      double d[5][5];  // fields: entropy, u-a, u+a, the two shear fields
#pragma unroll
      for (int p = 0; p < 5; p++) {
        double x[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) x[v] = cs[p + 1][S + v] - cs[p][S + v];
        const double w = s.v[0] * x[1] + s.v[1] * x[2] + s.v[2] * x[3] - x[4];
        const double h = gek * x[0] - kh * w, m = avn * x[0] - aih * x[1 + DIR];
        d[0][p] = x[0] - 2.0 * h;
        d[1][p] = h + m;
        d[2][p] = h - m;
        d[3][p] = CA * (x[1 + JA] - s.v[JA] * x[0]);
        d[4][p] = CB * (x[1 + JB] - s.v[JB] * x[0]);
      }
      // (R^T lambda_F)_k (columns of R, navierstokes3d.h:384-470)
      const double eb = lF[4];
      const double sumb = lF[0] + s.v[0] * lF[1] + s.v[1] * lF[2] + s.v[2] * lF[3];
      const double difb = lF[1 + DIR] + s.vn * eb;
      double g[5];  // this part's share of g_k
#pragma unroll
      for (int k = 0; k < 5; k++) {
        double gb;
        if (k == 0) gb = sumb + s.ek * eb;
        else if (k == 1) gb = sumb + s.h0 * eb - s.a * difb;
        else if (k == 2) gb = sumb + s.h0 * eb + s.a * difb;
        else if (k == 3) gb = CA * (lF[1 + JA] + s.v[JA] * eb);
        else gb = CB * (lF[1 + JB] + s.v[JB] * eb);
        const double l = k == 1 ? lk[1] : (k == 2 ? lk[2] : lk[0]);
        double jump, corr;
        if (part == 0) {
          weno5_lr_vjp<W>(d[k], eps34, 0.5 * gb, 0.5 * gb, d[k], jump, corr);
          g[k] = 0.5 * corr;
        } else {
          const double ob = 0.5 * l * gb;
          weno5_lr_vjp<W>(d[k], eps34, ob, -ob, d[k], jump, corr);
          d[k][2] -= ob;
          g[k] = -0.5 * l * jump;
          const double lb = -0.5 * jump * gb;  // adjoint of l_k: Harten's |lambda| (Roe) or the common Rusanov speed
          if (UPW == UPWIND_ROE) {
            const double hb = harten_d(k == 1 ? s.vn - s.a : (k == 2 ? s.vn + s.a : s.vn)) * lb;
            gv[DIR] += hb;
            if (k == 1) ab -= hb;
            if (k == 2) ab += hb;
          } else {
            alb += lb;
          }
        }
        // one field at a time: interleaved, the WENO adjoints of the heavier
        // weights do not fit the 256 registers of two waves per SIMD
        __builtin_amdgcn_sched_barrier(0);
      }
      // R g at the Roe state
      const double gsum = g[0] + g[1] + g[2], gdif = g[2] - g[1];
#pragma unroll
      for (int j = 0; j < 3; j++) gv[j] += (lF[1 + j] + eb * s.v[j]) * gsum;
      gv[DIR] += eb * s.a * gdif;
      gv[JA] += CA * eb * g[3];
      gv[JB] += CB * eb * g[4];
      ab += difb * gdif + eb * (g[1] + g[2]) * 2.0 * s.a * igm1;
      // back through the rows of L, and the rows' own derivatives: sums of the
      // adjoints of h and m above against x
      double hx0 = 0.0, hw = 0.0, mx0 = 0.0, mxd = 0.0, sa = 0.0, sb = 0.0;
      asm volatile("" ::: "memory");  // read the records again: held, the 25 differences take 50 registers
#pragma unroll
      for (int p = 0; p < 5; p++) {
        double x[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) x[v] = cs[p + 1][S + v] - cs[p][S + v];
        const double w = s.v[0] * x[1] + s.v[1] * x[2] + s.v[2] * x[3] - x[4];
        const double hb = (d[1][p] + d[2][p]) - 2.0 * d[0][p], mb = d[1][p] - d[2][p];
        const double a = CA * d[3][p], b = CB * d[4][p], wb = -kh * hb;
        hx0 += hb * x[0];
        hw += hb * w;
        mx0 += mb * x[0];
        mxd += mb * x[1 + DIR];
        sa += a * x[0];
        sb += b * x[0];
#pragma unroll
        for (int j = 0; j < 3; j++) gv[j] += wb * x[1 + j];
        xb[p][0] = d[0][p] + gek * hb + avn * mb - s.v[JA] * a - s.v[JB] * b;
#pragma unroll
        for (int j = 0; j < 3; j++) xb[p][1 + j] = s.v[j] * wb;
        xb[p][1 + DIR] -= aih * mb;
        xb[p][1 + JA] += a;
        xb[p][1 + JB] += b;
        xb[p][4] = -wb;
      }
      // h = kh (ek x_0 - w), m = aih (v_d x_0 - x_d), kh = (gamma-1)/(2a^2), aih = 1/(2a)
      const double khb = s.ek * hx0 - hw, ekb = kh * hx0;
#pragma unroll
      for (int j = 0; j < 3; j++) gv[j] += s.v[j] * ekb;
      gv[DIR] += aih * mx0;
      gv[JA] -= sa;
      gv[JB] -= sb;
      ab -= s.ia * (2.0 * kh * khb + aih * (s.vn * mx0 - mxd));
    }
    // post the adjoints of the six cells (differences of those of the
    // differences, and in part 0 the mean of the two cells' fluxes), take the
    // posts that touch this cell
#pragma unroll
    for (int v0 = 0; v0 < NV; v0 += VJP_CHAR_EV) {
      if (active)
#pragma unroll
        for (int v = v0; v < NV && v < v0 + VJP_CHAR_EV; v++)
#pragma unroll
          for (int p = 0; p < 6; p++)
            E[r0 * ES + p * VJP_CHAR_EV + v - v0] = (p > 0 ? xb[p - 1][v] : 0.0) - (p < 5 ? xb[p][v] : 0.0) +
                                                   (part == 0 && (p == 2 || p == 3) ? 0.5 * lF[v] : 0.0);
      __syncthreads();
      if (active)
#pragma unroll
        for (int v = v0; v < NV && v < v0 + VJP_CHAR_EV; v++)
#pragma unroll
          for (int p = 0; p < 6; p++) acc[v] += ei[p][v - v0];
      __syncthreads();
    }
    if (part == 0 && active) {
      double uc[NV], ub[NV] = {0, 0, 0, 0, 0};
#pragma unroll
      for (int v = 0; v < NV; v++) uc[v] = sC[r0 * CS + v];
      flux_jac_T<DIR>(uc, gamma, acc, ub);
#pragma unroll
      for (int v = 0; v < NV; v++) acc[v] = ub[v];
    }
  };
  take_back(std::integral_constant<int, 0>{});
  take_back(std::integral_constant<int, 1>{});
  // the Roe state's (and the Rusanov speed's) dependence on cells t-1 and t
  if (active) {
    double u2[NV], u3[NV], ub2[NV] = {0, 0, 0, 0, 0}, ub3[NV] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int v = 0; v < NV; v++) { u2[v] = cs[2][v]; u3[v] = cs[3][v]; }
    if (UPW == UPWIND_RUSANOV) {
      if (sel == 0) speed_vjp<DIR>(u2, gamma, alb, ub2);
      else if (sel == 1) speed_vjp<DIR>(u3, gamma, alb, ub3);
      else roe_speed_vjp<DIR>(u2, u3, gamma, alb, ub2, ub3);
    }
    // a = sqrt((H - |v|^2/2)(gamma-1)) -> (v, H) of the Roe average -> the two cells
    const double ka = 0.5 * ab * gm1 * s.ia;
    for (int j = 0; j < 3; j++) gv[j] -= ka * s.v[j];
    roe_avg_vjp(u2, u3, gamma, gv, ka, ub2, ub3);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      E[r0 * ES + v] = ub2[v];
      E[r0 * ES + NV + v] = ub3[v];
    }
  }
  __syncthreads();
  if (active) {
    const int tp = sl.at(1);
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] += E[tp * ES + v] + E[r0 * ES + NV + v];
    const size_t c = base + (size_t)t * stride;
    double vb[NV] = {0, 0, 0, 0, 0};
    if (VG) {
      double uc[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) uc[v] = sC[r0 * CS + v];
      visc_gather_cell(uc, QB, GB, nx, ny, nz, gamma, c, vb);
    }
    vjp_store(nu, L, lam, mode, ncell, c, acc, VG, vb);
  }
}

// ---------------------------------------------------------------------------
// viscous term
// ---------------------------------------------------------------------------
// par_i = sum_d dxinv_d(i) D_d[FV_d](i), D the 4th-order central difference
// over FV_d at i-2..i+2 along d, where FV_d is the viscous flux of the
// primitive variables Q = (u, v, w, T) and their gradients (4th-order central,
// periodic) inside the grid, and the ghost-layer flux (biased stencil in the
// second layer, zero derivatives across d) at the two positions on each side
// of a line (NavierStokes3DParabolicFunction.c:50-325,
// FirstDerivativeFourthOrder.c:36-129).  The reverse pass:
//  k_visc_vjp_tile   flux adjoints of every cell from its interior readers,
//                    back through the flux onto Q (stored in QB) and onto the
//                    gradients (stored in GB, already times dxinv), by tiles
//                    of VTX x VTY columns marching through vks z-planes: Q
//                    and the readers' adjoint weights of a plane sit in LDS
//                    with a 2-cell halo in x and y, the z stencil in
//                    registers, so each is read about once per tile;
//  k_visc_vjp_ghost  the same for the ghost-layer fluxes of each line, whose
//                    gradient adjoints are spread over their stencils into QB;
//  visc_gather_cell  QB plus the transposed gradient stencils over GB, then
//                    back through the primitive variables: the x line VJP,
//                    which runs last, adds this onto the nu that the z and y
//                    line VJPs left, before its own share.
struct ViscC {
  double gamma, inv_Re, inv_gm1, inv_Pr;
};

// adjoint of the viscous flux along DIR at a point: fb = adjoint of
// (tau_d1, tau_d2, tau_d3, energy flux); adds to qb (u, v, w, T values) and
// grb (gradient entries, grb[c][e] = d/d(dq_c/dx_e)); returns the adjoint of mu
template <int DIR>
__device__ __forceinline__ double visc_flux_vjp(const double q[4], const double (&gr)[4][3], double mu,
                                                const ViscC &vc, const double fb[4], double qb[4],
                                                double (&grb)[4][3]) {
  const double tt = 2.0 / 3.0;
  const double mr = mu * vc.inv_Re, kq = mr * vc.inv_gm1 * vc.inv_Pr;
  const double ux = gr[0][0], uy = gr[0][1], uz = gr[0][2];
  const double vx = gr[1][0], vy = gr[1][1], vz = gr[1][2];
  const double wx = gr[2][0], wy = gr[2][1], wz = gr[2][2];
  double b1, b2, b3;
  if (DIR == 0) { b1 = tt * (2 * ux - vy - wz); b2 = uy + vx; b3 = uz + wx; }
  else if (DIR == 1) { b1 = uy + vx; b2 = tt * (-ux + 2 * vy - wz); b3 = vz + wy; }
  else { b1 = uz + wx; b2 = vz + wy; b3 = tt * (-ux - vy + 2 * wz); }
  const double gT = gr[3][DIR];
  const double tb1 = fb[0] + q[0] * fb[3], tb2 = fb[1] + q[1] * fb[3], tb3 = fb[2] + q[2] * fb[3];
  qb[0] += fb[3] * (mr * b1);
  qb[1] += fb[3] * (mr * b2);
  qb[2] += fb[3] * (mr * b3);
  const double mub = (tb1 * b1 + tb2 * b2 + tb3 * b3) * vc.inv_Re + fb[3] * gT * (vc.inv_Re * vc.inv_gm1 * vc.inv_Pr);
  const double c1 = mr * tb1, c2 = mr * tb2, c3 = mr * tb3;
  if (DIR == 0) {
    grb[0][0] += 2 * tt * c1; grb[1][1] -= tt * c1; grb[2][2] -= tt * c1;
    grb[0][1] += c2; grb[1][0] += c2;
    grb[0][2] += c3; grb[2][0] += c3;
  } else if (DIR == 1) {
    grb[0][1] += c1; grb[1][0] += c1;
    grb[0][0] -= tt * c2; grb[1][1] += 2 * tt * c2; grb[2][2] -= tt * c2;
    grb[1][2] += c3; grb[2][1] += c3;
  } else {
    grb[0][2] += c1; grb[2][0] += c1;
    grb[1][2] += c2; grb[2][1] += c2;
    grb[0][0] -= tt * c3; grb[1][1] -= tt * c3; grb[2][2] += 2 * tt * c3;
  }
  grb[3][DIR] += kq * fb[3];
  return mub;
}

// mu_c at a cell: momentum and energy components of cb*lam + ca*nu_in
__device__ __forceinline__ void visc_mu(const double *__restrict__ lam, const double *__restrict__ nu_in, double ca,
                                        double cb, size_t ncell, size_t c, double m[4]) {
  // all loads before any use: a null check of nu_in inside the loop would
  // put a wait in each iteration
  double l[4], n[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 4; k++) l[k] = lam[(size_t)(1 + k) * ncell + c];
  if (nu_in)
#pragma unroll
    for (int k = 0; k < 4; k++) n[k] = nu_in[(size_t)(1 + k) * ncell + c];
#pragma unroll
  for (int k = 0; k < 4; k++) m[k] = cb * l[k] + (nu_in ? ca * n[k] : 0.0);
}

// A plane of Q and of the readers' adjoint weights with a 2-cell halo in x and
// y, and the tile's 1/dx and 1/dy, which are zero outside the grid: a reader
// there does not count.  Two planes: the next one is staged while the slower
// wavefronts still read this one, which leaves one barrier per plane.
// A thread stages its own column from the window in its registers and 304 of
// them one point of the halo, whose loads are in flight during the arithmetic
// of the plane before.  (When every plane was loaded whole, twice over the
// tile's halo, and waited for, in segments of 16 planes on any grid: 878 us for
// eight grids of together 9.3e6 cells against 532 us now.)
struct ViscVjpShared {
  double q[2][4][VHY][VHX], m[2][4][VHY][VHX];
  double dx[VHX], dy[VHY];
};

__device__ __forceinline__ void visc_vjp_tile(const double *__restrict__ Q, const double *__restrict__ lam,
                                              const double *__restrict__ nu_in, double ca, double cb,
                                              double *__restrict__ QB, double *__restrict__ GB, int nx, int ny,
                                              int nz, const double *__restrict__ dxg, const ViscC &vc, int b, int vks,
                                              ViscVjpShared &sh) {
  const size_t ncell = (size_t)nx * ny * nz;
  const size_t plane = (size_t)nx * ny;
  const int ntx = (nx + VTX - 1) / VTX, nty = (ny + VTY - 1) / VTY;
  const int tx = b % ntx, ty = (b / ntx) % nty, kz = b / (ntx * nty);
  const int x0 = tx * VTX, y0 = ty * VTY, k0 = kz * vks;
  const int t = threadIdx.x, lx = t % VTX, ly = t / VTX;
  const int i = x0 + lx, j = y0 + ly;
  const bool own = i < nx && j < ny;
  // columns past the grid hold the periodic copies, which tile columns next to
  // the grid's last ones read: x0 + ox spans [x0 - 2, x0 + VTX + 1] and y0 + oy
  // [y0 - 2, y0 + VTY + 1], which can exceed 2 nx and 2 ny.  The column is a
  // byte offset of 32 bits, added to a wave-uniform plane address: with 64-bit
  // lane offsets the compiler keeps one address per array and component in
  // registers through the loop.  A plane of 2^29 columns, where the offset
  // would overflow, makes u, lam and nu alone 322 GB (nz >= 5).
  auto column = [&](int ox, int oy) {
    return (unsigned)(((y0 + oy + 2 * ny) % ny) * (size_t)nx + (x0 + ox + 2 * nx) % nx) * 8u;
  };
  unsigned col = column(lx, ly);
  // 304 threads also stage a point of the halo: rows -2, -1, VTY, VTY+1 over
  // the full width, then columns -2, -1, VTX, VTX+1
  const bool halo = t < 4 * VHX + 4 * VTY;
  int hx = t % VHX, hy = t / VHX;
  if (hy >= 2) hy += VTY;
  if (t >= 4 * VHX) {
    const int u = t - 4 * VHX, r = u % 4;
    hx = r < 2 ? r : VTX + r;
    hy = 2 + u / 4;
  }
  unsigned hcol = halo ? column(hx - 2, hy - 2) : col;
  const double *dx = dxg + 3, *dy = dxg + (nx + 6) + 3, *dz = dxg + (nx + 6) + (ny + 6) + 3;
  const int k1 = min(k0 + vks, nz);
  if (t < VHX) sh.dx[t] = x0 + t >= 2 && x0 + t - 2 < nx ? dx[x0 + t - 2] : 0.0;
  else if (t < VHX + VHY) {
    const int r = y0 + t - VHX - 2;
    sh.dy[t - VHX] = r >= 0 && r < ny ? dy[r] : 0.0;
  }
  const int offs[4] = {-2, -1, 1, 2};
  // Q and the readers' weights of a column; a missing nu_in reads lam's lines
  // a second time, so that no branch holds the loads up
  const double *nu = nu_in ? nu_in : lam;
  auto at = [](const double *base, unsigned byte) { return *(const double *)((const char *)base + byte); };
  auto load = [&](size_t pl, unsigned c, double (&qo)[4], double (&l)[4], double (&n)[4]) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      qo[v] = at(Q + v * ncell + pl, c);
      l[v] = at(lam + (1 + v) * ncell + pl, c);
      n[v] = at(nu + (1 + v) * ncell + pl, c);
    }
  };
  auto weight = [&](double l, double n) { return cb * l + (nu_in ? ca * n : 0.0); };
  auto put = [](double *base, unsigned byte, double x) { *(double *)((char *)base + byte) = x; };
  // window: Q and the weights m of this column at planes k-2..k+2; l and n of
  // plane k+2 and the halo point of plane k arrive unweighted
  double q[5][4], m[5][4], l[4], n[4], hq[4] = {0, 0, 0, 0}, hl[4] = {0, 0, 0, 0}, hn[4] = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < 4; s++) {
    load((size_t)wrapn(k0 - 2 + s, nz) * plane, col, q[s], l, n);
#pragma unroll
    for (int v = 0; v < 4; v++) m[s][v] = weight(l[v], n[v]);
  }
  load((size_t)wrapn(k0 + 2, nz) * plane, col, q[4], l, n);
  if (halo) load((size_t)k0 * plane, hcol, hq, hl, hn);
  int buf = 0;
  for (int k = k0; k < k1; k++) {
    asm volatile("" : "+v"(col), "+v"(hcol));
    auto &sq = sh.q[buf];
    auto &sm = sh.m[buf];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      m[4][v] = weight(l[v], n[v]);
      sq[v][ly + 2][lx + 2] = q[2][v];
      sm[v][ly + 2][lx + 2] = m[2][v];
    }
    if (halo)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        sq[v][hy][hx] = hq[v];
        sm[v][hy][hx] = weight(hl[v], hn[v]);
      }
    __syncthreads();
    double qn[4] = {0, 0, 0, 0};
    if (k + 1 < k1) {
      load((size_t)wrapn(k + 3, nz) * plane, col, qn, l, n);
      if (halo) load((size_t)(k + 1) * plane, hcol, hq, hl, hn);
    }
    if (own) {
      double gr[4][3];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const double *r = &sq[c][ly + 2][0];
        gr[c][0] = d4c(r[lx], r[lx + 1], r[lx + 3], r[lx + 4]) * sh.dx[lx + 2];
        gr[c][1] = d4c(sq[c][ly][lx + 2], sq[c][ly + 1][lx + 2], sq[c][ly + 3][lx + 2], sq[c][ly + 4][lx + 2]) * sh.dy[ly + 2];
        gr[c][2] = d4c(q[0][c], q[1][c], q[3][c], q[4][c]) * dz[k];
      }
      const double qc[4] = {q[2][0], q[2][1], q[2][2], q[2][3]};
      const double mu = pow076(qc[3]);
      double zw[5];  // dz has ghost entries; a reader out there does not count
#pragma unroll
      for (int s = 0; s < 5; s++) {
        const double w = dz[k - 2 + s];
        zw[s] = (unsigned)(k - 2 + s) < (unsigned)nz ? w : 0.0;
      }
      double qb[4] = {0, 0, 0, 0}, grb[4][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, mub = 0.0;
      // direction by direction: reader r = pos - s reads this cell's flux
      // with weight d4w(s) dxinv(r), inside the grid only
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double fb[4] = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int o = offs[s];
          const double w = d4w(o) * (d == 0 ? sh.dx[lx + 2 - o]
                                            : (d == 1 ? sh.dy[ly + 2 - o] : zw[2 - o]));
#pragma unroll
          for (int c = 0; c < 4; c++)
            fb[c] += w * (d == 0 ? sm[c][ly + 2][lx + 2 - o] : (d == 1 ? sm[c][ly + 2 - o][lx + 2] : m[2 - o][c]));
        }
        if (d == 0) mub += visc_flux_vjp<0>(qc, gr, mu, vc, fb, qb, grb);
        else if (d == 1) mub += visc_flux_vjp<1>(qc, gr, mu, vc, fb, qb, grb);
        else mub += visc_flux_vjp<2>(qc, gr, mu, vc, fb, qb, grb);
        __builtin_amdgcn_sched_barrier(0);  // the next direction's weights are read after this one's use
      }
      qb[3] += mub * (0.76 * mu * nr_rcp(qc[3]));
      const size_t pl = (size_t)k * plane;
      const double dxe[3] = {sh.dx[lx + 2], sh.dy[ly + 2], dz[k]};
#pragma unroll
      for (int c = 0; c < 4; c++) {
        put(QB + c * ncell + pl, col, qb[c]);
#pragma unroll
        for (int e = 0; e < 3; e++) put(GB + (c * 3 + e) * ncell + pl, col, grb[c][e] * dxe[e]);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
#pragma unroll
      for (int s = 0; s < 4; s++) {
        q[s][v] = q[s + 1][v];
        m[s][v] = m[s + 1][v];
      }
      q[4][v] = qn[v];
    }
    buf ^= 1;
  }
}

// one thread per line along DIR: the four ghost-layer fluxes -2, -1, n, n+1
template <int DIR>
__device__ __forceinline__ void visc_vjp_ghost_line(const double *__restrict__ Q, const double *__restrict__ lam,
                                                    const double *__restrict__ nu_in, double ca, double cb,
                                                    double *__restrict__ QB, int nx, int ny, int nz,
                                                    const double *__restrict__ dxg, const ViscC &vc, size_t line) {
  const size_t ncell = (size_t)nx * ny * nz;
  const int n = DIR == 0 ? nx : (DIR == 1 ? ny : nz);
  const size_t nplane = ncell / n;
  if (line >= nplane) return;
  size_t base, stride;
  if (DIR == 0) { base = line * nx; stride = 1; }
  else if (DIR == 1) { base = (line % nx) + (line / nx) * (size_t)nx * ny; stride = nx; }
  else { base = line; stride = (size_t)nx * ny; }
  const double *dxd = dxg + (DIR >= 1 ? nx + 6 : 0) + (DIR == 2 ? ny + 6 : 0);  // entry 0: position -3
  // readers 0, 1, n-2, n-1, times their dxinv
  double a[4][4];
  const int rd[4] = {0, 1, n - 2, n - 1};
#pragma unroll
  for (int r = 0; r < 4; r++) {
    visc_mu(lam, nu_in, ca, cb, ncell, base + (size_t)rd[r] * stride, a[r]);
#pragma unroll
    for (int k = 0; k < 4; k++) a[r][k] *= dxd[3 + rd[r]];
  }
  // the seven cells gp-3 .. gp+3 of slot s (positions -2, -1, n, n+1,
  // periodic) are entries s .. s+6 of the window n-5 .. n-1, 0 .. 4 (n >= 5),
  // loaded once; the slots' adjoints onto Q accumulate per window entry and
  // reach QB with one read-modify-write each (entries that are the same cell
  // of a short line add in turn)
  double f[10][4], acc[10][4];
  size_t cw[10];
#pragma unroll
  for (int j = 0; j < 10; j++) {
    cw[j] = base + (size_t)(j < 5 ? n - 5 + j : j - 5) * stride;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      f[j][c] = Q[(size_t)c * ncell + cw[j]];
      acc[j][c] = 0.0;
    }
  }
  const double r12 = 1.0 / 12.0;
#pragma unroll
  for (int slot = 0; slot < 4; slot++) {
    const int gp = slot < 2 ? slot - 2 : n + slot - 2;
    double fb[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (slot == 0) fb[k] = d4w(-2) * a[0][k];
      else if (slot == 1) fb[k] = d4w(-1) * a[0][k] + d4w(-2) * a[1][k];
      else if (slot == 2) fb[k] = d4w(1) * a[3][k] + d4w(2) * a[2][k];
      else fb[k] = d4w(2) * a[3][k];
    }
    // the forward evaluation at this ghost position (ghost_flux of hm_kernels.hip)
    const double(*w)[4] = f + slot;  // positions gp-3 .. gp+3
    // stencil weights over positions gp-3 .. gp+3
    double w7[7] = {0, 0, 0, 0, 0, 0, 0};
    if (slot == 0) { w7[2] = -3 * r12; w7[3] = -10 * r12; w7[4] = 18 * r12; w7[5] = -6 * r12; w7[6] = r12; }
    else if (slot == 3) { w7[0] = -r12; w7[1] = 6 * r12; w7[2] = -18 * r12; w7[3] = 10 * r12; w7[4] = 3 * r12; }
    else { w7[1] = r12; w7[2] = -8 * r12; w7[4] = 8 * r12; w7[5] = -r12; }
    const double dxgh = dxd[3 + gp];
    double gr[4][3];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      double d = 0.0;
      if (slot == 0) d = (-3 * w[2][c] - 10 * w[3][c] + 18 * w[4][c] - 6 * w[5][c] + w[6][c]) * r12;
      else if (slot == 3) d = (-w[0][c] + 6 * w[1][c] - 18 * w[2][c] + 10 * w[3][c] + 3 * w[4][c]) * r12;
      else d = d4c(w[1][c], w[2][c], w[4][c], w[5][c]);
#pragma unroll
      for (int e = 0; e < 3; e++) gr[c][e] = e == DIR ? d * dxgh : 0.0;
    }
    const double q[4] = {w[3][0], w[3][1], w[3][2], w[3][3]};
    const double mu = pow076(q[3]);
    double qb[4] = {0, 0, 0, 0}, grb[4][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    const double mub = visc_flux_vjp<DIR>(q, gr, mu, vc, fb, qb, grb);
    qb[3] += mub * (0.76 * mu * nr_rcp(q[3]));
#pragma unroll
    for (int c = 0; c < 4; c++) acc[slot + 3][c] += qb[c];
#pragma unroll
    for (int s = 0; s < 7; s++) {
      if (w7[s] == 0.0) continue;
#pragma unroll
      for (int c = 0; c < 4; c++) acc[slot + s][c] += w7[s] * dxgh * grb[c][DIR];
    }
  }
  // on lines of 10 cells and more the entries are different cells, and the 40
  // loads go out together instead of each after the store before it: 10, 5.6
  // and 5.7 us (x, y, z) at 48x80x66, 15, 14 and 13 us one by one
  if (n >= 10) {
    double b[10][4];
#pragma unroll
    for (int j = 0; j < 10; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) b[j][c] = QB[(size_t)c * ncell + cw[j]];
#pragma unroll
    for (int j = 0; j < 10; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) QB[(size_t)c * ncell + cw[j]] = b[j][c] + acc[j][c];
    return;
  }
#pragma unroll
  for (int j = 0; j < 10; j++)
#pragma unroll
    for (int c = 0; c < 4; c++) QB[(size_t)c * ncell + cw[j]] += acc[j][c];
}

// ---------------------------------------------------------------------------
// kernels: one grid
// ---------------------------------------------------------------------------
// neighbouring lines share cache lines along x: keep them on one XCD
template <int DIR, int UPW, int W, bool VG>
__global__ void __launch_bounds__(VJP_LINE_MAX) k_rhs_vjp(const double *__restrict__ u, const double *__restrict__ lam,
                                                      const double *__restrict__ nu_in, double ca, double cb,
                                                      double *__restrict__ nu, double *__restrict__ L, int mode,
                                                      int nx, int ny, int nz, const double *__restrict__ dxg,
                                                      double gamma, double eps, const double *__restrict__ QB,
                                                      const double *__restrict__ GB) {
  extern __shared__ double smem[];
  const int n = DIR == 0 ? nx : (DIR == 1 ? ny : nz);
  const LineSlot s = line_slot(xcd_block(), n, (size_t)nx * ny * nz / n);
  rhs_vjp_line<DIR, UPW, W, VG>(u, lam, nu_in, ca, cb, nu, L, mode, nx, ny, nz, dxg, gamma, eps, QB, GB, s, smem);
}

template <int DIR, int UPW, int W, bool VG>
__global__ void __launch_bounds__(VJP_CHAR_LINE_MAX) __attribute__((amdgpu_waves_per_eu(2))) k_rhs_vjp_char(
    const double *__restrict__ u, const double *__restrict__ lam, const double *__restrict__ nu_in, double ca,
    double cb, double *__restrict__ nu, double *__restrict__ L, int mode, int nx, int ny, int nz,
    const double *__restrict__ dxg, double gamma, double eps, const double *__restrict__ QB,
    const double *__restrict__ GB) {
  extern __shared__ double smem[];
  const int n = DIR == 0 ? nx : (DIR == 1 ? ny : nz);
  const LineSlot s = line_slot(xcd_block(), n, (size_t)nx * ny * nz / n);
  rhs_vjp_char_line<DIR, UPW, W, VG>(u, lam, nu_in, ca, cb, nu, L, mode, nx, ny, nz, dxg, gamma, eps, QB, GB, s, smem);
}

__global__ void __launch_bounds__(VT) k_visc_vjp_tile(const double *__restrict__ Q, const double *__restrict__ lam,
                                                     const double *__restrict__ nu_in, double ca, double cb,
                                                     double *__restrict__ QB, double *__restrict__ GB, int nx, int ny,
                                                     int nz, const double *__restrict__ dxg, ViscC vc, int vks) {
  __shared__ ViscVjpShared sh;
  visc_vjp_tile(Q, lam, nu_in, ca, cb, QB, GB, nx, ny, nz, dxg, vc, blockIdx.x, vks, sh);
}

// one wavefront per block: a grid has few lines, and their scattered loads
// are spread over more CUs (x, 5280 lines of 48 cells: 15 us against 30 at
// four wavefronts)
template <int DIR>
__global__ void __launch_bounds__(64) k_visc_vjp_ghost(const double *__restrict__ Q, const double *__restrict__ lam,
                                                        const double *__restrict__ nu_in, double ca, double cb,
                                                        double *__restrict__ QB, int nx, int ny, int nz,
                                                        const double *__restrict__ dxg, ViscC vc) {
  visc_vjp_ghost_line<DIR>(Q, lam, nu_in, ca, cb, QB, nx, ny, nz, dxg, vc,
                           (size_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// ---------------------------------------------------------------------------
// kernels: all members of an ensemble
// ---------------------------------------------------------------------------
// Member m's state, adjoints and work space sit at 5*off, 5*off and 20*off;
// its stage coefficients are dt_m * (A, B).  Line work lists hold each
// member's first line along a direction (nmem + 1 entries).
struct EnsVjp {
  const EnsMember *mem;
  int nmem;
  const double *u, *lam, *nu_in;
  double A, B;
  double *nu, *L, *work;
  int mode;
  double gamma, eps;
  ViscC vc;
};

__device__ __forceinline__ int ens_find(const unsigned *first, int nmem, unsigned item) {
  int lo = 0, hi = nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first[mid] <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ int ens_find_cell(const EnsMember *mem, int nmem, size_t idx) {
  int lo = 0, hi = nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mem[mid].off <= idx) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Calls f(member index) for cell idx of a launch with one thread per cell.
// A block of consecutive cells nearly always lies in one member: the member
// is then found once for the block, the same for every lane (scalar loads
// of its table entry); otherwise every lane searches for its own.
template <class F>
__device__ __forceinline__ void with_cell_member(const EnsMember *mem, int nmem, size_t idx, const F &f) {
  const size_t b0 = (size_t)blockIdx.x * blockDim.x;
  const int m0 = ens_find_cell(mem, nmem, b0);
  if (b0 + blockDim.x <= mem[m0].off + mem[m0].ncell) f(m0);
  else f(ens_find_cell(mem, nmem, idx));
}

// with VG (the x lines of a viscous ensemble) also QB and GB of the member's
// work space, whose viscous share the lines add
#define ENS_MEMBER_ARGS(a, M)                                                                              \
  a.u + 5 * M.off, a.lam + 5 * M.off, a.nu_in ? a.nu_in + 5 * M.off : nullptr, M.dt * a.A, M.dt * a.B,     \
      a.nu + 5 * M.off, a.L ? a.L + 5 * M.off : nullptr, a.mode, M.n[0], M.n[1], M.n[2], M.dxg, a.gamma, a.eps, \
      VG ? a.work + 20 * M.off + 4 * M.ncell : nullptr, VG ? a.work + 20 * M.off + 8 * M.ncell : nullptr

template <int DIR, int UPW, int W, bool VG>
__global__ void __launch_bounds__(VJP_LINE_MAX) k_ens_rhs_vjp(EnsVjp a, const unsigned *__restrict__ first,
                                                          unsigned nitems) {
  extern __shared__ double smem[];
  const XcdItems r = xcd_items(nitems);
  for (unsigned item = r.first; item < r.end; item += r.step) {
    const int m = ens_find(first, a.nmem, item);
    const EnsMember M = a.mem[m];
    const LineSlot s = line_slot(item - first[m], M.n[DIR], M.ncell / M.n[DIR]);
    rhs_vjp_line<DIR, UPW, W, VG>(ENS_MEMBER_ARGS(a, M), s, smem);
    __syncthreads();
  }
}

template <int DIR, int UPW, int W, bool VG>
__global__ void __launch_bounds__(VJP_CHAR_LINE_MAX) __attribute__((amdgpu_waves_per_eu(2))) k_ens_rhs_vjp_char(EnsVjp a, const unsigned *__restrict__ first,
                                                                    unsigned nitems) {
  extern __shared__ double smem[];
  const XcdItems r = xcd_items(nitems);
  for (unsigned item = r.first; item < r.end; item += r.step) {
    const int m = ens_find(first, a.nmem, item);
    const EnsMember M = a.mem[m];
    const LineSlot s = line_slot(item - first[m], M.n[DIR], M.ncell / M.n[DIR]);
    rhs_vjp_char_line<DIR, UPW, W, VG>(ENS_MEMBER_ARGS(a, M), s, smem);
    __syncthreads();
  }
}

#undef ENS_MEMBER_ARGS

// primitive variables of every member's state into its work space
__global__ void __launch_bounds__(256) k_ens_vjp_prims(EnsVjp a, size_t ncell) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  with_cell_member(a.mem, a.nmem, idx, [&](int m) {
    const EnsMember &M = a.mem[m];
    const size_t c = idx - M.off;
    double s[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) s[v] = a.u[5 * M.off + (size_t)v * M.ncell + c];
    double q[4];
    visc_prims(s, a.gamma, q);
    double *Q = a.work + 20 * M.off;
#pragma unroll
    for (int v = 0; v < 4; v++) Q[(size_t)v * M.ncell + c] = q[v];
  });
}

// tiles of all members; tiles0 holds each member's first tile
__global__ void __launch_bounds__(VT) k_ens_visc_vjp_tile(EnsVjp a, const unsigned *__restrict__ tiles0,
                                                         unsigned ntiles, int vks) {
  __shared__ ViscVjpShared sh;
  const unsigned item = blockIdx.x;  // one block per tile (a loop over tiles spills 12 B per lane)
  if (item >= ntiles) return;
  const int m = ens_find(tiles0, a.nmem, item);
  const EnsMember M = a.mem[m];
  const double *Q = a.work + 20 * M.off;
  double *QB = a.work + 20 * M.off + 4 * M.ncell, *GB = a.work + 20 * M.off + 8 * M.ncell;
  visc_vjp_tile(Q, a.lam + 5 * M.off, a.nu_in ? a.nu_in + 5 * M.off : nullptr, M.dt * a.A, M.dt * a.B, QB, GB,
                M.n[0], M.n[1], M.n[2], M.dxg, a.vc, (int)(item - tiles0[m]), vks, sh);
}

template <int DIR>
__global__ void __launch_bounds__(64) k_ens_visc_vjp_ghost(EnsVjp a, const unsigned *__restrict__ first,
                                                            unsigned nitems) {
  const unsigned item = blockIdx.x * blockDim.x + threadIdx.x;
  if (item >= nitems) return;
  const int m = ens_find(first, a.nmem, item);
  const EnsMember M = a.mem[m];
  const double *Q = a.work + 20 * M.off;
  double *QB = a.work + 20 * M.off + 4 * M.ncell;
  visc_vjp_ghost_line<DIR>(Q, a.lam + 5 * M.off, a.nu_in ? a.nu_in + 5 * M.off : nullptr, M.dt * a.A,
                           M.dt * a.B, QB, M.n[0], M.n[1], M.n[2], M.dxg, a.vc, item - first[m]);
}

// ---------------------------------------------------------------------------
bool vjp_supported(const Grid &g, const Scheme &sc) {
  const int lmax = sc.interp == INTERP_CHAR ? VJP_CHAR_LINE_MAX : VJP_LINE_MAX;
  return g.n[0] <= lmax && g.n[1] <= lmax && g.n[2] <= lmax;
}

size_t vjp_work_size(const Grid &g, const Scheme &sc) { return sc.Re > 0 ? 20 * g.ncell : 0; }

// dynamic LDS beyond 64 KiB needs the kernel's opt-in (160 KiB per CU on gfx950)
static void allow_lds(const void *kernel, size_t bytes) {
  if (bytes > 65536) (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// calls f(tag) with the scheme's upwinding and WENO weights as compile-time
// constants tag.upw, tag.weno
template <int U, int Wt>
struct SchemeTag {
  static constexpr int upw = U, weno = Wt;
};

template <class F>
static void with_scheme(const Scheme &sc, F &&f) {
  const bool roe = sc.upwind == UPWIND_ROE;
  switch (sc.weno) {
    case WENO_MAPPED: roe ? f(SchemeTag<UPWIND_ROE, WENO_MAPPED>{}) : f(SchemeTag<UPWIND_RUSANOV, WENO_MAPPED>{}); break;
    case WENO_Z: roe ? f(SchemeTag<UPWIND_ROE, WENO_Z>{}) : f(SchemeTag<UPWIND_RUSANOV, WENO_Z>{}); break;
    case WENO_YC: roe ? f(SchemeTag<UPWIND_ROE, WENO_YC>{}) : f(SchemeTag<UPWIND_RUSANOV, WENO_YC>{}); break;
    case WENO_OPTIMAL:
      roe ? f(SchemeTag<UPWIND_ROE, WENO_OPTIMAL>{}) : f(SchemeTag<UPWIND_RUSANOV, WENO_OPTIMAL>{});
      break;
    default: roe ? f(SchemeTag<UPWIND_ROE, WENO_JS>{}) : f(SchemeTag<UPWIND_RUSANOV, WENO_JS>{}); break;
  }
}

template <int DIR>
static void launch_vjp_dir(const Grid &g, const Scheme &sc, const double *u, const double *lam, const double *nu_in,
                           double ca, double cb, double *nu, double *L, int mode, const double *dxg, hipStream_t st,
                           const double *QB = nullptr, const double *GB = nullptr) {
  const unsigned threads = (unsigned)vjp_threads(g.n[DIR]);
  const unsigned lpb = (unsigned)vjp_lines_per_block((int)threads, g.n[DIR]);
  const unsigned lines = (unsigned)((g.ncell / g.n[DIR] + lpb - 1) / lpb);  // work items
  with_scheme(sc, [&](auto tag) {
    constexpr int U = decltype(tag)::upw, W = decltype(tag)::weno;
    auto go = [&](auto vg) {
      constexpr bool VG = decltype(vg)::value;
      if (sc.interp == INTERP_COMP) {
        const size_t lds = (size_t)VJP_LDS * lpb * g.n[DIR] * sizeof(double);
        allow_lds((const void *)k_rhs_vjp<DIR, U, W, VG>, lds);
        hipLaunchKernelGGL((k_rhs_vjp<DIR, U, W, VG>), dim3(lines), dim3(threads), lds, st, u, lam, nu_in, ca, cb,
                           nu, L, mode, g.n[0], g.n[1], g.n[2], dxg, sc.gamma, sc.eps, QB, GB);
      } else {
        const size_t lds = (size_t)VJP_CHAR_LDS * lpb * g.n[DIR] * sizeof(double);
        allow_lds((const void *)k_rhs_vjp_char<DIR, U, W, VG>, lds);
        hipLaunchKernelGGL((k_rhs_vjp_char<DIR, U, W, VG>), dim3(lines), dim3(threads), lds, st, u, lam, nu_in, ca,
                           cb, nu, L, mode, g.n[0], g.n[1], g.n[2], dxg, sc.gamma, sc.eps, QB, GB);
      }
    };
    // only the x lines of a viscous run add the viscous share
    if (DIR == 0 && QB) go(std::integral_constant<bool, DIR == 0>{});
    else go(std::false_type{});
  });
}

void launch_rhs_vjp(const Grid &g, const Scheme &sc, const double *u, const double *lam, const double *nu_in,
                    double ca, double cb, double *nu, double *L, bool set_L, const double *dxg, double *work,
                    hipStream_t st) {
  const bool visc = sc.Re > 0;
  // z first and x last: the strided z lines take the plain store; the y
  // lines add into nu; the viscous kernels leave the flux and gradient
  // adjoints in QB and GB, and the contiguous x lines add the viscous share
  // and their own into nu (x also into L)
  const int last = L ? (set_L ? VJP_ADD_LSET : VJP_ADD_L) : VJP_ADD;
  launch_vjp_dir<2>(g, sc, u, lam, nu_in, ca, cb, nu, L, VJP_WRITE, dxg, st);
  launch_vjp_dir<1>(g, sc, u, lam, nu_in, ca, cb, nu, L, VJP_ADD, dxg, st);
  // work: Q [4], QB [4], GB [12] (times ncell)
  double *QB = visc ? work + 4 * g.ncell : nullptr, *GB = visc ? work + 8 * g.ncell : nullptr;
  if (visc) {
    double *Q = work;
    const ViscC vc = {sc.gamma, 1.0 / sc.Re, 1.0 / (sc.gamma - 1.0), 1.0 / sc.Pr};
    launch_prims(g, sc, u, Q, st);
    hipLaunchKernelGGL(k_visc_vjp_tile, dim3(visc_tiles(g.n[0], g.n[1], g.n[2], g.vks)), dim3(VT), 0, st, Q, lam, nu_in,
                       ca, cb, QB, GB, g.n[0], g.n[1], g.n[2], dxg, vc, g.vks);
    const unsigned gx = (unsigned)((g.ncell / g.n[0] + 63) / 64), gy = (unsigned)((g.ncell / g.n[1] + 63) / 64),
                   gz = (unsigned)((g.ncell / g.n[2] + 63) / 64);
    hipLaunchKernelGGL(k_visc_vjp_ghost<0>, dim3(gx), dim3(64), 0, st, Q, lam, nu_in, ca, cb, QB, g.n[0], g.n[1],
                       g.n[2], dxg, vc);
    hipLaunchKernelGGL(k_visc_vjp_ghost<1>, dim3(gy), dim3(64), 0, st, Q, lam, nu_in, ca, cb, QB, g.n[0], g.n[1],
                       g.n[2], dxg, vc);
    hipLaunchKernelGGL(k_visc_vjp_ghost<2>, dim3(gz), dim3(64), 0, st, Q, lam, nu_in, ca, cb, QB, g.n[0], g.n[1],
                       g.n[2], dxg, vc);
  }
  launch_vjp_dir<0>(g, sc, u, lam, nu_in, ca, cb, nu, L, last, dxg, st, QB, GB);
}

// a segment of p planes takes p + 2 plane times
int visc_vjp_segment(int count, const int (*n)[3]) { return plane_segment(count, n, 2, visc_tiles); }

bool ens_vjp_supported(const Scheme &sc, const int nmax[3]) {
  Grid g;
  for (int d = 0; d < 3; d++) g.n[d] = nmax[d];
  g.ncell = 1;
  return vjp_supported(g, sc);
}

size_t ens_vjp_work_size(const Scheme &sc, size_t ncell) { return sc.Re > 0 ? 20 * ncell : 0; }

int ens_vjp_threads(int nmax) { return nmax <= 256 ? 256 : vjp_threads(nmax); }
int ens_vjp_lines_per_item(int nmax, int n) { return vjp_lines_per_block(ens_vjp_threads(nmax), n); }

template <int DIR>
static void launch_ens_vjp_dir(const Scheme &sc, const EnsVjpPlan &p, const EnsVjp &a, hipStream_t st) {
  // work items: groups of vjp_lines_per_block(threads, n) lines of a member
  const unsigned items = p.nitems[DIR];
  const unsigned grid = items < 4096 ? items : 4096;  // persistent blocks stride over the items
  const unsigned threads = (unsigned)ens_vjp_threads(p.nmax[DIR]);
  with_scheme(sc, [&](auto tag) {
    constexpr int U = decltype(tag)::upw, W = decltype(tag)::weno;
    auto go = [&](auto vg) {
      constexpr bool VG = decltype(vg)::value;
      if (sc.interp == INTERP_COMP) {
        const size_t lds = (size_t)VJP_LDS * threads * sizeof(double);
        allow_lds((const void *)k_ens_rhs_vjp<DIR, U, W, VG>, lds);
        hipLaunchKernelGGL((k_ens_rhs_vjp<DIR, U, W, VG>), dim3(grid), dim3(threads), lds, st, a, p.items0[DIR],
                           items);
      } else {
        const size_t lds = (size_t)VJP_CHAR_LDS * threads * sizeof(double);
        allow_lds((const void *)k_ens_rhs_vjp_char<DIR, U, W, VG>, lds);
        hipLaunchKernelGGL((k_ens_rhs_vjp_char<DIR, U, W, VG>), dim3(grid), dim3(threads), lds, st, a,
                           p.items0[DIR], items);
      }
    };
    // only the x lines of a viscous ensemble add the viscous share (a.work)
    if (DIR == 0 && a.work) go(std::integral_constant<bool, DIR == 0>{});
    else go(std::false_type{});
  });
}

void launch_ens_rhs_vjp(const Scheme &sc, const EnsVjpPlan &p, const double *u, const double *lam,
                        const double *nu_in, double A, double B, double *nu, double *L, bool set_L, double *work,
                        hipStream_t st) {
  EnsVjp a;
  a.mem = p.mem;
  a.nmem = p.nmem;
  a.u = u;
  a.lam = lam;
  a.nu_in = nu_in;
  a.A = A;
  a.B = B;
  a.nu = nu;
  a.L = L;
  a.work = work;
  a.gamma = sc.gamma;
  a.eps = sc.eps;
  a.vc = {sc.gamma, sc.Re > 0 ? 1.0 / sc.Re : 0.0, 1.0 / (sc.gamma - 1.0), 1.0 / sc.Pr};
  const bool visc = sc.Re > 0;
  // the order of the single grid: z (plain store), y, the viscous kernels, x
  a.mode = VJP_WRITE;
  launch_ens_vjp_dir<2>(sc, p, a, st);
  a.mode = VJP_ADD;
  launch_ens_vjp_dir<1>(sc, p, a, st);
  if (visc) {
    const unsigned nb = (unsigned)((p.ncell + 255) / 256);
    hipLaunchKernelGGL(k_ens_vjp_prims, dim3(nb), dim3(256), 0, st, a, p.ncell);
    hipLaunchKernelGGL(k_ens_visc_vjp_tile, dim3(p.ntiles), dim3(VT), 0, st, a, p.tiles0, p.ntiles, p.vks);
    hipLaunchKernelGGL(k_ens_visc_vjp_ghost<0>, dim3((p.nlines[0] + 63) / 64), dim3(64), 0, st, a, p.lines0[0],
                       p.nlines[0]);
    hipLaunchKernelGGL(k_ens_visc_vjp_ghost<1>, dim3((p.nlines[1] + 63) / 64), dim3(64), 0, st, a, p.lines0[1],
                       p.nlines[1]);
    hipLaunchKernelGGL(k_ens_visc_vjp_ghost<2>, dim3((p.nlines[2] + 63) / 64), dim3(64), 0, st, a, p.lines0[2],
                       p.nlines[2]);
  }
  // the x lines add the viscous share (QB, GB of a.work) before their own
  a.mode = L ? (set_L ? VJP_ADD_LSET : VJP_ADD_L) : VJP_ADD;
  launch_ens_vjp_dir<0>(sc, p, a, st);
}

}  // namespace hm
