// hm_pass.hip -- fused direction passes of the NS3D WENO5 right-hand side
// and RK4 stage (gfx950, FP64).
//
// One RK stage is three launches, one per direction (after the viscous-term
// kernel of hm_kernels.hip when the run is viscous):
//   pass x:  R = dxinv (F_{i+1/2} - F_{i-1/2})
//   pass y:  R = R + dyinv (G_{j+1/2} - G_{j-1/2})
//   pass z:  r = -(R + dzinv (H_{k+1/2} - H_{k-1/2})) + par,
//            then the stage's update (or r itself for hm_rhs)
// i.e. rhs = -hyp + par of TimeRHSFunctionExplicit.c:88-93 summed in the
// reference's order, with the hyperbolic term of HyperbolicFunction.c:75-101
// accumulated direction by direction and the parabolic term par of
// NavierStokes3DParabolicFunction.c:50-325.
//
// Each pass stages the cells of its pencils in LDS once, evaluates what
// depends on one cell alone (its flux, the factors of the Roe average) once,
// computes the interface fluxes (WENO5, component-wise or characteristic, with Roe or Rusanov
// upwinding) from LDS, and differences them in LDS: interface fluxes never
// reach HBM.
//  * x pass: one wavefront per x-line, chunks of 64 interfaces along x.
//  * y, z passes: a block owns 64 consecutive columns (x fastest) of the
//    plane across y (z), which may span several x-rows of that plane, and
//    marches along y (z) four rows per step, with a 9-row ring of cell data
//    and a 5-row ring of interface fluxes in LDS; on grids with few columns
//    it marches one segment of its lines (march_segments).
// Output of cell c needs the interfaces c-1/2 and c+1/2; a step emits the
// cells one row (lane) behind its interfaces, and the last cell of a line,
// whose right interface is the periodic image of interface 0, is emitted
// after the march.
//
// Restatements relative to the reference arithmetic (equal in exact
// arithmetic; rounding-level differences only):
//  * 1/rho, the weights' normalisation, the Roe-average weights and the
//    square roots use hardware estimates refined to full precision (nr_rcp,
//    nr_rsq); velocities are m * (1/rho).
//  * The mass flux of a cell is its momentum m_d (the reference forms
//    rho * (m_d / rho)).
//  * An interpolated value is the value of the cell next to the interface
//    plus a correction formed from first differences (weno5_lr).
//  * The values the solution's interpolant takes are u itself: the modified
//    solution P/(gamma-1) + rho |v|^2/2 that the reference interpolates
//    (NavierStokes3DModifiedSolution.c:31-70, gravity 0) is u's energy.
//  * What depends on one cell alone (the factors of the Roe average, the
//    Rusanov speed) is formed once per cell; s H = (e + P)/s with s = sqrt(rho).
//  * The characteristic projections use the structure of the left
//    eigenvectors (navierstokes3d.h:288-374): with
//    w = v.x_{1..3} - x_4, rows 0, d and 4 are
//      L00 x0 + (g-1)/a^2 w,  Ld0 x0 - (g-1)/(2a^2) w -/+ 1/(2a) x_d,
//    and the two shear rows have two non-zero entries; the product with the
//    right eigenvectors (navierstokes3d.h:384-470) is expanded the same
//    way.  The speed of sound of the Roe state is sqrt((g-1)(H - |v|^2/2)),
//    the reference's sqrt(g P / rho) with P from H.
//  * Only differences between cells are projected; the mean of the two
//    cells' fluxes passes L and R unchanged (L R = I).
//
// FP64 issue bounds these passes: a wave64 FP64 instruction takes a SIMD 4
// cycles, and two waves per SIMD keep it busy 60-67% of the time (y), three
// 73-81% (x); the z pass at 256^3 also moves 224 B per cell, at close to the
// rate of a copy.
// The forms above take 946 FP64 (1050 VALU) instructions per interface of the
// characteristic JS/Roe x pass and 744 (843) of the component-wise JS/Rusanov
// one (915 and 1016 of the former since the reciprocals take one cubic step),
// where weights from second and one-sided differences, projected values and
// Roe averages formed at each interface took 1356 (1474) and 1072 (1188):
// 256^3 RK4 step 15.55 -> 13.54 ms, 201^3 SSPRK3/YC step 5.20 -> 4.18 ms,
// 64-member Euler ensemble 18.7 -> 15.2 ms per step by that alone.  At 256^3
// the characteristic passes now take 0.72 (x), 0.76 (y) and 0.92 ms (z).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "hm_device.h"
#include "hm_internal.h"

namespace hm {

namespace {

// per-cell LDS record: U0..U4, F1..F4 (F0 = U_d), 1/sqrt(rho), sqrt(rho) H
// and, for Rusanov upwinding, the cell's speed c + |v_d|.  What an interface
// needs of one cell alone (the factors of the Roe average, the speed) is so
// formed once per cell and not at both of its interfaces.
constexpr int nq(int upw) { return upw == UPWIND_RUSANOV ? 12 : 11; }

struct PassConst {
  int n[3];
  int seg;    // cells per march segment along the pass direction (y, z passes)
  size_t ncell;
  double gamma, gm1, eps34;  // eps34 = 3/4 of the WENO epsilon
  const double *dxg;  // ghosted dxinv x|y|z
};

struct PassIO {
  const double *U;    // stage state
  double *R;          // hyperbolic-term accumulator
  const double *par;  // viscous term, par[c*ncell + cell], c = momentum x, y, z, energy
  double *Q;
  StageUpdate upd;
  int visc, mode;
};

// per-cell record of the pass direction (NavierStokes3DFlux.c:23-57)
template <int DIR, int UPW>
__device__ __forceinline__ void cell_data(const double u[NV], const PassConst &k, double c[nq(UPW)]) {
  const double rho = u[0];
  const double ir = rho == 0.0 ? 0.0 : nr_rcp(rho), is = rho == 0.0 ? 0.0 : nr_rsq(rho);
  const double vx = u[1] * ir, vy = u[2] * ir, vz = u[3] * ir;
  const double vsq = vx * vx + vy * vy + vz * vz;
  const double P = (u[4] - 0.5 * rho * vsq) * k.gm1;
  const double vn = DIR == 0 ? vx : (DIR == 1 ? vy : vz);
  const double m = u[DIR + 1];
#pragma unroll
  for (int q = 0; q < NV; q++) c[q] = u[q];
  c[5] = m * vx + (DIR == 0 ? P : 0.0);
  c[6] = m * vy + (DIR == 1 ? P : 0.0);
  c[7] = m * vz + (DIR == 2 ? P : 0.0);
  c[8] = (u[4] + P) * vn;
  c[9] = is;
  c[10] = (u[4] + P) * is;
  if (UPW == UPWIND_RUSANOV) c[11] = nr_sqrt(k.gamma * P * ir) + fabs(vn);
}

// One side of WENO5 at an interface: twice the difference between the
// interpolated value and the value of the upwind cell next to the interface
// (include/interpolation.h:265-500, Interp1PrimFifthOrderWENO.c:146-158).
// l1..l3 = 3/4 (beta_k + eps); p1..p3 = the candidates' differences from that
// cell's value times 2, 12, 6 (the ratios 1, 6, 3 of the optimal weights);
// d4 the stencil's 4th difference (YC).  W selects the weights:
//  * WENO_JS:     a_k = c_k / (beta_k + eps)^2
//  * WENO_Z:      a_k = c_k (1 + (tau / (beta_k + eps))^2), tau = |beta_1 - beta_3|
//  * WENO_YC:     the same with tau = d4^2
//  * WENO_MAPPED: the JS weights w mapped by
//                 w (c + c^2 - 3 c w + w^2) / (c^2 + w (1 - 2c)) and renormalised
//  * WENO_OPTIMAL: the constant weights of no_limiting
//    (WENOFifthOrderInitializeWeights.c:33-228, HyperbolicFunction.c:62)
// The a_k are multiplied through by the product of all (beta_k + eps)^2 and
// applied with one reciprocal (two for the mapped weights).
template <int W>
__device__ __forceinline__ double weno_side(double l1, double l2, double l3, double p1, double p2, double p3,
                                            double d4) {
  if (W == WENO_OPTIMAL) return 0.1 * (p1 + p2 + p3);
  const double q1 = l2 * l3, q2 = l1 * l3, q3 = l1 * l2;
  double a1 = q1 * q1, a2 = q2 * q2, a3 = q3 * q3;
  if (W == WENO_Z || W == WENO_YC) {
    // tau in the scale of l; the YC tau is formed from the data itself
    const double tau = W == WENO_Z ? l3 - l1 : 0.75 * (d4 * d4);
    const double t2 = tau * tau;
    a1 *= l1 * l1 + t2;
    a2 *= l2 * l2 + t2;
    a3 *= l3 * l3 + t2;
  }
  const double k3 = scalar(3.0);
  if (W == WENO_MAPPED) {
    const double c1 = 0.1, c2 = 0.6, c3 = 0.3;
    const double in = nr_rcp(a1 + k3 * (2.0 * a2 + a3));
    const double w1 = a1 * in, w2 = a2 * (6.0 * in), w3 = a3 * (3.0 * in);
    const double n1 = w1 * (c1 + c1 * c1 - 3 * c1 * w1 + w1 * w1), e1 = c1 * c1 + w1 * (1.0 - 2.0 * c1);
    const double n2 = w2 * (c2 + c2 * c2 - 3 * c2 * w2 + w2 * w2), e2 = c2 * c2 + w2 * (1.0 - 2.0 * c2);
    const double n3 = w3 * (c3 + c3 * c3 - 3 * c3 * w3 + w3 * w3), e3 = c3 * c3 + w3 * (1.0 - 2.0 * c3);
    // n_k / e_k multiplied through by e1 e2 e3
    a1 = n1 * (e2 * e3);
    a2 = n2 * (e1 * e3);
    a3 = n3 * (e1 * e2);
    return (a1 * p1 + a2 * ((1.0 / 6.0) * p2) + a3 * ((1.0 / 3.0) * p3)) * nr_rcp(a1 + a2 + a3);
  }
  return (a1 * p1 + a2 * p2 + a3 * p3) * nr_rcp(a1 + k3 * (2.0 * a2 + a3));
}

// WENO5 on both sides of one interface from the five first differences
// D_s = b_{s+1} - b_s of cells I-3..I+2: the left-biased value is
// b_2 + cl/2, the right-biased one (the mirror image,
// WENOFifthOrderCalculateWeights.c:166-177) b_3 + cr/2.  With e the second
// difference of a candidate stencil and x its first difference nearest the
// interface, the smoothness indicators are
//   3/4 beta = e^2 + 3/4 x (x + e)       (outer stencils; e towards x)
//   3/4 beta = e^2 + 3/4 x y             (middle stencil, differences x, y),
// equal to 13/16 e^2 + 3/16 (..)^2 of the textbook form: 21 operations for
// all six with eps, where that form takes 38.
template <int W>
__device__ __forceinline__ void weno5_lr(const double (&D)[5], double eps34, double &cl, double &cr) {
  const double k34 = scalar(0.75), k23 = scalar(2.0 / 3.0);
  const double e0 = D[1] - D[0], e1 = D[2] - D[1], e2 = D[3] - D[2], e3 = D[4] - D[3];
  const double s0 = e0 * e0 + eps34, s1 = e1 * e1 + eps34, s2 = e2 * e2 + eps34, s3 = e3 * e3 + eps34;
  const double x1 = k34 * D[1], x2 = k34 * D[2], x3 = k34 * D[3];
  const double l1 = x1 * (D[1] + e0) + s0, l2 = x1 * D[2] + s1, l3 = x2 * (D[2] - e2) + s2;
  const double r1 = x3 * (D[3] - e3) + s3, r2 = x3 * D[2] + s2, r3 = x2 * (D[2] + e1) + s1;
  const double F = 4.0 * D[2];
  const double tl = W == WENO_YC ? (e0 + e2) - 2.0 * e1 : 0.0;
  const double tr = W == WENO_YC ? (e1 + e3) - 2.0 * e2 : 0.0;
  cl = weno_side<W>(l1, l2, l3, k23 * e0 + D[1], 2.0 * D[1] + F, F - D[3], tl);
  cr = -weno_side<W>(r1, r2, r3, D[3] - k23 * e3, 2.0 * D[3] + F, F - D[1], tr);
}

// Roe-averaged state of two cells (navierstokes3d.h:144-169) and the
// eigen-structure constants of the DIR flux Jacobian there.
struct RoeState {
  double vx, vy, vz, vn, a, ek, h0;
  double L00, Lm0, L40, k0, kh, aih;  // left-eigenvector entries (see top)
};

// L(q), R(q): quantity q of the records of the cells left and right of the
// interface.  With s = sqrt(rho) of each cell, the averages are
// (s_L x_L + s_R x_R) / (s_L + s_R), s v = m / s and s H = (e + P) / s.
template <int DIR, class LQ, class RQ>
__device__ __forceinline__ RoeState roe_state(const LQ &L, const RQ &R, const PassConst &k) {
  RoeState s;
  const double iL = L(9), iR = R(9);
  const double inv = nr_rcp(L(0) * iL + R(0) * iR);
  s.vx = (L(1) * iL + R(1) * iR) * inv;
  s.vy = (L(2) * iL + R(2) * iR) * inv;
  s.vz = (L(3) * iL + R(3) * iR) * inv;
  const double H = (L(10) + R(10)) * inv;
  s.ek = 0.5 * (s.vx * s.vx + s.vy * s.vy + s.vz * s.vz);
  const double a2 = (H - s.ek) * k.gm1;
  const double ra = nr_rsq(a2);  // 1/a
  s.a = sqrt_of(a2, ra);
  s.vn = DIR == 0 ? s.vx : (DIR == 1 ? s.vy : s.vz);
  s.h0 = H;
  s.aih = 0.5 * ra;
  s.k0 = k.gm1 * (ra * ra);
  s.kh = 0.5 * s.k0;
  const double gek = s.kh * s.ek, avn = s.aih * s.vn;
  s.L00 = 1.0 - 2.0 * gek;
  s.Lm0 = gek + avn;
  s.L40 = gek - avn;
  return s;
}

// rows 0, d, 4 of L x (u-a wave in row d = DIR+1)
template <int DIR>
__device__ __forceinline__ void proj_acoustic(const RoeState &s, double x0, double x1, double x2, double x3,
                                              double x4, double &p0, double &pm, double &p4) {
  const double w = s.vx * x1 + s.vy * x2 + s.vz * x3 - x4;
  const double xm = DIR == 0 ? x1 : (DIR == 1 ? x2 : x3);
  const double t = s.kh * w;
  p0 = s.L00 * x0 + s.k0 * w;
  pm = s.Lm0 * x0 - (t + s.aih * xm);
  p4 = s.L40 * x0 + (s.aih * xm - t);
}

// the two shear rows of L x, in row order
template <int DIR>
__device__ __forceinline__ void proj_shear(const RoeState &s, double x0, double x1, double x2, double x3,
                                           double &pa, double &pb) {
  if (DIR == 0) {        // rows 2, 3: (vy, 0, -1, 0, 0), (-vz, 0, 0, 1, 0)
    pa = s.vy * x0 - x2;
    pb = x3 - s.vz * x0;
  } else if (DIR == 1) { // rows 1, 3: (-vx, 1, 0, 0, 0), (vz, 0, 0, -1, 0)
    pa = x1 - s.vx * x0;
    pb = s.vz * x0 - x3;
  } else {               // rows 1, 2: (vx, -1, 0, 0, 0), (-vy, 0, 1, 0, 0)
    pa = s.vx * x0 - x1;
    pb = x2 - s.vy * x0;
  }
}

// f = R g, with g0 (entropy), gm (u-a), g4 (u+a), ga, gb (shear rows in
// row order)
template <int DIR>
__device__ __forceinline__ void right_mult(const RoeState &s, double g0, double gm, double g4, double ga,
                                           double gb, double f[NV]) {
  const double sum = g0 + gm + g4;
  const double dif = s.a * (g4 - gm);
  f[0] = sum;
  f[1] = s.vx * sum;
  f[2] = s.vy * sum;
  f[3] = s.vz * sum;
  f[DIR + 1] += dif;
  double e = s.ek * g0 + s.h0 * (gm + g4) + s.vn * dif;
  if (DIR == 0) {        // columns 2, 3: (0,0,-1,0,-vy), (0,0,0,1,vz)
    f[2] -= ga;
    f[3] += gb;
    e += s.vz * gb - s.vy * ga;
  } else if (DIR == 1) { // columns 1, 3: (0,1,0,0,vx), (0,0,0,-1,-vz)
    f[1] += ga;
    f[3] -= gb;
    e += s.vx * ga - s.vz * gb;
  } else {               // columns 1, 2: (0,-1,0,0,-vx), (0,0,1,0,vy)
    f[1] -= ga;
    f[2] += gb;
    e += s.vy * gb - s.vx * ga;
  }
  f[4] = e;
}

// Interface flux at I-1/2 from the LDS records of cells I-3..I+2;
// ld(s, q) returns quantity q of cell I-3+s.  The flux is written as the mean
// of the two cells' fluxes plus a correction from the differences between
// neighbouring cells.  In the characteristic scheme only the differences are
// projected: L R = I, so the mean passes through L and R unchanged.
template <int DIR, int INTERP, int UPW, int W, class LD>
__device__ __forceinline__ void iface(const LD &ld, const PassConst &k, double fI[NV]) {
  const RoeState s = roe_state<DIR>([&](int q) { return ld(2, q); }, [&](int q) { return ld(3, q); }, k);
  double alpha = 0.0;
  if (UPW == UPWIND_RUSANOV) {  // NavierStokes3DUpwind.c:349-420
    const double cL = ld(2, 11), cR = ld(3, 11), aA = s.a + fabs(s.vn);
    alpha = fmax(fmax(cL, cR), fmax(cR, aA));
  }
  // half of |lambda|
  const double l0 = 0.5 * (UPW == UPWIND_ROE ? harten(s.vn) : alpha);
  const double lm = UPW == UPWIND_ROE ? 0.5 * harten(s.vn - s.a) : l0;
  const double l4 = UPW == UPWIND_ROE ? 0.5 * harten(s.vn + s.a) : l0;
  double cl, cr;

  if (INTERP == INTERP_CHAR) {
    // fluxes, then states: projected differences of the five fields (rows 0,
    // d, 4, then the two shear rows; WENOFifthOrderCalculateWeightsChar,
    // Interp1PrimFifthOrderWENOChar.c:86-198)
    double g[5];
#pragma unroll
    for (int part = 0; part < 2; part++) {
      double d[5][5];
#pragma unroll
      for (int p = 0; p < 5; p++) {
        double x[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const int q = part == 1 ? v : (v == 0 ? DIR + 1 : 4 + v);
          x[v] = ld(p + 1, q) - ld(p, q);
        }
        proj_acoustic<DIR>(s, x[0], x[1], x[2], x[3], x[4], d[0][p], d[1][p], d[2][p]);
        proj_shear<DIR>(s, x[0], x[1], x[2], x[3], d[3][p], d[4][p]);
      }
#pragma unroll
      for (int f = 0; f < 5; f++) {
        weno5_lr<W>(d[f], k.eps34, cl, cr);
        if (part == 0) g[f] = 0.25 * (cl + cr);
        else g[f] -= (f == 1 ? lm : (f == 2 ? l4 : l0)) * (d[f][2] + 0.5 * (cr - cl));
      }
    }
    right_mult<DIR>(s, g[0], g[1], g[2], g[3], g[4], fI);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int q = v == 0 ? DIR + 1 : 4 + v;
      fI[v] += 0.5 * (ld(2, q) + ld(3, q));
    }
  } else {
    // component-wise (Interp1PrimFifthOrderWENO.c:74-168)
    double fh[NV], du[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      double b[6], D[5];
#pragma unroll
      for (int p = 0; p < 6; p++) b[p] = ld(p, v == 0 ? DIR + 1 : 4 + v);
#pragma unroll
      for (int p = 0; p < 5; p++) D[p] = b[p + 1] - b[p];
      weno5_lr<W>(D, k.eps34, cl, cr);
      fh[v] = 0.5 * ((b[2] + b[3]) + 0.5 * (cl + cr));
#pragma unroll
      for (int p = 0; p < 6; p++) b[p] = ld(p, v);
#pragma unroll
      for (int p = 0; p < 5; p++) D[p] = b[p + 1] - b[p];
      weno5_lr<W>(D, k.eps34, cl, cr);
      du[v] = D[2] + 0.5 * (cr - cl);
    }
    if (UPW == UPWIND_RUSANOV) {
#pragma unroll
      for (int v = 0; v < NV; v++) fI[v] = fh[v] - l0 * du[v];
    } else {
      // R |Lambda|/2 L (uR - uL) (NavierStokes3DUpwind.c:40-124)
      double p0, pm, p4, pa, pb;
      proj_acoustic<DIR>(s, du[0], du[1], du[2], du[3], du[4], p0, pm, p4);
      proj_shear<DIR>(s, du[0], du[1], du[2], du[3], pa, pb);
      double d[NV];
      right_mult<DIR>(s, l0 * p0, lm * pm, l4 * p4, l0 * pa, l0 * pb, d);
#pragma unroll
      for (int v = 0; v < NV; v++) fI[v] = fh[v] - d[v];
    }
  }
}

// The hyperbolic-term accumulator R, read and written plainly by the
// per-pass kernels.  In the one-launch-per-stage kernel (COH) blocks hand R
// to each other within the launch, so there R goes through agent-scope
// relaxed atomics: coherent loads and write-through stores (sc1) that
// bypass the stale lines of the eight non-coherent XCD L2s.  The stage
// kernel's dependency counters then need no L2 write-back or invalidate.
template <bool COH>
__device__ __forceinline__ double load_r(const double *p) {
  if (COH) return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return *p;
}
template <bool COH>
__device__ __forceinline__ void store_r(double *p, double v) {
  if (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// Inputs of cell idx's output that come from global memory: its dxinv, the
// hyperbolic term so far (y, z), the viscous term and the update's operands (z).
// The marching passes issue these loads in one block with the next ring
// row's, so that their latencies overlap.
struct EmitIn {
  double dxi, par[NV], rin[NV], a[NV], b[NV], c[NV];
};

template <int DIR, bool COH = false>
__device__ __forceinline__ EmitIn emit_load(const PassConst &k, const PassIO &io, size_t idx, int pos) {
  EmitIn in;
  in.dxi = k.dxg[(DIR >= 1 ? k.n[0] + 6 : 0) + (DIR == 2 ? k.n[1] + 6 : 0) + 3 + pos];
#pragma unroll
  for (int v = 0; v < NV; v++) in.par[v] = in.rin[v] = in.a[v] = in.b[v] = in.c[v] = 0.0;
  if (DIR > 0)
#pragma unroll
    for (int v = 0; v < NV; v++) in.rin[v] = load_r<COH>(io.R + (size_t)v * k.ncell + idx);
  if (DIR == 2 && io.visc && io.mode != OUT_HYP)
#pragma unroll
    for (int c = 0; c < 4; c++) in.par[c + 1] = io.par[(size_t)c * k.ncell + idx];
  // the operands of the update, one uniform branch per kind, each with its
  // loads in one block
  if (DIR == 2 && io.mode == OUT_STAGE) {
    if (io.upd.kind == UPD_MIX) {
#pragma unroll
      for (int v = 0; v < NV; v++) in.a[v] = io.upd.a0[(size_t)v * k.ncell + idx];
    } else if (io.upd.kind == UPD_RK4) {
#pragma unroll
      for (int v = 0; v < NV; v++) {
        in.a[v] = io.upd.a0[(size_t)v * k.ncell + idx];
        in.b[v] = io.upd.a1[(size_t)v * k.ncell + idx];
        in.c[v] = io.upd.a2[(size_t)v * k.ncell + idx];
      }
    }
  }
  return in;
}

// Finish cell idx of the pass: flux difference and the pass's output.  uc is
// the cell's stage state (z pass).  Every mode and kind of update stores one
// array through one pointer: the compiler merged the stores of branches that
// chose among outputs into one store whose address register one path never
// set.
template <int DIR, bool COH = false>
__device__ __forceinline__ void emit_store(const PassConst &k, const PassIO &io, size_t idx, const EmitIn &in,
                                           const double (&fm)[NV], const double (&fp)[NV], const double (&uc)[NV]) {
  double r[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const double h = in.dxi * (fp[v] - fm[v]);
    // hyp = (hx + hy) + hz and rhs = (-hyp) + par (TimeRHSFunctionExplicit.c:88-93)
    if (DIR == 0) r[v] = h;
    else if (DIR == 1 || io.mode == OUT_HYP) r[v] = in.rin[v] + h;
    else r[v] = (-(in.rin[v] + h)) + in.par[v];
  }
  if (DIR < 2) {
#pragma unroll
    for (int v = 0; v < NV; v++) store_r<COH>(io.R + (size_t)v * k.ncell + idx, r[v]);
    return;
  }
  if (io.mode == OUT_STAGE) {
    const double c = io.upd.c;
    if (io.upd.kind == UPD_SELF) {
#pragma unroll
      for (int v = 0; v < NV; v++) r[v] = uc[v] + c * r[v];
    } else if (io.upd.kind == UPD_MIX) {
#pragma unroll
      for (int v = 0; v < NV; v++) r[v] = in.a[v] + (io.upd.k * (uc[v] - in.a[v]) + c * r[v]);
    } else {
#pragma unroll
      for (int v = 0; v < NV; v++)
        r[v] = in.b[v] + (((in.c[v] - in.b[v]) + (uc[v] - in.a[v])) * (1.0 / 3.0) + c * r[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < NV; v++) io.upd.out[(size_t)v * k.ncell + idx] = r[v];
  if (io.visc && io.mode == OUT_STAGE) {
    // primitive variables (u, v, w, T) of the new state for the next
    // viscous-term evaluation (NavierStokes3DParabolicFunction.c:85-108)
    double q[4];
    visc_prims(r, k.gamma, q);
#pragma unroll
    for (int c = 0; c < 4; c++) io.Q[(size_t)c * k.ncell + idx] = q[c];
  }
}

template <int DIR, bool COH = false>
__device__ __forceinline__ void emit(const PassConst &k, const PassIO &io, size_t idx, int pos,
                                     const double (&fm)[NV], const double (&fp)[NV], const double (&uc)[NV]) {
  emit_store<DIR, COH>(k, io, idx, emit_load<DIR, COH>(k, io, idx, pos), fm, fp, uc);
}

// ---------------------------------------------------------------------------
// x pass: one wavefront per x-line, LPB lines per block
// ---------------------------------------------------------------------------
constexpr int XCH = 64;        // interfaces per chunk
constexpr int XNC = XCH + 6;   // cells per chunk
constexpr int XPAD = 72;

template <int LPB, int UPW>
struct XShared {
  double sC[LPB][nq(UPW)][XPAD];
  double sF[LPB][NV][XCH + 1];  // slot 0: fI[x0-1]; slot 1+l: fI[x0+l]
  double sF0[LPB][NV];          // fI[0] of the line
};

// lines LPB*group .. LPB*group + LPB-1 of the grid (line = j + ny*k)
template <int INTERP, int UPW, int LPB, int W, bool COH = false>
__device__ __forceinline__ void pass_x_body(const PassConst &k, const PassIO &io, size_t group,
                                            XShared<LPB, UPW> &sh) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = k.n[0];
  const size_t nlines = (size_t)k.n[1] * k.n[2];
  const size_t line = group * LPB + w;
  const bool active = line < nlines;
  const size_t base = (active ? line : 0) * (size_t)nx;
  int x0 = 0;
  for (; x0 < nx; x0 += XCH) {
    if (x0 > 0) {
      // carry fI[x0-1] into slot 0 (the previous chunk's output phase is done)
      if (lane < NV) sh.sF[w][lane][0] = sh.sF[w][lane][XCH];
    }
    const int ncells = min(XNC, nx + 6 - x0);
    for (int c = lane; c < ncells; c += 64) {
      const size_t cell = base + wrap(x0 - 3 + c, nx);
      double u[NV], cd[nq(UPW)];
#pragma unroll
      for (int v = 0; v < NV; v++) u[v] = io.U[(size_t)v * k.ncell + cell];
      cell_data<0, UPW>(u, k, cd);
#pragma unroll
      for (int q = 0; q < nq(UPW); q++) sh.sC[w][q][c] = cd[q];
    }
    __syncthreads();
    if (active && x0 + lane < nx) {
      auto ld = [&](int s, int q) { return sh.sC[w][q][lane + s]; };
      double f[NV];
      iface<0, INTERP, UPW, W>(ld, k, f);
#pragma unroll
      for (int v = 0; v < NV; v++) sh.sF[w][v][lane + 1] = f[v];
      if (x0 == 0 && lane == 0)
#pragma unroll
        for (int v = 0; v < NV; v++) sh.sF0[w][v] = f[v];
    }
    __syncthreads();
    const int cell = x0 - 1 + lane;
    if (active && cell >= 0 && cell <= nx - 2) {
      double fm[NV], fp[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) {
        fm[v] = sh.sF[w][v][lane];
        fp[v] = sh.sF[w][v][lane + 1];
      }
      emit<0, COH>(k, io, base + cell, cell, fm, fp, fm);
    }
    __syncthreads();
  }
  // last cell: fI[nx-1] of the last chunk, fI[nx] = fI[0]
  x0 -= XCH;
  if (active && lane == 0) {
    double fm[NV], fp[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      fm[v] = sh.sF[w][v][nx - x0];
      fp[v] = sh.sF0[w][v];
    }
    emit<0, COH>(k, io, base + nx - 1, nx - 1, fm, fp, fm);
  }
}

// ---------------------------------------------------------------------------
// y, z passes: 64 columns marching along DIR, MR rows per step
// ---------------------------------------------------------------------------
constexpr int MW = 64;  // columns

template <int MR, int UPW>
struct MShared {
  static constexpr int NRING = MR + 5;  // cell rows t0-3 .. t0+MR+1
  static constexpr int NFR = MR + 1;    // interface rows t0-1 .. t0+MR-1
  double sC[nq(UPW)][NRING][MW];
  double sF[NV][NFR][MW];
  double sF0[NV][MW];
};

// item = group + groups * segment: columns MW*group .. MW*group + MW-1 of the
// plane across DIR, and the cells c0 .. c1-1 of the segment along DIR.  A
// segment that is a whole line keeps the flux of interface 0 for its last
// cell; any other evaluates interfaces c0 .. c1, one more than its cells,
// and starts on six rows of its neighbour.
template <int DIR, int INTERP, int UPW, int MR, int W, bool COH = false>
__device__ __forceinline__ void pass_m_body(const PassConst &k, const PassIO &io, size_t item,
                                            MShared<MR, UPW> &sh) {
  constexpr int NRING = MShared<MR, UPW>::NRING, NFR = MShared<MR, UPW>::NFR;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = k.n[0], ny = k.n[1];
  const int n = k.n[DIR];
  // the 64 lanes take 64 consecutive columns c = i + nx*o of the plane
  // across DIR (o = z index in the y pass, y index in the z pass)
  const size_t ncol = k.ncell / n;
  const unsigned groups = (unsigned)((ncol + MW - 1) / MW);
  const bool whole = k.seg >= n;
  const unsigned sg = whole ? 0u : (unsigned)item / groups;
  const int c0 = (int)sg * k.seg, c1 = min(c0 + k.seg, n);
  const int tend = whole ? n : c1 + 1;        // interfaces c0 .. tend-1
  const int elast = whole ? n - 2 : c1 - 1;   // last cell the march emits
  const size_t c = ((unsigned)item - sg * groups) * (size_t)MW + lane;
  const bool col = c < ncol;
  const size_t line = col ? c : ncol - 1;
  const size_t o = line / nx;
  const size_t stride = DIR == 1 ? (size_t)nx : (size_t)nx * ny;
  const size_t cbase = DIR == 1 ? o * nx * ny + (line - o * nx) : line;  // cell at position 0

  auto load_row = [&](int r) {  // r in [c0-3, c0+MR+1]
    const size_t cell = cbase + (size_t)wrap(r, n) * stride;
    double u[NV], cd[nq(UPW)];
#pragma unroll
    for (int v = 0; v < NV; v++) u[v] = io.U[(size_t)v * k.ncell + cell];
    cell_data<DIR, UPW>(u, k, cd);
    const int slot = (r + NRING) % NRING;
#pragma unroll
    for (int q = 0; q < nq(UPW); q++) sh.sC[q][slot][lane] = cd[q];
  };

  // ring row r's state, loaded one march step ahead in the same block as
  // the output's operands, so that their latencies overlap
  auto fetch_row = [&](int r, double (&u)[NV]) {  // r in [-3, n+MR+1]
    const size_t cell = cbase + (size_t)wrap(r, n) * stride;
#pragma unroll
    for (int v = 0; v < NV; v++) u[v] = io.U[(size_t)v * k.ncell + cell];
  };
  auto stage_row = [&](int r, const double (&u)[NV]) {
    double cd[nq(UPW)];
    cell_data<DIR, UPW>(u, k, cd);
    const int slot = (r + NRING) % NRING;
#pragma unroll
    for (int q = 0; q < nq(UPW); q++) sh.sC[q][slot][lane] = cd[q];
  };

  // rows c0-3..c0+MR+1
  for (int r = w; r < MR + 5; r += MR) load_row(c0 + r - 3);
  for (int t0 = c0; t0 < tend; t0 += MR) {
    __syncthreads();
    const int t = t0 + w;
    double uc[NV] = {0, 0, 0, 0, 0};  // stage state of cell t-1, which this wavefront emits
    if (t < tend) {
      const int sl0 = (t - 3 + NRING) % NRING;
      auto ld = [&](int s, int q) {
        int sl = sl0 + s;
        sl = sl >= NRING ? sl - NRING : sl;
        return sh.sC[q][sl][lane];
      };
      double f[NV];
      iface<DIR, INTERP, UPW, W>(ld, k, f);
      if (DIR == 2)
#pragma unroll
        for (int v = 0; v < NV; v++) uc[v] = ld(2, v);
      const int fs = t % NFR;
#pragma unroll
      for (int v = 0; v < NV; v++) sh.sF[v][fs][lane] = f[v];
      if (t == 0)
#pragma unroll
        for (int v = 0; v < NV; v++) sh.sF0[v][lane] = f[v];
    }
    const int e = t0 - 1 + w;  // row emitted by this wavefront
    const bool emits = col && e >= c0 && e <= elast;
    __syncthreads();
    // the next step's ring row (its slot held row t0-3+w, which no later
    // step reads) and the output's operands, loaded by every lane (a stand-in
    // row 0 after the last step, output rows clamped into the line) so that
    // no divergent branch separates the loads
    const bool more = t0 + MR < tend;
    const int rn = more ? t0 + MR + 2 + w : 0;  // at most n+MR (n+MR+1 in a segment)
    double un[NV];
    fetch_row(rn, un);
    const int ec = e < 0 ? 0 : (e > elast ? elast : e);
    const EmitIn in = emit_load<DIR, COH>(k, io, cbase + (size_t)ec * stride, ec);
    if (more) stage_row(rn, un);
    if (emits) {
      double fm[NV], fp[NV];
      const int a = e % NFR, b = (e + 1) % NFR;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        fm[v] = sh.sF[v][a][lane];
        fp[v] = sh.sF[v][b][lane];
      }
      emit_store<DIR, COH>(k, io, cbase + (size_t)e * stride, in, fm, fp, uc);
    }
  }
  // last row of a whole line: fI[n-1] and fI[n] = fI[0]
  if (whole && w == 0 && col) {
    double fm[NV], fp[NV], uc[NV];
    const int a = (n - 1) % NFR;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      fm[v] = sh.sF[v][a][lane];
      fp[v] = sh.sF0[v][lane];
      uc[v] = sh.sC[v][(n - 1) % NRING][lane];
    }
    emit<DIR, COH>(k, io, cbase + (size_t)(n - 1) * stride, n - 1, fm, fp, uc);
  }
}

// three waves per SIMD (168 registers; left alone the characteristic passes
// take 170-194 and two waves), except with the mapped weights, which would
// spill 20 registers and more
constexpr int x_waves(int interp, int weno) { return interp == INTERP_CHAR && weno == WENO_MAPPED ? 2 : 3; }

template <int INTERP, int UPW, int W>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(x_waves(INTERP, W)))) k_pass_x(PassConst k, PassIO io) {
  __shared__ XShared<4, UPW> sh;
  pass_x_body<INTERP, UPW, 4, W>(k, io, blockIdx.x, sh);
}

// at most 256 registers: two waves per SIMD, which is what the LDS allows.
// Three, as blocks of 6 or 12 wavefronts with 6 or 12 rows per step, are slower:
// six wavefronts sit 2, 2, 1, 1 on the SIMDs (256^3 characteristic step 11.8 ->
// 14.1 ms), twelve wait for each other at every barrier (y 0.76 -> 0.83 ms).
template <int DIR, int INTERP, int UPW, int W>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_pass_m(PassConst k, PassIO io) {
  __shared__ MShared<4, UPW> sh;
  pass_m_body<DIR, INTERP, UPW, 4, W>(k, io, blockIdx.x, sh);
}

// ---------------------------------------------------------------------------
// batched passes: all members of an ensemble in one persistent launch
// ---------------------------------------------------------------------------
struct EnsArgs {
  const EnsMember *mem;    // member table
  int nmem;
  const unsigned *item0;   // first work item of each member, nmem + 1 entries
  unsigned nitems;
  double gamma, gm1, eps34;  // eps34 = 3/4 of the WENO epsilon
  const double *U;         // stage states of all members (member m at 5*off)
  double *R;
  StageUpdate upd;
  int visc;
};

// the member of a work item and the item's index within the member
__device__ __forceinline__ int ens_member(const EnsArgs &a, unsigned item) {
  int lo = 0, hi = a.nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.item0[mid] <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ void ens_setup(const EnsArgs &a, int m, int dir, PassConst &k, PassIO &io) {
  const EnsMember M = a.mem[m];
  for (int d = 0; d < 3; d++) k.n[d] = M.n[d];
  k.seg = M.seg[dir];
  k.ncell = M.ncell;
  k.gamma = a.gamma;
  k.gm1 = a.gm1;
  k.eps34 = a.eps34;
  k.dxg = M.dxg;
  const size_t o = 5 * M.off;
  io.U = a.U + o;
  io.R = a.R + o;
  io.par = M.par;
  io.Q = M.q;
  io.upd = a.upd;
  io.upd.c = M.dt * a.upd.c;
  io.upd.a0 = a.upd.a0 + o;
  io.upd.a1 = a.upd.a1 + o;
  io.upd.a2 = a.upd.a2 + o;
  io.upd.out = a.upd.out + o;
  io.visc = a.visc;
  io.mode = OUT_STAGE;
}

template <int INTERP, int UPW, int LPB, int W>
__global__ void __launch_bounds__(64 * LPB) __attribute__((amdgpu_waves_per_eu(x_waves(INTERP, W)))) k_ens_x(EnsArgs a) {
  __shared__ XShared<LPB, UPW> sh;
  for (unsigned item = blockIdx.x; item < a.nitems; item += gridDim.x) {
    const int m = ens_member(a, item);
    PassConst k;
    PassIO io;
    ens_setup(a, m, 0, k, io);
    pass_x_body<INTERP, UPW, LPB, W>(k, io, item - a.item0[m], sh);
    __syncthreads();
  }
}

template <int DIR, int INTERP, int UPW, int MR, int W>
__global__ void __launch_bounds__(64 * MR) __attribute__((amdgpu_waves_per_eu(2))) k_ens_m(EnsArgs a) {
  __shared__ MShared<MR, UPW> sh;
  for (unsigned item = blockIdx.x; item < a.nitems; item += gridDim.x) {
    const int m = ens_member(a, item);
    PassConst k;
    PassIO io;
    ens_setup(a, m, DIR, k, io);
    pass_m_body<DIR, INTERP, UPW, MR, W>(k, io, item - a.item0[m], sh);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// one persistent launch per RK stage: the x, y and z work items of all members
// ---------------------------------------------------------------------------
// Blocks take items in ticket order: every x item of every member (xg
// groups of x-lines each), then the y items, then the z items.  A member's y items add to the rhs its x items
// wrote, and its z items read what its y items left, so a y (z) item first
// waits until all x (y) items of its member are done, as counted in ctr.
// Every item a block waits on holds a smaller ticket, taken by a block that
// is running and that waits only on smaller tickets in turn, so the waits
// end whatever the number of resident blocks.  Each wait is bounded: after
// spin_limit polls it sets the error flag ctr[2] and goes on, so the kernel
// always exits, and the host reports the flag.  The last block to leave
// zeroes the ticket and the counters for the next launch, so graph replays
// need no memset.
struct EnsStageArgs {
  EnsArgs a;                 // item0 and nitems of a are not used
  const unsigned *item0[3];  // first item of each member per direction
  unsigned nitems[3];
  const unsigned *xgroups0;  // first x-line group of each member
  unsigned xg;               // x-line groups per x item
  unsigned *ctr;             // [0] ticket, [1] blocks done, [2] error flag, [3] unused,
                             // [4, 4+nmem) x items done, [4+nmem, 4+2nmem) y items done
  unsigned spin_limit;
};

template <int SH, int UPW>
union StageShared {
  XShared<SH, UPW> x;
  MShared<SH, UPW> m;
};

// the member of item `item` of a direction whose first items are item0
__device__ __forceinline__ int stage_member(const unsigned *item0, int nmem, unsigned item) {
  int lo = 0, hi = nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (item0[mid] <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Wave 0 acts for the block: all 64 of its lanes take the same branches and
// only lane 0 contributes to the counters (the others add 0).  A branch on
// threadIdx.x == 0 between two barriers of the item loop would let the
// compiler move lane 0's atomics out of the loop (a loop that lanes leave
// one by one), so that the rest of the block passed the next barrier before
// lane 0 had counted its item or fetched the next ticket.
__device__ __forceinline__ bool lead_wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x) < 64u; }

__device__ __forceinline__ unsigned lane0_one() { return (threadIdx.x & 63u) == 0u ? 1u : 0u; }

// The only data blocks of the launch hand to each other is R, and every
// access to it here is an agent-scope atomic (load_r / store_r with COH):
// the stores write through the XCD's L2, the loads bypass stale lines of
// the L1 and the L2.  A count of finished items therefore needs only each
// wave's stores acknowledged before it, and a wait only the count seen
// before the block's first load of R; neither writes back nor invalidates
// an L2 (the fences a release or acquire at agent scope would add, once per
// work item, for every XCD).
//
// Whole block: wait until *c >= need (bounded).  The barrier keeps the
// block's loads after the poll that saw the count.
__device__ __forceinline__ void stage_wait(const unsigned *c, unsigned need, unsigned *err, unsigned limit) {
  if (lead_wave()) {
    for (unsigned polls = 0;; polls++) {
      const unsigned v =
          __builtin_amdgcn_readfirstlane(__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      if (v >= need) break;
      if (polls >= limit) {
        __hip_atomic_fetch_or(err, lane0_one(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
  }
  __syncthreads();
}

// Whole block: every wave waits until its write-through stores of R are
// acknowledged, then one wave counts the item.
__device__ __forceinline__ void stage_signal(unsigned *c) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (lead_wave()) __hip_atomic_fetch_add(c, lane0_one(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int INTERP, int UPW, int SH, int W>
__global__ void __launch_bounds__(64 * SH) __attribute__((amdgpu_waves_per_eu(2))) k_ens_stage(EnsStageArgs s) {
  __shared__ StageShared<SH, UPW> sh;
  __shared__ unsigned s_ticket, s_last;
  const int nmem = s.a.nmem;
  unsigned *const done_x = s.ctr + 4, *const done_y = s.ctr + 4 + nmem;
  const unsigned nx_items = s.nitems[0], nxy_items = s.nitems[0] + s.nitems[1];
  const unsigned total = nxy_items + s.nitems[2];
  for (;;) {
    if (lead_wave()) {
      const unsigned old = __hip_atomic_fetch_add(&s.ctr[0], lane0_one(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_ticket = __builtin_amdgcn_readfirstlane(old);  // lane 0's: the value before its add
    }
    __syncthreads();
    const unsigned t = __builtin_amdgcn_readfirstlane(s_ticket);
    if (t >= total) break;
    const int phase = t < nx_items ? 0 : (t < nxy_items ? 1 : 2);
    const unsigned item = t - (phase == 0 ? 0u : (phase == 1 ? nx_items : nxy_items));
    const unsigned *const item0 = s.item0[phase];
    const int m = stage_member(item0, nmem, item);
    if (phase > 0) {
      const unsigned *before = s.item0[phase - 1];
      stage_wait(phase == 1 ? &done_x[m] : &done_y[m], before[m + 1] - before[m], &s.ctr[2], s.spin_limit);
    }
    const unsigned local = item - item0[m];
    if (phase == 0) {
      PassConst k;
      PassIO io;
      ens_setup(s.a, m, 0, k, io);
      const unsigned g1 = min((local + 1) * s.xg, s.xgroups0[m + 1] - s.xgroups0[m]);
      for (unsigned g = local * s.xg; g < g1; g++) {
        pass_x_body<INTERP, UPW, SH, W, true>(k, io, g, sh.x);
        __syncthreads();
      }
      stage_signal(&done_x[m]);
    } else if (phase == 1) {
      PassConst k;
      PassIO io;
      ens_setup(s.a, m, 1, k, io);
      pass_m_body<1, INTERP, UPW, SH, W, true>(k, io, local, sh.m);
      stage_signal(&done_y[m]);
    } else {
      PassConst k;
      PassIO io;
      ens_setup(s.a, m, 2, k, io);
      pass_m_body<2, INTERP, UPW, SH, W, true>(k, io, local, sh.m);
      __syncthreads();
    }
  }
  // the last block out resets the counters (every other block has stopped
  // touching them)
  if (lead_wave()) {
    const unsigned old = __hip_atomic_fetch_add(&s.ctr[1], lane0_one(), __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    s_last = __builtin_amdgcn_readfirstlane(old) == gridDim.x - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(s_last)) {
    for (unsigned i = threadIdx.x; i < 2u * (unsigned)nmem; i += blockDim.x) s.ctr[4 + i] = 0u;
    if (threadIdx.x < 2u) s.ctr[threadIdx.x] = 0u;  // ticket, blocks done
  }
}

// primitive variables (u, v, w, T) of a state
__global__ void __launch_bounds__(256) k_prims(const double *__restrict__ u, double *__restrict__ Q, size_t ncell,
                                               double gamma) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  double s[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) s[v] = u[(size_t)v * ncell + idx];
  double q[4];
  visc_prims(s, gamma, q);
#pragma unroll
  for (int c = 0; c < 4; c++) Q[(size_t)c * ncell + idx] = q[c];
}

// work items of a y or z pass: groups of MW columns times segments
size_t march_items(size_t ncol, int n, int seg) {
  return ((ncol + MW - 1) / MW) * (size_t)(seg >= n ? 1 : (n + seg - 1) / seg);
}

template <int DIR, int INTERP, int UPW, int W>
void launch_t(const Grid &g, const PassConst &k, const PassIO &io, hipStream_t st) {
  if (DIR == 0) {
    const size_t nlines = (size_t)g.n[1] * g.n[2];
    hipLaunchKernelGGL((k_pass_x<INTERP, UPW, W>), dim3((unsigned)((nlines + 3) / 4)), dim3(256), 0, st, k, io);
  } else {
    const size_t nb = march_items(g.ncell / g.n[DIR], g.n[DIR], k.seg);
    hipLaunchKernelGGL((k_pass_m<DIR == 0 ? 1 : DIR, INTERP, UPW, W>), dim3((unsigned)nb), dim3(256), 0, st, k, io);
  }
}

template <int DIR, int INTERP, int UPW>
void launch_w(const Grid &g, const Scheme &sc, const PassConst &k, const PassIO &io, hipStream_t st) {
  if (sc.weno == WENO_MAPPED) launch_t<DIR, INTERP, UPW, WENO_MAPPED>(g, k, io, st);
  else if (sc.weno == WENO_Z) launch_t<DIR, INTERP, UPW, WENO_Z>(g, k, io, st);
  else if (sc.weno == WENO_YC) launch_t<DIR, INTERP, UPW, WENO_YC>(g, k, io, st);
  else if (sc.weno == WENO_OPTIMAL) launch_t<DIR, INTERP, UPW, WENO_OPTIMAL>(g, k, io, st);
  else launch_t<DIR, INTERP, UPW, WENO_JS>(g, k, io, st);
}

template <int DIR>
void launch_d(const Grid &g, const Scheme &sc, const PassConst &k, const PassIO &io, hipStream_t st) {
  if (sc.interp == INTERP_CHAR) {
    if (sc.upwind == UPWIND_ROE) launch_w<DIR, INTERP_CHAR, UPWIND_ROE>(g, sc, k, io, st);
    else launch_w<DIR, INTERP_CHAR, UPWIND_RUSANOV>(g, sc, k, io, st);
  } else {
    if (sc.upwind == UPWIND_ROE) launch_w<DIR, INTERP_COMP, UPWIND_ROE>(g, sc, k, io, st);
    else launch_w<DIR, INTERP_COMP, UPWIND_RUSANOV>(g, sc, k, io, st);
  }
}

}  // namespace

void launch_pass(const Grid &g, const Scheme &sc, int dir, const PassBuffers &b, int mode, const double *dxg,
                 hipStream_t st) {
  PassConst k;
  PassIO io;
  for (int d = 0; d < 3; d++) k.n[d] = g.n[d];
  k.seg = dir == 0 ? 0 : g.seg[dir];
  k.ncell = g.ncell;
  k.gamma = sc.gamma;
  k.gm1 = sc.gamma - 1.0;
  k.eps34 = 0.75 * sc.eps;
  k.dxg = dxg;
  io.U = b.U;
  io.R = b.R;
  io.par = b.par;
  io.Q = b.Q;
  io.upd = b.upd;
  io.visc = sc.Re > 0 ? 1 : 0;
  io.mode = mode;
  if (dir == 0) launch_d<0>(g, sc, k, io, st);
  else if (dir == 1) launch_d<1>(g, sc, k, io, st);
  else launch_d<2>(g, sc, k, io, st);
}

namespace {
template <int INTERP, int UPW, int W>
void ens_launch_w(int dir, int shape, const EnsArgs &a, unsigned grid, hipStream_t st) {
  if (dir == 0) {
    if (shape == 0) hipLaunchKernelGGL((k_ens_x<INTERP, UPW, 4, W>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_ens_x<INTERP, UPW, 2, W>), dim3(grid), dim3(128), 0, st, a);
  } else if (dir == 1) {
    if (shape == 0) hipLaunchKernelGGL((k_ens_m<1, INTERP, UPW, 4, W>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_ens_m<1, INTERP, UPW, 2, W>), dim3(grid), dim3(128), 0, st, a);
  } else {
    if (shape == 0) hipLaunchKernelGGL((k_ens_m<2, INTERP, UPW, 4, W>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_ens_m<2, INTERP, UPW, 2, W>), dim3(grid), dim3(128), 0, st, a);
  }
}

template <int INTERP, int UPW>
void ens_launch_t(int weno, int dir, int shape, const EnsArgs &a, unsigned grid, hipStream_t st) {
  if (weno == WENO_MAPPED) ens_launch_w<INTERP, UPW, WENO_MAPPED>(dir, shape, a, grid, st);
  else if (weno == WENO_Z) ens_launch_w<INTERP, UPW, WENO_Z>(dir, shape, a, grid, st);
  else if (weno == WENO_YC) ens_launch_w<INTERP, UPW, WENO_YC>(dir, shape, a, grid, st);
  else if (weno == WENO_OPTIMAL) ens_launch_w<INTERP, UPW, WENO_OPTIMAL>(dir, shape, a, grid, st);
  else ens_launch_w<INTERP, UPW, WENO_JS>(dir, shape, a, grid, st);
}
}  // namespace

unsigned ens_items_per_member(int dir, int shape, const int n[3], const int seg[3]) {
  const size_t ncell = (size_t)n[0] * n[1] * n[2];
  if (dir == 0) {
    const size_t lpb = shape == 0 ? 4 : 2;
    return (unsigned)(((size_t)n[1] * n[2] + lpb - 1) / lpb);
  }
  return (unsigned)march_items(ncell / n[dir], n[dir], seg[dir]);
}

void launch_ens_pass(const Scheme &sc, int dir, int shape, const EnsMember *mem, int nmem, const unsigned *item0,
                     unsigned nitems, unsigned grid, const double *U, double *R, const StageUpdate &upd,
                     hipStream_t st) {
  EnsArgs a;
  a.mem = mem;
  a.nmem = nmem;
  a.item0 = item0;
  a.nitems = nitems;
  a.gamma = sc.gamma;
  a.gm1 = sc.gamma - 1.0;
  a.eps34 = 0.75 * sc.eps;
  a.U = U;
  a.R = R;
  a.upd = upd;
  a.visc = sc.Re > 0;
  if (grid == 0 || grid > nitems) grid = nitems;
  if (sc.interp == INTERP_CHAR) {
    if (sc.upwind == UPWIND_ROE) ens_launch_t<INTERP_CHAR, UPWIND_ROE>(sc.weno, dir, shape, a, grid, st);
    else ens_launch_t<INTERP_CHAR, UPWIND_RUSANOV>(sc.weno, dir, shape, a, grid, st);
  } else {
    if (sc.upwind == UPWIND_ROE) ens_launch_t<INTERP_COMP, UPWIND_ROE>(sc.weno, dir, shape, a, grid, st);
    else ens_launch_t<INTERP_COMP, UPWIND_RUSANOV>(sc.weno, dir, shape, a, grid, st);
  }
}

namespace {
// blocks of `kern` that one CU holds at once
template <class K>
unsigned resident_per_cu(K kern, int threads) {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, threads, 0) != hipSuccess || nb < 1) nb = 1;
  return (unsigned)nb;
}

template <int INTERP, int UPW, int W>
void stage_launch_w(int rows, const EnsStageArgs &s, unsigned grid, int cus, hipStream_t st) {
  const unsigned total = s.nitems[0] + s.nitems[1] + s.nitems[2];
  if (rows == 4) {
    static const unsigned per_cu = resident_per_cu(k_ens_stage<INTERP, UPW, 4, W>, 256);
    if (grid == 0) grid = per_cu * (unsigned)cus;
    hipLaunchKernelGGL((k_ens_stage<INTERP, UPW, 4, W>), dim3(std::min(grid, total)), dim3(256), 0, st, s);
  } else {
    static const unsigned per_cu = resident_per_cu(k_ens_stage<INTERP, UPW, 2, W>, 128);
    if (grid == 0) grid = per_cu * (unsigned)cus;
    hipLaunchKernelGGL((k_ens_stage<INTERP, UPW, 2, W>), dim3(std::min(grid, total)), dim3(128), 0, st, s);
  }
}

template <int INTERP, int UPW>
void stage_launch_t(int weno, int rows, const EnsStageArgs &s, unsigned grid, int cus, hipStream_t st) {
  if (weno == WENO_MAPPED) stage_launch_w<INTERP, UPW, WENO_MAPPED>(rows, s, grid, cus, st);
  else if (weno == WENO_Z) stage_launch_w<INTERP, UPW, WENO_Z>(rows, s, grid, cus, st);
  else if (weno == WENO_YC) stage_launch_w<INTERP, UPW, WENO_YC>(rows, s, grid, cus, st);
  else if (weno == WENO_OPTIMAL) stage_launch_w<INTERP, UPW, WENO_OPTIMAL>(rows, s, grid, cus, st);
  else stage_launch_w<INTERP, UPW, WENO_JS>(rows, s, grid, cus, st);
}
}  // namespace

void launch_ens_stage(const Scheme &sc, int rows, const EnsMember *mem, int nmem, const unsigned *const item0[3],
                      const unsigned nitems[3], const unsigned *xgroups0, unsigned xg, unsigned grid, int cus,
                      unsigned *ctr, unsigned spin_limit, const double *U, double *R, const StageUpdate &upd,
                      hipStream_t st) {
  EnsStageArgs s;
  EnsArgs &a = s.a;
  a.mem = mem;
  a.nmem = nmem;
  a.item0 = nullptr;
  a.nitems = 0;
  a.gamma = sc.gamma;
  a.gm1 = sc.gamma - 1.0;
  a.eps34 = 0.75 * sc.eps;
  a.U = U;
  a.R = R;
  a.upd = upd;
  a.visc = sc.Re > 0;
  for (int d = 0; d < 3; d++) {
    s.item0[d] = item0[d];
    s.nitems[d] = nitems[d];
  }
  s.xgroups0 = xgroups0;
  s.xg = xg;
  s.ctr = ctr;
  s.spin_limit = spin_limit;
  if (sc.interp == INTERP_CHAR) {
    if (sc.upwind == UPWIND_ROE) stage_launch_t<INTERP_CHAR, UPWIND_ROE>(sc.weno, rows, s, grid, cus, st);
    else stage_launch_t<INTERP_CHAR, UPWIND_RUSANOV>(sc.weno, rows, s, grid, cus, st);
  } else {
    if (sc.upwind == UPWIND_ROE) stage_launch_t<INTERP_COMP, UPWIND_ROE>(sc.weno, rows, s, grid, cus, st);
    else stage_launch_t<INTERP_COMP, UPWIND_RUSANOV>(sc.weno, rows, s, grid, cus, st);
  }
}

// Segments of the y (z) march.  A block marches 64 columns; a grid (or an
// ensemble) with few columns leaves CUs idle and ends on a long tail, so its
// lines are cut into segments, each of which evaluates one interface more
// than its cells and stages six rows of its neighbour again.  The length is
// the one with the least estimated time
//   max(0.9 work/256 + longest/2, 1.1 longest)
// in march steps of MR rows, a segment costing its steps plus 2 for its
// start (work: all segments' steps; 256 CUs of two blocks each); a shorter
// one has to win 3%, and lines under 8 cells stay whole (the row indices of
// a segment reach n + 5).  Measured, y / z pass, whole lines -> segments: 64^3
// component-wise 45 / 60 -> 17 / 20 us, 128^3 106 / 159 -> 86 / 125 us, 201^3
// 403 / 539 -> 340 / 456 us; 256^3 stays whole (666 / 866 us, 656-672 / 866-900
// in segments of 47 to 127 cells).  The formula's shape and its factors are a
// fit to such sweeps, not derived.  MR is the four-row blocks'; the two-row
// blocks an ensemble can choose take the same segments (64 members of 32 to 64
// a side, step with whole lines -> segments and the present arithmetic: four
// rows 4.58 -> 3.55 ms, two rows 5.40 -> 4.17 ms).
void march_segments(int count, const int (*n)[3], int dir, int *seg) {
  constexpr int MR = 4, CUS = 256;
  int nmax = 0;
  for (int m = 0; m < count; m++) nmax = std::max(nmax, n[m][dir]);
  auto cut = [](int N, int len) {  // cells per segment: equal parts of at most len cells
    if (N < 8 || len >= N) return N;
    const int parts = (N + len - 1) / len;
    return (N + parts - 1) / parts;
  };
  int best = nmax;
  double tbest = 0.0;
  for (int parts = 1; parts <= std::max(1, nmax / 3); parts++) {
    const int len = (nmax + parts - 1) / parts;
    if (parts > 1 && len == (nmax + parts - 2) / (parts - 1)) continue;
    double work = 0.0;
    int longest = 0;
    for (int m = 0; m < count; m++) {
      const int N = n[m][dir], c = cut(N, len);
      const int steps = 2 + ((c < N ? c + 1 : N) + MR - 1) / MR;
      work += (double)march_items((size_t)n[m][0] * n[m][1] * n[m][2] / N, N, c) * steps;
      longest = std::max(longest, steps);
    }
    const double t = std::max(0.9 * work / CUS + 0.5 * longest, 1.1 * longest);
    if (parts == 1 || t < 0.97 * tbest) {
      tbest = t;
      best = len;
    }
  }
  for (int m = 0; m < count; m++) seg[m] = cut(n[m][dir], best);
}

void launch_prims(const Grid &g, const Scheme &sc, const double *u, double *Q, hipStream_t st) {
  hipLaunchKernelGGL(k_prims, dim3((unsigned)((g.ncell + 255) / 256)), dim3(256), 0, st, u, Q, g.ncell, sc.gamma);
}

}  // namespace hm
