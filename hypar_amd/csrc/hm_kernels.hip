// hm_kernels.hip -- gfx950 kernels of the NS3D WENO5 + RK4 path besides the
// direction passes (hm_pass.hip).
//
// State layout: structure of arrays without ghosts (see include/hypar_mi355x.h).
// All boundaries are periodic; stencil indices wrap.
//
//   k_visc_par, k_ens_visc  the viscous term of every cell from the primitive
//                           variables the previous z pass stored
//                           (NavierStokes3DParabolicFunction.c:50-325), with
//                           the reference's ghost-layer fluxes at the faces
//   k_par_out               the viscous term as a five-variable array
//   k_cfl, k_sqdiff, k_volint  reductions: CFL number, step norm, volume
//                           integrals (NavierStokes3DComputeCFL.c:16-55,
//                           TimePostStep.c:43-63, VolumeIntegral.c:14-50)
//   k_aos_to_soa, k_soa_to_aos  layout conversion at the host transfers
#include <hip/hip_runtime.h>

#include <cmath>

#include "hm_device.h"
#include "hm_internal.h"

namespace hm {

// ---------------------------------------------------------------------------
// viscous terms
// ---------------------------------------------------------------------------
// Primitive variables used by the viscous term: (u, v, w, T) with
// T = gamma*P/rho (NavierStokes3DParabolicFunction.c:85-108).
struct QT {
  double u, v, w, T;
};

struct ViscParams {
  double gamma, inv_Re, inv_gm1, inv_Pr;
};

// Viscous flux along DIR at a point from the primitive values and the
// gradient components (derivatives already scaled by dxinv).
// grad[c][e] = d(q_c)/dx_e for c in (u,v,w,T).
template <int DIR>
__device__ __forceinline__ void visc_flux(double fv[4], const QT &q, const double (&gr)[4][3],
                                          double mu, const ViscParams &vp) {
  const double two_third = 2.0 / 3.0;
  const double mr = mu * vp.inv_Re;
  const double kq = mu * vp.inv_Re * vp.inv_gm1 * vp.inv_Pr;
  const double ux = gr[0][0], uy = gr[0][1], uz = gr[0][2];
  const double vx = gr[1][0], vy = gr[1][1], vz = gr[1][2];
  const double wx = gr[2][0], wy = gr[2][1], wz = gr[2][2];
  double t1, t2, t3, qd;
  if (DIR == 0) {
    t1 = two_third * mr * (2 * ux - vy - wz);
    t2 = mr * (uy + vx);
    t3 = mr * (uz + wx);
    qd = kq * gr[3][0];
  } else if (DIR == 1) {
    t1 = mr * (uy + vx);
    t2 = two_third * mr * (-ux + 2 * vy - wz);
    t3 = mr * (vz + wy);
    qd = kq * gr[3][1];
  } else {
    t1 = mr * (uz + wx);
    t2 = mr * (vz + wy);
    t3 = two_third * mr * (-ux - vy + 2 * wz);
    qd = kq * gr[3][2];
  }
  fv[0] = t1; fv[1] = t2; fv[2] = t3;
  fv[3] = q.u * t1 + q.v * t2 + q.w * t3 + qd;
}

// Viscous term of the right-hand side (NavierStokes3DParabolicFunction.c:50-325):
//   par = dxinv Dx FVx + dyinv Dy FVy + dzinv Dz FVz,
// the x and y terms added to each other first and the z fluxes one by one
// around their sum (the reference adds the three terms), with FVd the viscous flux along d of the
// primitive variables (u, v, w, T) and their gradient (4th-order central
// differences with periodic neighbours, scaled by the point's dxinv;
// FirstDerivativeFourthOrder.c:103) and Dd the same central difference of
// the flux.  par[c*ncell + cell], c = momentum x, y, z, energy (the mass
// component is zero).  Q holds u, v, w, T of every cell, Q[c*ncell + cell];
// the viscosity is mu = T^0.76 (pow076).
//
// Where the stencil of Dd leaves the grid (positions -2, -1, n, n+1 along
// d) the reference reads the fluxes of its ghost layers: the primitive
// values there are the periodic copies, the derivative along d uses the
// biased stencils of FirstDerivativeFourthOrder.c:74-93/106-125 in the outer
// layer and the central one in the inner layer, scaled by the ghost dxinv
// (a copy of the nearest interior value, InitialSolution.c:101-113), and the
// derivatives across d are zero, because the reference computes those only
// on lines whose other indices are interior.  The kernel evaluates these
// ghost-layer fluxes where its stencils need them.
//
// A block owns a TX x TY tile of (x, y) columns and marches through the
// planes of one z segment [k0, k1) (pks planes).  A thread evaluates the
// gradient and the fluxes of one point: a column of the tile, or one of the
// halo points whose x or y flux the tile's differences read (the rows y0-2,
// y0-1, y0+TY, y0+TY+1 and the columns x0-2, x0-1, x0+TX, x0+TX+1); the halo
// points take whole wavefronts.  A thread holds its point's values on planes
// q-2..q+2 in registers: the z derivative comes from there, and the plane q+1
// among them is what it stages in LDS for the others' x and y derivatives in
// the next step, so only the 208 points beyond those of the block's threads
// are loaded for LDS alone.  The x and y fluxes of plane q go to LDS, where
// their x and y differences are formed.  Plane and fluxes are double-buffered,
// which leaves one barrier per plane.  The z flux of plane q goes at once into
// the sums of the planes q-2..q+2 whose z difference reads it, five running
// sums per component, to which the x + y part of plane q is added; the sum of
// plane q-2 is then complete.  The z differences of the segment need FVz on
// planes k0-2..k1+1, so the march covers them; on the ghost planes (-2, -1,
// nz, nz+1) the z flux comes from direct loads of the column.
//
// LDS bandwidth (3000 cycles per plane and CU) and vector issue (3200) bound
// it, hardly overlapped because the block's wavefronts go through them
// together: 3.3 us per plane.  Its 11 wavefronts allow a thread 168 registers,
// of which k_visc_par spills 4 and k_ens_visc 2 (20 and 12 B of scratch a lane).
// Tiles of 16 x 16, two blocks per CU, took 603 us
// at 256^3, this one 430 us; a form with 512 threads, two barriers per plane
// and the halo points evaluated after the columns by some of the threads, 497
// us (before that, with log and exp, a flux ring and a buffer of x + y parts,
// 670 us).  64^3 takes 21 us, 16x12x20 14 us (87 and 91 us with segments of 16
// planes and more).
template <int TX, int TY>
struct ViscParShared {
  double q[2][4][TY + 8][TX + 8];  // a plane of Q: x0-4..x0+TX+3, y0-4..y0+TY+3
  double fx[2][4][TY][TX + 4];     // x fluxes of the tile's rows at x0-2..x0+TX+1
  double fy[2][4][TY + 4][TX];     // y fluxes of the tile's columns at y0-2..y0+TY+1
};

__device__ __forceinline__ int wrapi(int p, int n) {
  const int r = p % n;
  return r < 0 ? r + n : r;
}

// Stencil of d/dx_d at the ghost position of slot s (0..3 for the positions
// -2, -1, n, n+1): 12 times the weights of the five points from offset
// ghost_first(slot) on (periodic copies).  The weighted values are summed
// before the sum is scaled by dxinv/12: scaled weights are rounded, so that
// equal values no longer cancel.
__device__ __forceinline__ int ghost_first(int slot) { return slot == 0 ? -1 : (slot == 3 ? -3 : -2); }
__device__ __forceinline__ double ghost_weight(int slot, int k) {
  const double lo[5] = {-3, -10, 18, -6, 1}, hi[5] = {-1, 6, -18, 10, 3}, mid[5] = {1, -8, 0, 8, -1};
  return slot == 0 ? lo[k] : (slot == 3 ? hi[k] : mid[k]);
}

// Viscous flux along DIR at a ghost position: derivative along DIR only
// (d[c], already scaled), primitive values q, viscosity mu.
template <int DIR>
__device__ __forceinline__ void ghost_flux(double fv[4], const QT &q, const double (&d)[4], double mu,
                                           const ViscParams &vp) {
  double gr[4][3];
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int e = 0; e < 3; e++) gr[c][e] = e == DIR ? d[c] : 0.0;
  visc_flux<DIR>(fv, q, gr, mu, vp);
}

// 12 times the 4th-order central difference, summed in the reference's order:
// T is close to 1 and its differences small, so another order differs from
// the reference by more than the term's other roundings
__device__ __forceinline__ double d4u(double fm2, double fm1, double fp1, double fp2) {
  return fm2 - 8 * fm1 + 8 * fp1 - fp2;
}

// tile b of the grid; every thread of the block takes part
template <int TX, int TY>
__device__ __forceinline__ void visc_par_tile(const double *__restrict__ Q, double *__restrict__ par, int nx,
                                              int ny, int nz,
                                              const double *__restrict__ dxg,  // ghosted dxinv x|y|z
                                              const ViscParams &vp, int b, int pks, ViscParShared<TX, TY> &sh) {
  static_assert(TX * TY % 64 == 0 && 4 * TX % 64 == 0, "each kind of point takes whole wavefronts");
  const size_t ncell = (size_t)nx * ny * nz;
  const size_t plane = (size_t)nx * ny;
  const int ntx = (nx + TX - 1) / TX, nty = (ny + TY - 1) / TY;
  const int tx = b % ntx, ty = (b / ntx) % nty, kz = b / (ntx * nty);
  const int x0 = tx * TX, y0 = ty * TY, k0 = kz * pks;
  const int k1 = min(k0 + pks, nz);
  const double *dxa = dxg, *dya = dxg + (nx + 6), *dza = dxg + (nx + 6) + (ny + 6);  // entry 3+p: position p
  const int t = threadIdx.x;
  // this thread's point: 2 a column of the tile, 1 a halo row's, 0 a halo column's
  const int wt = __builtin_amdgcn_readfirstlane(t);
  const int kind = wt < TX * TY ? 2 : (wt < TX * TY + 4 * TX ? 1 : 0);
  int ox, oy;
  if (kind == 2) {
    ox = t % TX;
    oy = t / TX;
  } else if (kind == 1) {
    const int u = t - TX * TY, r = u / TX;
    ox = u % TX;
    oy = r < 2 ? r - 2 : TY + r - 2;
  } else {
    const int u = t - TX * TY - 4 * TX, r = u % 4;
    ox = r < 2 ? r - 2 : TX + r - 2;
    oy = u / 4;
  }
  const int i = x0 + ox, j = y0 + oy;
  const size_t col = (size_t)wrapi(j, ny) * nx + wrapi(i, nx);
  const bool inx = i >= 0 && i < nx, iny = j >= 0 && j < ny;
  const bool own = kind == 2 && inx && iny;
  // does the tile read this point's x (y) flux; it is a ghost-layer flux where
  // the point lies beyond the grid along x (y)
  const bool wantx = kind != 1 && iny && i < nx + 2, wanty = kind != 0 && inx && j < ny + 2;
  const bool regular = inx && iny && (wantx || wanty);
  const double r12 = 1.0 / 12.0;
  // also for the ghost positions: read in the march, they cost the border tiles
  // 1 us a plane (256^3: 515 us against 430, 128^3: 76 against 71)
  const double dxi = i < nx + 2 ? dxa[3 + i] * r12 : 0.0, dyi = j < ny + 2 ? dya[3 + j] * r12 : 0.0;

  // a further point of the staged plane, beyond those of the block's threads:
  // rows y0-4, y0-3, y0+TY+2, y0+TY+3, columns alike, and the 16 points
  // across the corners
  const int e = t >= TX * TY ? t - TX * TY : (t < 16 ? 4 * TX + 4 * TY + t : -1);
  int ex = 0, ey = 0;
  if (e >= 0 && e < 4 * TX) {
    const int r = e / TX;
    ex = e % TX;
    ey = r < 2 ? r - 4 : TY + r;
  } else if (e >= 0 && e < 4 * TX + 4 * TY) {
    const int u = e - 4 * TX, r = u % 4;
    ex = r < 2 ? r - 4 : TX + r;
    ey = u / 4;
  } else if (e >= 0) {
    const int u = e - 4 * TX - 4 * TY, r = u % 4, w = u / 4;
    ex = r < 2 ? r - 2 : TX + r - 2;
    ey = w < 2 ? w - 2 : TY + w - 2;
  }
  const size_t ecol = (size_t)wrapi(y0 + ey, ny) * nx + wrapi(x0 + ex, nx);

  auto ldq = [&](size_t c, int k, double (&r)[4]) {  // k in [-4, nz + 4]
    const size_t o = (size_t)wrap(k, nz) * plane + c;
#pragma unroll
    for (int v = 0; v < 4; v++) r[v] = Q[(size_t)v * ncell + o];
  };

  // planes q-2..q+2 of the point, plane q+1 of the further point, and the
  // sums of planes q-2..q+1 so far
  double rq[5][4], pe[4] = {0.0, 0.0, 0.0, 0.0}, sum[4][4];
#pragma unroll
  for (int s = 0; s < 5; s++) ldq(col, k0 - 4 + s, rq[s]);
  if (e >= 0) ldq(ecol, k0 - 2, pe);
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int v = 0; v < 4; v++) sum[s][v] = 0.0;
  int buf = 0;
  auto stage = [&](int bq, const double (&r)[4]) {
#pragma unroll
    for (int v = 0; v < 4; v++) sh.q[bq][v][oy + 4][ox + 4] = r[v];
    if (e >= 0)
#pragma unroll
      for (int v = 0; v < 4; v++) sh.q[bq][v][ey + 4][ex + 4] = pe[v];
  };
  stage(buf, rq[2]);  // plane k0-2
  if (e >= 0) ldq(ecol, k0 - 1, pe);
  __syncthreads();
  for (int q = k0 - 2; q < k1 + 2; q++) {
    const bool gz = q < 0 || q >= nz;     // a ghost plane along z (uniform)
    const bool outq = q >= k0 && q < k1;  // a plane whose x and y terms are formed
    // the middle entries hold the periodic copy of every point, also beyond
    // the grid, so one evaluation serves interior and ghost fluxes
    const QT qv = {rq[2][0], rq[2][1], rq[2][2], rq[2][3]};
    const double mu = pow076(qv.T);
    double fzq[4] = {0.0, 0.0, 0.0, 0.0};
    if (gz) {
      if (own) {
        const int slot = q < 0 ? q + 2 : q - nz + 2, o0 = ghost_first(slot);
        double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 5; k++) {
          double r[4];
          ldq(col, q + o0 + k, r);
          const double w = ghost_weight(slot, k);
#pragma unroll
          for (int v = 0; v < 4; v++) d[v] += w * r[v];
        }
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] *= r12 * dza[3 + q];
        ghost_flux<2>(fzq, qv, d, mu, vp);
      }
    } else {
      // Q on LDS at offsets (a, c) from the point
      auto sq = [&](int v, int a, int c) { return sh.q[buf][v][oy + 4 + c][ox + 4 + a]; };
      double fv[4];
      if (regular && (outq || kind == 2)) {
        double gr[4][3];
        const double dzi = dza[3 + q] * r12;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          gr[v][0] = d4u(sq(v, -2, 0), sq(v, -1, 0), sq(v, 1, 0), sq(v, 2, 0)) * dxi;
          gr[v][1] = d4u(sq(v, 0, -2), sq(v, 0, -1), sq(v, 0, 1), sq(v, 0, 2)) * dyi;
          gr[v][2] = d4u(rq[0][v], rq[1][v], rq[3][v], rq[4][v]) * dzi;
        }
        if (kind == 2) visc_flux<2>(fzq, qv, gr, mu, vp);
        if (outq && kind != 1) {
          visc_flux<0>(fv, qv, gr, mu, vp);
#pragma unroll
          for (int v = 0; v < 4; v++) sh.fx[buf][v][oy][ox + 2] = fv[v];
        }
        if (outq && kind != 0) {
          visc_flux<1>(fv, qv, gr, mu, vp);
#pragma unroll
          for (int v = 0; v < 4; v++) sh.fy[buf][v][oy + 2][ox] = fv[v];
        }
      }
      // ghost-layer fluxes: x at i = -2, -1, nx, nx+1, y at j = -2, -1, ny, ny+1
      if (outq && wantx && !inx) {
        const int slot = i < 0 ? i + 2 : i - nx + 2, o0 = ghost_first(slot);
        double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 5; k++) {
          const double w = ghost_weight(slot, k);
#pragma unroll
          for (int v = 0; v < 4; v++) d[v] += w * sq(v, o0 + k, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] *= dxi;
        ghost_flux<0>(fv, qv, d, mu, vp);
#pragma unroll
        for (int v = 0; v < 4; v++) sh.fx[buf][v][oy][ox + 2] = fv[v];
      }
      if (outq && wanty && !iny) {
        const int slot = j < 0 ? j + 2 : j - ny + 2, o0 = ghost_first(slot);
        double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 5; k++) {
          const double w = ghost_weight(slot, k);
#pragma unroll
          for (int v = 0; v < 4; v++) d[v] += w * sq(v, 0, o0 + k);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] *= dyi;
        ghost_flux<1>(fv, qv, d, mu, vp);
#pragma unroll
        for (int v = 0; v < 4; v++) sh.fy[buf][v][oy + 2][ox] = fv[v];
      }
    }
    // stage plane q+1; the loads for the next plane are in flight during the
    // barrier and the differences
    stage(buf ^ 1, rq[3]);
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int v = 0; v < 4; v++) rq[s][v] = rq[s + 1][v];
    if (q + 1 < k1 + 2) {
      ldq(col, q + 3, rq[4]);
      if (e >= 0) ldq(ecol, q + 2, pe);
    }
    __syncthreads();
    if (kind == 2) {
      // plane p = q-2+s reads FVz(q) with weight -1/12, 8/12, 0, -8/12, 1/12
      // times its dzinv (planes outside the segment are not stored; their
      // metric index is clamped into the array)
      const double z0 = -r12 * dza[3 + max(q - 2, -3)], z1 = 8.0 * r12 * dza[3 + max(q - 1, -3)];
      const double z3 = -8.0 * r12 * dza[3 + min(q + 1, nz + 2)], z4 = r12 * dza[3 + min(q + 2, nz + 2)];
      if (q - 2 >= k0 && own) {  // the sum of plane q-2 is now complete
        const size_t o = (size_t)(q - 2) * plane + col;
#pragma unroll
        for (int v = 0; v < 4; v++) par[(size_t)v * ncell + o] = sum[0][v] + z0 * fzq[v];
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        sum[0][v] = sum[1][v] + z1 * fzq[v];
        sum[1][v] = sum[2][v];
        sum[2][v] = sum[3][v] + z3 * fzq[v];
        sum[3][v] = z4 * fzq[v];
      }
      if (outq && own) {
        const auto &fx = sh.fx[buf];
        const auto &fy = sh.fy[buf];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double px = dxi * d4u(fx[v][oy][ox], fx[v][oy][ox + 1], fx[v][oy][ox + 3], fx[v][oy][ox + 4]);
          const double py = dyi * d4u(fy[v][oy][ox], fy[v][oy + 1][ox], fy[v][oy + 3][ox], fy[v][oy + 4][ox]);
          sum[1][v] += px + py;
        }
      }
    }
    buf ^= 1;
  }
}

__global__ void __launch_bounds__(PAR_THREADS) k_visc_par(const double *__restrict__ Q, double *__restrict__ par,
                                                         int nx, int ny, int nz, int pks,
                                                         const double *__restrict__ dxg, ViscParams vp) {
  __shared__ ViscParShared<PTX, PTY> sh;
  visc_par_tile<PTX, PTY>(Q, par, nx, ny, nz, dxg, vp, blockIdx.x, pks, sh);
}

// Viscous terms of all members of an ensemble: one launch with a block per
// (member, tile) work item; ptiles0 holds each member's first item.
struct EnsViscArgs {
  const EnsMember *mem;
  int nmem;
  const unsigned *ptiles0;
  unsigned nitems;
  int pks;
  ViscParams vp;
};

__global__ void __launch_bounds__(PAR_THREADS) k_ens_visc(EnsViscArgs a) {
  __shared__ ViscParShared<PTX, PTY> sh;
  const unsigned item = blockIdx.x;  // one block per item (a loop over items spills 13 registers)
  if (item >= a.nitems) return;
  int lo = 0, hi = a.nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.ptiles0[mid] <= item) lo = mid;
    else hi = mid - 1;
  }
  const EnsMember &M = a.mem[lo];
  visc_par_tile<PTX, PTY>(M.q, M.par, M.n[0], M.n[1], M.n[2], M.dxg, a.vp, (int)(item - a.ptiles0[lo]), a.pks, sh);
}

// primitive variables of every member's state
__global__ void __launch_bounds__(256) k_ens_prims(const EnsMember *__restrict__ mem, int nmem,
                                                   const double *__restrict__ u, size_t ncell, double gamma) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  int lo = 0, hi = nmem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mem[mid].off <= idx) lo = mid;
    else hi = mid - 1;
  }
  const EnsMember &M = mem[lo];
  const size_t c = idx - M.off;
  const double *um = u + 5 * M.off;
  double s[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) s[v] = um[(size_t)v * M.ncell + c];
  double q[4];
  visc_prims(s, gamma, q);
#pragma unroll
  for (int v = 0; v < 4; v++) M.q[(size_t)v * M.ncell + c] = q[v];
}

// ---------------------------------------------------------------------------
// the parabolic term on its own (hm_parabolic): par, with the zero mass
// component, into a five-variable array
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_par_out(const double *__restrict__ par, double *__restrict__ out,
                                                 size_t ncell) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  out[idx] = 0.0;
#pragma unroll
  for (int v = 0; v < 4; v++) out[(size_t)(v + 1) * ncell + idx] = par[(size_t)v * ncell + idx];
}

// ---------------------------------------------------------------------------
// reductions: CFL max, squared-difference sum, volume integrals
//
// Bound by the reads of the states.  512 blocks of 1024 threads fill the 256
// CUs and leave 512 partials (five of each for the integrals), few enough for
// the host to fold: the kernels write them into pinned host memory, without a
// copy.  At 128^3: k_cfl 17.4 us (84 MB, 4.8 TB/s; 20.1 before), k_volint 14.7
// (22.0 before, on 409 blocks of 256), k_sqdiff 25.3 for 168 MB; the three calls
// 123 -> 109 us, the rest of it launches and waits.  (A last block that folds on
// the GPU costs each block a release to memory behind its XCD's cache: 45 us
// over 2048 blocks.)
// ---------------------------------------------------------------------------
constexpr int RED_THREADS = 1024, RED_WAVES = RED_THREADS / 64;

__device__ __forceinline__ double wave_max(double v) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// The cells t, t + T, t + 2T, ... of thread t of a launch of T threads, as
// (i, j, k): T < 2^20, so the divisions are of 32 bits and once a thread, and
// a step is additions with a carry instead of three 64-bit remainders a cell.
struct CellWalk {
  int i, j, k, si, sj, sk, nx, ny;
  __device__ __forceinline__ CellWalk(int nx_, int ny_) : nx(nx_), ny(ny_) {
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x, T = gridDim.x * blockDim.x;
    const unsigned r = t / (unsigned)nx, R = T / (unsigned)nx;
    i = (int)(t - r * nx);
    k = (int)(r / (unsigned)ny);
    j = (int)(r - (unsigned)k * ny);
    si = (int)(T - R * nx);
    sk = (int)(R / (unsigned)ny);
    sj = (int)(R - (unsigned)sk * ny);
  }
  __device__ __forceinline__ void step() {
    i += si;
    j += sj;
    k += sk;
    if (i >= nx) { i -= nx; j++; }
    if (j >= ny) { j -= ny; k++; }
  }
};

// per-block partial maxima of the local CFL; NaN propagates as +Inf flag
__global__ void __launch_bounds__(RED_THREADS) k_cfl(const double *__restrict__ u, double *__restrict__ part,
                                             int nx, int ny, int nz, const double *__restrict__ dxg,
                                             double gamma, double dt) {
  const size_t ncell = (size_t)nx * ny * nz;
  __shared__ double red[RED_WAVES];
  double m = 0.0;
  CellWalk cell(nx, ny);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < ncell;
       idx += (size_t)gridDim.x * blockDim.x, cell.step()) {
    double s[NV];
    for (int v = 0; v < NV; v++) s[v] = u[(size_t)v * ncell + idx];
    Prim q = flowvar(s, gamma);
    const double c = sqrt(gamma * q.P / q.rho);
    const double lx = (fabs(q.vx) + c) * dt * dxg[3 + cell.i];
    const double ly = (fabs(q.vy) + c) * dt * dxg[(nx + 6) + 3 + cell.j];
    const double lz = (fabs(q.vz) + c) * dt * dxg[(nx + 6) + (ny + 6) + 3 + cell.k];
    double l = fmax(fmax(lx, ly), lz);
    if (!(l == l) || l > 1.0e300) l = __builtin_inf();
    m = fmax(m, l);
  }
  m = wave_max(m);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int q = 1; q < RED_WAVES; q++) r = fmax(r, red[q]);
    part[blockIdx.x] = r;
  }
}

__global__ void __launch_bounds__(RED_THREADS) k_sqdiff(const double *__restrict__ a, const double *__restrict__ b,
                                                double *__restrict__ part, size_t n) {
  __shared__ double red[RED_WAVES];
  double s = 0.0;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
       idx += (size_t)gridDim.x * blockDim.x) {
    const double d = a[idx] - b[idx];
    s += d * d;
  }
  s = wave_sum(s);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = 0.0;
    for (int q = 0; q < RED_WAVES; q++) r += red[q];
    part[blockIdx.x] = r;
  }
}

// ---------------------------------------------------------------------------
// layout conversion (reference AoS with ghosts <-> hm SoA)
// ---------------------------------------------------------------------------
__global__ void k_aos_to_soa(const double *__restrict__ aos, double *__restrict__ soa, int nx, int ny,
                             int nz, int g) {
  const size_t ncell = (size_t)nx * ny * nz;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  const int i = (int)(idx % nx);
  const int j = (int)((idx / nx) % ny);
  const int k = (int)(idx / ((size_t)nx * ny));
  const size_t p = ((size_t)(k + g) * (ny + 2 * g) + (j + g)) * (nx + 2 * g) + (i + g);
  for (int v = 0; v < NV; v++) soa[(size_t)v * ncell + idx] = aos[p * NV + v];
}

__global__ void k_soa_to_aos(const double *__restrict__ soa, double *__restrict__ aos, int nx, int ny,
                             int nz, int g) {
  const size_t ncell = (size_t)nx * ny * nz;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncell) return;
  const int i = (int)(idx % nx);
  const int j = (int)((idx / nx) % ny);
  const int k = (int)(idx / ((size_t)nx * ny));
  const size_t p = ((size_t)(k + g) * (ny + 2 * g) + (j + g)) * (nx + 2 * g) + (i + g);
  for (int v = 0; v < NV; v++) aos[p * NV + v] = soa[(size_t)v * ncell + idx];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline unsigned nblocks(size_t n, unsigned bs) { return (unsigned)((n + bs - 1) / bs); }

static ViscParams visc_params(const Scheme &sc) {
  ViscParams vp;
  vp.gamma = sc.gamma;
  vp.inv_Re = sc.Re > 0 ? 1.0 / sc.Re : 0.0;
  vp.inv_gm1 = 1.0 / (sc.gamma - 1.0);
  vp.inv_Pr = 1.0 / sc.Pr;
  return vp;
}

// A segment of p planes marches p + 4 and starts on 4 more.  (For grids that run
// together, total work over 256 plus half a block chose segments too long: 463
// us against 349 for the eight of 9.3e6 cells.)
int visc_segment(int count, const int (*n)[3]) { return plane_segment(count, n, 6, par_tiles); }

void launch_visc_par(const Grid &g, const Scheme &sc, const double *Q, double *par, const double *dxg,
                     hipStream_t st) {
  const unsigned nb = par_tiles(g.n[0], g.n[1], g.n[2], g.pks);
  hipLaunchKernelGGL(k_visc_par, dim3(nb), dim3(PAR_THREADS), 0, st, Q, par, g.n[0], g.n[1], g.n[2], g.pks, dxg,
                     visc_params(sc));
}

void launch_ens_visc(const Scheme &sc, const EnsMember *mem, int nmem, const unsigned *ptiles0, unsigned nitems,
                     int pks, hipStream_t st) {
  EnsViscArgs a;
  a.pks = pks;
  a.mem = mem;
  a.nmem = nmem;
  a.ptiles0 = ptiles0;
  a.nitems = nitems;
  a.vp = visc_params(sc);
  hipLaunchKernelGGL(k_ens_visc, dim3(nitems), dim3(PAR_THREADS), 0, st, a);
}

void launch_ens_prims(const Scheme &sc, const EnsMember *mem, int nmem, const double *u, size_t ncell,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_ens_prims, dim3(nblocks(ncell, 256)), dim3(256), 0, st, mem, nmem, u, ncell, sc.gamma);
}

void launch_par_out(const Grid &g, const double *par, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_par_out, dim3(nblocks(g.ncell, 256)), dim3(256), 0, st, par, out, g.ncell);
}

// Volume integral of every conserved variable: sum of u dV over the
// interior cells with dV = 1/dxinv_x 1/dxinv_y 1/dxinv_z
// (src/HyParFunctions/VolumeIntegral.c:14-50); one partial per block and
// variable, part[5*block + v].
__global__ void __launch_bounds__(RED_THREADS) k_volint(const double *__restrict__ u, double *__restrict__ part, int nx,
                                                int ny, int nz, const double *__restrict__ dxg) {
  const size_t ncell = (size_t)nx * ny * nz;
  __shared__ double red[NV][RED_WAVES];
  double acc[NV] = {0, 0, 0, 0, 0};
  CellWalk cell(nx, ny);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < ncell;
       idx += (size_t)gridDim.x * blockDim.x, cell.step()) {
    double dV = 1.0;
    dV *= 1.0 / dxg[3 + cell.i];
    dV *= 1.0 / dxg[(nx + 6) + 3 + cell.j];
    dV *= 1.0 / dxg[(nx + 6) + (ny + 6) + 3 + cell.k];
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] += u[(size_t)v * ncell + idx] * dV;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const double t = wave_sum(acc[v]);
    if (lane == 0) red[v][w] = t;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double r = 0.0;
    for (int q = 0; q < RED_WAVES; q++) r += red[threadIdx.x][q];
    part[(size_t)blockIdx.x * NV + threadIdx.x] = r;
  }
}

unsigned reduction_blocks(size_t n) {
  unsigned b = nblocks(n, RED_THREADS);
  return b > 512 ? 512 : (b == 0 ? 1 : b);
}

void launch_volint(const Grid &g, const double *u, double *part, unsigned nb, const double *dxg, hipStream_t st) {
  hipLaunchKernelGGL(k_volint, dim3(nb), dim3(RED_THREADS), 0, st, u, part, g.n[0], g.n[1], g.n[2], dxg);
}

void launch_cfl(const Grid &g, const Scheme &sc, const double *u, double *part, unsigned nb,
                const double *dxg, double dt, hipStream_t st) {
  hipLaunchKernelGGL(k_cfl, dim3(nb), dim3(RED_THREADS), 0, st, u, part, g.n[0], g.n[1], g.n[2], dxg, sc.gamma, dt);
}

void launch_sqdiff(const double *a, const double *b, double *part, unsigned nb, size_t n,
                   hipStream_t st) {
  hipLaunchKernelGGL(k_sqdiff, dim3(nb), dim3(RED_THREADS), 0, st, a, b, part, n);
}

void launch_aos_to_soa(const Grid &g, const double *aos, double *soa, int ghosts, hipStream_t st) {
  hipLaunchKernelGGL(k_aos_to_soa, dim3(nblocks(g.ncell, 256)), dim3(256), 0, st, aos, soa, g.n[0], g.n[1],
                     g.n[2], ghosts);
}

void launch_soa_to_aos(const Grid &g, const double *soa, double *aos, int ghosts, hipStream_t st) {
  hipLaunchKernelGGL(k_soa_to_aos, dim3(nblocks(g.ncell, 256)), dim3(256), 0, st, soa, aos, g.n[0], g.n[1],
                     g.n[2], ghosts);
}

}  // namespace hm
