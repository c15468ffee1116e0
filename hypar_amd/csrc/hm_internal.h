// hm_internal.h -- declarations shared by the C-ABI and the kernel launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include <cmath>
#include <string>

struct hm_solver;

namespace hm {

// drops every slot binding of s (hm_bind.hip); hm_destroy calls it
void drop_bindings(const ::hm_solver *s);

enum { INTERP_COMP = 0, INTERP_CHAR = 1 };
enum { UPWIND_ROE = 0, UPWIND_RUSANOV = 1 };
enum { OUT_STAGE = 0, OUT_RHS = 1, OUT_HYP = 2, OUT_PAR = 3 };
enum { WENO_JS = 0, WENO_MAPPED = 1, WENO_Z = 2, WENO_YC = 3, WENO_OPTIMAL = 4 };

struct Grid {
  int n[3];
  size_t ncell;
  int seg[3];  // cells per march segment of the y and z passes (march_segments)
  int pks;     // planes per segment of the viscous-term kernel (visc_segment)
  int vks;     // planes per segment of its adjoint (visc_vjp_segment)
};

struct Scheme {
  int interp, upwind;
  double gamma;
  double Re;  // as the solver uses it (physics.inp Re / Minf); <= 0 inviscid
  double Pr;
  double eps;
  int weno;   // WENO_*
};

// records msg as the calling thread's hm_last_error() and returns code
int set_error(int code, const std::string &msg);

// Metrics of the uniform periodic grid x_i = i*(2*pi/n) with g ghost points
// per side: ghost coordinates extrapolated linearly (ReadArray.c:59-90),
// dxinv = 2/(x[i+1]-x[i-1]) inside and copies of the edge value in the
// ghosts (InitialSolution.c:74-113).  X is caller scratch of n + 2g doubles;
// out receives n + 2g doubles.  Host code (compiled without FMA contraction
// on x86-64), so the values are those of the reference's own host code.
inline void uniform_dxinv(int n, int g, double *X, double *out) {
  const double h = 2.0 * M_PI / n;
  for (int i = 0; i < n; i++) X[g + i] = (double)i * h;
  for (int i = 0; i < g; i++) {
    int delta = g - i;
    X[i] = X[g] + ((double)delta) * (X[g] - X[g + 1]);
  }
  for (int i = n + g; i < n + 2 * g; i++) {
    int delta = i - (n + g - 1);
    X[i] = X[n + g - 1] + ((double)delta) * (X[n + g - 1] - X[n + g - 2]);
  }
  for (int i = 0; i < n; i++) out[i + g] = 2.0 / (X[i + 1 + g] - X[i - 1 + g]);
  for (int i = 0; i < g; i++) out[i] = out[g];
  for (int i = n + g; i < n + 2 * g; i++) out[i] = out[n + g - 1];
}

// the viscous term par (4*ncell: momentum x, y, z, energy) of the state
// whose primitive variables (u, v, w, T) are in Q (4*ncell)
void launch_visc_par(const Grid &g, const Scheme &sc, const double *Q, double *par, const double *dxg,
                     hipStream_t st);
// par as a five-variable array with a zero mass component
void launch_par_out(const Grid &g, const double *par, double *out, hipStream_t st);
unsigned reduction_blocks(size_t n);
// volume integral partials: part[5*block + v], 5*nb entries
void launch_volint(const Grid &g, const double *u, double *part, unsigned nb, const double *dxg, hipStream_t st);
void launch_cfl(const Grid &g, const Scheme &sc, const double *u, double *part, unsigned nb,
                const double *dxg, double dt, hipStream_t st);
void launch_sqdiff(const double *a, const double *b, double *part, unsigned nb, size_t n,
                   hipStream_t st);
void launch_aos_to_soa(const Grid &g, const double *aos, double *soa, int ghosts, hipStream_t st);
void launch_soa_to_aos(const Grid &g, const double *soa, double *aos, int ghosts, hipStream_t st);

// per-slot operators (hm_slots.hip)
void launch_flux(const Grid &g, const Scheme &sc, int dir, const double *u, double *f, hipStream_t st);
void launch_modsol(const Grid &g, const Scheme &sc, const double *u, double *uC, hipStream_t st);
void launch_interp(const Grid &g, const Scheme &sc, int dir, double *fI, const double *fC,
                   const double *u, int upw, int uflag, hipStream_t st);
void launch_upwind(const Grid &g, const Scheme &sc, int dir, double *fI, const double *fL,
                   const double *fR, const double *uL, const double *uR, const double *u,
                   hipStream_t st);
void launch_fluxdiff(const Grid &g, int dir, double *hyp, const double *fI, const double *dxg,
                     int accumulate, hipStream_t st);
void launch_axpy(const double *x, double a, double *y, size_t n, hipStream_t st);
void launch_fill(double *x, double value, size_t n, hipStream_t st);

// Update of a Runge-Kutta stage by the z pass.  With r the stage's right-hand
// side and U its state,
//   UPD_SELF  out = U + c r                                  (the first stage)
//   UPD_MIX   out = a0 + (k (U - a0) + c r)
//   UPD_RK4   out = a1 + (((a2 - a1) + (U - a0))/3 + c r)
// RK4 with the stage states U2 = u + dt/2 k1, U3 = u + dt/2 k2, U4 = u + dt k3
// ends in u + dt (k1 + 2 k2 + 2 k3 + k4)/6 = U3 + ((U2 - U3) + (U4 - u))/3 +
// dt/6 k4, and SSPRK3 (its tableau of TimeExplicitRKInitialize.c:69-79) is
// U2 = u + dt k1, U3 = u + ((U2 - u) + dt k2)/4, u + 2/3 ((U3 - u) + dt k3).
// The updates so need no accumulator: a stage reads at most u, the last RK4
// stage u, U2 and U3, and writes one state.
enum { UPD_SELF = 0, UPD_MIX = 1, UPD_RK4 = 2 };
struct StageUpdate {
  int kind;
  double c, k;                  // c in units of dt for an ensemble, whose members have their own
  const double *a0, *a1, *a2;   // operands the kind reads
  double *out;
};

// fused direction passes (hm_pass.hip)
struct PassBuffers {
  const double *U;        // stage state
  double *R;              // hyperbolic-term accumulator, 5*ncell
  const double *par;      // viscous term, 4*ncell (viscous runs; read by the z pass)
  double *Q;              // u, v, w, T of the new state (z pass, viscous OUT_STAGE)
  StageUpdate upd;        // z pass: the stage's update (OUT_STAGE); out also takes OUT_RHS and OUT_HYP
};
// pass along dir: x stores its flux differences in R, y adds its own, z adds
// its own and forms rhs = -hyp + par, then finishes the stage (mode
// OUT_STAGE) or writes rhs (OUT_RHS) or hyp (OUT_HYP)
void launch_pass(const Grid &g, const Scheme &sc, int dir, const PassBuffers &b, int mode, const double *dxg,
                 hipStream_t st);
// primitive variables (u, v, w, T) of u into Q
void launch_prims(const Grid &g, const Scheme &sc, const double *u, double *Q, hipStream_t st);

// tiles of the viscous adjoint kernel (hm_adjoint.hip): a block owns VTX x VTY
// (x, y) columns and marches through a z segment of vks planes
constexpr int VTX = 64, VTY = 8;
constexpr int VT = VTX * VTY;  // threads of a viscous block
constexpr int VHX = VTX + 4, VHY = VTY + 4;
__host__ __device__ inline unsigned visc_tiles(int nx, int ny, int nz, int vks) {
  return (unsigned)(((nx + VTX - 1) / VTX) * ((ny + VTY - 1) / VTY) * ((nz + vks - 1) / vks));
}
// segment length of that kernel over `count` grids that run together
int visc_vjp_segment(int count, const int (*n)[3]);

// tiles of the viscous-term kernel (hm_kernels.hip): a block owns PTX x PTY
// (x, y) columns and marches through a z segment of pks planes
constexpr int PTX = 32, PTY = 16;
constexpr int PAR_THREADS = PTX * PTY + 4 * PTX + 4 * PTY;  // the tile's columns and its halo points
__host__ __device__ inline unsigned par_tiles(int nx, int ny, int nz, int pks) {
  return (unsigned)(((nx + PTX - 1) / PTX) * ((ny + PTY - 1) / PTY) * ((nz + pks - 1) / pks));
}
// segment length of the viscous-term kernel over `count` grids that run together
int visc_segment(int count, const int (*n)[3]);

// The z segment of these two kernels, whose blocks march p planes of a tile in
// p + start plane times, one block on each of the 256 CUs: W blocks take
// ceil(W/256) (p + start).  The length with the least such time is taken; a
// shorter one has to win 3%.
template <class Tiles>
int plane_segment(int count, const int (*n)[3], int start, Tiles tiles) {
  constexpr int CUS = 256;
  int nmax = 0;
  for (int m = 0; m < count; m++) nmax = n[m][2] > nmax ? n[m][2] : nmax;
  int best = nmax;
  double tbest = 0.0;
  for (int parts = 1; parts <= nmax; parts++) {
    const int p = (nmax + parts - 1) / parts;
    if (parts > 1 && p == (nmax + parts - 2) / (parts - 1)) continue;
    double blocks = 0.0;
    for (int m = 0; m < count; m++) blocks += tiles(n[m][0], n[m][1], n[m][2], p);
    const double t = std::ceil(blocks / CUS) * (p + start);
    if (parts == 1 || t < 0.97 * tbest) {
      tbest = t;
      best = p;
    }
  }
  return best;
}

// batched ensemble passes (hm_pass.hip): members of one scheme
struct EnsMember {
  int n[3];
  int seg[3];         // cells per march segment of the y and z passes
  size_t ncell;
  size_t off;         // first cell of the member; its state is u[5*off .. 5*(off+ncell))
  const double *dxg;  // ghosted dxinv x|y|z of the member (device)
  double dt;          // the member's time step
  // viscous members: viscous term (4*ncell) and primitive variables
  // (4*ncell); null when inviscid
  double *par, *q;
};
// work items of one member in pass dir with tile shape `shape` (0: 4
// wavefronts per block, 1: 2 wavefronts per block)
unsigned ens_items_per_member(int dir, int shape, const int n[3], const int seg[3]);
// cells per march segment of the pass along dir (1 or 2) of `count` grids that
// run together, into seg[count]
void march_segments(int count, const int (*n)[3], int dir, int *seg);
// one pass of an RK stage over all members; grid = number of persistent
// blocks (0: one block per work item)
void launch_ens_pass(const Scheme &sc, int dir, int shape, const EnsMember *mem, int nmem, const unsigned *item0,
                     unsigned nitems, unsigned grid, const double *U, double *R, const StageUpdate &upd,
                     hipStream_t st);
// all three passes of an RK stage over all members in one persistent
// launch (rows = 4 or 2 wavefronts per block, the tile shapes of the split
// passes; grid 0 = the blocks the GPU holds at once, cus CUs).  An x item
// is ENS_STAGE_XG groups of x-lines: item0[0] lists each member's first x
// item, xgroups0 its first x-line group (the split x pass's items).  ctr
// holds 4 + 2*nmem zeroed counters and is zero again when the launch ends;
// a dependency wait that polls more than spin_limit times sets ctr[2].
#ifndef HM_ENS_XG
#define HM_ENS_XG 64
#endif
constexpr unsigned ENS_STAGE_XG = HM_ENS_XG;
void launch_ens_stage(const Scheme &sc, int rows, const EnsMember *mem, int nmem, const unsigned *const item0[3],
                      const unsigned nitems[3], const unsigned *xgroups0, unsigned xg, unsigned grid, int cus,
                      unsigned *ctr, unsigned spin_limit, const double *U, double *R, const StageUpdate &upd,
                      hipStream_t st);

// viscous terms of all members (hm_kernels.hip): one launch over the
// (member, par_tiles) items of pks planes, ptiles0 = each member's first item
// (nmem + 1 entries); primitive variables of all members
void launch_ens_visc(const Scheme &sc, const EnsMember *mem, int nmem, const unsigned *ptiles0, unsigned nitems,
                     int pks, hipStream_t st);
void launch_ens_prims(const Scheme &sc, const EnsMember *mem, int nmem, const double *u, size_t ncell,
                      hipStream_t st);

// discrete adjoint (hm_adjoint.hip)
bool vjp_supported(const Grid &g, const Scheme &sc);
// doubles of device work space launch_rhs_vjp needs (viscous schemes)
size_t vjp_work_size(const Grid &g, const Scheme &sc);
// nu = (d rhs/d u)^T mu at u with mu = cb*lam + ca*nu_in (nu_in may be
// null); when L is not null the finished nu is also added into L (set_L:
// L = lam + nu); work holds vjp_work_size doubles
void launch_rhs_vjp(const Grid &g, const Scheme &sc, const double *u, const double *lam, const double *nu_in,
                    double ca, double cb, double *nu, double *L, bool set_L, const double *dxg, double *work,
                    hipStream_t st);

// the same for all members of an ensemble at once: member m's stage
// coefficients are dt_m*A and dt_m*B; lines0[d] lists each member's first
// line along d (nmem + 1 entries), nmax[d] the longest line along d, and
// items0[d] each member's first work item of the line VJPs along d, an item
// being ens_vjp_lines_per_item(nmax[d], n[d]) consecutive lines of the member
struct EnsVjpPlan {
  const EnsMember *mem;  // device member table
  int nmem;
  size_t ncell;
  const unsigned *lines0[3];
  unsigned nlines[3];
  const unsigned *items0[3];
  unsigned nitems[3];
  int nmax[3];
  const unsigned *tiles0;  // viscous members: each member's first viscous tile (nmem + 1 entries)
  unsigned ntiles;
  int vks;                 // planes per tile
};
bool ens_vjp_supported(const Scheme &sc, const int nmax[3]);
int ens_vjp_threads(int nmax);                 // block size of the line VJPs along a direction
int ens_vjp_lines_per_item(int nmax, int n);  // lines of length n per work item
size_t ens_vjp_work_size(const Scheme &sc, size_t ncell);
void launch_ens_rhs_vjp(const Scheme &sc, const EnsVjpPlan &p, const double *u, const double *lam,
                        const double *nu_in, double A, double B, double *nu, double *L, bool set_L, double *work,
                        hipStream_t st);

}  // namespace hm
