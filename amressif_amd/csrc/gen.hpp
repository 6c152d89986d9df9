// The general path: the fractional step on n^dim cells (dim 2 or 3) with
// periodic directions (phy_bc 111) beside the wall codes, FP64.  Used by a
// context whose inputs are 3D or name a periodic direction; the 2D wall-only
// configurations keep the fused single-level kernels.
//
// Layout in HBM (one box, i fastest, then j, then k; no padding):
//   face array of direction d: n + 1 along d, n along the others
//   cell arrays (p, phi, b, multigrid levels): n^dim
//   cell velocities X: dim comps with two ghost layers, (n + 4)^dim each
//   (in 2D the k extent is 1 and has no ghosts)
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "internal.hpp"

namespace amr {
namespace gen {

constexpr int kBlock = 256;
constexpr int kMaxGenLevels = 16;

// Ghost rule of a wall side (cont2cart, utilities.cpp:87-346): 0 every comp
// -mirror (135), 1 slip: the normal comp -mirror, the others +mirror (-135;
// the east side's code 1), 2 unit inflow 2 - mirror (165 on W, E, S, B, F,
// -165 on W), 3 the north side's 2 inflow - mirror (165).
struct Geom {
    int dim, n, nk;        // nk: cells along k (n in 3D, 1 in 2D)
    int per[3];            // periodic directions
    int kind_lo[3], kind_hi[3];
    double inflow[3];
    double idx[3], idx2[3];  // 1/dx, 1/dx^2
    double iren, c15, dt;
    int pseudo;            // PSEUDO_TIMESTEPPING
    int64_t nf[3];         // faces per direction
    int64_t ncell;         // n^dim
    int64_t xs;            // cells per component of X ((n + 4)^dim)
};

struct Level {
    int n;            // cells per side
    double a[3];      // 1/h_d^2 of this level
    double *e, *r;    // the down leg's correction and the right-hand side (n^dim)
    double *out;      // the up leg's (or the exact solve's) correction
    int64_t ncell;
};

struct Ctx {
    Geom g{};
    double rk[4]{};
    double *U[3]{}, *Up[3]{}, *C[3]{}, *B[3]{}, *S[3]{};  // u^n, u^{n-1}, BDF2 constant, pseudo bases (u* ends in S)
    double *X = nullptr;   // cell velocities with ghosts
    double *p = nullptr, *phi = nullptr, *b = nullptr;
    Level lev[kMaxGenLevels]{};
    int nlev = 0;
    double *exact = nullptr;  // coarsest level: eigenvectors and eigenvalues of its 1D operators
    double *phi2 = nullptr;   // the solve's iterates alternate between phi and phi2
    double *partials = nullptr;
    int64_t npartials = 0;
    int nb_face[3]{};        // blocks per face direction of a launch over every face
    int last_P = 8, last_V = 8;
    int s3_ntx = 0, s3_nty = 0, s3_zc = 0;  // 3D stage: tiles in x and y, planes per workgroup
};

// ---- launchers (kernels_gen.hip); every guarded kernel returns at once once
// its loop's flag in the control block is set
hipError_t cells(const Ctx &c, hipStream_t s, double *const *faces, double *X);
// 2D: the step's pseudo-iteration `it` (or the explicit update), out <- the last stage from base, with its norm
// partials; chained: it also takes the norm of the launch before and ends the loop
hipError_t iteration2(const Ctx &c, hipStream_t s, double *const *base, double *const *out, int it, bool chained,
                      Ctl *ctl);
// 3D: one RK4 stage in one pass, out <- base + rk (R(in) - c15 in + C); out
// aliases neither in nor base.  last: the norm partials of base - out as well
hipError_t stage3(const Ctx &c, hipStream_t s, double *const *in, double *const *base, double *const *out, double rk,
                  int last, const Ctl *guard);
void stage3_shape(int n, int *ntx, int *nty, int *zc);
int stage3_blocks(const Ctx &c);
hipError_t fin_pseudo(const Ctx &c, hipStream_t s, int it, Ctl *ctl);
hipError_t bdf2(const Ctx &c, hipStream_t s);
// b = (1.5/dt) D(faces) (b may be null: the norm only); partials of max|D|, sum b
hipError_t divergence(const Ctx &c, hipStream_t s, double *const *faces, double *b, int *nblocks);
// which 0: div_star, rhs_sum and b's mean (the step's Poisson RHS), 1: div_new
hipError_t fin_div(const Ctx &c, hipStream_t s, int nblocks, Ctl *ctl, int which);
hipError_t mg_start(const Ctx &c, hipStream_t s, Ctl *ctl);
// one V-cycle for L e = lev[0].r into lev[0].out (kernels_gen_mg.hip)
hipError_t vcycle(const Ctx &c, hipStream_t s, const Ctl *ctl);
// phi2 = phi + e, lev[0].r = (b - mean) - L phi2 and the stopping test (e null: phi2 = 0)
hipError_t outer(const Ctx &c, hipStream_t s, const double *phi, const double *e, double *phi2, Ctl *ctl);
int outer_blocks(int dim, int n);
// the exact 2D solve of a level of at most 64^2 cells (kernels_mg.hip's k_tail_dct)
hipError_t launch_exact2(hipStream_t s, const double *r, double *e, int n, const double *tab, const Ctl *ctl);
// u = u* - (dt/1.5) G phi and p += phi - mean (the solve's)
hipError_t project(const Ctx &c, hipStream_t s, Ctl *ctl);
hipError_t fin_step(const Ctx &c, hipStream_t s, Ctl *ctl, amressif_step_stats *log);
hipError_t fill(hipStream_t s, double *dst, int64_t count, double value);
// Array4 views <-> internal arrays: a box region [0, ext) with the view's lo/hi
hipError_t pack(hipStream_t s, const amr_array4 &a, int comp, double *dst, int ex, int ey, int ez);
hipError_t unpack(hipStream_t s, const double *src, const amr_array4 &a, int comp, int ex, int ey, int ez);
// the window [lo, hi] of a view <-> the same cells of an internal array of
// extents ex x ey x .. (unpack 0: view -> array)
hipError_t pack_window(hipStream_t s, const amr_array4 &a, int comp, double *dst, int ex, int ey, const int *lo,
                       const int *hi, int unpack);
// userCtx / velCart views with ghosts: the cells the view holds, ghosts by the
// rules (p, phi: Neumann mirror / periodic image; phi shifted by -mean)
hipError_t unpack_cells_ghosted(const Ctx &c, hipStream_t s, const double *src, const amr_array4 &a, int comp,
                                const double *shift);
hipError_t unpack_velcart(const Ctx &c, hipStream_t s, const double *X, const amr_array4 &a);
hipError_t phi_mean(const Ctx &c, hipStream_t s, Ctl *ctl);

}  // namespace gen
}  // namespace amr
