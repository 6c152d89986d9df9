// Host side of the general path (gen.hpp): context set-up, state load/store
// and the time step on n^dim cells (dim 2 or 3) with periodic directions.
// The C-ABI entry points of api.cpp hand a context to these functions when
// its inputs are 3D or name a periodic direction.
//
// The step follows main.cpp:875-1202 as the single-level path does: the BDF2
// history with -G p folded into the constant, the RK4 dual-time loop (or the
// explicit update of PSEUDO_TIMESTEPPING = 0) under device-side control with
// one host poll per batch of pseudo-iterations, the Poisson RHS, the V-cycle
// iteration to ||r||inf <= tol_rel ||b||inf (poisson.cpp:41-186; one poll per
// batch of cycles), and the projection with p += phi - mean(phi).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include <cstdlib>

#include "gen.hpp"
#include "iter_tile.hpp"

namespace {

using amr::Ctx;
namespace G = amr::gen;

int gfail(amressif_ctx *ctx, int code, const std::string &msg) { return amr_fail(ctx, code, msg); }

#define GCHK(expr)                                                                               \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess) return gfail(ctx, AMRESSIF_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <class T>
hipError_t alloc(Ctx &c, T **ptr, size_t count)
{
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, count * sizeof(T) + 256);
    if (e != hipSuccess) return e;
    c.allocs.push_back(p);
    c.bytes += (int64_t)(count * sizeof(T) + 256);
    *ptr = (T *)p;
    return hipSuccess;
}

// cont2cart's wall rule of one side (utilities.cpp:87-346): the kind of
// gen.hpp, or -1 where the reference aborts, -3 where it leaves the ghosts
// unfilled
int side_kind(int d, int hi, int code)
{
    if (code == 135) return 0;
    if (code == 195 || code == -195) return -1;
    if (d == 0 && !hi) {
        if (code == -135) return 1;
        if (code == 165 || code == -165) return 2;
        return -3;
    }
    if (d == 0 && hi) {
        if (code == -165) return -1;
        if (code == 1) return 1;
        if (code == 165) return 2;
        return -3;
    }
    if (code == -165) return -1;
    if (code == -135) return 1;
    if (code == 165) return (d == 1 && hi) ? 3 : 2;
    return -3;
}

// Orthonormal eigenvectors Q[i][k] (row stride ld) and eigenvalues of the 1D second
// difference a (e(i + 1) - 2 e(i) + e(i - 1)) on m cells: DCT-II vectors with Neumann
// ends, cosines and sines of the same wave number with periodic ones.  Vector 0 is
// the constant.
void modes_1d(int m, double a, bool per, std::vector<double> &Q, std::vector<double> &lam)
{
    const double pi = 3.14159265358979323846;
    Q.assign((size_t)m * m, 0.0);
    lam.assign(m, 0.0);
    for (int k = 0; k < m; ++k) {
        const int f = per ? (k + 1) / 2 : k;  // wave number
        double nrm = 0.0;
        for (int i = 0; i < m; ++i) {
            double v;
            if (!per) v = std::cos(pi * (double)(((int64_t)(2 * i + 1) * f) % (4 * m)) / (2 * m));
            else if (k % 2 == 1 || k == 0) v = std::cos(2 * pi * (double)((int64_t)i * f % m) / m);
            else v = std::sin(2 * pi * (double)((int64_t)i * f % m) / m);
            Q[(size_t)i * m + k] = v;
            nrm += v * v;
        }
        for (int i = 0; i < m; ++i) Q[(size_t)i * m + k] /= std::sqrt(nrm);
        const double h = std::sin(pi * f / (per ? m : 2.0 * m));
        lam[k] = -4.0 * a * h * h;
    }
}

// the tables of the coarsest level's exact solve (k_gen_exact3 in 3D, k_tail_dct in 2D)
std::vector<double> exact_tables(const G::Geom &g, const G::Level &L)
{
    const int m = L.n;
    std::vector<double> Q[3], lam[3], t;
    for (int d = 0; d < g.dim; ++d) modes_1d(m, L.a[d], g.per[d] != 0, Q[d], lam[d]);
    if (g.dim == 3) {
        const int ld = 24;
        t.assign((size_t)6 * m * ld + (size_t)m * m * m, 0.0);
        for (int d = 0; d < 3; ++d) {
            double *q = t.data() + (size_t)2 * d * m * ld, *qt = q + (size_t)m * ld;
            for (int i = 0; i < m; ++i)
                for (int k = 0; k < m; ++k) q[i * ld + k] = qt[k * ld + i] = Q[d][(size_t)i * m + k];
        }
        double *dinv = t.data() + (size_t)6 * m * ld;
        for (int q = 1; q < m * m * m; ++q)  // the constant mode's stays 0
            dinv[q] = 1.0 / (lam[0][q % m] + lam[1][(q / m) % m] + lam[2][q / (m * m)]);
        return t;
    }
    const int ld = 64;
    t.assign((size_t)3 * ld * ld, 0.0);
    for (int i = 0; i < m; ++i)
        for (int k = 0; k < m; ++k) {
            t[i * ld + k] = Q[0][(size_t)i * m + k];
            t[ld * ld + i * ld + k] = Q[1][(size_t)i * m + k];
            t[2 * ld * ld + i * ld + k] = i + k == 0 ? 0.0 : 1.0 / (lam[0][k] + lam[1][i]);
        }
    return t;
}

int poll(amressif_ctx *ctx)
{
    Ctx &c = ctx->c;
    GCHK(hipMemcpyAsync(c.ctl_host, c.ctl, sizeof(amr::Ctl), hipMemcpyDeviceToHost, c.stream));
    GCHK(hipStreamSynchronize(c.stream));
    return 0;
}

int check_view3(amressif_ctx *ctx, const amr_array4 *a, const int *lo, const int *hi, int ncomp, const char *what)
{
    if (!a || !a->ptr) return gfail(ctx, AMRESSIF_ERR_ARG, std::string(what) + ": null view");
    if (a->dtype != 0) return gfail(ctx, AMRESSIF_ERR_ARG, std::string(what) + ": double views only");
    for (int d = 0; d < 3; ++d)
        if (a->lo[d] > lo[d] || a->hi[d] < hi[d])
            return gfail(ctx, AMRESSIF_ERR_ARG, std::string(what) + ": view does not cover the box");
    if (a->ncomp < ncomp) return gfail(ctx, AMRESSIF_ERR_ARG, std::string(what) + ": too few components");
    return 0;
}

void face_ext(const G::Geom &g, int d, int *ext)
{
    for (int e = 0; e < 3; ++e) ext[e] = e < g.dim ? g.n + (e == d) : 1;
}

}  // namespace

// ================================================================== set-up
bool amr_gen_wanted(const amressif_inputs *in)
{
    if (in->spacedim == 3) return true;
    for (int d = 0; d < 2; ++d)
        if (in->phy_bc_lo[d] == 111 || in->phy_bc_hi[d] == 111) return true;
    return false;
}

int amr_gen_create(amressif_ctx *ctx)
{
    Ctx &c = ctx->c;
    const amressif_inputs &in = c.in;
    const int dim = in.spacedim, n = in.n_cell;
    if (dim != 2 && dim != 3) return gfail(ctx, AMRESSIF_ERR_ARG, "spacedim must be 2 or 3");
    if (n < 4 || (dim == 3 && n > 1024)) return gfail(ctx, AMRESSIF_ERR_ARG, "n_cell out of range for the general path");
    if (in.precision != AMRESSIF_FP64)
        return gfail(ctx, AMRESSIF_ERR_UNSUPPORTED, "3D and periodic runs are FP64 only (precision = 0)");
    if (in.poisson_solver != 0)
        return gfail(ctx, AMRESSIF_ERR_UNSUPPORTED, "3D and periodic runs use the multigrid Poisson solve");
    auto *gp = new G::Ctx();
    c.gen = gp;
    G::Ctx &gc = *gp;
    G::Geom &g = gc.g;
    g.dim = dim;
    g.n = n;
    g.nk = dim == 3 ? n : 1;
    // BCRec mapping (main.cpp:810-835) and the cont2cart branches per side
    for (int d = 0; d < dim; ++d) {
        const int lo = in.phy_bc_lo[d], hi = in.phy_bc_hi[d];
        if ((lo == 111) != (hi == 111))
            return gfail(ctx, AMRESSIF_ERR_UNSUPPORTED, "a periodic direction needs 111 on both sides");
        if (!(lo == 111 || std::abs(lo) == 135 || std::abs(lo) == 165 || std::abs(lo) == 195))
            return gfail(ctx, AMRESSIF_ERR_BC, "Invalid bc_lo");
        // the reference's hi-side test reads phy_bc_lo for the 135 case (main.cpp:827)
        if (!(hi == 111 || std::abs(lo) == 135 || std::abs(hi) == 165 || std::abs(hi) == 195))
            return gfail(ctx, AMRESSIF_ERR_BC, "Invalid bc_hi");
        g.per[d] = lo == 111;
        if (!g.per[d])
            for (int side = 0; side < 2; ++side) {
                const int k = side_kind(d, side, side ? hi : lo);
                if (k == -1) return gfail(ctx, AMRESSIF_ERR_BC, "boundary code: Not yet implemented");
                if (k == -3)
                    return gfail(ctx, AMRESSIF_ERR_UNSUPPORTED,
                                 "boundary code leaves the reference's ghost cells unfilled (utilities.cpp:87-346)");
                (side ? g.kind_hi : g.kind_lo)[d] = k;
            }
        g.inflow[d] = in.inflow_waveform[d];
        const double dx = (in.hi_phy_dim[d] - in.lo_phy_dim[d]) / n;
        if (!(dx > 0)) return gfail(ctx, AMRESSIF_ERR_ARG, "hi_phy_dim must exceed lo_phy_dim");
        g.idx[d] = 1.0 / dx;
        g.idx2[d] = 1.0 / (dx * dx);
    }
    g.dt = amressif_dt(&in);
    g.c15 = 1.5 / g.dt;
    g.iren = 1.0 / in.ren;
    g.pseudo = in.PSEUDO_TIMESTEPPING;
    g.ncell = (int64_t)n * n * g.nk;
    g.xs = (int64_t)(n + 4) * (n + 4) * (dim == 3 ? n + 4 : 1);
    const double dtau = 0.4 * g.dt;  // main.cpp:861-869
    gc.rk[0] = dtau * 0.25;
    gc.rk[1] = dtau * (1.0 / 3.0);
    gc.rk[2] = dtau * 0.5;
    gc.rk[3] = dtau * 1.0;
    for (int d = 0; d < dim; ++d) {
        int ext[3];
        face_ext(g, d, ext);
        g.nf[d] = (int64_t)ext[0] * ext[1] * ext[2];
        gc.nb_face[d] = (int)((g.nf[d] + G::kBlock - 1) / G::kBlock);
    }
    // multigrid hierarchy: halve while the side is even and the level holds more
    // than 512 cells; the first level of at most 20 (3D) or 64 (2D) cells per side is
    // solved exactly and ends it
    {
        int nl = n, l = 0;
        for (;;) {
            G::Level &L = gc.lev[l];
            L.n = nl;
            L.ncell = (int64_t)nl * nl * (dim == 3 ? nl : 1);
            for (int d = 0; d < 3; ++d) {
                const double h = d < dim ? (in.hi_phy_dim[d] - in.lo_phy_dim[d]) / nl : 1.0;
                L.a[d] = 1.0 / (h * h);
            }
            ++l;
            if ((nl & 1) || L.ncell <= 512 || l == G::kMaxGenLevels) break;
            nl /= 2;
        }
        gc.nlev = l;
        if (gc.lev[l - 1].ncell > 1024)
            return gfail(ctx, AMRESSIF_ERR_UNSUPPORTED,
                         "coarsest multigrid level above 1024 cells (n_cell = m 2^k with m^dim > 1024, m odd)");
        while (gc.nlev > 1 && gc.lev[gc.nlev - 2].n <= (dim == 3 ? 20 : 64)) gc.nlev -= 1;
    }
    if (dim == 3) {
        G::stage3_shape(n, &gc.s3_ntx, &gc.s3_nty, &gc.s3_zc);
        if (const char *e = std::getenv("AMRESSIF_GEN_S3ZC")) gc.s3_zc = std::max(1, std::min(n + 1, std::atoi(e)));
    }
    const size_t cellsz = (size_t)g.ncell;
#define GALLOC(p, cnt)                                                                     \
    do {                                                                                   \
        hipError_t e_ = alloc(c, p, cnt);                                                  \
        if (e_ != hipSuccess) return gfail(ctx, AMRESSIF_ERR_HIP, hipGetErrorString(e_)); \
    } while (0)
    for (int d = 0; d < dim; ++d) {
        GALLOC(&gc.U[d], g.nf[d]); GALLOC(&gc.Up[d], g.nf[d]); GALLOC(&gc.C[d], g.nf[d]);
        GALLOC(&gc.B[d], g.nf[d]); GALLOC(&gc.S[d], g.nf[d]);
    }
    GALLOC(&gc.X, (size_t)g.xs * dim);
    GALLOC(&gc.p, cellsz); GALLOC(&gc.phi, cellsz); GALLOC(&gc.phi2, cellsz); GALLOC(&gc.b, cellsz);
    for (int l = 0; l < gc.nlev; ++l) {
        if (l + 1 < gc.nlev) GALLOC(&gc.lev[l].e, (size_t)gc.lev[l].ncell);
        GALLOC(&gc.lev[l].r, (size_t)gc.lev[l].ncell);
        GALLOC(&gc.lev[l].out, (size_t)gc.lev[l].ncell);
    }
    gc.npartials = std::max<int64_t>(std::max<int64_t>(2 * ((g.ncell + G::kBlock - 1) / G::kBlock), 2 * G::outer_blocks(dim, n)),
                                     3 * (int64_t)(dim == 3 ? G::stage3_blocks(gc) : 2 * amr::iter_tile_blocks(n))) + 64;
    GALLOC(&gc.partials, (size_t)gc.npartials);
    {
        const std::vector<double> tab = exact_tables(g, gc.lev[gc.nlev - 1]);
        GALLOC(&gc.exact, tab.size());
        GCHK(hipMemcpy(gc.exact, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
    }
    GALLOC(&c.ctl, 1);
    {
        hipError_t e = hipHostMalloc((void **)&c.ctl_host, sizeof(amr::Ctl), hipHostMallocDefault);
        if (e != hipSuccess) return gfail(ctx, AMRESSIF_ERR_HIP, hipGetErrorString(e));
        std::memset(c.ctl_host, 0, sizeof(amr::Ctl));
        GCHK(hipMemcpy(c.ctl, c.ctl_host, sizeof(amr::Ctl), hipMemcpyHostToDevice));
    }
#undef GALLOC
    // a cavity at rest until a state is loaded
    for (int d = 0; d < dim; ++d) {
        GCHK(G::fill(c.stream, gc.U[d], g.nf[d], 0.0));
        GCHK(G::fill(c.stream, gc.Up[d], g.nf[d], 0.0));
    }
    GCHK(G::fill(c.stream, gc.p, g.ncell, 0.0));
    GCHK(G::fill(c.stream, gc.phi, g.ncell, 0.0));
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

// ================================================================== state
int amr_gen_load_state(amressif_ctx *ctx, const amr_array4 *vel, const amr_array4 *velPrev, const amr_array4 *userCtx)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    if (!vel || !velPrev) return gfail(ctx, AMRESSIF_ERR_ARG, "null argument");
    for (int d = 0; d < g.dim; ++d) {
        int ext[3], lo[3] = {0, 0, 0}, hi[3];
        face_ext(g, d, ext);
        for (int e = 0; e < 3; ++e) hi[e] = ext[e] - 1;
        if (int rc = check_view3(ctx, &vel[d], lo, hi, 1, "velCont")) return rc;
        if (int rc = check_view3(ctx, &velPrev[d], lo, hi, 1, "velContPrev")) return rc;
        GCHK(G::pack(c.stream, vel[d], 0, gc.U[d], ext[0], ext[1], ext[2]));
        GCHK(G::pack(c.stream, velPrev[d], 0, gc.Up[d], ext[0], ext[1], ext[2]));
    }
    if (userCtx) {
        const int lo[3] = {0, 0, 0}, hi[3] = {g.n - 1, g.n - 1, g.nk - 1};
        if (int rc = check_view3(ctx, userCtx, lo, hi, 2, "userCtx")) return rc;
        GCHK(G::pack(c.stream, *userCtx, 0, gc.p, g.n, g.n, g.nk));
        GCHK(G::pack(c.stream, *userCtx, 1, gc.phi, g.n, g.n, g.nk));
    } else {
        GCHK(G::fill(c.stream, gc.p, g.ncell, 0.0));
        GCHK(G::fill(c.stream, gc.phi, g.ncell, 0.0));
    }
    c.pred_valid = 0;
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

int amr_gen_store_state(amressif_ctx *ctx, amr_array4 *vel, amr_array4 *velPrev, amr_array4 *userCtx,
                        amr_array4 *velCart)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    for (int d = 0; d < g.dim; ++d) {
        int ext[3], lo[3] = {0, 0, 0}, hi[3];
        face_ext(g, d, ext);
        for (int e = 0; e < 3; ++e) hi[e] = ext[e] - 1;
        if (vel) {
            if (int rc = check_view3(ctx, &vel[d], lo, hi, 1, "velCont")) return rc;
            GCHK(G::unpack(c.stream, gc.U[d], vel[d], 0, ext[0], ext[1], ext[2]));
        }
        if (velPrev) {
            if (int rc = check_view3(ctx, &velPrev[d], lo, hi, 1, "velContPrev")) return rc;
            GCHK(G::unpack(c.stream, gc.Up[d], velPrev[d], 0, ext[0], ext[1], ext[2]));
        }
    }
    if (userCtx) {
        const int lo[3] = {0, 0, 0}, hi[3] = {g.n - 1, g.n - 1, g.nk - 1};
        if (int rc = check_view3(ctx, userCtx, lo, hi, 2, "userCtx")) return rc;
        for (int d = 0; d < 3; ++d)
            if ((d < g.dim && (userCtx->lo[d] < -1 || userCtx->hi[d] > g.n)) ||
                (d >= g.dim && (userCtx->lo[d] != 0 || userCtx->hi[d] != 0)))
                return gfail(ctx, AMRESSIF_ERR_ARG, "userCtx: at most one ghost layer");
        GCHK(G::phi_mean(gc, c.stream, c.ctl));
        GCHK(G::unpack_cells_ghosted(gc, c.stream, gc.p, *userCtx, 0, nullptr));
        GCHK(G::unpack_cells_ghosted(gc, c.stream, gc.phi, *userCtx, 1, &c.ctl->phi_mean));
    }
    if (velCart) {
        const int lo[3] = {0, 0, 0}, hi[3] = {g.n - 1, g.n - 1, g.nk - 1};
        if (int rc = check_view3(ctx, velCart, lo, hi, g.dim, "velCart")) return rc;
        for (int d = 0; d < 3; ++d)
            if ((d < g.dim && (velCart->lo[d] < -2 || velCart->hi[d] > g.n + 1)) ||
                (d >= g.dim && (velCart->lo[d] != 0 || velCart->hi[d] != 0)))
                return gfail(ctx, AMRESSIF_ERR_ARG, "velCart: at most two ghost layers");
        GCHK(G::cells(gc, c.stream, gc.U, gc.X));
        GCHK(G::unpack_velcart(gc, c.stream, gc.X, *velCart));
    }
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

// ---- MultiFabs of several boxes (amressif_load_state_mf / _store_state_mf)
namespace {

struct Box3 {
    int lo[3], hi[3];
};

// The valid boxes of a MultiFab (nodal: the face direction, or -1 for cells):
// inside the domain, pairwise disjoint and covering it; faces also returns
// the boxes' face windows (the cell box with hi + 1 along the nodal direction)
int check_mf3(amressif_ctx *ctx, const amr_multifab *mf, int nodal, int ncomp, int max_grow, const char *what,
              std::vector<Box3> &win)
{
    const G::Geom &g = ctx->c.gen->g;
    const std::string w(what);
    if (!mf || mf->nbox < 1 || !mf->fab) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": empty MultiFab");
    if (mf->ngrow < 0 || mf->ngrow > max_grow)
        return gfail(ctx, AMRESSIF_ERR_ARG, w + ": ngrow must be in [0, " + std::to_string(max_grow) + "]");
    const int ext[3] = {g.n, g.n, g.nk};
    std::vector<Box3> cells;
    win.clear();
    int64_t vol = 0;
    for (int b = 0; b < mf->nbox; ++b) {
        const amr_array4 &a = mf->fab[b];
        if (!a.ptr) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": null fab");
        if (a.dtype != 0) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": double views only");
        if (a.ncomp < ncomp) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": too few components");
        Box3 c{};
        for (int d = 0; d < 3; ++d) {
            const int gr = d < g.dim ? mf->ngrow : 0;
            c.lo[d] = a.lo[d] + gr;
            c.hi[d] = a.hi[d] - gr - (d == nodal ? 1 : 0);
            if (c.lo[d] < 0 || c.hi[d] >= ext[d] || c.hi[d] < c.lo[d])
                return gfail(ctx, AMRESSIF_ERR_ARG, w + ": a valid box lies outside the domain");
        }
        for (const Box3 &o : cells) {
            bool disjoint = false;
            for (int d = 0; d < 3; ++d) disjoint = disjoint || c.hi[d] < o.lo[d] || o.hi[d] < c.lo[d];
            if (!disjoint) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": valid boxes overlap");
        }
        vol += (int64_t)(c.hi[0] - c.lo[0] + 1) * (c.hi[1] - c.lo[1] + 1) * (c.hi[2] - c.lo[2] + 1);
        cells.push_back(c);
        Box3 f = c;
        if (nodal >= 0) f.hi[nodal] += 1;
        win.push_back(f);
    }
    if (vol != g.ncell) return gfail(ctx, AMRESSIF_ERR_ARG, w + ": valid boxes do not cover the domain");
    return 0;
}

}  // namespace

int amr_gen_load_state_mf(amressif_ctx *ctx, const amr_multifab *vel, const amr_multifab *velPrev,
                          const amr_multifab *userCtx)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    if (!vel || !velPrev) return gfail(ctx, AMRESSIF_ERR_ARG, "null argument");
    // validate everything before the first copy: a failed load leaves the state as it was
    std::vector<Box3> bx[7];
    for (int d = 0; d < g.dim; ++d) {
        if (int rc = check_mf3(ctx, &vel[d], d, 1, 0, "velCont", bx[2 * d])) return rc;
        if (int rc = check_mf3(ctx, &velPrev[d], d, 1, 0, "velContPrev", bx[2 * d + 1])) return rc;
    }
    if (userCtx)
        if (int rc = check_mf3(ctx, userCtx, -1, 2, 1 << 20, "userCtx", bx[6])) return rc;
    for (int d = 0; d < g.dim; ++d) {
        int ext[3];
        face_ext(g, d, ext);
        for (int k = 0; k < 2; ++k) {
            const amr_multifab &mf = k ? velPrev[d] : vel[d];
            double *dst = k ? gc.Up[d] : gc.U[d];
            for (int b = 0; b < mf.nbox; ++b) {
                const Box3 &q = bx[2 * d + k][b];
                GCHK(G::pack_window(c.stream, mf.fab[b], 0, dst, ext[0], ext[1], q.lo, q.hi, 0));
            }
        }
    }
    if (userCtx) {
        for (int b = 0; b < userCtx->nbox; ++b) {
            const Box3 &q = bx[6][b];
            GCHK(G::pack_window(c.stream, userCtx->fab[b], 0, gc.p, g.n, g.n, q.lo, q.hi, 0));
            GCHK(G::pack_window(c.stream, userCtx->fab[b], 1, gc.phi, g.n, g.n, q.lo, q.hi, 0));
        }
    } else {
        GCHK(G::fill(c.stream, gc.p, g.ncell, 0.0));
        GCHK(G::fill(c.stream, gc.phi, g.ncell, 0.0));
    }
    c.pred_valid = 0;
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

int amr_gen_store_state_mf(amressif_ctx *ctx, amr_multifab *vel, amr_multifab *velPrev, amr_multifab *userCtx,
                           amr_multifab *velCart)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    std::vector<Box3> bx[6], cb;
    for (int d = 0; d < g.dim; ++d) {
        if (vel)
            if (int rc = check_mf3(ctx, &vel[d], d, 1, 0, "velCont", bx[2 * d])) return rc;
        if (velPrev)
            if (int rc = check_mf3(ctx, &velPrev[d], d, 1, 0, "velContPrev", bx[2 * d + 1])) return rc;
    }
    if (userCtx)
        if (int rc = check_mf3(ctx, userCtx, -1, 2, 1, "userCtx", cb)) return rc;
    if (velCart)
        if (int rc = check_mf3(ctx, velCart, -1, g.dim, 2, "velCart", cb)) return rc;
    for (int d = 0; d < g.dim; ++d) {
        int ext[3];
        face_ext(g, d, ext);
        for (int k = 0; k < 2; ++k) {
            amr_multifab *mf = k ? velPrev : vel;
            if (!mf) continue;
            const double *src = k ? gc.Up[d] : gc.U[d];
            for (int b = 0; b < mf[d].nbox; ++b) {
                const Box3 &q = bx[2 * d + k][b];
                GCHK(G::pack_window(c.stream, mf[d].fab[b], 0, const_cast<double *>(src), ext[0], ext[1], q.lo, q.hi,
                                    1));
            }
        }
    }
    // cell views are written whole, ghosts by global index: the neighbouring
    // box's values inside the domain, the mirror or periodic image outside it
    if (userCtx) {
        GCHK(G::phi_mean(gc, c.stream, c.ctl));
        for (int b = 0; b < userCtx->nbox; ++b) {
            GCHK(G::unpack_cells_ghosted(gc, c.stream, gc.p, userCtx->fab[b], 0, nullptr));
            GCHK(G::unpack_cells_ghosted(gc, c.stream, gc.phi, userCtx->fab[b], 1, &c.ctl->phi_mean));
        }
    }
    if (velCart) {
        GCHK(G::cells(gc, c.stream, gc.U, gc.X));
        for (int b = 0; b < velCart->nbox; ++b) GCHK(G::unpack_velcart(gc, c.stream, gc.X, velCart->fab[b]));
    }
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

int amr_gen_init_state(amressif_ctx *ctx)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    for (int d = 0; d < g.dim; ++d) {
        GCHK(G::fill(c.stream, gc.U[d], g.nf[d], 0.0));
        GCHK(G::fill(c.stream, gc.Up[d], g.nf[d], 0.0));
    }
    GCHK(G::fill(c.stream, gc.p, g.ncell, 0.0));
    GCHK(G::fill(c.stream, gc.phi, g.ncell, 0.0));
    c.pred_valid = 0;
    GCHK(hipStreamSynchronize(c.stream));
    return AMRESSIF_OK;
}

// ================================================================== step
int amr_gen_advance(amressif_ctx *ctx, int nsteps, amressif_step_stats *stats)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    if (nsteps < 0) return gfail(ctx, AMRESSIF_ERR_ARG, "bad argument");
    if (nsteps == 0) return AMRESSIF_OK;
    if (c.log_cap < nsteps) {
        if (c.log) GCHK(hipFree(c.log));
        c.log = nullptr;
        GCHK(hipMalloc((void **)&c.log, sizeof(amressif_step_stats) * (size_t)nsteps));
        c.log_cap = nsteps;
    }
    GCHK(amr::launch_ctl_set(c, c.in.momentum_tolerance, c.in.poisson_tol_rel, c.in.poisson_tol_abs, c.in.IterNum,
                             c.in.mg_max_iter));
    int status = AMRESSIF_OK;
    const bool dim3 = g.dim == 3;
    for (int s = 0; s < nsteps; ++s) {
        GCHK(G::bdf2(gc, c.stream));
        GCHK(amr::launch_ctl_reset_step(c));
        // ---- momentum predictor: pseudo-iteration k writes the array (k odd: B, even: S)
        // that is the base of the next one.  u^{n-1}'s array is free once the constant
        // holds it: the scratch of the 3D stages 1 and 3
        double **scratch = gc.Up;
        auto iter_out = [&](int k) { return (k & 1) ? gc.B : gc.S; };
        int count = 1;
        if (!g.pseudo) {
            if (dim3) GCHK(G::stage3(gc, c.stream, gc.U, gc.U, iter_out(1), g.dt / 1.5, 1, c.ctl));
            else GCHK(G::iteration2(gc, c.stream, gc.U, iter_out(1), 0, false, c.ctl));
            GCHK(G::fin_pseudo(gc, c.stream, 0, c.ctl));
        } else {
            int done = 0, batch = std::max(1, gc.last_P), k = 0;
            while (!done) {
                for (int it = 0; it < batch; ++it) {
                    double **base = k == 0 ? gc.U : iter_out(k), **out = iter_out(k + 1);
                    if (dim3) {
                        GCHK(G::stage3(gc, c.stream, base, base, scratch, gc.rk[0], 0, c.ctl));
                        GCHK(G::stage3(gc, c.stream, scratch, base, out, gc.rk[1], 0, c.ctl));
                        GCHK(G::stage3(gc, c.stream, out, base, scratch, gc.rk[2], 0, c.ctl));
                        GCHK(G::stage3(gc, c.stream, scratch, base, out, gc.rk[3], 1, c.ctl));
                    } else {
                        // each launch takes the norm of the one before: the finalizer follows the batch
                        GCHK(G::iteration2(gc, c.stream, base, out, k, it > 0, c.ctl));
                    }
                    if (dim3 || it == batch - 1) GCHK(G::fin_pseudo(gc, c.stream, k, c.ctl));
                    ++k;
                }
                if (int rc = poll(ctx)) return rc;
                done = c.ctl_host->mom_done;
                batch = std::max(2, batch / 2);
            }
            count = std::max(1, c.ctl_host->mom_count);  // launches past it left every array as it was
            gc.last_P = count;
        }
        // u* is iter_out(count)'s; u^n becomes u^{n-1}, and the projection writes
        // u^{n+1} into the scratch
        for (int d = 0; d < g.dim; ++d) {
            if (count & 1) std::swap(gc.B[d], gc.S[d]);
            std::swap(gc.U[d], gc.Up[d]);
        }
        // ---- Poisson: b = (1.5/dt) D(u*), its mean removed in the residual
        int nb = 0;
        GCHK(G::divergence(gc, c.stream, gc.S, gc.b, &nb));
        GCHK(G::fin_div(gc, c.stream, nb, c.ctl, 0));
        GCHK(G::mg_start(gc, c.stream, c.ctl));
        {   // from phi0 = 0 (poisson.cpp:63); the iterate alternates between phi2 (even cycles) and phi
            int done = 0, batch = std::max(1, gc.last_V), k = 0;
            auto iter = [&](int q) { return (q & 1) ? gc.phi : gc.phi2; };
            GCHK(G::outer(gc, c.stream, nullptr, nullptr, iter(0), c.ctl));
            while (!done) {
                for (int it = 0; it < batch; ++it, ++k) {
                    GCHK(G::vcycle(gc, c.stream, c.ctl));
                    GCHK(G::outer(gc, c.stream, iter(k), gc.lev[0].out, iter(k + 1), c.ctl));
                }
                if (int rc = poll(ctx)) return rc;
                done = c.ctl_host->mg_done;
                batch = 2;
            }
            gc.last_V = std::max(1, c.ctl_host->mg_iters);
            if (c.ctl_host->mg_iters % 2 == 0) std::swap(gc.phi, gc.phi2);
        }
        // ---- projection, p += phi - mean, divergence of u^{n+1}
        GCHK(G::project(gc, c.stream, c.ctl));
        GCHK(G::divergence(gc, c.stream, gc.U, nullptr, &nb));
        GCHK(G::fin_div(gc, c.stream, nb, c.ctl, 1));
        GCHK(G::fin_step(gc, c.stream, c.ctl, c.log + s));
        if (c.ctl_host->flags & AMRESSIF_FLAG_NONFINITE) {
            status = gfail(ctx, AMRESSIF_ERR_NONFINITE, "non-finite pseudo-iteration norm at step " + std::to_string(s));
            nsteps = s + 1;
            break;
        }
        c.pred_valid = 1;
    }
    if (stats)
        GCHK(hipMemcpyAsync(stats, c.log, sizeof(amressif_step_stats) * (size_t)nsteps, hipMemcpyDeviceToHost,
                            c.stream));
    GCHK(hipStreamSynchronize(c.stream));
    return status;
}

// ================================================================== timing
// which: 0 cells; 1: 3D one stage, 2: with the norm partials; 2D 1 and 2: one pseudo-iteration
int amr_gen_time_kernel(amressif_ctx *ctx, int which, int reps, double *avg_ms, double *bytes_per_launch)
{
    Ctx &c = ctx->c;
    G::Ctx &gc = *c.gen;
    const G::Geom &g = gc.g;
    if (which < 0 || which > 2) return gfail(ctx, AMRESSIF_ERR_ARG, "unknown general-path kernel");
    hipEvent_t e0, e1;
    GCHK(hipEventCreate(&e0));
    GCHK(hipEventCreate(&e1));
    // a realistic state: the pseudo base another array than the stencil input
    for (int d = 0; d < g.dim; ++d)
        GCHK(hipMemcpyAsync(gc.B[d], gc.U[d], g.nf[d] * 8, hipMemcpyDeviceToDevice, c.stream));
    GCHK(G::bdf2(gc, c.stream));
    auto launch = [&]() -> hipError_t {
        if (which == 0) return G::cells(gc, c.stream, gc.U, gc.X);
        if (g.dim == 3) return G::stage3(gc, c.stream, gc.U, gc.B, gc.S, gc.rk[0], which == 2, nullptr);
        return G::iteration2(gc, c.stream, gc.B, gc.S, 0, false, nullptr);
    };
    GCHK(launch());
    GCHK(hipEventRecord(e0, c.stream));
    for (int r = 0; r < reps; ++r) GCHK(launch());
    GCHK(hipEventRecord(e1, c.stream));
    GCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    GCHK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *avg_ms = ms / reps;
    // algorithmic bytes (FP64), each array read or written once per launch:
    // cells: dim face arrays in, dim ghosted cell comps out; the 3D stage: u*,
    // u^k, C in, u* out; the 2D pseudo-iteration: u^k, C in, u^{k+1} out
    const double faces = (double)(g.nf[0] + g.nf[1] + (g.dim == 3 ? g.nf[2] : 0));
    const double bytes = which == 0 ? 8.0 * (faces + (double)g.xs * g.dim) : 8.0 * (g.dim == 3 ? 4.0 : 3.0) * faces;
    if (bytes_per_launch) *bytes_per_launch = bytes;
    c.pred_valid = 0;
    return AMRESSIF_OK;
}
