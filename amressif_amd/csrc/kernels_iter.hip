// One FP64 pseudo-iteration of a 2D step in one launch: the four RK4 dual-time
// stages (momentum.cpp:9-94 with the stage sequence of main.cpp:929-1017) on a
// tile kept in registers from the first load to the last store.
//
// A workgroup holds 64 columns x K W rows of both face arrays, K rows per thread
// of W waves; each stage uses up three rings of them (u* on a face reads faces
// three away), so 40 columns x (K W - 24) rows are written.  In a stage
//  * x neighbours come from adjacent lanes (DPP);
//  * y neighbours are the thread's own rows, and for its first and last rows the
//    neighbouring waves' through LDS: each wave publishes its outer faces, one
//    barrier per stage, double-buffered.  T_v of the row below a wave's first is
//    formed again from those instead of taking a second barrier;
//  * a face's QUICK flux is con s + cp D(-) + cm D(+): the sum s and the second
//    differences D of the two cells, scaled by the face velocity's factors, so the D
//    serve the fluxes on both sides of a cell and the Laplacian;
//  * cell velocities are kept doubled (the sum of a cell's two faces).
// Ghost cells: past a wall the rule of the mirror cell, which is a lane or a row of
// the same wave's window, set in every stage; periodic halos are loaded as images
// and evolve as such.  Halo columns and rows past a wall's ghosts hold values that
// nothing kept reads.
//
// Against two launches of two stages each (k_stage_pair) this moves half the bytes
// and, where the grid is too small to fill the chip with row marches, shortens the
// chain: a march's wave walks 24 rows (30 us a launch at any n up to 768), a tile's
// 4 K.  Bound by its dependent chains (3 us per stage at K = 4) with two waves per SIMD:
// where a workgroup runs the VALU is busy 28% of the time at 128^2 and 54% at 1024^2,
// where 2.56 times the faces written are computed and the last of three rounds of
// workgroups is two thirds full.
#include "device_common.hpp"
#include "iter_tile.hpp"

namespace amr {

namespace {

constexpr int kItH = 12;            // halo of four stages
constexpr int kItX = 64 - 2 * kItH;  // columns written per workgroup
constexpr int kItW = 8;             // waves

struct FaceVel2 {
    double con, cp, cm;
};
__device__ __forceinline__ FaceVel2 face_vel2(double vel, double kq)
{
    const double q = kq * vel;
    FaceVel2 f;
    f.con = -4.0 * q;
    f.cp = fmin(q, 0.0);
    f.cm = fmax(q, 0.0);
    return f;
}
__device__ __forceinline__ double face_flux2(const FaceVel2 &f, double xm, double xp, double dm, double dp)
{
    return f.con * (xm + xp) + (f.cp * dm + f.cm * dp);
}

template <int K>
__global__ __launch_bounds__(64 * kItW) void k_iter_tile(IterTile a)
{
    static_assert(K >= 3, "a wave's halo rows are those of the next wave alone");
    constexpr int W = kItW, ROWS = K * W, TY = ROWS - 2 * kItH;
    // the rows of a wave its neighbours read: the first two x-faces and three y-faces, the last three of both
    constexpr int NU = K < 5 ? K : 5, NV = K < 6 ? K : 6;
    __shared__ double shU[2][W][NU][64], shV[2][W][NV][64];
    __shared__ double shN[32];
    const int n = a.n, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int tx = blk % a.ntx, ty = blk / a.ntx;
    const int x0 = tx * kItX - kItH, i = x0 + lane, y = ty * TY - kItH + w * K;  // column, first row
    const bool px = a.per[0], py = a.per[1];
    auto wrap = [n](int q) {
        const int m = q % n;
        return m < 0 ? m + n : m;
    };
    auto cell = [&](int q, bool per) { return per ? wrap(q) : min(max(q, 0), n - 1); };
    auto face = [&](int q, bool per) { return q >= 0 && q <= n ? q : (per ? wrap(q) : min(max(q, 0), n)); };
    const int xf = face(i, px), xc = cell(i, px);
    const bool lanO = lane >= kItH && lane < kItH + kItX;
    const bool uo = lanO && i <= n, vo = lanO && i < n;
    auto row_out = [&](int k) { return w * K + k >= kItH && w * K + k < ROWS - kItH; };
    double u[K], v[K], ub[K], vb[K], cu[K], cv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const size_t ku = xf + (size_t)a.su * cell(y + k, py), kv = xc + (size_t)a.sv * face(y + k, py);
        u[k] = ub[k] = a.u[ku];
        v[k] = vb[k] = a.v[kv];
        cu[k] = a.cu[ku];
        cv[k] = a.cv[kv];
    }
    bool done = false;
    if (a.prev) {
        // the norm of the launch before and the loop control of main.cpp:898-1039, as
        // k_fin_pseudo: every workgroup reduces the records itself, in the same order,
        // and the first one writes the control block.  One thread reads mom_done for its
        // workgroup, since the first one may be writing it meanwhile (either value gives
        // the same decision).  -4 us per pseudo-iteration, the finalizer's launch:
        // 128^2 FP64 step 8.5 -> 8.0 ms.
        double r[2] = {0.0, 0.0};
        for (int q = threadIdx.x; q < (int)gridDim.x; q += 64 * W) {
            r[0] += a.prev[(size_t)a.rec * q];
            r[1] += a.prev[(size_t)a.rec * q + 1];
        }
        block_reduce_n<0u>(r, shN);
        if (threadIdx.x == 0) {
            bool end = __hip_atomic_load(&a.ctl->mom_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            if (!end) {
                const double npts = (double)n * (double)n;
                const double ex = sqrt(r[0]) / sqrt(npts), ey = sqrt(r[1]) / sqrt(npts);
                const double ne = (ex < ey) ? ey : ex;
                const bool cap = a.it > a.ctl->iter_num, div = ne > 1.e2;
                end = cap || div || !(ne > a.ctl->tol_mom);
                if (blockIdx.x == 0) {
                    a.ctl->norm_error = ne;
                    a.ctl->mom_count = a.it;
                    int f = 0;
                    if (!(ne == ne) || isinf(ne)) f |= AMRESSIF_FLAG_NONFINITE;
                    if (cap) f |= AMRESSIF_FLAG_CAP;
                    else if (div) f |= AMRESSIF_FLAG_DIVERGED;
                    if (f) a.ctl->flags |= f;
                    if (end) a.ctl->mom_done = 1;
                }
            }
            shN[0] = end ? 1.0 : 0.0;
        }
        __syncthreads();
        done = shN[0] != 0.0;
        __syncthreads();  // shN is used again
    } else {
        done = a.ctl && a.ctl->mom_done;  // no launch of this kernel without prev writes it
    }
    const int nst = done ? 0 : a.nst;
    const bool xedge = !px && (x0 < 0 || x0 + 63 >= n);
    const bool yedge = !py && (y - 3 < 0 || y + K + 1 >= n);
    const int ml = min(max(i < 0 ? lane - 2 * i - 1 : lane + 2 * (n - i) - 1, 0), 63);  // the mirror cell's lane
    // the north rule's constant of U: twice the lid's velocity (the cells are doubled)
    const double lidc = a.kind[3] == 3 ? 4.0 * ((a.lid && i >= 0 && i < n) ? a.lid[i] : a.inflow[0]) : a.ct[3][0];
    double sq[2] = {0.0, 0.0};
    for (int s = 0; s < nst; ++s) {
        const int bf = s & 1;
#pragma unroll
        for (int q = 0; q < NU; ++q) shU[bf][w][q][lane] = u[q < 2 ? q : K - NU + q];
#pragma unroll
        for (int q = 0; q < NV; ++q) shV[bf][w][q][lane] = v[q < 3 ? q : K - NV + q];
        __syncthreads();
        if (w * K + K - 1 < 3 * (s + 1) || w * K >= ROWS - 3 * (s + 1)) continue;  // no row of this wave counts any more
        const int wm = max(w - 1, 0), wp = min(w + 1, W - 1);
        // doubled cell velocities of rows -3 .. K + 1 (index r + 3)
        double X[K + 5][2], vm1;
        {
            double f[K + 6];
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] = shU[bf][wm][NU - 3 + q][lane];
#pragma unroll
            for (int k = 0; k < K; ++k) f[3 + k] = u[k];
            f[K + 3] = shU[bf][wp][0][lane];
            f[K + 4] = shU[bf][wp][1][lane];
#pragma unroll
            for (int r = 0; r < K + 5; ++r) X[r][0] = f[r] + lane_next(f[r]);
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] = shV[bf][wm][NV - 3 + q][lane];
            vm1 = f[2];
#pragma unroll
            for (int k = 0; k < K; ++k) f[3 + k] = v[k];
#pragma unroll
            for (int q = 0; q < 3; ++q) f[K + 3 + q] = shV[bf][wp][q][lane];
#pragma unroll
            for (int r = 0; r < K + 5; ++r) X[r][1] = f[r] + f[r + 1];
        }
        const double um1 = shU[bf][wm][NU - 1][lane];  // u of row -1
        const double vK = shV[bf][wp][0][lane];   // v of row K
        if (xedge) {
            const int side = i < 0 ? 0 : 1;
            const bool out = i < 0 || i >= n;
#pragma unroll
            for (int r = 0; r < K + 5; ++r)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const double m = __shfl(X[r][c], ml, 64);
                    const double gst = (side ? a.sg[1][c] : a.sg[0][c]) * m + (side ? a.ct[1][c] : a.ct[0][c]);
                    X[r][c] = out ? gst : X[r][c];
                }
        }
        if (yedge) {
#pragma unroll
            for (int r = 0; r < K + 5; ++r) {
                const int q = y + r - 3;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if (q == -1 && r + 1 < K + 5) X[r][c] = a.sg[2][c] * X[r + 1 < K + 5 ? r + 1 : r][c] + a.ct[2][c];
                    if (q == -2 && r + 3 < K + 5) X[r][c] = a.sg[2][c] * X[r + 3 < K + 5 ? r + 3 : r][c] + a.ct[2][c];
                    const double cn = c == 0 ? lidc : a.ct[3][1];
                    if (q == n && r >= 1) X[r][c] = a.sg[3][c] * X[r >= 1 ? r - 1 : r][c] + cn;
                    if (q == n + 1 && r >= 3) X[r][c] = a.sg[3][c] * X[r >= 3 ? r - 3 : r][c] + cn;
                }
            }
        }
        const double rk = a.rk[s], rkh = 0.5 * rk;
        const bool last = s == nst - 1;
        // march up the rows -1 .. K - 1: the lower face's flux and the second
        // differences along y carried, T_v of the row below
        double Dm[2], D0[2], Fs[2], tv = 0.0;
        {
            const FaceVel2 f = face_vel2(vm1, a.kq[1]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                Dm[c] = (X[0][c] - 2.0 * X[1][c]) + X[2][c];  // row -2
                D0[c] = (X[1][c] - 2.0 * X[2][c]) + X[3][c];  // row -1
                Fs[c] = face_flux2(f, X[1][c], X[2][c], Dm[c], D0[c]);
            }
        }
#pragma unroll
        for (int r = -1; r < K; ++r) {
            const double uf = r < 0 ? um1 : u[r < 0 ? 0 : r];
            const FaceVel2 fx = face_vel2(uf, a.kq[0]), fn = face_vel2(r + 1 < K ? v[r + 1 < K ? r + 1 : 0] : vK, a.kq[1]);
            double T[2] = {0.0, 0.0};
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const double C = X[r + 3][c], Xn = X[r + 4][c];
                const double Dn = -2.0 * Xn + (C + X[r + 5][c]);
                const double Fn = face_flux2(fn, C, Xn, D0[c], Dn);
                if (r >= 0 || c == 1) {
                    const double xm = lane_prev(C);
                    const double D = -2.0 * C + (xm + lane_next(C));
                    const double F = face_flux2(fx, xm, C, lane_prev(D), D);
                    T[c] = a.kv[1] * D0[c] + (a.kv[0] * D + (((Fs[c] - Fn) + F) - lane_next(F)));
                }
                Fs[c] = Fn;
                D0[c] = Dn;
            }
            if (r >= 0) {
                const int k = r, yk = y + r;
                // without R first: what a wall face keeps
                const double Tw = lane_prev(T[0]);
                const double uw = ub[k] + rk * (cu[k] - a.c15 * u[k]), vw = vb[k] + rk * (cv[k] - a.c15 * v[k]);
                u[k] = uw + rkh * (Tw + T[0]);
                v[k] = vw + rkh * (tv + T[1]);
                // wall faces: R = 0; in the explicit form half of the inner T (fluxTotal's wall ghosts keep 0)
                // (the empty asm keeps these few waves' selects out of the others' rows)
                if (xedge) {
                    asm volatile("");
                    if (i == 0 || i == n) u[k] = a.expl ? uw + rkh * (i == 0 ? T[0] : Tw) : uw;
                }
                if (yedge && (yk == 0 || yk == n)) {
                    asm volatile("");
                    v[k] = a.expl ? vw + rkh * (yk == 0 ? T[1] : tv) : vw;
                }
                if (last && row_out(k)) {
                    const double du = ub[k] - u[k], dv = vb[k] - v[k];
                    if (uo && yk < n) sq[0] += ((i == 0 || i == n) ? 0.5 : 1.0) * du * du;
                    if (vo && yk <= n) sq[1] += ((yk == 0 || yk == n) ? 0.5 : 1.0) * dv * dv;
                }
            }
            tv = T[1];
        }
    }
    if (done && !a.copy_done) return;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!row_out(k)) continue;
        if (uo && y + k < n) a.uo[i + (size_t)a.su * (y + k)] = u[k];
        if (vo && y + k <= n) a.vo[i + (size_t)a.sv * (y + k)] = v[k];
    }
    if (done) return;
    block_reduce_n<0u>(sq, shN);
    if (threadIdx.x == 0) {
        double *p = a.partials + (size_t)a.rec * blk;
        p[0] = sq[0];
        p[1] = sq[1];
        if (a.rec > 2) p[2] = 0.0;
    }
}

// Rows per thread.  A round of 256 workgroups takes about 1.5 us per row held plus 5,
// over a launch's 6 us (128^2: 17.6, 24.0 and 29.8 us with 4, 6 and 8 rows), and a
// tile writes 8, 24 and 40 rows of its 32, 48 and 64: the height whose rounds are
// shortest, 4 up to n = 279, 6 to 479 and from 640 to 679, 8 elsewhere.  (Sixteen waves of half the
// rows each are no faster: 24.2 us for 48 rows, 33.6 for 64.)
int rows_per_thread(int n)
{
    const int ntx = (n + 1 + kItX - 1) / kItX;
    int best = 0, cost = 0;
    for (int k = 4; k <= 8; k += 2) {
        const int ty = k * kItW - 2 * kItH, rounds = (ntx * ((n + 1 + ty - 1) / ty) + 255) / 256;
        if (!best || rounds * (3 * k + 10) < cost) { best = k; cost = rounds * (3 * k + 10); }
    }
    return best;
}

}  // namespace

int iter_tile_blocks(int n)
{
    const int ntx = (n + 1 + kItX - 1) / kItX, ty = rows_per_thread(n) * kItW - 2 * kItH;
    return ntx * ((n + 1 + ty - 1) / ty);
}

hipError_t launch_iter_tile(IterTile a, hipStream_t s)
{
    if (a.n < 4 || a.nst < 1 || a.nst > 4 || a.uo == a.u || a.vo == a.v) return hipErrorInvalidValue;
    a.ntx = (a.n + 1 + kItX - 1) / kItX;
    for (int d = 0; d < 2; ++d) {
        a.kq[d] = -0.0625 * a.idx[d];  // of doubled cells: half of -1/(8 dx)
        a.kv[d] = 0.5 * a.idx2[d] * a.iren;
        for (int hi = 0; hi < 2; ++hi) {
            const int side = 2 * d + hi, kind = a.kind[side];
            for (int c = 0; c < 2; ++c) {
                a.sg[side][c] = kind == 1 && c != d ? 1.0 : -1.0;
                a.ct[side][c] = kind == 2 ? 4.0 : (kind == 3 ? 4.0 * a.inflow[c] : 0.0);
            }
        }
    }
    const dim3 grid(iter_tile_blocks(a.n));
    const int k = rows_per_thread(a.n);
    const dim3 block(64 * kItW);
    if (k == 4) hipLaunchKernelGGL(k_iter_tile<4>, grid, block, 0, s, a);
    else if (k == 6) hipLaunchKernelGGL(k_iter_tile<6>, grid, block, 0, s, a);
    else hipLaunchKernelGGL(k_iter_tile<8>, grid, block, 0, s, a);
    return hipGetLastError();
}

// a record of two doubles per workgroup, two sets of them in c.partials (n <= 10239)
bool iteration_fits(const Ctx &c) { return c.g.n >= 4 && iter_tile_blocks(c.g.n) <= kMaxPartials; }

// The sizes at which a pseudo-iteration runs as one k_iter_tile launch: measured
// against the two k_stage_pair launches, 18 against 59 us up to 256^2, 30 against 60
// at 512^2, 48 against 65 at 768^2, 66 against 69 at 1024^2; above, the halo's
// recomputation costs more than the march (103 against 73 us at 1280^2).
bool iter_tile_wanted(const Ctx &c)
{
    return c.iter_tile && iteration_fits(c) && (c.g.n <= 1024 || c.iter_tile == 2);
}

constexpr int kHalf = 2 * kMaxPartials;  // doubles; c.partials holds twice as many
const double *iteration_partials(const Ctx &c, int it) { return c.partials + (it & 1) * kHalf; }

hipError_t launch_iteration(const Ctx &c, const StageLaunch &s, int *nblocks)
{
    const Geometry &g = c.g;
    if (!iteration_fits(c)) return hipErrorInvalidValue;
    IterTile a{};
    a.u = s.ub; a.v = s.vb;
    a.cu = s.cu; a.cv = s.cv;
    a.uo = s.uo; a.vo = s.vo;
    a.lid = c.lid;
    // two sets of records in turn: a launch reads the one before's while it writes its own
    a.partials = c.partials + (s.it & 1) * kHalf;
    a.prev = s.chained ? c.partials + (1 - (s.it & 1)) * kHalf : nullptr;
    a.it = s.it;
    a.ctl = s.unguarded ? nullptr : c.ctl;
    a.n = g.n;
    a.su = a.sv = g.P;
    a.rec = 2;
    a.copy_done = 1;
    a.nst = 4;
    // ghost_rule's codes as kinds: 135 -mirror; -135 (east: 1) slip; else the inflow of 165
    a.kind[0] = g.bc_lo0 == 135 ? 0 : (g.bc_lo0 == -135 ? 1 : 2);
    a.kind[1] = g.bc_hi0 == 135 ? 0 : (g.bc_hi0 == 1 ? 1 : 2);
    a.kind[2] = g.bc_lo1 == 135 ? 0 : (g.bc_lo1 == -135 ? 1 : 2);
    a.kind[3] = g.bc_hi1 == 135 ? 0 : (g.bc_hi1 == -135 ? 1 : 3);
    a.inflow[0] = g.inflow0;
    a.inflow[1] = g.inflow1;
    for (int k = 0; k < 4; ++k) a.rk[k] = c.rk[k];
    a.c15 = 1.5 / g.dt;
    a.iren = 1.0 / g.ren;
    a.idx[0] = 1.0 / g.dx;
    a.idx[1] = 1.0 / g.dy;
    a.idx2[0] = 1.0 / (g.dx * g.dx);
    a.idx2[1] = 1.0 / (g.dy * g.dy);
    if (nblocks) *nblocks = iter_tile_blocks(g.n);
    return launch_iter_tile(a, c.stream);
}

}  // namespace amr
