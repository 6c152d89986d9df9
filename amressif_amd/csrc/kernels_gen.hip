// Kernels of the general path (gen.hpp): the fractional step on n^dim cells,
// dim 2 or 3, with periodic directions beside the wall codes, FP64.
//
// The RK4 dual-time loop (momentum.cpp:9-94): in 3D one launch per stage
// (k_gen_stage3), in 2D one per pseudo-iteration of four stages (k_iter_tile,
// kernels_iter.hip).  A stage forms cell velocities with the wall rules or
// periodic images (cont2cart, utilities.cpp:16-350), fluxTotal T = -C + V per
// cell (QUICK, fn_flux_calc.cpp:11-202, and the viscous Laplacian :695-766), and
// on every face R = (T(left) + T(right))/2 with the flux ghosts of
// main.cpp:939-1014 (wall faces R = 0, periodic images), u* <- u^k + rk (R -
// (1.5/dt) u* + C), the BDF2 constant C holding -G p (momentum.cpp:68-87,
// fn_rhs.cpp:8-68); on the last stage the Error_Computation partials
// (utilities.cpp:421-493).  k_gen_cells writes the cell velocities for output.
// Then the Poisson RHS (fn_rhs.cpp:71-125), the multigrid solve
// (kernels_gen_mg.hip), and the projection (poisson.cpp:192-392).  Blocks are handed to the XCDs in contiguous ranges
// (xcd_block), so the rows and planes a stencil shares sit in one L2.
#include "device_common.hpp"
#include "gen.hpp"
#include "iter_tile.hpp"

namespace amr {
namespace gen {

namespace {

constexpr int B = kBlock;

__device__ __forceinline__ int64_t gid() { return (int64_t)xcd_block(blockIdx.x, gridDim.x) * B + threadIdx.x; }

// (i, j, k) of the linear index q over an nx x ny x .. box (x fastest) in
// 32-bit unsigned arithmetic: every box here has fewer than 2^31 points
// (n <= 1024 in 3D, n <= 16384 in 2D), and two 32-bit divisions cost a
// fraction of the 64-bit div/mod sequence.
__device__ __forceinline__ void split3(int64_t q, int nx, int ny, int *x)
{
    const unsigned u = (unsigned)q, a = u / (unsigned)nx, b = a / (unsigned)ny;
    x[0] = (int)(u - a * (unsigned)nx);
    x[1] = (int)(a - b * (unsigned)ny);
    x[2] = (int)b;
}

__device__ __forceinline__ int64_t fidx(const Geom &g, int d, int i, int j, int k)
{
    const int64_t nx = g.n + (d == 0), ny = g.n + (d == 1);
    return i + nx * (j + ny * (int64_t)k);
}
__device__ __forceinline__ int64_t cidx(const Geom &g, int i, int j, int k)
{
    return i + (int64_t)g.n * (j + (int64_t)g.n * k);
}
__device__ __forceinline__ int64_t cidx(const Geom &g, const int *x) { return cidx(g, x[0], x[1], x[2]); }
__device__ __forceinline__ int64_t xidx(const Geom &g, int i, int j, int k)
{
    const int64_t s = g.n + 4;
    const int gk = g.dim == 3 ? 2 : 0;
    return (i + 2) + s * ((j + 2) + s * (int64_t)(k + gk));
}

// apply a wall rule to the mirror values v (one ghost layer crossing of dim d)
__device__ __forceinline__ void wall_rule(const Geom &g, int kind, int d, double *v)
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (c >= g.dim) break;
        if (kind == 0) v[c] = -v[c];
        else if (kind == 1) v[c] = c == d ? -v[c] : v[c];
        else if (kind == 2) v[c] = 2.0 - v[c];
        else v[c] = 2.0 * g.inflow[c] - v[c];
    }
}

// ------------------------------------------------------------ cell velocities
__global__ __launch_bounds__(B) void k_gen_cells(Geom g, const double *f0, const double *f1, const double *f2,
                                                 double *X)
{
    const int64_t s = g.n + 4, sk = g.dim == 3 ? s : 1;
    const int64_t q = gid();
    if (q >= s * s * sk) return;
    const int n = g.n;
    int x[3];
    split3(q, (int)s, (int)s, x);
    x[0] -= 2;
    x[1] -= 2;
    x[2] = g.dim == 3 ? x[2] - 2 : 0;
    int b[3] = {x[0], x[1], x[2]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= g.dim) break;
        if (x[d] < 0 || x[d] >= n) b[d] = g.per[d] ? (x[d] + n) % n : (x[d] < 0 ? -x[d] - 1 : 2 * n - 1 - x[d]);
    }
    const double *f[3] = {f0, f1, f2};
    double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (c >= g.dim) break;
        int e[3] = {b[0], b[1], b[2]};
        e[c] += 1;
        v[c] = 0.5 * (f[c][fidx(g, c, b[0], b[1], b[2])] + f[c][fidx(g, c, e[0], e[1], e[2])]);
    }
    // the wall passes in the reference's order W, E, S, N, B, F: the rule of
    // the lowest direction applies first (corners are the later passes'
    // rules of the earlier passes' ghosts)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= g.dim) break;
        if ((x[d] < 0 || x[d] >= n) && !g.per[d]) wall_rule(g, x[d] < 0 ? g.kind_lo[d] : g.kind_hi[d], d, v);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
        if (c < g.dim) X[q + (int64_t)c * g.xs] = v[c];
}

// A face's velocity as the three factors its QUICK fluxes share: with X(-), X(+) the
// cells at the face and D their second differences, QUICK's flux
// vel ((X(-) + X(+))/2 - D(upwind)/8) is con (X(-) + X(+)) + cp D(-) + cm D(+).
// kq = -1/(8 dx), so that a cell's divergence is a plain difference of fluxes.
struct FaceVel {
    double con, cp, cm;
};
__device__ __forceinline__ FaceVel face_vel(double vel, double kq)
{
    const double q = kq * vel;
    FaceVel f;
    f.con = -4.0 * q;
    f.cp = fmin(q, 0.0);
    f.cm = fmax(q, 0.0);
    return f;
}
__device__ __forceinline__ double face_flux(const FaceVel &f, double xm, double xp, double dm, double dp)
{
    return f.con * (xm + xp) + (f.cp * dm + f.cm * dp);
}

// ------------------------------------------------ one RK4 stage in one pass (3D)
// u* <- u^k + rk (R(u*) - (1.5/dt) u* + C) on every face, from the faces
// alone: 96 B per cell (u*, u^k and C in, the new u* out; 72 B where u* is
// u^k), where the three passes it replaces (cell velocities, fluxTotal, update)
// moved 2.4 times that.  At 256^3 a launch takes 426 us (with the norm partials 445)
// against 162 + 390 + 374 us of the three passes, at 144^3 77 us against 34 + 69 +
// 60, at 64^3 22 against 5.5 + 22 + 7.  Bound by memory at 256^3: the counters give
// 1.36 GB read and 0.43 written (1.62 GB without the halo), 4.2 TB/s where a large
// copy reaches 4.9, with the VALU busy 38% of the time (FP64 instructions 20%); on
// small grids by a plane's chain and the planes of prologue.
//
// A workgroup owns 58 columns x kS3Y rows and marches up a chunk of planes.  Wave r
// works on rows y0 - 3 + 2 r and the next, lane l on column x0 - 3 + l, so the
// stencil's three faces on either side are waves and lanes of the same workgroup:
//  * x neighbours come from adjacent lanes (DPP);
//  * y neighbours are the thread's other row or come through LDS: a plane's cell
//    velocities, double-buffered, one barrier per plane.  The y-flux total T_v of
//    the wave below takes the same barrier one plane later, so the lower row's
//    v-faces of plane z are written at plane z + 1;
//  * z neighbours stay in registers: cell velocities of planes z .. z + 2, the
//    second difference and the flux at the plane's lower face.  The planes' x- and
//    y-faces wait in an LDS ring until their plane is the march's.
// One wait for memory per plane, at its top: for the faces of plane z + 2 and the
// base and constant of plane z, loaded a plane ago; then the next plane's loads
// and the last plane's results go out.  Waves with one row each (16 of them, up to
// 128 VGPRs) had to load the base and constant in the plane that uses them: 620 us
// at 256^3.  Planes are addressed as buffers (scalar base, 32-bit offsets): with
// 64-bit addresses the compiler kept one per array and row in registers and
// spilled them, and each reload waited for every load in flight (934 us).
// A face's flux is con s + cp D(-) + cm D(+) (FaceVel): the second differences serve
// QUICK on both sides of a cell and the Laplacian.
// Ghosts: periodic directions wrap a load's index; past a wall it is mirrored
// (face -q for q < 0, 2n - q for q > n: the average of a ghost cell's two faces is
// then its mirror cell's) and the cell takes the wall's rule, affine in the mirror
// cell: sg X + ct.  The output must not alias the stencil input.
// One workgroup per CU; the chunk of planes is chosen on the host so that the grid
// fills the CUs in whole rounds (stage3_shape).
typedef unsigned Dwords2 __attribute__((ext_vector_type(2)));
constexpr int kS3X = 58, kS3W = 8, kS3Y = 2 * kS3W - 5;
struct Stage3 {
    const double *s[3], *b[3], *c[3];
    double *o[3];
    double *partials;
    double rk;
    double kq[3], kv[3];        // -1/(8 dx), 1/(dx^2 Re)
    double sg[6][3], ct[6][3];  // wall rules: sides W, E, S, N, B, F
    int ntx, nty, zc;
};

template <bool LAST>
__global__ __launch_bounds__(64 * kS3W) void k_gen_stage3(Geom g, Stage3 a, const Ctl *guard)
{
    __shared__ double shX[2][3][2 * kS3W][64];
    __shared__ double shT[2][kS3W][64];
    __shared__ double shF[4][2][2 * kS3W][64];  // x- and y-faces of planes z .. z + 2 (slot: plane mod 4)
    // the rules in LDS: only edge waves and planes use them, and as kernel arguments
    // they would hold 72 scalar registers through the march
    __shared__ double shR[6][3][2];
    if (guard && guard->mom_done) return;  // the same for every thread of the launch
    const int n = g.n, lane = threadIdx.x & 63;
    const int r = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int tx = blk % a.ntx, ty = (blk / a.ntx) % a.nty, tz = blk / (a.ntx * a.nty);
    const int x0 = tx * kS3X - 3, i = x0 + lane, y = ty * kS3Y + 2 * r - 3;  // column, lower row
    const int z0 = tz * a.zc, z1 = min(z0 + a.zc, n + 1);  // face planes z0 .. z1 - 1 (plane n: z-faces only)
    const bool px = g.per[0], py = g.per[1], pz = g.per[2];
    if (threadIdx.x < 18) {
        shR[threadIdx.x / 3][threadIdx.x % 3][0] = a.sg[threadIdx.x / 3][threadIdx.x % 3];
        shR[threadIdx.x / 3][threadIdx.x % 3][1] = a.ct[threadIdx.x / 3][threadIdx.x % 3];
    }
    __syncthreads();
    auto cell_of = [n](int q, bool per) {  // -3 <= q; past n + 2: any cell (nothing that is kept reads it)
        q = min(q, n + 2);
        if (per) return q < 0 ? q + n : (q >= n ? q - n : q);
        return q < 0 ? -1 - q : (q >= n ? 2 * n - 1 - q : q);
    };
    auto face_of = [n](int q, bool per) {  // periodic: face n keeps its own copy of face 0
        q = min(q, n + 3);
        if (per) return q < 0 ? q + n : (q > n ? q - n : q);
        return q < 0 ? -q : (q > n ? 2 * n - q : q);
    };
    const unsigned su = (unsigned)(n + 1) * n, sw = (unsigned)n * n;  // plane strides (x- and y-faces alike; z-faces)
    // byte offsets in a plane: x- and z-faces of the two rows, y-faces of the three; on
    // output rows and lanes they are the thread's own faces
    unsigned ou[2], oc[2], ov[3];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        ou[q] = 8u * (unsigned)(face_of(i, px) + (n + 1) * cell_of(y + q, py));
        oc[q] = 8u * (unsigned)(cell_of(i, px) + n * cell_of(y + q, py));
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) ov[q] = 8u * (unsigned)(cell_of(i, px) + n * face_of(y + q, py));
    // a plane of `count` doubles as a buffer resource: a scalar base and 32-bit byte
    // offsets (64-bit addresses would be kept in registers per array), and an access
    // past it reads 0 or writes nothing, so that masks are offsets
    auto plane = [](const double *base, unsigned first, unsigned count) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(base + first), 0, 8 * count, 0x00020000);
    };
    auto ld = [](__amdgpu_buffer_rsrc_t p, unsigned off) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(p, off, 0, 0));
    };
    auto st = [](__amdgpu_buffer_rsrc_t p, unsigned off, double v) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Dwords2, v), p, off, 0, 0);
    };
    auto rule = [&](int side, double *X) {
#pragma unroll
        for (int c = 0; c < 3; ++c) X[c] = shR[side][c][0] * X[c] + shR[side][c][1];
    };
    const bool xedge = !px && (x0 < 0 || x0 + 63 >= n), yedge = !py && (y < 0 || y + 1 >= n);
    struct Plane {  // x-faces and y-faces of one plane, z-faces above it
        double u[2], v[3], w[2];
    };
    auto load = [&](int z, Plane &P) {
        const auto u = plane(a.s[0], cell_of(z, pz) * su, su), v = plane(a.s[1], cell_of(z, pz) * su, su),
                   w = plane(a.s[2], face_of(z + 1, pz) * sw, sw);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            P.u[q] = ld(u, ou[q]);
            P.w[q] = ld(w, oc[q]);
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) P.v[q] = ld(v, ov[q]);
    };
    // cell velocities of plane z from its faces and the z-faces below it
    auto cells = [&](int z, const Plane &P, const double *wl, double (*X)[3]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            X[q][0] = 0.5 * (P.u[q] + lane_next(P.u[q]));
            X[q][1] = 0.5 * (P.v[q] + P.v[q + 1]);
            X[q][2] = 0.5 * (wl[q] + P.w[q]);
        }
        if (xedge) {
            if (i < 0) {
                rule(0, X[0]);
                rule(0, X[1]);
            } else if (i >= n) {
                rule(1, X[0]);
                rule(1, X[1]);
            }
        }
        if (yedge) {
            if (y < 0) rule(2, X[0]);
            if (y >= n) rule(3, X[0]);
            if (y + 1 < 0) rule(2, X[1]);
            if (y + 1 >= n) rule(3, X[1]);
        }
        if (!pz && (z < 0 || z >= n)) {
            rule(z < 0 ? 4 : 5, X[0]);
            rule(z < 0 ? 4 : 5, X[1]);
        }
    };
    auto keep = [&](int z, const Plane &P) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            shF[z & 3][0][2 * r + q][lane] = P.u[q];
            shF[z & 3][1][2 * r + q][lane] = P.v[q];
        }
    };
    // output rows 3 .. 2 kS3W - 3 of the workgroup's: both rows of waves 2 .. kS3W - 2, wave 1's upper one
    const bool rowT = r >= 1 && r <= kS3W - 2;
    const bool lanO = rowT && lane >= 3 && lane <= 60;
    unsigned fu[2], fv[2], fw[2];  // the faces this thread updates: their offsets, or past the plane
    constexpr unsigned kNone = 0x80000000u;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const bool o = lanO && (q == 1 || r >= 2);
        fu[q] = o && y + q < n && i <= n ? ou[q] : kNone;
        fv[q] = o && y + q <= n && i < n ? ov[q] : kNone;
        fw[q] = o && y + q < n && i < n ? oc[q] : kNone;
    }
    struct Upd {  // base and constant of the three faces of both rows
        double ub[2], uc[2], vb[2], vc[2], wb[2], wc[2];
    };
    auto load_upd = [&](int z, Upd &U) {  // z >= 0; plane n has z-faces only
        const unsigned o = z * su, m = z < n ? su : 0, p = z * sw, k = z <= n ? sw : 0;
        const auto ub = plane(a.b[0], o, m), uc = plane(a.c[0], o, m), vb = plane(a.b[1], o, m),
                   vc = plane(a.c[1], o, m), wb = plane(a.b[2], p, k), wc = plane(a.c[2], p, k);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            U.ub[q] = ld(ub, fu[q]);
            U.uc[q] = ld(uc, fu[q]);
            U.vb[q] = ld(vb, fv[q]);
            U.vc[q] = ld(vc, fv[q]);
            U.wb[q] = ld(wb, fw[q]);
            U.wc[q] = ld(wc, fw[q]);
        }
    };
    // the norm's sums, per thread in LDS: in registers they would spill inside the march, where
    // a reload waits for every load in flight
    __shared__ double shS[3][64 * kS3W];
    if (LAST)
#pragma unroll
        for (int d = 0; d < 3; ++d) shS[d][threadIdx.x] = 0.0;
    // one face at position q along d from T on its two sides: u^k + rk (R + e), e = C - (1.5/dt) u*, R = (tl + tr)/2;
    // at wall faces R = 0, in the explicit form half of the inner T (ends: whether this wave, row or plane
    // can hold one; the empty asm keeps their selects out of the others' path)
    const double rkh = 0.5 * a.rk;
    auto face = [&](int d, bool ends, int q, double tl, double tr, double base, double e) {
        const double uw = base + a.rk * e;
        double unew = uw + rkh * (tl + tr);
        if (ends && !g.per[d]) {
            if (!LAST) asm volatile("");  // (with the norm it would spill)
            if (q == 0 || q == n) unew = g.pseudo ? uw : uw + rkh * (q == 0 ? tr : tl);
        }
        return unew;
    };
    auto norm = [&](int q, bool on, double base, double unew) {
        const double df = on ? base - unew : 0.0;
        return ((q == 0 || q == n) ? 0.5 : 1.0) * df * df;
    };
    // cell velocities of planes z .. z + 2, and of plane z its second difference and lower flux along z;
    // z-faces z .. z + 2; the march starts at T of plane z0 - 1
    double X0[2][3], X1[2][3], X2[2][3], dz[2][3], fz[2][3], w0[2], w1[2], w2[2];
    Plane pn;  // plane z + 2 (z-faces z + 3), loaded at plane z - 1
    {
        Plane pa, pb, p0, p1;
        double wa[2], xa[2][3], xb[2][3];
#pragma unroll
        for (int q = 0; q < 2; ++q) wa[q] = ld(plane(a.s[2], face_of(z0 - 3, pz) * sw, sw), oc[q]);
        load(z0 - 3, pa);
        load(z0 - 2, pb);
        load(z0 - 1, p0);
        load(z0, p1);
        load(z0 + 1, pn);
        cells(z0 - 3, pa, wa, xa);
        cells(z0 - 2, pb, pa.w, xb);
        cells(z0 - 1, p0, pb.w, X0);
        cells(z0, p1, p0.w, X1);
        keep(z0 - 1, p0);
        keep(z0, p1);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            w0[q] = pb.w[q];
            w1[q] = p0.w[q];
            w2[q] = p1.w[q];
            const FaceVel f = face_vel(w0[q], a.kq[2]);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                dz[q][c] = (xb[q][c] - 2.0 * X0[q][c]) + X1[q][c];
                fz[q][c] = face_flux(f, xb[q][c], X0[q][c], (xa[q][c] - 2.0 * xb[q][c]) + X0[q][c], dz[q][c]);
            }
        }
    }
    Upd nxt{};                                      // of plane z at its top
    double tv[2] = {0.0, 0.0}, tw[2] = {0.0, 0.0};  // plane z - 1: T_v, T_w
    double vbl = 0.0, vel = 0.0;                    // and its lower row's v-face: base and e
    double ru[2], rv[2], rw[2];                     // results to store
    // the results formed at plane z (the lower row's v-faces are plane z - 1's)
    auto flush = [&](int z) {
        const unsigned o = z * su, m = z < n ? su : 0;
        const auto u = plane(a.o[0], o, m), v = plane(a.o[1], o, m), vl = plane(a.o[1], o - su, z > z0 ? su : 0),
                   w = plane(a.o[2], z * sw, sw);
        st(vl, fv[0], rv[0]);
        st(v, fv[1], rv[1]);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            st(u, fu[q], ru[q]);
            st(w, fw[q], rw[q]);
        }
    };
    for (int z = z0 - 1; z < z1; ++z) {
        const int bf = z & 1;
        cells(z + 2, pn, w2, X2);
        keep(z + 2, pn);
        const double w3[2] = {pn.w[0], pn.w[1]};
        const Upd cur = nxt;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) shX[bf][c][2 * r + q][lane] = X0[q][c];
        shT[bf][r][lane] = tv[1];
        load(z + 3, pn);
        load_upd(z + 1, nxt);
        if (z > z0) flush(z - 1);
        __syncthreads();
        if (rowT) {
            const double pu[2] = {shF[z & 3][0][2 * r][lane], shF[z & 3][0][2 * r + 1][lane]};
            const double pv[3] = {shF[z & 3][1][2 * r][lane], shF[z & 3][1][2 * r + 1][lane], shF[z & 3][1][2 * r + 2][lane]};
            double T[2][3];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                {   // z: the flux of the upper face
                    const FaceVel f = face_vel(w1[q], a.kq[2]);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const double D = (X0[q][c] - 2.0 * X1[q][c]) + X2[q][c];
                        const double F = face_flux(f, X0[q][c], X1[q][c], dz[q][c], D);
                        T[q][c] = a.kv[2] * dz[q][c] + (fz[q][c] - F);
                        fz[q][c] = F;
                        dz[q][c] = D;
                    }
                }
                {   // x: the east face's flux is the next lane's
                    const FaceVel f = face_vel(pu[q], a.kq[0]);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const double X = X0[q][c], xm = lane_prev(X);
                        const double D = -2.0 * X + (xm + lane_next(X));
                        const double F = face_flux(f, xm, X, lane_prev(D), D);
                        T[q][c] = a.kv[0] * D + ((T[q][c] + F) - lane_next(F));
                    }
                }
            }
            {   // y: the faces below, between and above the two rows
                const FaceVel fs = face_vel(pv[0], a.kq[1]), fm = face_vel(pv[1], a.kq[1]), fn = face_vel(pv[2], a.kq[1]);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double XA = X0[0][c], XB = X0[1][c];
                    const double s1 = shX[bf][c][2 * r - 1][lane], s2 = shX[bf][c][2 * r - 2][lane];
                    const double n1 = shX[bf][c][2 * r + 2][lane], n2 = shX[bf][c][2 * r + 3][lane];
                    const double DA = (s1 - 2.0 * XA) + XB, DB = (XA - 2.0 * XB) + n1;
                    const double Fs = face_flux(fs, s1, XA, (s2 - 2.0 * s1) + XA, DA);
                    const double Fm = face_flux(fm, XA, XB, DA, DB);
                    const double Fn = face_flux(fn, XB, n1, DB, (XB - 2.0 * n1) + n2);
                    T[0][c] = a.kv[1] * DA + ((T[0][c] + Fs) - Fm);
                    T[1][c] = a.kv[1] * DB + ((T[1][c] + Fm) - Fn);
                }
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                ru[q] = face(0, xedge, i, lane_prev(T[q][0]), T[q][0], cur.ub[q], cur.uc[q] - g.c15 * pu[q]);
                rw[q] = face(2, z == 0 || z == n, z, tw[q], T[q][2], cur.wb[q], cur.wc[q] - g.c15 * w0[q]);
            }
            rv[0] = face(1, y == 0 || y == n, y, shT[bf][r - 1][lane], tv[0], vbl, vel);
            rv[1] = face(1, y + 1 == 0 || y + 1 == n, y + 1, T[0][1], T[1][1], cur.vb[1], cur.vc[1] - g.c15 * pv[1]);
            if (LAST && z >= z0) {
                shS[0][threadIdx.x] += norm(i, fu[0] != kNone && z < n, cur.ub[0], ru[0]) +
                                       norm(i, fu[1] != kNone && z < n, cur.ub[1], ru[1]);
                shS[1][threadIdx.x] += norm(y, fv[0] != kNone && z > z0, vbl, rv[0]) +
                                       norm(y + 1, fv[1] != kNone && z < n, cur.vb[1], rv[1]);
                shS[2][threadIdx.x] += norm(z, fw[0] != kNone, cur.wb[0], rw[0]) +
                                       norm(z, fw[1] != kNone, cur.wb[1], rw[1]);
            }
            vbl = cur.vb[0];
            vel = cur.vc[0] - g.c15 * pv[0];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                tv[q] = T[q][1];
                tw[q] = T[q][2];
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                X0[q][c] = X1[q][c];
                X1[q][c] = X2[q][c];
            }
            w0[q] = w1[q];
            w1[q] = w2[q];
            w2[q] = w3[q];
        }
    }
    flush(z1 - 1);
    if (z1 <= n) {  // the lower rows' v-faces of the last plane
        shT[z1 & 1][r][lane] = tv[1];
        __syncthreads();
        if (rowT) {
            rv[0] = face(1, y == 0 || y == n, y, shT[z1 & 1][r - 1][lane], tv[0], vbl, vel);
            if (LAST) shS[1][threadIdx.x] += norm(y, fv[0] != kNone, vbl, rv[0]);
            st(plane(a.o[1], (unsigned)(z1 - 1) * su, su), fv[0], rv[0]);
        }
    }
    if (LAST) {
        double sq[3] = {shS[0][threadIdx.x], shS[1][threadIdx.x], shS[2][threadIdx.x]};
        __syncthreads();
        block_reduce_n<0u>(sq, &shX[0][0][0][0]);
        if (threadIdx.x == 0)
#pragma unroll
            for (int d = 0; d < 3; ++d) a.partials[3 * (int64_t)blk + d] = sq[d];
    }
}

// block range of face direction d in a grid over every face (nb[d] blocks each)
__device__ __forceinline__ int face_dir(const int *nb, int blk, int &lb)
{
    if (blk < nb[0]) { lb = blk; return 0; }
    if (blk < nb[0] + nb[1]) { lb = blk - nb[0]; return 1; }
    lb = blk - nb[0] - nb[1];
    return 2;
}
__device__ __forceinline__ void face_coords(const Geom &g, int d, int64_t q, int *x)
{
    split3(q, g.n + (d == 0), g.n + (d == 1), x);
}

// Error_Computation from the block partials (records of three, one sum per
// direction); the loop control of main.cpp:898-1039 (countIter, IterNum cap,
// divergence guard), or for PSEUDO_TIMESTEPPING = 0 the single update's norm
// with countIter 0
__global__ __launch_bounds__(1024) void k_gen_fin_pseudo(Geom g, const double *partials, int nrec, Ctl *ctl)
{
    __shared__ double sh[48];
    if (ctl->mom_done) return;
    double v[3] = {0.0, 0.0, 0.0}, e[3] = {0.0, 0.0, 0.0};
    for_records<3, 3>(partials, nrec, [&](const double *a) {
        v[0] += a[0];
        v[1] += a[1];
        v[2] += a[2];
    });
    block_reduce_n<0u>(v, sh);
    if (threadIdx.x != 0) return;
    const double npts = (double)g.ncell;
    for (int d = 0; d < g.dim; ++d) e[d] = sqrt(v[d]) / sqrt(npts);
    double ne = (e[0] < e[1]) ? e[1] : e[0];
    if (g.dim == 3) ne = (ne < e[2]) ? e[2] : ne;
    ctl->norm_error = ne;
    if (!(ne == ne) || isinf(ne)) ctl->flags |= AMRESSIF_FLAG_NONFINITE;
    if (!g.pseudo) {
        ctl->mom_done = 1;
        return;
    }
    ctl->mom_count += 1;
    if (ctl->mom_count > ctl->iter_num) { ctl->flags |= AMRESSIF_FLAG_CAP; ctl->mom_done = 1; }
    else if (ne > 1.e2) { ctl->flags |= AMRESSIF_FLAG_DIVERGED; ctl->mom_done = 1; }
    else if (!(ne > ctl->tol_mom)) ctl->mom_done = 1;
}

// ------------------------------------------------------------ BDF2 constant
// main.cpp:879-884 with the pressure term folded: C = (1.5/dt) u^n + (0.5/dt)
// (u^n - u^{n-1}) - G p (p's ghosts: Neumann mirror, so G p = 0 on wall
// faces; periodic images).  The stages then read u^n in place, and the face arrays
// change roles instead of being copied (amr_gen_advance).
struct Bdf2Arrays {
    const double *u[3], *up[3];
    double *c[3];
    const double *p;
    int nb[3];
};
__global__ __launch_bounds__(B) void k_gen_bdf2(Geom g, Bdf2Arrays a)
{
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    int lb;
    const int d = face_dir(a.nb, blk, lb);
    const int64_t q = (int64_t)lb * B + threadIdx.x;
    if (q >= g.nf[d]) return;
    const int n = g.n;
    int x[3];
    face_coords(g, d, q, x);
    const int xd = x[d];
    double gp = 0.0;
    if (g.per[d] || (xd > 0 && xd < n)) {
        int l[3] = {x[0], x[1], x[2]}, r[3] = {x[0], x[1], x[2]};
        l[d] = xd == 0 ? n - 1 : xd - 1;
        r[d] = xd == n ? 0 : xd;
        gp = (a.p[cidx(g, r)] - a.p[cidx(g, l)]) * g.idx[d];
    }
    const double un = a.u[d][q], um = a.up[d][q];
    a.c[d][q] = g.c15 * un + (0.5 / g.dt) * (un - um) - gp;
}

// ------------------------------------------------------------ divergence
__global__ __launch_bounds__(B) void k_gen_div(Geom g, const double *f0, const double *f1, const double *f2,
                                               double *b, double *partials)
{
    __shared__ double sh[B / 64];
    const int64_t q = gid();
    double m = 0.0, sum = 0.0;
    if (q < g.ncell) {
        const int n = g.n;
        int x[3];
        split3(q, n, n, x);
        const double *f[3] = {f0, f1, f2};
        double D = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d >= g.dim) break;
            int e[3] = {x[0], x[1], x[2]};
            e[d] += 1;
            const double t = (f[d][fidx(g, d, e[0], e[1], e[2])] - f[d][fidx(g, d, x[0], x[1], x[2])]) * g.idx[d];
            D = d == 0 ? t : D + t;
        }
        m = fabs(D);
        if (D != D) m = D;
        if (b) {
            const double bv = g.c15 * D;
            b[q] = bv;
            sum = bv;
        }
    }
    const double rm = block_reduce<true>(m, sh);
    const double rs = block_reduce<false>(sum, sh);
    if (threadIdx.x == 0) {
        partials[2 * (int64_t)blockIdx.x] = rm;
        partials[2 * (int64_t)blockIdx.x + 1] = rs;
    }
}

__global__ __launch_bounds__(1024) void k_gen_fin_div(const double *partials, int nb, Ctl *ctl, double ncell, int which)
{
    __shared__ double sh[32];
    double v[2] = {0.0, 0.0};
    for_records<2, 2>(partials, nb, [&](const double *a) {
        v[0] = (a[0] > v[0] || a[0] != a[0]) ? a[0] : v[0];
        v[1] += a[1];
    });
    block_reduce_n<1u>(v, sh);
    const double m = v[0], s = v[1];
    if (threadIdx.x != 0) return;
    if (which == 0) {
        ctl->div_star = m;
        ctl->rhs_sum = s;
        ctl->b_mean = s / ncell;
    } else {
        ctl->div_new = m;
    }
}

// ------------------------------------------------------------ Poisson control
__global__ void k_gen_mg_start(Ctl *ctl)
{
    ctl->mg_done = 0;
    ctl->mg_iters = 0;
    ctl->mg_started = 0;
}

// ------------------------------------------------------------ projection
__global__ __launch_bounds__(B) void k_gen_sum(int64_t m, const double *x, double *partials)
{
    __shared__ double sh[B / 64];
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    const double v = q < m ? x[q] : 0.0;
    const double s = block_reduce<false>(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ __launch_bounds__(B) void k_gen_fin_mean(const double *partials, int nb, double m, Ctl *ctl)
{
    __shared__ double sh[B / 64];
    double s = 0.0;
    for (int k = threadIdx.x; k < nb; k += B) s += partials[k];
    s = block_reduce<false>(s, sh);
    if (threadIdx.x == 0) ctl->phi_mean = s / m;
}

// update_solution: u_d = u*_d - (G_d phi) dt/1.5 on the faces (G phi = 0 on
// wall faces: phi's ghosts mirror), then p += phi - mean(phi) on the cells
struct ProjArrays {
    double *u[3];
    const double *s[3];
    double *p;
    const double *phi;
    int nb[4];  // face blocks per direction, then cell blocks
};
__global__ __launch_bounds__(B) void k_gen_project(Geom g, ProjArrays a, const Ctl *ctl)
{
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int n = g.n;
    if (blk >= a.nb[0] + a.nb[1] + a.nb[2]) {
        const int64_t q = (int64_t)(blk - a.nb[0] - a.nb[1] - a.nb[2]) * B + threadIdx.x;
        if (q < g.ncell) a.p[q] = a.p[q] + (a.phi[q] - ctl->phi_mean);
        return;
    }
    int lb;
    const int d = face_dir(a.nb, blk, lb);
    const int64_t q = (int64_t)lb * B + threadIdx.x;
    if (q >= g.nf[d]) return;
    int x[3];
    face_coords(g, d, q, x);
    const int xd = x[d];
    double gphi = 0.0;
    if (g.per[d] || (xd > 0 && xd < n)) {
        int l[3] = {x[0], x[1], x[2]}, r[3] = {x[0], x[1], x[2]};
        l[d] = xd == 0 ? n - 1 : xd - 1;
        r[d] = xd == n ? 0 : xd;
        gphi = (a.phi[cidx(g, r)] - a.phi[cidx(g, l)]) * g.idx[d];
    }
    a.u[d][q] = a.s[d][q] - (gphi * g.dt / 1.5);
}

__global__ void k_gen_fin_step(Ctl *ctl, amressif_step_stats *log)
{
    amressif_step_stats st;
    st.pseudo_iters = ctl->mom_count;
    st.vcycles = ctl->mg_iters;
    st.flags = ctl->flags;
    st.pad = 0;
    st.norm_error = ctl->norm_error;
    st.div_star = ctl->div_star;
    st.rhs_sum = ctl->rhs_sum;
    st.poisson_res = ctl->b_norm > 0 ? ctl->res_norm / ctl->b_norm : ctl->res_norm;
    st.div_new = ctl->div_new;
    *log = st;
}

__global__ __launch_bounds__(B) void k_gen_fill(double *dst, int64_t count, double value)
{
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    if (q < count) dst[q] = value;
}

// ------------------------------------------------------------ Array4 views
struct V4 {
    double *ptr;
    int lo[3], hi[3];
    int64_t js, ks, ns;
};
V4 view(const amr_array4 &a)
{
    V4 v;
    v.ptr = (double *)a.ptr;
    for (int d = 0; d < 3; ++d) {
        v.lo[d] = a.lo[d];
        v.hi[d] = a.hi[d];
    }
    v.js = a.hi[0] - a.lo[0] + 1;
    v.ks = v.js * (a.hi[1] - a.lo[1] + 1);
    v.ns = v.ks * (a.hi[2] - a.lo[2] + 1);
    return v;
}
__device__ __forceinline__ int64_t vidx(const V4 &v, int i, int j, int k, int c)
{
    return (i - v.lo[0]) + v.js * (j - v.lo[1]) + v.ks * (k - v.lo[2]) + v.ns * c;
}

__global__ __launch_bounds__(B) void k_gen_pack(V4 v, int comp, double *dst, int ex, int ey, int ez, int unpack)
{
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    if (q >= (int64_t)ex * ey * ez) return;
    const int i = (int)(q % ex), j = (int)((q / ex) % ey), k = (int)(q / ((int64_t)ex * ey));
    const int64_t e = vidx(v, i, j, k, comp);
    if (unpack) v.ptr[e] = dst[q];
    else dst[q] = v.ptr[e];
}

// every cell of the view: ghosts by the Neumann mirror or the periodic image
__global__ __launch_bounds__(B) void k_gen_unpack_ghosted(Geom g, const double *src, V4 v, int comp,
                                                          const double *shift)
{
    const int64_t wx = v.hi[0] - v.lo[0] + 1, wy = v.hi[1] - v.lo[1] + 1, wz = v.hi[2] - v.lo[2] + 1;
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    if (q >= wx * wy * wz) return;
    int x[3] = {v.lo[0] + (int)(q % wx), v.lo[1] + (int)((q / wx) % wy), v.lo[2] + (int)(q / (wx * wy))};
    int m[3] = {x[0], x[1], x[2]};
    const int n = g.n;
    for (int d = 0; d < g.dim; ++d)
        if (x[d] < 0 || x[d] >= n) {
            if (g.per[d]) m[d] = ((x[d] % n) + n) % n;
            else m[d] = x[d] < 0 ? -x[d] - 1 : 2 * n - 1 - x[d];
        }
    const double s = shift ? *shift : 0.0;
    v.ptr[vidx(v, x[0], x[1], x[2], comp)] = src[cidx(g, m)] - s;
}

__global__ __launch_bounds__(B) void k_gen_unpack_velcart(Geom g, const double *X, V4 v)
{
    const int64_t wx = v.hi[0] - v.lo[0] + 1, wy = v.hi[1] - v.lo[1] + 1, wz = v.hi[2] - v.lo[2] + 1;
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    if (q >= wx * wy * wz) return;
    const int x[3] = {v.lo[0] + (int)(q % wx), v.lo[1] + (int)((q / wx) % wy), v.lo[2] + (int)(q / (wx * wy))};
    for (int c = 0; c < g.dim; ++c) v.ptr[vidx(v, x[0], x[1], x[2], c)] = X[xidx(g, x[0], x[1], x[2]) + (int64_t)c * g.xs];
}

inline int nblk(int64_t m) { return (int)((m + B - 1) / B); }

}  // namespace

// ============================================================ launchers
hipError_t cells(const Ctx &c, hipStream_t s, double *const *f, double *X)
{
    hipLaunchKernelGGL(k_gen_cells, dim3(nblk(c.g.xs)), dim3(B), 0, s, c.g, f[0], f[1], c.g.dim == 3 ? f[2] : f[0], X);
    return hipGetLastError();
}

void stage3_shape(int n, int *ntx, int *nty, int *zc)
{
    *ntx = (n + 1 + kS3X - 1) / kS3X;
    *nty = (n + 1 + kS3Y - 1) / kS3Y;
    // one workgroup per CU: the chunk of planes for which the rounds of 256
    // workgroups, each of zc planes and about five planes of prologue, are
    // shortest
    int64_t best = -1;
    *zc = n + 1;
    for (int q = 1; q <= n + 1; ++q) {
        const int64_t blocks = (int64_t)*ntx * *nty * ((n + 1 + q - 1) / q);
        const int64_t cost = (blocks + 255) / 256 * (q + 5);
        if (best < 0 || cost <= best) { best = cost; *zc = q; }
    }
}

int stage3_blocks(const Ctx &c)
{
    return c.s3_ntx * c.s3_nty * ((c.g.n + 1 + c.s3_zc - 1) / c.s3_zc);
}

// 2D: a pseudo-iteration is one tile launch at every size: 17 us at 384^2, 56 at 1024^2, 200 at
// 2048^2 and 780 at 4096^2, where four stages of three passes each took 48, 131, 409 and 2300.
// Two sets of norm records in turn (a launch reads the one before's while it writes its own).
static double *records2(const Ctx &c, int it) { return c.partials + (it & 1) * 3 * (int64_t)iter_tile_blocks(c.g.n); }

hipError_t iteration2(const Ctx &c, hipStream_t s, double *const *base, double *const *out, int it, bool chained,
                      Ctl *ctl)
{
    IterTile a{};
    const Geom &g = c.g;
    a.u = base[0]; a.v = base[1];
    a.cu = c.C[0]; a.cv = c.C[1];
    a.uo = out[0]; a.vo = out[1];
    a.partials = records2(c, it);
    a.prev = chained ? records2(c, it + 1) : nullptr;
    a.it = it;
    a.ctl = ctl;
    a.n = g.n;
    a.su = g.n + 1;
    a.sv = g.n;
    a.rec = 3;
    a.nst = g.pseudo ? 4 : 1;
    a.expl = !g.pseudo;
    for (int k = 0; k < 4; ++k) a.rk[k] = g.pseudo ? c.rk[k] : g.dt / 1.5;
    a.c15 = g.c15;
    a.iren = g.iren;
    for (int d = 0; d < 2; ++d) {
        a.per[d] = g.per[d];
        a.kind[2 * d] = g.kind_lo[d];
        a.kind[2 * d + 1] = g.kind_hi[d];
        a.inflow[d] = g.inflow[d];
        a.idx[d] = g.idx[d];
        a.idx2[d] = g.idx2[d];
    }
    return launch_iter_tile(a, s);
}

hipError_t stage3(const Ctx &c, hipStream_t s, double *const *in, double *const *base, double *const *out, double rk,
                  int last, const Ctl *guard)
{
    Stage3 a{};
    for (int d = 0; d < 3; ++d) {
        if (out[d] == in[d] || out[d] == base[d]) return hipErrorInvalidValue;
        a.s[d] = in[d];
        a.b[d] = base[d];
        a.c[d] = c.C[d];
        a.o[d] = out[d];
    }
    a.partials = c.partials;
    a.rk = rk;
    for (int d = 0; d < 3; ++d) {
        a.kq[d] = -0.125 * c.g.idx[d];
        a.kv[d] = c.g.idx2[d] * c.g.iren;
        for (int hi = 0; hi < 2; ++hi) {
            // 0: -mirror, 1: slip, 2: 2 - mirror, 3: 2 inflow - mirror
            const int kind = hi ? c.g.kind_hi[d] : c.g.kind_lo[d];
            for (int q = 0; q < 3; ++q) {
                a.sg[2 * d + hi][q] = kind == 1 && q != d ? 1.0 : -1.0;
                a.ct[2 * d + hi][q] = kind == 2 ? 2.0 : (kind == 3 ? 2.0 * c.g.inflow[q] : 0.0);
            }
        }
    }
    a.ntx = c.s3_ntx;
    a.nty = c.s3_nty;
    a.zc = c.s3_zc;
    const dim3 grid(stage3_blocks(c));
    if (last) hipLaunchKernelGGL(k_gen_stage3<true>, grid, dim3(64 * kS3W), 0, s, c.g, a, guard);
    else hipLaunchKernelGGL(k_gen_stage3<false>, grid, dim3(64 * kS3W), 0, s, c.g, a, guard);
    return hipGetLastError();
}

hipError_t fin_pseudo(const Ctx &c, hipStream_t s, int it, Ctl *ctl)
{
    const int nrec = c.g.dim == 3 ? stage3_blocks(c) : iter_tile_blocks(c.g.n);
    hipLaunchKernelGGL(k_gen_fin_pseudo, dim3(1), dim3(1024), 0, s, c.g, c.g.dim == 3 ? c.partials : records2(c, it), nrec,
                       ctl);
    return hipGetLastError();
}

hipError_t bdf2(const Ctx &c, hipStream_t s)
{
    Bdf2Arrays a{};
    for (int d = 0; d < 3; ++d) {
        const bool on = d < c.g.dim;
        a.u[d] = on ? c.U[d] : nullptr;
        a.up[d] = on ? c.Up[d] : nullptr;
        a.c[d] = on ? c.C[d] : nullptr;
        a.nb[d] = on ? c.nb_face[d] : 0;
    }
    a.p = c.p;
    hipLaunchKernelGGL(k_gen_bdf2, dim3(a.nb[0] + a.nb[1] + a.nb[2]), dim3(B), 0, s, c.g, a);
    return hipGetLastError();
}

hipError_t divergence(const Ctx &c, hipStream_t s, double *const *f, double *b, int *nblocks)
{
    *nblocks = nblk(c.g.ncell);
    hipLaunchKernelGGL(k_gen_div, dim3(*nblocks), dim3(B), 0, s, c.g, f[0], f[1], c.g.dim == 3 ? f[2] : f[0], b,
                       c.partials);
    return hipGetLastError();
}

hipError_t fin_div(const Ctx &c, hipStream_t s, int nblocks, Ctl *ctl, int which)
{
    hipLaunchKernelGGL(k_gen_fin_div, dim3(1), dim3(1024), 0, s, c.partials, nblocks, ctl, (double)c.g.ncell, which);
    return hipGetLastError();
}

hipError_t mg_start(const Ctx &c, hipStream_t s, Ctl *ctl)
{
    hipLaunchKernelGGL(k_gen_mg_start, dim3(1), dim3(1), 0, s, ctl);
    return hipGetLastError();
}

hipError_t phi_mean(const Ctx &c, hipStream_t s, Ctl *ctl)
{
    const int nb = nblk(c.g.ncell);
    hipLaunchKernelGGL(k_gen_sum, dim3(nb), dim3(B), 0, s, c.g.ncell, c.phi, c.partials);
    hipLaunchKernelGGL(k_gen_fin_mean, dim3(1), dim3(B), 0, s, c.partials, nb, (double)c.g.ncell, ctl);
    return hipGetLastError();
}

hipError_t project(const Ctx &c, hipStream_t s, Ctl *ctl)
{
    ProjArrays a{};
    for (int d = 0; d < 3; ++d) {
        const bool on = d < c.g.dim;
        a.u[d] = on ? c.U[d] : nullptr;
        a.s[d] = on ? c.S[d] : nullptr;
        a.nb[d] = on ? c.nb_face[d] : 0;
    }
    a.nb[3] = nblk(c.g.ncell);
    a.p = c.p;
    a.phi = c.phi;
    hipLaunchKernelGGL(k_gen_project, dim3(a.nb[0] + a.nb[1] + a.nb[2] + a.nb[3]), dim3(B), 0, s, c.g, a, ctl);
    return hipGetLastError();
}

hipError_t fin_step(const Ctx &c, hipStream_t s, Ctl *ctl, amressif_step_stats *log)
{
    hipLaunchKernelGGL(k_gen_fin_step, dim3(1), dim3(1), 0, s, ctl, log);
    return hipGetLastError();
}

hipError_t fill(hipStream_t s, double *dst, int64_t count, double value)
{
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gen_fill, dim3(nblk(count)), dim3(B), 0, s, dst, count, value);
    return hipGetLastError();
}

hipError_t pack(hipStream_t s, const amr_array4 &a, int comp, double *dst, int ex, int ey, int ez)
{
    hipLaunchKernelGGL(k_gen_pack, dim3(nblk((int64_t)ex * ey * ez)), dim3(B), 0, s, view(a), comp, dst, ex, ey, ez,
                       0);
    return hipGetLastError();
}

hipError_t unpack(hipStream_t s, const double *src, const amr_array4 &a, int comp, int ex, int ey, int ez)
{
    hipLaunchKernelGGL(k_gen_pack, dim3(nblk((int64_t)ex * ey * ez)), dim3(B), 0, s, view(a), comp,
                       const_cast<double *>(src), ex, ey, ez, 1);
    return hipGetLastError();
}

// the window [lo, hi] (inclusive, inside the view) between a view and an
// internal array of extents ex x ey x ..: view -> array (unpack 0) or back
__global__ __launch_bounds__(B) void k_gen_pack_window(V4 v, int comp, double *dst, int ex, int ey, int lo0, int lo1,
                                                       int lo2, int wx, int wy, int wz, int unpack)
{
    const int64_t q = (int64_t)blockIdx.x * B + threadIdx.x;
    if (q >= (int64_t)wx * wy * wz) return;
    const int i = lo0 + (int)(q % wx), j = lo1 + (int)((q / wx) % wy), k = lo2 + (int)(q / ((int64_t)wx * wy));
    const int64_t e = vidx(v, i, j, k, comp), d = i + (int64_t)ex * (j + (int64_t)ey * k);
    if (unpack) v.ptr[e] = dst[d];
    else dst[d] = v.ptr[e];
}

hipError_t pack_window(hipStream_t s, const amr_array4 &a, int comp, double *dst, int ex, int ey, const int *lo,
                       const int *hi, int unpack)
{
    const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
    hipLaunchKernelGGL(k_gen_pack_window, dim3(nblk((int64_t)wx * wy * wz)), dim3(B), 0, s, view(a), comp, dst, ex, ey,
                       lo[0], lo[1], lo[2], wx, wy, wz, unpack);
    return hipGetLastError();
}

hipError_t unpack_cells_ghosted(const Ctx &c, hipStream_t s, const double *src, const amr_array4 &a, int comp,
                                const double *shift)
{
    const V4 v = view(a);
    const int64_t m = (int64_t)(v.hi[0] - v.lo[0] + 1) * (v.hi[1] - v.lo[1] + 1) * (v.hi[2] - v.lo[2] + 1);
    hipLaunchKernelGGL(k_gen_unpack_ghosted, dim3(nblk(m)), dim3(B), 0, s, c.g, src, v, comp, shift);
    return hipGetLastError();
}

hipError_t unpack_velcart(const Ctx &c, hipStream_t s, const double *X, const amr_array4 &a)
{
    const V4 v = view(a);
    const int64_t m = (int64_t)(v.hi[0] - v.lo[0] + 1) * (v.hi[1] - v.lo[1] + 1) * (v.hi[2] - v.lo[2] + 1);
    hipLaunchKernelGGL(k_gen_unpack_velcart, dim3(nblk(m)), dim3(B), 0, s, c.g, X, v);
    return hipGetLastError();
}

}  // namespace gen
}  // namespace amr
