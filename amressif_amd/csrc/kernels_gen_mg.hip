// The general path's multigrid (poisson.cpp:41-186 solves the same problem with
// AMReX's MLMG): the V-cycle's two legs per level and the outer step as one launch
// each, the coarsest level solved exactly.
//
//   k_gen_leg<.., false> : two red-black Gauss-Seidel sweeps from zero, then the
//                          residual's 2^dim-cell average on the next level
//   k_gen_leg<.., true>  : (bi/tri)linear prolongation of the next level's
//                          correction added, two sweeps
//   k_gen_exact3, and k_tail_dct in 2D : e = L^+ r on the coarsest level by the
//                          eigenvectors of its 1D operators
//   k_gen_outer          : phi' = phi + e, r = (b - mean) - L phi', max |r|, sum phi'
//
// L e = sum_d (e(x + 1) - 2 e + e(x - 1))/h_d^2 with Neumann walls (the neighbour
// past a wall is the cell itself: its term drops) and periodic images.
#include "device_common.hpp"
#include "gen.hpp"

namespace amr {
namespace gen {

namespace {

// Legs.  A workgroup owns a tile of T^dim cells and holds it with a halo of 5 in LDS:
// each of the four half-sweeps makes one ring stale and the residual one more.  Cell
// k of a thread is number t + NT k of the box; its right-hand side, already divided
// by the diagonal, stays in registers.  Cells outside a wall hold 0 and are never
// updated, so their terms drop; periodic halos are images and evolve as such (a
// level that is smoothed has an even side, so colours match across the wrap).
// Five launches per leg (four half-sweeps and a transfer) became one: on small
// levels a launch is 4 us whatever it does (2D legs of 96^2 to 384^2: 6.3 us against
// 18, the 384^2 solve's cycle 55 us against 195).
template <int DIM>
struct LegShape;
template <>
struct LegShape<2> {
    static constexpr int T = 32, NT = 512;
};
template <>
struct LegShape<3> {
    static constexpr int T = 8, NT = 512;
};

template <int DIM, bool UP>
__global__ __launch_bounds__(LegShape<DIM>::NT) void k_gen_leg(Geom g, Level F, Level Cl, int nt, const Ctl *ctl)
{
    constexpr int T = LegShape<DIM>::T, NT = LegShape<DIM>::NT, H = 5, E = T + 2 * H, E2 = E * E;
    constexpr int N = DIM == 3 ? E2 * E : E2, K = (N + NT - 1) / NT;
    constexpr int TC = T / 2, CE = TC + 6, NC = DIM == 3 ? CE * CE * CE : CE * CE;  // coarse cells the prolongation reads
    constexpr int NR = DIM == 3 ? T * T * T : T * T;
    __shared__ double sh[N];
    __shared__ double aux[UP ? NC : NR];
    if (ctl->mg_done) return;
    const int t = threadIdx.x, n = F.n;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int o[3] = {(blk % nt) * T, ((blk / nt) % nt) * T, DIM == 3 ? (blk / (nt * nt)) * T : 0};
    if (UP) {  // stage the coarse correction: cells o/2 - 3 .. of each direction, clamped at walls
        const int m = Cl.n;
        for (int q = t; q < NC; q += NT) {
            const int c[3] = {q % CE, (q / CE) % CE, DIM == 3 ? q / (CE * CE) : 0};
            int64_t k = 0;
#pragma unroll
            for (int d = DIM - 1; d >= 0; --d) {
                int x = o[d] / 2 - 3 + c[d];
                x = g.per[d] ? ((x % m) + m) % m : min(max(x, 0), m - 1);
                k = k * m + x;
            }
            aux[q] = Cl.out[k];
        }
        __syncthreads();
    }
    double rs[K], rd[K];  // r / diag and 1 / diag
    int info[K];          // half-sweeps the cell stays exact for (0: outside, not updated), colour in bit 8
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int id = t + NT * k;
        const int l[3] = {id % E, (id / E) % E, DIM == 3 ? id / E2 : H};
        double e = 0.0, r = 0.0, diag = 0.0;
        int ring = E, col = 0;
        bool in = id < N;
        int64_t q = 0;
#pragma unroll
        for (int d = DIM - 1; d >= 0; --d) {
            const int x = o[d] + l[d] - H;
            int y = x;
            if (g.per[d]) {
                y = x < 0 ? x + n : (x >= n ? x - n : x);  // images up to n cells away; beyond (a tile past n) unused
                y = min(max(y, 0), n - 1);
                diag += 2.0 * F.a[d];
            } else {
                in = in && x >= 0 && x < n;
                diag += ((x > 0) + (x < n - 1)) * F.a[d];
            }
            ring = min(ring, min(l[d], E - 1 - l[d]));
            col += x;
            q = q * n + y;
        }
        rd[k] = 0.0;
        info[k] = 0;
        if (in) {
            r = F.r[q];
            rd[k] = 1.0 / diag;
            info[k] = ring | ((col & 1) << 8);
            if (UP) {
                e = F.e[q];
                // per direction 3/4 of the coarse cell and 1/4 of its neighbour on the fine cell's side
                int c[3] = {0, 0, 0}, s[3] = {0, 0, 0};
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    const int x = l[d] - H;  // tile origins are even: parities are the cell's own
                    c[d] = (x >> 1) + 3;
                    s[d] = (x & 1) ? 1 : -1;
                }
                double p = 0.0;
#pragma unroll
                for (int v = 0; v < (1 << DIM); ++v) {
                    const int i = c[0] + ((v & 1) ? s[0] : 0), j = c[1] + ((v & 2) ? s[1] : 0);
                    const int kk = DIM == 3 ? c[2] + ((v & 4) ? s[2] : 0) : 0;
                    const double w = ((v & 1) ? 0.25 : 0.75) * ((v & 2) ? 0.25 : 0.75) * (DIM == 3 ? ((v & 4) ? 0.25 : 0.75) : 1.0);
                    p += w * aux[i + CE * (j + CE * kk)];
                }
                e += p;
            }
        }
        rs[k] = r * rd[k];
        if (id < N) sh[id] = e;
    }
    __syncthreads();
    auto nbs = [&](int id) {
        double s = F.a[0] * (sh[id - 1] + sh[id + 1]) + F.a[1] * (sh[id - E] + sh[id + E]);
        if (DIM == 3) s += F.a[2] * (sh[id - E2] + sh[id + E2]);
        return s;
    };
#pragma unroll
    for (int h = 0; h < 4; ++h) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int id = t + NT * k;
            if ((info[k] & 255) > h && (info[k] >> 8) == (h & 1))
                sh[id] = (!UP && h == 0 ? 0.0 : nbs(id) * rd[k]) - rs[k];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int id = t + NT * k;
        const int l[3] = {id % E - H, (id / E) % E - H, DIM == 3 ? id / E2 - H : 0};
        const bool own = id < N && l[0] >= 0 && l[0] < T && l[1] >= 0 && l[1] < T && l[2] >= 0 && l[2] < T &&
                         o[0] + l[0] < n && o[1] + l[1] < n && (DIM == 2 || o[2] + l[2] < n);
        if (own) {
            const int64_t q = o[0] + l[0] + (int64_t)n * (o[1] + l[1] + (int64_t)n * (o[2] + l[2]));
            if (UP) {
                F.out[q] = sh[id];
            } else {
                F.e[q] = sh[id];
                aux[l[0] + T * (l[1] + T * l[2])] = (rs[k] - nbs(id) * rd[k] + sh[id]) / rd[k];
            }
        }
    }
    if (UP) return;
    __syncthreads();
    constexpr int NCO = DIM == 3 ? TC * TC * TC : TC * TC;
    for (int q = t; q < NCO; q += NT) {
        const int c[3] = {q % TC, (q / TC) % TC, DIM == 3 ? q / (TC * TC) : 0}, m = Cl.n;
        const int x = o[0] / 2 + c[0], y = o[1] / 2 + c[1], z = o[2] / 2 + c[2];
        if (x >= m || y >= m || (DIM == 3 && z >= m)) continue;
        const double *f = aux + 2 * c[0] + T * (2 * c[1] + T * 2 * c[2]);
        double s = f[0] + f[1] + f[T] + f[T + 1];
        if (DIM == 3) s += f[T * T] + f[T * T + 1] + f[T * T + T] + f[T * T + T + 1];
        Cl.r[x + (int64_t)m * (y + (int64_t)m * z)] = (DIM == 3 ? 0.125 : 0.25) * s;
    }
}

// The same legs of a large 3D level, marched along z: the tile form reads and smooths
// 11 times its cells there.  A workgroup holds 64 columns x 32 rows (two rows per
// thread of 16 waves) and pipelines the half-sweeps: with plane p loaded, half-sweep s
// works on plane p - 1 - s, so the z neighbours are the thread's own registers and
// already carry the sweeps they must.  x neighbours come from adjacent lanes, y
// neighbours are the thread's other row or, published a step before, the next wave's
// row in LDS: one barrier per plane.  Outside a wall the loads give 0 and 1/diag is 0,
// so nothing moves there.  Halos: 4 rings for four half-sweeps; going down one more for
// the residual and one to start on even cells.  A workgroup loads each plane of its
// tile once: 17 B per cell down, 25 up (coarse cells with them) are what a leg cannot
// do without.  The halo's loads are 1.97 times that down and 1.52 up, plus nine and
// seven planes a chunk, most of them from the L2: the counters give 20 and 28 B (five
// launches moved about 140).  163 us a leg at 256^3 against 477 down and 527 up, at 2.1
// and 2.9 TB/s.  Bound by the instructions of a plane (1.7 us; where a workgroup runs
// the VALU is busy 77% of the time down, 65% up) with half the lanes idle in each
// half-sweep.
template <bool UP>
__global__ __launch_bounds__(1024) void k_gen_leg3(Geom g, Level F, Level Cl, int ntx, int nty, int zc, const Ctl *ctl)
{
    constexpr int HX = UP ? 4 : 6, OX = 64 - 2 * HX, OY = 32 - 2 * HX, NE = UP ? 6 : 7, NR = UP ? 5 : 6;
    constexpr unsigned kNone = 0x80000000u;
    __shared__ double shY[2][4][16][2][64];
    if (ctl->mg_done) return;
    const int n = F.n, m = Cl.n, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int tx = blk % ntx, ty = (blk / ntx) % nty, tz = blk / (ntx * nty);
    const int x = tx * OX - HX + lane, y = ty * OY - HX + 2 * w;  // column, first row (even)
    const int z0 = tz * zc, z1 = min(z0 + zc, n);                 // zc even
    const bool px = g.per[0], py = g.per[1], pz = g.per[2];
    auto wrap = [](int q, int k) {
        const int v = q % k;
        return v < 0 ? v + k : v;
    };
    // byte offsets in a plane of the two rows' cells (past the plane: 0) and, going up, of the
    // six coarse cells around them: rows y/2 - 1 .. y/2 + 1, the column's cell and its side's neighbour
    unsigned off[2], offc[3][2];
    double rdi[2], rdb[2], dxy[2];  // 1/diag inside and on the first and last plane; the diagonal without z
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const bool in = (px || (x >= 0 && x < n)) && (py || (y + q >= 0 && y + q < n));
        const int xx = px ? wrap(x, n) : x, yy = py ? wrap(y + q, n) : y + q;
        off[q] = in ? 8u * (unsigned)(xx + n * yy) : kNone;
        dxy[q] = (px ? 2.0 : (x > 0) + (x < n - 1)) * F.a[0] + (py ? 2.0 : (y + q > 0) + (y + q < n - 1)) * F.a[1];
        rdi[q] = in ? 1.0 / (dxy[q] + 2.0 * F.a[2]) : 0.0;
        rdb[q] = in ? 1.0 / (dxy[q] + F.a[2]) : 0.0;
    }
    if (UP) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                int cx = (x >> 1) + (v ? ((x & 1) ? 1 : -1) : 0), cy = (y >> 1) + j - 1;
                cx = px ? wrap(cx, m) : min(max(cx, 0), m - 1);
                cy = py ? wrap(cy, m) : min(max(cy, 0), m - 1);
                offc[j][v] = 8u * (unsigned)(cx + m * cy);
            }
    }
    auto plane = [](const double *base, int64_t first, unsigned count) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(base + first), 0, 8 * count, 0x00020000);
    };
    auto ld = [](__amdgpu_buffer_rsrc_t r, unsigned o) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0));
    };
    const unsigned sn = (unsigned)n * n, sm = (unsigned)m * m;
    auto load = [&](const double *f, int p, double *v) {  // plane p of a fine array
        const bool in = pz || (p >= 0 && p < n);
        const auto r = plane(f, (int64_t)(pz ? wrap(p, n) : (in ? p : 0)) * sn, in ? sn : 0);
        v[0] = ld(r, off[0]);
        v[1] = ld(r, off[1]);
    };
    double cf[3][2];
    auto load_coarse = [&](int k) {
        const int kk = pz ? wrap(k, m) : min(max(k, 0), m - 1);
        const auto r = plane(Cl.out, (int64_t)kk * sm, sm);
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int v = 0; v < 2; ++v) cf[j][v] = ld(r, offc[j][v]);
    };
    // the rows' coarse values interpolated in x and y
    auto rows_of = [&](double *h) {
        double c[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) c[j] = 0.75 * cf[j][0] + 0.25 * cf[j][1];
        h[0] = 0.75 * c[1] + 0.25 * c[0];
        h[1] = 0.75 * c[1] + 0.25 * c[2];
    };
    double E[2][NE], R[2][NR], ne[2] = {0.0, 0.0}, nr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int k = 0; k < NE; ++k) E[q][k] = 0.0;
#pragma unroll
        for (int k = 0; k < NR; ++k) R[q][k] = 0.0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) shY[0][j][w][0][lane] = shY[0][j][w][1][lane] = 0.0;
    const bool lanO = lane >= HX && lane < HX + OX && x < n;
    const bool rowO = 2 * w >= HX && 2 * w < HX + OY && y < n;  // both rows (n even); x, y >= 0 there
    const bool even = (lane & 1) == 0;
    const int ps = z0 - (UP ? 4 : 5), pe = z1 + (UP ? 3 : 4);
    // the two coarse planes around plane p: (p / 2 - 1, p / 2) for even p, (p / 2, p / 2 + 1) for odd
    double hlo[2] = {0.0, 0.0}, hhi[2] = {0.0, 0.0}, acc = 0.0;
    load(F.r, ps, nr);
    if (UP) {
        load(F.e, ps, ne);  // ps is even, as zc is
        load_coarse((ps >> 1) - 1);
        rows_of(hlo);
        load_coarse(ps >> 1);
        rows_of(hhi);
        load_coarse((ps >> 1) + 1);
    }
    __syncthreads();
    int bf = 0;
    for (int p = ps; p <= pe; ++p, bf ^= 1) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
#pragma unroll
            for (int k = NE - 1; k > 0; --k) E[q][k] = E[q][k - 1];
#pragma unroll
            for (int k = NR - 1; k > 0; --k) R[q][k] = R[q][k - 1];
            E[q][0] = 0.0;
            R[q][0] = nr[q];
            if (UP) {
                const double c = (p & 1) ? 0.75 * hlo[q] + 0.25 * hhi[q] : 0.75 * hhi[q] + 0.25 * hlo[q];
                E[q][0] = off[q] != kNone && (pz || (p >= 0 && p < n)) ? ne[q] + c : 0.0;
            }
        }
        // plane p + 1: an odd one needs the next coarse plane, which was loaded two planes ago
        load(F.r, p + 1, nr);
        if (UP) {
            load(F.e, p + 1, ne);
            if (!(p & 1)) {
#pragma unroll
                for (int q = 0; q < 2; ++q) hlo[q] = hhi[q];
                rows_of(hhi);
                load_coarse((p >> 1) + 2);
            }
        }
        // the sum of the six neighbours' terms at row q of window plane c (y neighbours from slot j)
        auto nbs = [&](int q, int c, int j) {
            const double C = E[q][c];
            const double yo = shY[bf][j][q == 0 ? max(w - 1, 0) : min(w + 1, 15)][1 - q][lane];
            return F.a[0] * (lane_prev(C) + lane_next(C)) + (F.a[1] * (yo + E[1 - q][c]) + F.a[2] * (E[q][c - 1] + E[q][c + 1]));
        };
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int z = p - 1 - s;
            const bool zi = pz || (z > 0 && z < n - 1), zin = pz || (z >= 0 && z < n);
            // lanes of the colour in the first row: x + y + z of parity s (x and lane, y and 0 alike)
            const bool mine = ((z + s) & 1) == 0 ? even : !even;
            double v[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double rd = zi ? rdi[q] : (zin ? rdb[q] : 0.0);
                v[q] = (!UP && s == 0) ? -R[q][1] * rd : (nbs(q, s + 1, UP ? s : s - 1) - R[q][s + 1]) * rd;
            }
            E[0][s + 1] = mine ? v[0] : E[0][s + 1];
            E[1][s + 1] = mine ? E[1][s + 1] : v[1];
        }
        if (UP) {
            const int z = p - 4;
            if (lanO && rowO && z >= z0) {
#pragma unroll
                for (int q = 0; q < 2; ++q) F.out[x + (int64_t)n * (y + q + (int64_t)n * z)] = E[q][4];
            }
        } else {
            const int ze = p - 4, z = p - 5;
            if (lanO && rowO && ze >= z0 && ze < z1) {
#pragma unroll
                for (int q = 0; q < 2; ++q) F.e[x + (int64_t)n * (y + q + (int64_t)n * ze)] = E[q][4];
            }
            if (z >= z0) {
                const double dz = (pz ? 2.0 : (z > 0) + (z < n - 1)) * F.a[2];
                double res = 0.0;
#pragma unroll
                for (int q = 0; q < 2; ++q) res += R[q][5] - (nbs(q, 5, 3) - (dxy[q] + dz) * E[q][5]);
                res += lane_next(res);
                acc = (z & 1) ? acc + res : res;
                if ((z & 1) && even && lanO && rowO)
                    Cl.r[(x >> 1) + (int64_t)m * ((y >> 1) + (int64_t)m * (z >> 1))] = 0.125 * acc;
            }
        }
        // what the next step's neighbours read
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) shY[bf ^ 1][j][w][q][lane] = E[q][UP ? j : j + 1];
        __syncthreads();
    }
}

// e = L^+ r on a 3D level of m <= 20 cells per side, in one workgroup: three products
// with the eigenvectors of the 1D operators (DCT-II, or the real Fourier modes), the
// inverse eigenvalues (the constant mode 0), three products back.  Each product
// contracts the slowest axis of a cube in LDS and writes the result as the fastest
// (rows padded to m + 1), so three of them bring the axes back in order.  The products
// run on the matrix cores: 16 outputs x 16 lines per v_mfma_f64_16x16x4f64 tile, a
// wave keeping its 16 outputs' factors of all six products in registers: 13.4 us at
// 16^3, 24 at 18^3, a chain of barriers.  (On the
// VALU with the factors in LDS 18.5 us at 16^3 and 30 at 18^3, bound by LDS reads.)
// tab: per direction Q[i][k] and Q[k][i] transposed, m x 24 each (zero padded), then
// the m^3 inverse eigenvalues.
constexpr int kExM = 20, kExLd = 24, kExK = kExM / 4;
typedef double Mfma4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(1024) void k_gen_exact3(const double *r, double *e, int m, const double *tab,
                                                     const Ctl *ctl)
{
    __shared__ double A[kExM * kExM * (kExM + 1)], B[kExM * kExM * (kExM + 1)];
    if (ctl->mg_done) return;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), m2 = m * m, ld = m + 1;
    // q / m by a reciprocal (exact: q < 2^13, m <= 20); the compiler's division is 20 times as long
    const unsigned rm = 0xffffffffu / (unsigned)m + 1u;
    auto pad = [&](int q) { return (int)__umulhi((unsigned)q, rm) + q; };  // (q / m) ld + q % m
    const int sz = m * kExLd, mt = m > 16 ? 2 : 1, k0 = 16 * (w % mt);  // this wave's outputs k0 .. k0 + 15
    // the products' tables in order: z, y, x forward, z, y, x back
    double P[6][kExK];
#pragma unroll
    for (int g = 0; g < 6; ++g) {
        const double *T = tab + (g < 3 ? 4 - 2 * g : 5 - 2 * (g - 3)) * sz;
#pragma unroll
        for (int s = 0; s < kExK; ++s) {
            const int a = 4 * s + (lane >> 4), k = k0 + (lane & 15);
            P[g][s] = a < m && k < m ? T[a * kExLd + k] : 0.0;
        }
    }
    for (int q = t; q < m2 * m; q += 1024) A[pad(q)] = r[q];
    __syncthreads();
    // in[a][b][c] (c fastest, padded), contracted over a: out[b][c][k] = sum_a P[a][k] in[a][b][c]
    auto product = [&](const double *in, double *out, const double (&p)[kExK]) {
        for (int q = w / mt; 16 * q < m2; q += 16 / mt) {
            const int line = 16 * q + (lane & 15), bc = pad(min(line, m2 - 1));
            Mfma4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < kExK; ++s)
                if (4 * s < m) {
                    const int a = min(4 * s + (lane >> 4), m - 1);  // (past m the factor is 0)
                    d = __builtin_amdgcn_mfma_f64_16x16x4f64(p[s], in[a * m * ld + bc], d, 0, 0, 0);
                }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int k = k0 + (lane >> 4) + 4 * v;
                if (line < m2 && k < m) out[line * ld + k] = d[v];
            }
        }
        __syncthreads();
    };
    product(A, B, P[0]);  // z: (z, y, x) -> (y, x, kz)
    product(B, A, P[1]);  // y: -> (x, kz, ky)
    product(A, B, P[2]);  // x: -> (kz, ky, kx)
    const double *dinv = tab + 6 * sz;  // by (kz, ky, kx)
    for (int q = t; q < m2 * m; q += 1024) B[pad(q)] *= dinv[q];
    __syncthreads();
    product(B, A, P[3]);  // kz back: (kz, ky, kx) -> (ky, kx, z)
    product(A, B, P[4]);  // ky: -> (kx, z, y)
    product(B, A, P[5]);  // kx: -> (z, y, x)
    for (int q = t; q < m2 * m; q += 1024) e[q] = A[pad(q)];
}

// phi' = phi + e and r = (b - mean b) - L phi', with max |r| and sum phi' per
// workgroup.  e null: the start from phi = 0 (phi' = 0, r = b - mean b).  A thread
// marches zc planes of a column (3D) or zc rows (2D, its y) and keeps the previous,
// current and next values along the march.
__global__ __launch_bounds__(256) void k_gen_outer(Geom g, Level L, const double *phi, const double *e, const double *b,
                                                   double *phi2, double *partials, int ntx, int nty, int zc,
                                                   const Ctl *ctl)
{
    __shared__ double sh[32];
    if (ctl->mg_done) return;
    const int n = L.n, dim = g.dim;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int x = (blk % ntx) * 64 + (int)(threadIdx.x & 63);
    const int y = ((blk / ntx) % nty) * 4 + (int)(threadIdx.x >> 6);  // 3D: the row; 2D: unused
    // the march's direction: z in 3D, y in 2D (4 chunks per workgroup there)
    const int chunk = dim == 3 ? blk / (ntx * nty) : 4 * (blk / ntx) + (int)(threadIdx.x >> 6);
    const int s0 = chunk * zc, s1 = min(s0 + zc, n), md = dim - 1;
    const int64_t sm = dim == 3 ? (int64_t)n * n : n;  // stride of the march
    double mx = 0.0, sum = 0.0;
    if (x < n && s0 < n && (dim == 2 || y < n)) {
        const int64_t base = x + (dim == 3 ? (int64_t)n * y : 0);
        auto val = [&](int64_t q) { return phi[q] + e[q]; };
        const double mean = ctl->b_mean;
        if (!e) {
            for (int s = s0; s < s1; ++s) {
                const int64_t q = base + sm * s;
                const double r = b[q] - mean;
                L.r[q] = r;
                phi2[q] = 0.0;
                mx = (fabs(r) > mx || r != r) ? fabs(r) : mx;
            }
        } else {
            // neighbours past a wall are the cell itself: offset 0
            const int64_t xm = x > 0 ? -1 : (g.per[0] ? n - 1 : 0), xp = x < n - 1 ? 1 : (g.per[0] ? -(n - 1) : 0);
            const int64_t ym = dim == 3 ? (y > 0 ? -n : (g.per[1] ? (int64_t)n * (n - 1) : 0)) : 0;
            const int64_t yp = dim == 3 ? (y < n - 1 ? n : (g.per[1] ? -(int64_t)n * (n - 1) : 0)) : 0;
            auto wrap = [&](int s) { return g.per[md] ? (s < 0 ? s + n : (s >= n ? s - n : s)) : min(max(s, 0), n - 1); };
            double lo = val(base + sm * wrap(s0 - 1)), c = val(base + sm * s0);
            for (int s = s0; s < s1; ++s) {
                const int64_t q = base + sm * s;
                const double hi = val(base + sm * wrap(s + 1));
                double lap = (val(q + xp) - 2.0 * c + val(q + xm)) * L.a[0];
                if (dim == 3) lap += (val(q + yp) - 2.0 * c + val(q + ym)) * L.a[1];
                lap += (hi - 2.0 * c + lo) * L.a[md];
                const double r = (b[q] - mean) - lap;
                L.r[q] = r;
                phi2[q] = c;
                sum += c;
                mx = (fabs(r) > mx || r != r) ? fabs(r) : mx;
                lo = c;
                c = hi;
            }
        }
    }
    double red[2] = {mx, sum};
    block_reduce_n<1u>(red, sh);
    if (threadIdx.x == 0) {
        partials[2 * (int64_t)blk] = red[0];
        partials[2 * (int64_t)blk + 1] = red[1];
    }
}

// the stopping test ||r||inf <= max(tol_abs, tol_rel ||b - mean||inf)
// (poisson.cpp:181-182); the first residual (phi = 0) is b - mean itself.  Also
// the mean of phi, for the projection.
__global__ __launch_bounds__(1024) void k_gen_fin_outer(const double *partials, int nb, double ncell, Ctl *ctl)
{
    __shared__ double sh[32];
    if (ctl->mg_done) return;
    double v[2] = {0.0, 0.0};
    for_records<2, 2>(partials, nb, [&](const double *a) {
        v[0] = (a[0] > v[0] || a[0] != a[0]) ? a[0] : v[0];
        v[1] += a[1];
    });
    block_reduce_n<1u>(v, sh);
    if (threadIdx.x != 0) return;
    const double m = v[0];
    if (!ctl->mg_started) {
        ctl->b_norm = m;
        ctl->mg_started = 1;
    }
    ctl->res_norm = m;
    ctl->phi_mean = v[1] / ncell;
    const double thr = fmax(ctl->tol_abs, ctl->tol_rel * ctl->b_norm);
    if (m <= thr || !(m == m)) ctl->mg_done = 1;
    else if (ctl->mg_iters >= ctl->mg_max_iter) {
        ctl->flags |= AMRESSIF_FLAG_MG_CAP;
        ctl->mg_done = 1;
    } else ctl->mg_iters += 1;
}

}  // namespace

// ============================================================ launchers
// The legs of a 3D level march above 64 cells per side: 163 us a leg at 256^3, 40 at
// 128^3, 25 at 72^3, 23 at 64^3, 22 at 32^3 against 1218, 153, 31, 23 and 14 of the tiles
static bool leg_march(int n) { return n > 64; }

// Planes per workgroup of k_gen_leg3 (even: a coarse plane's two children are one workgroup's,
// and the march up starts on an even plane): the shortest rounds of 256 workgroups, each of
// zc planes and about nine to fill and drain the half-sweeps
static int leg_chunk(int n, int tiles)
{
    int best = 2;
    int64_t cost = -1;
    for (int q = 2; q <= n; q += 2) {
        const int64_t v = ((int64_t)tiles * ((n + q - 1) / q) + 255) / 256 * (q + 9);
        if (cost < 0 || v <= cost) { cost = v; best = q; }
    }
    return best;
}

hipError_t vcycle(const Ctx &c, hipStream_t s, const Ctl *ctl)
{
    const int L = c.nlev;
    auto leg = [&](int l, bool up) -> hipError_t {
        const Level &F = c.lev[l], &Cl = c.lev[l + 1];
        if (c.g.dim == 3 && leg_march(F.n)) {
            const int h = up ? 4 : 6, ntx = (F.n + 63 - 2 * h) / (64 - 2 * h), nty = (F.n + 31 - 2 * h) / (32 - 2 * h);
            const int zc = leg_chunk(F.n, ntx * nty);
            if (zc & 1) return hipErrorInvalidValue;
            const dim3 grid(ntx * nty * ((F.n + zc - 1) / zc)), block(1024);
            if (up) hipLaunchKernelGGL(k_gen_leg3<true>, grid, block, 0, s, c.g, F, Cl, ntx, nty, zc, ctl);
            else hipLaunchKernelGGL(k_gen_leg3<false>, grid, block, 0, s, c.g, F, Cl, ntx, nty, zc, ctl);
        } else if (c.g.dim == 3) {
            const int nt = (F.n + LegShape<3>::T - 1) / LegShape<3>::T;
            const dim3 grid(nt * nt * nt), block(LegShape<3>::NT);
            if (up) hipLaunchKernelGGL((k_gen_leg<3, true>), grid, block, 0, s, c.g, F, Cl, nt, ctl);
            else hipLaunchKernelGGL((k_gen_leg<3, false>), grid, block, 0, s, c.g, F, Cl, nt, ctl);
        } else {
            const int nt = (F.n + LegShape<2>::T - 1) / LegShape<2>::T;
            const dim3 grid(nt * nt), block(LegShape<2>::NT);
            if (up) hipLaunchKernelGGL((k_gen_leg<2, true>), grid, block, 0, s, c.g, F, Cl, nt, ctl);
            else hipLaunchKernelGGL((k_gen_leg<2, false>), grid, block, 0, s, c.g, F, Cl, nt, ctl);
        }
        return hipGetLastError();
    };
    for (int l = 0; l + 1 < L; ++l)
        if (hipError_t e = leg(l, false)) return e;
    const Level &B = c.lev[L - 1];
    if (c.g.dim == 3) hipLaunchKernelGGL(k_gen_exact3, dim3(1), dim3(1024), 0, s, B.r, B.out, B.n, c.exact, ctl);
    else if (hipError_t e = launch_exact2(s, B.r, B.out, B.n, c.exact, ctl)) return e;
    for (int l = L - 2; l >= 0; --l)
        if (hipError_t e = leg(l, true)) return e;
    return hipSuccess;
}

static int outer_chunk(int dim, int n) { return dim == 3 ? (n >= 128 ? 16 : 4) : (n >= 1024 ? 8 : 2); }

int outer_blocks(int dim, int n)
{
    const int zc = outer_chunk(dim, n), ntx = (n + 63) / 64, nc = (n + zc - 1) / zc;
    return dim == 3 ? ntx * ((n + 3) / 4) * nc : ntx * ((nc + 3) / 4);
}

hipError_t outer(const Ctx &c, hipStream_t s, const double *phi, const double *e, double *phi2, Ctl *ctl)
{
    const int dim = c.g.dim, n = c.g.n, zc = outer_chunk(dim, n), ntx = (n + 63) / 64, nb = outer_blocks(dim, n);
    hipLaunchKernelGGL(k_gen_outer, dim3(nb), dim3(256), 0, s, c.g, c.lev[0], phi, e, c.b, phi2, c.partials, ntx,
                       dim == 3 ? (n + 3) / 4 : 1, zc, ctl);
    hipLaunchKernelGGL(k_gen_fin_outer, dim3(1), dim3(1024), 0, s, c.partials, nb, (double)c.g.ncell, ctl);
    return hipGetLastError();
}

}  // namespace gen
}  // namespace amr
