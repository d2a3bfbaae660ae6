// Geometry kernels: cell centres, level-set hooks, normals, fluid/solid/ghost
// classification and the ghost-fluid donor records, run once per solve.
//
// All of it is integer logic and IEEE +,-,*,/,sqrt in the reference's order
// (no contraction), so flags, mirror points, donor indices and weights are bit
// identical to the reference's Src/Geometry and Scheme_Index results.
#include "ibtfo_geom.h"

namespace ibtfo {

// Psy_coord.cpp:25-35: x_i = Li + i*dx, y_j = Hi + j*dx (the reference spaces y
// with dx as well).
__device__ __forceinline__ double xc(const GeomArgs& g, int i) { return g.Li + i * g.dx; }
__device__ __forceinline__ double yc(const GeomArgs& g, int j) { return g.Hi + j * g.dx; }

__device__ double hook_phi(const GeomArgs& g, double x, double y, long long q) {
    switch (g.kind) {
        case 1: {  // Test/InclineSod/Level_Set_function.cpp:8-20, :48-51
            double k = g.p[0], nrm = g.p[1], b1 = g.p[2], b2 = g.p[3];
            double p1 = (y > k * x + b1) ? 1 * ib_fabs(k * x - y + b1) / nrm : -1 * ib_fabs(k * x - y + b1) / nrm;
            double p2 = (y > k * x + b2) ? -1 * ib_fabs(k * x - y + b2) / nrm : 1 * ib_fabs(k * x - y + b2) / nrm;
            return (p1 < p2) ? p1 : p2;
        }
        case 2: {  // Test/Vortex/Level_Set_function.cpp:31-38
            double r = ib_sqrt((x - 0.50) * (x - 0.50) + (y - 0.50) * (y - 0.50));
            double p1 = g.p[1] - r, p2 = r - g.p[0];
            return (p1 < p2) ? p1 : p2;
        }
        case 3:
            return g.phi_in[q];
        case 4: {  // ellipse body: phi > 0 outside; |phi| approximates the distance
            double cx = g.p[0], cy = g.p[1], a = g.p[2], b = g.p[3], ca = g.p[4], sa = g.p[5];
            double dxp = x - cx, dyp = y - cy;
            double xr = dxp * ca + dyp * sa, yr = -dxp * sa + dyp * ca;
            double s = ib_sqrt((xr / a) * (xr / a) + (yr / b) * (yr / b));
            // first-order distance: (s - 1) / |grad s|
            double gx = xr / (a * a), gy = yr / (b * b);
            double gn = ib_sqrt(gx * gx + gy * gy);
            return (s > 0.0 && gn > 0.0) ? (s * s - 1.0) / (2.0 * gn) : -((a < b) ? a : b);
        }
        case 5: {  // union of circles and convex polygons; exact signed distance (< 0 inside a body)
            double best = 1e300;
            for (int k = 0; k < g.nshapes; k++) {
                const double* sh = g.shapes + k * SHAPE_STRIDE;
                double d;
                if (sh[0] == 0.0) {
                    d = ib_sqrt((x - sh[1]) * (x - sh[1]) + (y - sh[2]) * (y - sh[2])) - sh[3];
                } else {
                    int nv = (int)sh[4];
                    double dmin = 1e300;
                    bool inside = true;
                    for (int e = 0; e < nv; e++) {
                        double ax = sh[5 + 2 * e], ay = sh[6 + 2 * e];
                        double bx = sh[5 + 2 * ((e + 1) % nv)], by = sh[6 + 2 * ((e + 1) % nv)];
                        double ex = bx - ax, ey = by - ay, px = x - ax, py = y - ay;
                        double t = (px * ex + py * ey) / (ex * ex + ey * ey);
                        t = t < 0.0 ? 0.0 : (t > 1.0 ? 1.0 : t);
                        double qx = px - t * ex, qy = py - t * ey;
                        double dd = qx * qx + qy * qy;
                        dmin = dd < dmin ? dd : dmin;
                        if (ex * py - ey * px < 0.0) inside = false;  // vertices counter-clockwise
                    }
                    d = inside ? -ib_sqrt(dmin) : ib_sqrt(dmin);
                }
                best = d < best ? d : best;
            }
            return best;
        }
        default:
            return 1.0;
    }
}

__global__ void k_geom_phi(GeomArgs g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= g.L.M) return;
    long long o = g.L.at(i, j);
    double x = xc(g, i), y = yc(g, j);
    g.phi[o] = hook_phi(g, x, y, (long long)j * g.L.M + i);
}

// Level_Set.cpp:71-86 (normals, ring left at 0) and :90-158 (classification in
// gather form: a solid cell is a ghost when a fluid cell lies within ng cells
// along x or y; the domain ring is ghost).
__global__ void k_geom_classify(GeomArgs g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    const Layout L = g.L;
    if (i >= L.M) return;
    const long long o = L.at(i, j);
    double nxv = 0.0, nyv = 0.0;
    if (i >= 1 && i < L.M - 1 && j >= 1 && j < L.N - 1) {
        nxv = (g.phi[L.at(i + 1, j)] - g.phi[L.at(i - 1, j)]) / ((xc(g, i + 1) - xc(g, i - 1)));
        nyv = (g.phi[L.at(i, j + 1)] - g.phi[L.at(i, j - 1)]) / ((yc(g, j + 1) - yc(g, j - 1)));
    }
    if (g.unit_normals) {  // corrected mode: unit normals (no reference counterpart)
        const double r = ib_sqrt(nxv * nxv + nyv * nyv);
        if (r > 0) { nxv = nxv / r; nyv = nyv / r; }
    }
    g.nx[o] = nxv;
    g.ny[o] = nyv;
    const int ng = L.ng;
    auto interior = [&](int ii, int jj) { return ii >= ng && ii < L.nx + ng && jj >= ng && jj < L.ny + ng; };
    uint8_t t;
    if (!interior(i, j)) t = 2;
    else if (g.phi[o] >= 0) t = 0;
    else {
        t = 1;
        for (int k = 1; k <= ng; k++) {
            const int ci[4] = {i - k, i + k, i, i};
            const int cj[4] = {j, j, j - k, j + k};
            for (int q = 0; q < 4; q++)
                if (interior(ci[q], cj[q]) && g.phi[L.at(ci[q], cj[q])] >= 0) t = 2;
        }
    }
    g.type[o] = t;
}

// Mirror_IDX.cpp:21-40: the ii in [0, M-1) with x_ii <= xm < x_{ii+1}; the same
// half-open test on the candidates around the closed-form estimate. No match
// leaves 0 (the value a zero-initialised record keeps in the reference).
__device__ int donor_idx(double v, double base, double h, int n) {
    double t = __builtin_floor((v - base) / h);
    int r = 0;
    if (!(t == t)) return 0;
    int t0 = (int)fmax(fmin(t, (double)n + 4.0), -4.0);
    for (int ii = t0 - 2; ii <= t0 + 2; ii++)
        if (ii >= 0 && ii < n - 1 && v < base + (ii + 1) * h && v >= base + ii * h) r = ii;
    return r;
}

// Lists of the interior cells that need a record (ghosts, cut cells, merge groups):
// a block lists its tile's cells in LDS, takes their slots with one atomic and
// shares the records among its threads. An atomic per wave on the one counter was
// what bounded these passes: on the 2048x1024 bodies grid 51 us a pass over the
// ghosts, 82 over the cut cells; now 8 and 29.
constexpr int TILE_X = 64, TILE_Y = 32, TILE_THREADS = 256;
struct TileList {
    int n;
    unsigned int base;
    unsigned short cell[TILE_X * TILE_Y];
};
__device__ __forceinline__ void tile_cell(const Layout& L, int k, int& i, int& j) {
    i = L.ng + blockIdx.x * TILE_X + k % TILE_X;
    j = L.ng + blockIdx.y * TILE_Y + k / TILE_X;
}
template <class F> __device__ __forceinline__ void tile_each(const Layout& L, F f) {
    for (int k = threadIdx.x; k < TILE_X * TILE_Y; k += TILE_THREADS) {
        int i, j;
        tile_cell(L, k, i, j);
        if (i < L.nx + L.ng && j < L.ny + L.ng) f(k, i, j);
    }
}
__device__ __forceinline__ void tile_push(TileList& l, int k) { l.cell[atomicAdd(&l.n, 1)] = (unsigned short)k; }
__device__ __forceinline__ void tile_claim(TileList& l, unsigned int* count) {  // one thread
    if (l.n) l.base = atomicAdd(count, (unsigned)l.n);
}
static dim3 tile_grid(const Layout& L) { return dim3((L.nx + TILE_X - 1) / TILE_X, (L.ny + TILE_Y - 1) / TILE_Y); }

__device__ void ghost_record(const GeomArgs& g, int i, int j, unsigned int slot);
__global__ __launch_bounds__(TILE_THREADS) void k_geom_ghosts(GeomArgs g) {
    __shared__ TileList l;
    if (threadIdx.x == 0) l.n = 0;
    __syncthreads();
    tile_each(g.L, [&](int k, int i, int j) {
        if (g.type[g.L.at(i, j)] == 2) tile_push(l, k);
    });
    __syncthreads();
    if (threadIdx.x == 0) tile_claim(l, g.count);
    if (g.cap == 0) return;  // counting only
    __syncthreads();
    for (int q = threadIdx.x; q < l.n; q += TILE_THREADS) {
        int i, j;
        tile_cell(g.L, l.cell[q], i, j);
        if (l.base + q < (unsigned)g.cap) ghost_record(g, i, j, l.base + q);
    }
}

// Scheme_Index for one ghost: IDWBaseGFM/GFM_Method.cpp:20-110,
// LinearBaseGFM/GFM_Method.cpp:19-44 + GFM_Bound.cpp:93-575 (donor choice),
// BCGFM/BCGFM_Method.cpp:49-205, HBCGFM/HBCGFM_Method.cpp:56-91.
__device__ void ghost_record(const GeomArgs& g, int i, int j, unsigned int slot) {
    const Layout L = g.L;
    const int ng = L.ng;
    const long long o = L.at(i, j);
    Ghost gh;
    gh.cell = o;
    gh.nx = g.nx[o];
    gh.ny = g.ny[o];
    double ph = ib_fabs(g.phi[o]);
    gh.phi = ph;
    double x = xc(g, i), y = yc(g, j);
    const int bc = g.bc;
    double dxg = xc(g, 1) - xc(g, 0), dyg = yc(g, 2) - yc(g, 1);
    if (bc == IBTFO_SIMPLE_BOUND) {
        // SimpleBound/Scheme_Index.cpp:12-66: the nearest fluid cell within ng
        // along -x (else +x) and -y (else +y); k cells away -> donor offset 1 - 2k
        // (2k - 1). Dependencies on earlier-filled ghosts are resolved on the host.
        auto t = [&](int ii, int jj) { return g.type[L.at(ii, jj)]; };
        int IDX = 0, IDY = 0;
        for (int k = 0; k < ng + 1; k++)
            if (t(i - k, j) < 1) { IDX = 1 - 2 * k; break; }
        if (IDX == 0)
            for (int k = 0; k < ng + 1; k++)
                if (t(i + k, j) < 1) { IDX = 2 * k - 1; break; }
        for (int k = 0; k < ng + 1; k++)
            if (t(i, j - k) < 1) { IDY = 1 - 2 * k; break; }
        if (IDY == 0)
            for (int k = 0; k < ng + 1; k++)
                if (t(i, j + k) < 1) { IDY = 2 * k - 1; break; }
        auto ring_cell = [&](int ii, int jj) { return ii < ng || ii >= L.nx + ng || jj < ng || jj >= L.ny + ng; };
        gh.idx = IDX; gh.idy = IDY;
        gh.d1 = L.at(i + IDX, j);
        gh.d1e = L.at(i, j + IDY);
        gh.idxe = gh.idye = -1;
        gh.pick = 0;
        gh.ring = (ring_cell(i + IDX, j) ? 1 : 0) | (ring_cell(i, j + IDY) ? 16 : 0);
        gh.xm = gh.ym = gh.xe = gh.ye = 0.0;
        for (int q = 0; q < 4; q++) { gh.a[q] = 0.0; gh.ae[q] = 0.0; }
        g.ghosts[slot] = gh;
        return;
    }
    if (bc == 1 || bc == 2 || bc == 3) {
        gh.xm = x + 2 * gh.nx * ph;
        gh.ym = y + 2 * gh.ny * ph;
        gh.xe = gh.ye = 0.0;
    } else {
        double delta = ib_sqrt(dxg * dxg + dyg * dyg) / 2;
        if (bc == 5 && ph > delta) {
            gh.xm = x + gh.nx * (2 * ph); gh.ym = y + gh.ny * (2 * ph);
            gh.xe = x + gh.nx * (2 * ph); gh.ye = y + gh.ny * (2 * ph);
        } else {
            gh.xm = x + gh.nx * (ph + delta); gh.ym = y + gh.ny * (ph + delta);
            gh.xe = x + gh.nx * (ph + 2.0 * delta); gh.ye = y + gh.ny * (ph + 2.0 * delta);
        }
    }
    gh.idx = donor_idx(gh.xm, g.Li, g.dx, L.M);
    gh.idy = donor_idx(gh.ym, g.Hi, g.dx, L.N);
    gh.d1 = L.at(gh.idx, gh.idy);
    const int di[4] = {0, 0, 1, 1}, dj[4] = {0, 1, 1, 0};
    for (int q = 0; q < 4; q++) { gh.a[q] = 0.0; gh.ae[q] = 0.0; }
    gh.idxe = gh.idye = 0;
    gh.d1e = gh.d1;
    if (bc == 1 || bc >= 4) {
        for (int q = 0; q < 4; q++) {
            int ii = gh.idx + di[q], jj = gh.idy + dj[q];
            uint8_t t = g.type[L.at(ii, jj)];
            bool keep = (bc == 1) ? (g.cut ? (t == 0 || t == 3) : (t < 1)) : (t != 1);
            if (keep) {
                double ddx = xc(g, ii) - gh.xm, ddy = yc(g, jj) - gh.ym;
                gh.a[q] = 1 / ib_sqrt(ddx * ddx + ddy * ddy);
            }
        }
    }
    if (bc >= 4) {
        gh.idxe = donor_idx(gh.xe, g.Li, g.dx, L.M);
        gh.idye = donor_idx(gh.ye, g.Hi, g.dx, L.N);
        gh.d1e = L.at(gh.idxe, gh.idye);
        for (int q = 0; q < 4; q++) {
            int ii = gh.idxe + di[q], jj = gh.idye + dj[q];
            if (g.type[L.at(ii, jj)] != 1) {
                double ddx = xc(g, ii) - gh.xe, ddy = yc(g, jj) - gh.ye;
                gh.ae[q] = 1 / ib_sqrt(ddx * ddx + ddy * ddy);
            }
        }
    }
    gh.ring = 0;
    // the ring's type is 2 as well, so the type decides both cases
    auto from_prev = [&](int ii, int jj) {
        const uint8_t t = g.type[L.at(ii, jj)];
        return t != 0 && !(g.cut && t == 3);
    };
    for (int q = 0; q < 4; q++) {
        if (from_prev(gh.idx + di[q], gh.idy + dj[q])) gh.ring |= 1 << q;
        if (bc >= 4 && from_prev(gh.idxe + di[q], gh.idye + dj[q])) gh.ring |= 1 << (4 + q);
    }
    gh.pick = -1;
    if (bc == 2 || bc == 3) {
        bool f[4];
        for (int q = 0; q < 4; q++) f[q] = g.type[L.at(gh.idx + di[q], gh.idy + dj[q])] < 1;
        bool f1 = f[0], f2 = f[1], f3 = f[2], f4 = f[3];
        double x_d = gh.xm - xc(g, gh.idx);
        double y_d = gh.xm - xc(g, gh.idx);  // the reference measures y_d with the x mirror too
        bool xr = x_d > dxg / 2, yu = y_d > dyg / 2;
        int pick = -1;
        if (f1 && f4 && f2 && f3) pick = yu ? (xr ? 2 : 1) : (xr ? 3 : 0);
        else if (!f1 && f4 && f2 && f3) pick = yu ? (xr ? 2 : 1) : 3;
        else if (f1 && !f4 && f2 && f3) pick = yu ? (xr ? 2 : 1) : 0;
        else if (f1 && f4 && !f2 && f3) pick = yu ? 2 : (xr ? 3 : 0);
        else if (f1 && f4 && f2 && !f3) pick = yu ? 1 : (xr ? 3 : 0);
        else if (f1 && f4 && !f2 && !f3) pick = xr ? 3 : 0;
        else if (!f1 && !f4 && f2 && f3) pick = xr ? 2 : 1;
        else if (f1 && !f4 && f2 && !f3) pick = yu ? 1 : 0;
        else if (!f1 && f4 && !f2 && f3) pick = yu ? 2 : 3;
        else if (f1 && !f4 && !f2 && f3) pick = yu ? 2 : 0;
        else if (!f1 && f4 && f2 && !f3) pick = yu ? 1 : 3;
        else if (f1 && !f4 && !f2 && !f3) pick = 0;
        else if (!f1 && !f4 && f2 && !f3) pick = 1;
        else if (!f1 && !f4 && !f2 && f3) pick = 2;
        else if (!f1 && f4 && !f2 && !f3) pick = 3;
        gh.pick = pick;
        gh.a[0] = pick;
    }
    g.ghosts[slot] = gh;
}

hipError_t geom_run(GeomArgs& g, hipStream_t s) {
    dim3 blk(128), grd((g.L.M + 127) / 128, g.L.N);
    if (g.kind != IBTFO_LS_FIELD || g.phi_in) hipLaunchKernelGGL(k_geom_phi, grd, blk, 0, s, g);
    hipLaunchKernelGGL(k_geom_classify, grd, blk, 0, s, g);
    return hipGetLastError();
}
hipError_t geom_ghosts(GeomArgs& g, hipStream_t s) {
    hipLaunchKernelGGL(k_geom_ghosts, tile_grid(g.L), dim3(TILE_THREADS), 0, s, g);
    return hipGetLastError();
}



// ------------------------------------------------------------ cut cells
// No reference counterpart. From the cell-centred phi: corner values are the
// means of the four surrounding cells' phi, a face's aperture is its fluid
// fraction under linear interpolation between its corners, the volume fraction
// is the area of the fluid polygon those crossings cut from the cell, and the
// wall vector S = -((aE - aW) dy, (aN - aS) dx) closes the faces.
__device__ __forceinline__ double cut_frac(double p, double q) {
    if (p >= 0 && q >= 0) return 1.0;
    if (p < 0 && q < 0) return 0.0;
    return p >= 0 ? p / (p - q) : q / (q - p);
}
__device__ __forceinline__ double corner_phi(const GeomArgs& g, int i, int j) {  // corner (i+1/2, j+1/2)
    const Layout& L = g.L;
    return 0.25 * (((g.phi[L.at(i, j)] + g.phi[L.at(i + 1, j)]) + g.phi[L.at(i, j + 1)]) + g.phi[L.at(i + 1, j + 1)]);
}
// Volume fraction and face apertures of an interior cell: a function of phi alone,
// so the passes below evaluate it again where they need it (cut cells are few).
// Records of all cells kept between the passes were 135 MB on a 2048x1024 grid,
// written once and read four times: a set-up took 1.97 ms with them, 1.30 without.
struct CutShape { double alpha, a[4]; };  // apertures W, E, S, N
__device__ __forceinline__ CutShape cut_shape(const GeomArgs& g, int i, int j) {
    const double sw = corner_phi(g, i - 1, j - 1), se = corner_phi(g, i, j - 1), ne = corner_phi(g, i, j),
                 nw = corner_phi(g, i - 1, j);
    CutShape c;
    c.a[0] = cut_frac(sw, nw); c.a[1] = cut_frac(se, ne); c.a[2] = cut_frac(sw, se); c.a[3] = cut_frac(nw, ne);
    if (sw >= 0 && se >= 0 && ne >= 0 && nw >= 0) c.alpha = 1.0;
    else if (sw < 0 && se < 0 && ne < 0 && nw < 0) c.alpha = 0.0;
    else {
        const double cx[4] = {0, 1, 1, 0}, cy[4] = {0, 0, 1, 1}, cv[4] = {sw, se, ne, nw};
        double px[8], py[8];
        int n = 0;
        for (int e = 0; e < 4; e++) {
            const int f = (e + 1) % 4;
            if (cv[e] >= 0) { px[n] = cx[e]; py[n] = cy[e]; n++; }
            if ((cv[e] >= 0) != (cv[f] >= 0)) {
                const double t = cv[e] / (cv[e] - cv[f]);
                px[n] = cx[e] + t * (cx[f] - cx[e]);
                py[n] = cy[e] + t * (cy[f] - cy[e]);
                n++;
            }
        }
        double a2 = 0.0;
        for (int k = 0; k < n; k++) {
            const int l = (k + 1) % n;
            a2 += px[k] * py[l] - px[l] * py[k];
        }
        c.alpha = 0.5 * a2;
    }
    return c;
}

// A cell's mark: which neighbour it merges into (0 none, 1-4 W, E, S, N), and
// whether one of its apertures is zero
constexpr uint8_t CUT_INTO = 7, CUT_ZERO_FACE = 8;

__global__ void k_cut_cells(GeomArgs g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    const Layout L = g.L;
    if (i >= L.M) return;
    const long long o = L.at(i, j);
    g.cmark[o] = 0;
    const int ng = L.ng;
    if (i < ng || i >= L.nx + ng || j < ng || j >= L.ny + ng) { g.type[o] = 2; return; }
    const CutShape c = cut_shape(g, i, j);
    if (c.a[0] == 0.0 || c.a[1] == 0.0 || c.a[2] == 0.0 || c.a[3] == 0.0) g.cmark[o] = CUT_ZERO_FACE;
    g.type[o] = c.alpha >= 1.0 ? 0 : (c.alpha > 0.0 ? 3 : 1);
}

// A cut cell with alpha < 1/2 picks a neighbour with alpha >= 1/2: along the
// normal's dominant axis first, then the other axis, then the opposite
// directions; without one it becomes inactive.
__global__ void k_cut_target(GeomArgs g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    const Layout L = g.L;
    const int ng = L.ng;
    if (i < ng || i >= L.nx + ng || j < ng || j >= L.ny + ng) return;
    const long long o = L.at(i, j);
    if (g.type[o] != 3 || cut_shape(g, i, j).alpha >= 0.5) return;
    const double n_x = g.nx[o], n_y = g.ny[o];
    const int sx = n_x >= 0 ? 1 : -1, sy = n_y >= 0 ? 1 : -1;
    int ci[4], cj[4];
    if (ib_fabs(n_x) >= ib_fabs(n_y)) {
        ci[0] = i + sx; cj[0] = j; ci[1] = i; cj[1] = j + sy; ci[2] = i - sx; cj[2] = j; ci[3] = i; cj[3] = j - sy;
    } else {
        ci[0] = i; cj[0] = j + sy; ci[1] = i + sx; cj[1] = j; ci[2] = i; cj[2] = j - sy; ci[3] = i - sx; cj[3] = j;
    }
    for (int q = 0; q < 4; q++) {
        if (ci[q] < ng || ci[q] >= L.nx + ng || cj[q] < ng || cj[q] >= L.ny + ng) continue;
        // a neighbour that another thread makes inactive has alpha < 1/2 either way
        const uint8_t tq = g.type[L.at(ci[q], cj[q])];
        if (tq == 0 || (tq == 3 && cut_shape(g, ci[q], cj[q]).alpha >= 0.5)) {
            g.cmark[o] |= ci[q] < i ? 1 : ci[q] > i ? 2 : cj[q] < j ? 3 : 4;
            return;
        }
    }
    g.type[o] = 1;  // no partner: inactive
}

// inactive cells within ng of an active cell along an axis are ghosts
__global__ void k_cut_ghosts(GeomArgs g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    const Layout L = g.L;
    const int ng = L.ng;
    if (i < ng || i >= L.nx + ng || j < ng || j >= L.ny + ng) return;
    const long long o = L.at(i, j);
    if (g.type[o] != 1) return;
    for (int k = 1; k <= ng; k++) {
        const int ci[4] = {i - k, i + k, i, i}, cj[4] = {j, j, j - k, j + k};
        for (int q = 0; q < 4; q++) {
            if (ci[q] < ng || ci[q] >= L.nx + ng || cj[q] < ng || cj[q] >= L.ny + ng) continue;
            const uint8_t tq = g.type[L.at(ci[q], cj[q])];
            if (tq == 0 || tq == 3) { g.type[o] = 2; return; }
        }
    }
}

// Records of the cut cells and merge groups gathered by each target from its W, E,
// S, N neighbours; run twice, counting them first. A face between an active cell
// and an inactive interior one (zero-area polygons where corners are exactly 0,
// small cells without a partner) is a wall: its aperture becomes 0 and the wall
// vector closes the faces again, so no flux leaves the fluid through it. A full
// cell with a zero aperture takes the cut-cell update: type 3 with alpha = 1 (set by
// the counting pass; its neighbours take types 0 and 3 alike). The filling pass also
// marks the groups' cells in the step kernel's type plane.
struct CutFaces {
    bool cut;      // the cell takes the cut-cell update
    int members;   // neighbours that merge into it: bits W, E, S, N
    int walls;     // inactive interior neighbours: bits W, E, S, N
};
__device__ __forceinline__ void cut_neighbour(int q, int& i, int& j) {
    i += q == 0 ? -1 : q == 1 ? 1 : 0;
    j += q == 2 ? -1 : q == 3 ? 1 : 0;
}
__device__ __forceinline__ CutFaces cut_faces(const GeomArgs& g, int i, int j) {
    const Layout& L = g.L;
    const int ng = L.ng;
    CutFaces c = {false, 0, 0};
    const long long o = L.at(i, j);
    const uint8_t t = g.type[o];
    if (t != 0 && t != 3) return c;
    for (int q = 0; q < 4; q++) {
        int ni = i, nj = j;
        cut_neighbour(q, ni, nj);
        if (ni < ng || ni >= L.nx + ng || nj < ng || nj >= L.ny + ng) continue;
        const long long nq = L.at(ni, nj);
        const uint8_t tq = g.type[nq];
        const int into = g.cmark[nq] & CUT_INTO;
        if (tq != 0 && tq != 3) c.walls |= 1 << q;
        else if (into == (q ^ 1) + 1) c.members |= 1 << q;  // the opposite direction's mark
    }
    c.cut = t == 3 || c.walls || (g.cmark[o] & CUT_ZERO_FACE);
    return c;
}

__global__ __launch_bounds__(TILE_THREADS) void k_cut_records(GeomArgs g) {
    __shared__ TileList cuts, groups;
    const Layout& L = g.L;
    const bool fill = g.cuts != nullptr;
    if (threadIdx.x == 0) cuts.n = groups.n = 0;
    __syncthreads();
    tile_each(L, [&](int k, int i, int j) {
        const CutFaces c = cut_faces(g, i, j);
        if (c.cut) tile_push(cuts, k);
        if (c.members) tile_push(groups, k);
    });
    __syncthreads();
    if (threadIdx.x == 0) {
        tile_claim(cuts, &g.ccount[0]);
        tile_claim(groups, &g.ccount[1]);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < cuts.n; q += TILE_THREADS) {
        int i, j;
        tile_cell(L, cuts.cell[q], i, j);
        const long long o = L.at(i, j);
        if (!fill) {
            g.type[o] = 3;
            continue;
        }
        const unsigned int slot = cuts.base + q;
        if (slot >= (unsigned int)g.ccap) continue;
        CutShape c = cut_shape(g, i, j);
        const int walls = cut_faces(g, i, j).walls, into = g.cmark[o] & CUT_INTO;
        for (int f = 0; f < 4; f++)
            if (walls >> f & 1) c.a[f] = 0.0;
        CutCell r;
        r.alpha = c.alpha; r.aw = c.a[0]; r.ae = c.a[1]; r.as = c.a[2]; r.an = c.a[3];
        r.sbx = -((r.ae - r.aw) * g.cdy);
        r.sby = -((r.an - r.as) * g.cdx);
        r.target = -1;
        if (into) {
            cut_neighbour(into - 1, i, j);
            r.target = L.at(i, j);
            g.stype[o] = 3 | MERGED_BIT;
        }
        g.cuts[slot] = r;
        g.cut_index[o] = (int)slot;
    }
    if (!fill) return;
    for (int q = threadIdx.x; q < groups.n; q += TILE_THREADS) {
        int i, j;
        tile_cell(L, groups.cell[q], i, j);
        const unsigned int slot = groups.base + q;
        if (slot >= (unsigned int)g.gcap) continue;
        const long long o = L.at(i, j);
        const int members = cut_faces(g, i, j).members;
        MergeGroup& gr = g.groups[slot];
        int n = 0;
        gr.pad = 0;
        gr.target = o;
        gr.at = cut_shape(g, i, j).alpha;
        for (int f = 0; f < 4; f++) {
            if (!(members >> f & 1)) continue;
            int ni = i, nj = j;
            cut_neighbour(f, ni, nj);
            gr.member[n] = L.at(ni, nj);
            gr.am[n] = cut_shape(g, ni, nj).alpha;
            n++;
        }
        gr.n = n;
        for (; n < 4; n++) {
            gr.member[n] = o;
            gr.am[n] = 0.0;
        }
        g.stype[o] = g.type[o] | MERGED_BIT;
    }
}

hipError_t cut_run(GeomArgs& g, hipStream_t s) {
    dim3 blk(128), grd((g.L.M + 127) / 128, g.L.N);
    hipLaunchKernelGGL(k_cut_cells, grd, blk, 0, s, g);
    hipLaunchKernelGGL(k_cut_target, grd, blk, 0, s, g);
    hipLaunchKernelGGL(k_cut_ghosts, grd, blk, 0, s, g);
    return hipGetLastError();
}
hipError_t cut_records(GeomArgs& g, hipStream_t s) {
    hipLaunchKernelGGL(k_cut_records, tile_grid(g.L), dim3(TILE_THREADS), 0, s, g);
    return hipGetLastError();
}

// ------------------------------------------------------------ mask level set
// Test/PNGGeo/Level_Set.cpp:31-149 on the device. The reference computes, for
// every cell, the distance to every edge pixel (O(cells x edges)); here the
// nearest edge pixel is found by a separable exact search (per pixel column the
// nearest edge row to each cell row, then per cell row the least of the parabolas
// (x_q - x_e)^2 + g(x_e) over pixel columns), and the distance to that pixel is
// evaluated with the reference's expression.

// Level_Set.cpp:36-48: a pixel's sign, +1 where R + G + B > 0 (here as a bool), else
// -1; image rows flipped so that row 0 is the bottom of the domain
__device__ __forceinline__ bool mask_sign(const MaskArgs& m, int x, int y) {
    return (m.rgba[(long long)(m.H - y - 1) * m.W + x] & 0xffffffu) != 0;  // the fourth byte is alpha
}
__device__ __forceinline__ double edge_x(const MaskArgs& m, int x) { return m.exo + m.dxp * x; }
__device__ __forceinline__ double edge_y(const MaskArgs& m, int y) { return m.eyo + m.dyp * y; }

// Level_Set.cpp:51-76: edge pixel where max(|v - v_left|, |v - v_below|) > 0.1 (signs
// that differ), pixels 1..W-2 x 1..H-2 only: one bit each, a word per 32 rows of a
// column. With the next pass and the row search's share 39 us for a 2052x1028 mask;
// planes of signs, edge bytes and column distances took 95.
__global__ void k_mask_edges(MaskArgs m) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, sg = blockIdx.y;
    if (x >= m.W) return;
    unsigned w = 0;
    if (x >= 1 && x < m.W - 1) {
        const int y0 = max(sg * MASK_SEG, 1), y1 = min((sg + 1) * MASK_SEG, m.H - 1);
        bool below = y0 < y1 && mask_sign(m, x, y0 - 1);
#pragma unroll 8
        for (int y = y0; y < y1; y++) {
            const bool c = mask_sign(m, x, y);
            if (c != below || c != mask_sign(m, x - 1, y)) w |= 1u << (y % MASK_SEG);
            below = c;
        }
    }
    m.bits[(long long)sg * m.W + x] = w;
}

// Per word: the column's last edge row below its rows and the first above them.
__global__ void k_mask_beyond(MaskArgs m) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, sg = blockIdx.y;
    if (x >= m.W) return;
    int b = -1, a = -1;
    for (int s = sg - 1; s >= 0 && b < 0; s--) {
        const unsigned w = m.bits[(long long)s * m.W + x];
        if (w) b = s * MASK_SEG + 31 - __clz((int)w);
    }
    for (int s = sg + 1; s < m.nseg && a < 0; s++) {
        const unsigned w = m.bits[(long long)s * m.W + x];
        if (w) a = s * MASK_SEG + __ffs((int)w) - 1;
    }
    m.before[(long long)sg * m.W + x] = b;
    m.after[(long long)sg * m.W + x] = a;
}

// The last pixel row whose edge height is <= yq (-1: none); the heights increase
// with the row, so a rounded estimate is corrected by single steps.
__device__ __forceinline__ int row_below(const MaskArgs& m, double yq) {
    int y0 = (int)floor((yq - m.eyo) / m.dyp);
    y0 = min(max(y0, -1), m.H - 1);
    while (y0 >= 0 && edge_y(m, y0) > yq) y0--;
    while (y0 + 1 < m.H && edge_y(m, y0 + 1) <= yq) y0++;
    return y0;
}
// Column x: the squared height difference of yq and the nearer of its edge rows just
// below and just above (infinite without an edge). In rounded arithmetic too no other
// edge of the column is nearer: the squares grow with the distance.
__device__ __forceinline__ double column_g(const MaskArgs& m, int x, int y0, double yq) {
    double best = HUGE_VAL;
    if (y0 >= 0) {
        const long long o = (long long)(y0 / MASK_SEG) * m.W + x;
        const unsigned w = m.bits[o] & (~0u >> (MASK_SEG - 1 - y0 % MASK_SEG));
        const int e = w ? y0 / MASK_SEG * MASK_SEG + 31 - __clz((int)w) : m.before[o];
        const double d = edge_y(m, e) - yq;
        if (e >= 0) best = d * d;
    }
    if (y0 + 1 < m.H) {
        const int y1 = y0 + 1;
        const long long o = (long long)(y1 / MASK_SEG) * m.W + x;
        const unsigned w = m.bits[o] & (~0u << (y1 % MASK_SEG));
        const int e = w ? y1 / MASK_SEG * MASK_SEG + __ffs((int)w) - 1 : m.after[o];
        const double d = edge_y(m, e) - yq;
        if (e >= 0 && d * d < best) best = d * d;
    }
    return best;
}

// Per cell row j: phi of its cells, +- the distance to the nearest edge pixel, which
// is the root of the least (x_e - X)^2 + g over the pixel columns that hold an edge
// (the root is monotone, so it is taken once, of the least radicand; every radicand
// is rounded as the reference rounds it). The columns whose parabola is least move
// to the right with X: f_a - f_b of two columns is linear in X. So the row is cut
// into intervals of `stride` cells; the least column is found between intervals (a
// wave per point, its lanes over all columns), and each cell of an interval then
// scans only the columns between its ends' (a lane per cell, all lanes the same
// column): n + W*nq/64 steps of a wave for the row, whatever the shape. The points
// lie half a cell from any cell, which makes the bound hold in rounded arithmetic:
// at a cell, a column outside it is worse by at least a column spacing times a cell
// size, the domain squared over W*M, against rounding of some 1e-16 of it.
// A serial lower envelope (one lane per row, a division per column) took 1.49 ms for
// a 2052x1028 mask; this takes 0.084, bound by the scans' LDS latency (0.147 with 256
// threads a block and no unrolling: LDS holds four blocks on a CU, and 1028 of them
// then leave a second round nearly empty; 0.088 with 1024 threads).
constexpr int EDT_THREADS = 512;
template <bool LDS> __global__ __launch_bounds__(EDT_THREADS) void k_edt_rows(MaskArgs m, int stride, int nq) {
    extern __shared__ double lds[];
    __shared__ int wsum[EDT_THREADS / 64];
    const int j = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6, W = m.W;
    const double yq = m.Hi + j * m.dxc;
    const int y0 = row_below(m, yq);
    double* ps = lds;                               // LDS: positions and g of the columns with an edge
    double* gs = ps + W;
    int* arg = (int*)(LDS ? (void*)(gs + W) : (void*)lds);  // nq + 1 bounds
    int n = W;
    if (LDS) {  // compacted in order
        n = 0;
        for (int x0 = 0; x0 < W; x0 += EDT_THREADS) {
            const int x = x0 + threadIdx.x;
            const double f = x < W ? column_g(m, x, y0, yq) : HUGE_VAL;
            const bool has = f < HUGE_VAL;
            const unsigned long long b = __ballot(has);
            if (lane == 0) wsum[wv] = __popcll(b);
            __syncthreads();
            int at = n;
            for (int u = 0; u < EDT_THREADS / 64; u++) {
                if (u < wv) at += wsum[u];
                n += wsum[u];
            }
            at += __popcll(b & ((1ull << lane) - 1));
            if (has) {
                ps[at] = edge_x(m, x);
                gs[at] = f;
            }
            __syncthreads();
        }
    }
    auto radicand = [&](int x, double X) {
        const double d = (LDS ? ps[x] : edge_x(m, x)) - X;
        return d * d + (LDS ? gs[x] : column_g(m, x, y0, yq));
    };
    if (threadIdx.x == 0) {
        arg[0] = 0;
        arg[nq] = n - 1;
    }
    for (int q = 1 + wv; q < nq; q += EDT_THREADS / 64) {
        const double X = m.Li + ((double)((long long)q * stride) - 0.5) * m.dxc;
        double best = HUGE_VAL;
        int at = 0;
#pragma unroll 8
        for (int x = lane; x < n; x += 64) {
            const double v = radicand(x, X);
            if (v < best) { best = v; at = x; }
        }
        for (int o = 32; o > 0; o >>= 1) {
            const double v = __shfl_xor(best, o, 64);
            const int a = __shfl_xor(at, o, 64);
            if (v < best || (v == best && a < at)) { best = v; at = a; }
        }
        if (lane == 0) arg[q] = at;
    }
    __syncthreads();
    const int ys = (int)((j + 0.5) * (m.H) / (m.N));
    for (int q = wv; q < nq; q += EDT_THREADS / 64) {
        const int lo = arg[q], hi = min(arg[q + 1], n - 1);  // none without an edge
        const int iend = min((q + 1) * stride, m.M);
        for (int i = q * stride + lane; i < iend; i += 64) {
            const double X = m.Li + i * m.dxc;
            double best = HUGE_VAL;
#pragma unroll 8
            for (int x = lo; x <= hi; x++) {
                const double v = radicand(x, X);
                best = v < best ? v : best;
            }
            const double d = ib_sqrt(best);
            const double dmin = d < 100.0 ? d : 100.0;  // Level_Set.cpp:131 starts every search at 100
            // the sign sampled at pixel (int((i+0.5) W / M), int((j+0.5) H / N))
            const int xs = (int)((i + 0.5) * (W) / (m.M));
            m.phi[m.L.at(i, j)] = (mask_sign(m, xs, ys) ? 1 : -1) * dmin;
        }
    }
}

hipError_t mask_run(MaskArgs& m, bool lds, hipStream_t s) {
    const dim3 cols((m.W + 255) / 256, m.nseg);
    hipLaunchKernelGGL(k_mask_edges, cols, dim3(256), 0, s, m);
    hipLaunchKernelGGL(k_mask_beyond, cols, dim3(256), 0, s, m);
    const int stride = edt_stride(m.M), nq = edt_intervals(m.M);
    if (lds) {
        hipLaunchKernelGGL(k_edt_rows<true>, dim3(m.N), dim3(EDT_THREADS), mask_lds_bytes(m.W, m.M), s, m, stride, nq);
    } else {
        hipLaunchKernelGGL(k_edt_rows<false>, dim3(m.N), dim3(EDT_THREADS), (nq + 1) * sizeof(int), s, m, stride, nq);
    }
    return hipGetLastError();
}
const void* mask_rows_kernel() { return (const void*)k_edt_rows<true>; }

}  // namespace ibtfo
