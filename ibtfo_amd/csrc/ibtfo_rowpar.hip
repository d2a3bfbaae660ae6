// Row-parallel step kernel (k_step_rowpar): the small-grid form of the step
// kernel, each row of a strip on its own wave. It lives in a translation unit
// of its own: compiled beside the marching strip kernels, its instantiations
// changed their register allocation (mixed-precision variants from 124 to 131
// VGPRs, four waves per SIMD to three).
#include "ibtfo_internal.h"
#include "ibtfo_face.h"

namespace ibtfo {

// The update of cell (c, j), of type tc, from its face fluxes (F, G on its upper
// x / y faces; fm_lds[k * 64], gm_lds[k * 64] on its lower faces, in the LDS slots
// of the lanes that computed them): the conservative or cut-cell update, floors,
// dt/mass partial terms, the RK2 stage average (with U^n in uo), the store and the
// fused Global_Boundary ring writes. The same statements as the update inside
// step_strip, which keeps its own inline copy (LDS slots for the cell and the
// fluxes); the row-parallel tests hold the two equal, comparing the two kernels'
// states bit for bit over every scheme, flux, boundary and stage.
template <int SCH, int RS, int LIM, typename T, bool CUT>
__device__ __forceinline__ void update_cell(const StepArgs& a, const Layout& L, const int c, const int j,
                                            const uint8_t tc, const double (&u0)[4], const double (&uo)[4],
                                            const T (&F)[4], const T (&G)[4], const T* fm_lds, const T* gm_lds,
                                            const double dt, const int quirks, const Rcp<double>& r_dx,
                                            const Rcp<double>& r_dy, const Rcp<double>& r_gm1, const double dtdx,
                                            const double dtdy, double* __restrict__ Uo, const int stage,
                                            double& amax, double& umax, double& vmax, double& msum, int& bad) {
    constexpr bool FP64 = sizeof(T) == sizeof(double);
    const long long PL = L.plane;
    const double dx = a.dx, dy = a.dy;
    const int ng = L.ng, nx = L.nx, ny = L.ny;
    const long long o = L.at(c, j);
    const bool fluid = CUT ? (tc & 3) == 0 : tc == 0;
    const bool merged = CUT && (tc & MERGED_BIT);
    bool floors = fluid;
    double vol = 1.0;
    double un[4] = {u0[0], u0[1], u0[2], u0[3]};
    if (fluid) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double dF = (double)F[k] - (double)fm_lds[k * 64];
            const double dG = (double)G[k] - (double)gm_lds[k * 64];
            // FP64, or FP32 fluxes with FP64 accumulation
            if (FP64) un[k] = (u0[k] - dq(dt * dF, r_dx)) - dq(dt * dG, r_dy);
            else un[k] = u0[k] - dtdx * dF - dtdy * dG;
        }
    } else if (CUT && (tc & 3) == 3) {
        // cut cell: aperture-weighted face fluxes and the wall's pressure
        // force S p (S closes the cell's faces), over the fluid volume
        // alpha dx dy; small cells are merged (and floored) afterwards
        const CutCell cc = a.cut[a.cut_index[o]];
        const PState<double> s0 = pstate(a.gm1, u0);
        const double wall[4] = {0.0, s0.p * cc.sbx, s0.p * cc.sby, 0.0};
        const Rcp<double> rv = rcp_of(cc.alpha * dx * dy);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double Fk = (double)F[k], Fm = (double)fm_lds[k * 64];
            const double Gk = (double)G[k], Gm = (double)gm_lds[k * 64];
            const double v = u0[k] - dq(dt * ((cc.ae * Fk - cc.aw * Fm) * dy), rv);
            un[k] = v - dq(dt * ((cc.an * Gk - cc.as * Gm) * dx + wall[k]), rv);
        }
        // a merge-group cell (small cell or target) takes its floors and
        // partials from the merge; the others are floored and counted here
        floors = !merged || cc.alpha >= 0.5;
        vol = cc.alpha;
    }
    if (floors) {
        double am = 0.0, um = 0.0, vm = 0.0;
        int nb = 0;
        floor_and_dt(a.gam, a.gm1, r_gm1, un, quirks, am, um, vm, nb);
        if (stage >= 2) {
            // RK2 (Heun): each stage's update takes the floors; the second stage
            // then averages with U^n, which the output buffer holds
#pragma unroll
            for (int k = 0; k < 4; k++) un[k] = 0.5 * (uo[k] + un[k]);
            am = um = vm = 0.0;
            nb = 0;
            dt_terms(a.gam, a.gm1, un, am, um, vm, nb);
        }
        if (!merged) {
            amax = am;
            umax = um;
            vmax = vm;
            bad = nb;
            msum = fluid ? un[0] * dx * dy : vol * un[0] * dx * dy;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) Uo[o + k * PL] = un[k];
    if (a.edge_fused == 2) periodic_images(Uo, L, c, j, un);
    if (a.edge_fused == 1) {
        // Test/Sod/Global_Boudary.cpp:24-59 (rows) and :62-75 (columns), which
        // read U_NEW: the updated state, or for a non-fluid cell under
        // SimpleBound the value its U_NEW kept
        double e[4] = {un[0], un[1], un[2], un[3]};
        if (a.unew_nf && !fluid)
            for (int k = 0; k < 4; k++) e[k] = a.unew_nf[o + k * PL];
        if (j < 2 * ng) Uo[L.at(c, 2 * ng - 1 - j) + 2 * PL] = -e[2];
        if (j == 2 * ng - 1)
            for (int r = 0; r < ng; r++) {
                long long q = L.at(c, r);
                Uo[q] = e[0]; Uo[q + PL] = e[1]; Uo[q + 3 * PL] = e[3];
            }
        if (j >= ny) Uo[L.at(c, 2 * (ny + ng) - 1 - j) + 2 * PL] = -e[2];
        if (j == ny + ng - 1)
            for (int r = 0; r < ng; r++) {
                long long q = L.at(c, ny + ng + r);
                Uo[q] = e[0]; Uo[q + PL] = e[1]; Uo[q + 3 * PL] = e[3];
            }
        if (c == ng)
            for (int r = 0; r < ng; r++) {
                long long q = L.at(r, j);
                for (int k = 0; k < 4; k++) Uo[q + k * PL] = e[k];
            }
        if (c == nx + ng - 1)
            for (int r = 0; r < ng; r++) {
                long long q = L.at(nx + ng + r, j);
                for (int k = 0; k < 4; k++) Uo[q + k * PL] = e[k];
            }
    }
}

// Deferred finish: the dt / mass reduction of a step's nrec <= DF_MAX_REC
// partial records by one wave, in the order of the one-wave finish kernel
// (k_finish_small: lane t takes records t, t + 64, ... in turn, then the
// cross-lane max / sum), so dt, mass and the clock come out bit for bit as
// they do with a finish kernel between the steps.
__device__ __forceinline__ void df_reduce(const double* part, const int nrec, double& A, double& Um, double& Vm,
                                          double& m, int& bad) {
    lane_records<DF_MAX_REC>(nrec, [&](int q) { return part + PART_STRIDE * (long long)q; }, A, Um, Vm, m, bad);
    A = wave_max(A);
    Um = wave_max(Um);
    Vm = wave_max(Vm);
    m = wave_sum(m);
    bad = __any(bad);
}

// The finish of the step that ran with head `h` (the finish kernel's clock
// bookkeeping): dt from the reduced partials, the reference's clock order
// (now_t advances by the new dt), the log entry of that step by `log_lane`.
__device__ __forceinline__ DfHead df_advance(const StepArgs& a, const DfHead& h, double A2, double Um, double Vm,
                                             double m, int bad, bool log_lane) {
    const double A = ib_sqrt(A2);
    const double dt = a.cfl * a.dx / (A + ((Um < Vm) ? Vm : Um));
    DfHead n;
    n.dt = dt;
    n.now_t = h.now_t + dt;
    n.iter = h.iter + 1;
    n.mass = m;
    n.done = !(n.now_t < a.t_end && n.iter < a.max_iter);
    n.cur = h.cur ^ 1;
    n.pending = 0;
    if (log_lane) {
        Ctl* ctl = a.ctl;
        const int slot = h.iter % LOGCAP;
        ctl->log_dt[slot] = dt;
        ctl->log_t[slot] = n.now_t;
        ctl->log_mass[slot] = m;
        if (bad) ctl->status |= 1;
    }
    return n;
}

// The head of this launch: from the control block for the first kernel of a
// batch, else the previous kernel's head advanced over its partial records.
// Every wave computes it alike; block (0,0) stores it for the next kernel.
__device__ __forceinline__ DfHead df_head(const StepArgs& a, const bool first_block) {
    Ctl* ctl = a.ctl;
    DfHead h;
    if (a.df == 1) {
        h.dt = ctl->dt; h.now_t = ctl->now_t; h.mass = ctl->mass_now;
        h.iter = ctl->iter; h.done = ctl->done; h.cur = ctl->cur; h.pending = 0;
    } else {
        const int p = a.df_k ^ 1;
        const DfHead* q = &ctl->df[p];
        static_assert(offsetof(DfHead, iter) % 8 == 0 && offsetof(DfHead, cur) % 8 == 0, "pairs read as 8 bytes");
        const unsigned long long l[5] = {ld8_here(&q->dt), ld8_here(&q->now_t), ld8_here(&q->mass),
                                         ld8_here(&q->iter), ld8_here(&q->cur)};
        double A, Um, Vm, m;
        int bad;
        df_reduce(a.df_part + (long long)p * DF_MAX_REC * PART_STRIDE, a.nbx * a.nby, A, Um, Vm, m, bad);
        const DfHead prev{uniform_double(l[0]), uniform_double(l[1]), uniform_double(l[2]), uniform_half(l[3], 0),
                          uniform_half(l[3], 1), uniform_half(l[4], 0), uniform_half(l[4], 1)};
        h = prev.pending ? df_advance(a, prev, A, Um, Vm, m, bad, first_block && threadIdx.x == 0) : prev;
    }
    h.pending = !h.done;
    if (first_block && threadIdx.x == 0) ctl->df[a.df_k] = h;
    return h;
}

// Orders a wave's own LDS exchanges: its LDS operations execute in order, so only
// the compiler has to keep them so.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row-parallel strip (small grids, where a strip's rows marching one after the
// other set the step's latency): the block has rows + 1 waves over the same
// 60-column x `rows` strip as step_strip; wave w takes row j = j0 - 1 + w at
// once. It loads rows j-1 .. j+1 of its column (the top wave one more),
// reconstructs row j in y and hands the lower-face state to the wave below (the
// top wave reconstructs row j+1's itself), computes the x faces of row j (for
// j >= j0, or in quirks mode where the y face may take the aliased x flux) and,
// after a block barrier, the y face j+1/2; after another the waves of rows
// j0 .. j1-1 update their cells with the y flux of face j-1/2 from the wave below.
// Every face is computed by the same statements as in
// step_strip, so the state is bit for bit the same; only the grouping of the
// mass partial sum differs. Block barriers are reached by every wave.
// The kernel is a chain of latencies. Everything it reads from memory is asked
// for at its start, in one round trip (the cell types and RK2's U^n too, which
// used to be read where the update needed them); the x exchange is within a wave
// and takes no block barrier; the limiters are evaluated without branches (FLAT).
// LDS per wave: 2 KB for the x exchange (cells, face states and fluxes in turn), 2 KB
// for its lower-face states and its y fluxes, sized by the launch: with the 64 KB of
// four arrays for 8 waves, two blocks filled a CU whatever their height.
constexpr int rowpar_lds(int rows, size_t flux) { return (rows + 1) * 4 * 64 * (int)(2 * sizeof(double) + flux); }
template <int SCH, int RS, int LIM, typename T, bool CUT>
__device__ __forceinline__ void step_rowpar(const StepArgs& a, const int bx, const int by, const int stage) {
    constexpr bool FP64 = sizeof(T) == sizeof(double);
    // the cut-cell and mixed-precision forms exist in corrected mode only
    const int quirks = CUT || !FP64 ? 0 : a.quirks;
    Ctl* ctl = a.ctl;
    // the wave's number as a scalar: its row, addresses and branches are wave-uniform
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Layout L = a.L;
    const long long PL = L.plane;
    const int ng = L.ng, nx = L.nx, ny = L.ny;
    const int cb = ng + STRIP_W * bx;
    const int c = cb - 2 + lane;
    const int cl = min(max(c, 0), L.M - 1);
    const int j0 = ng + a.rows * by;
    const int j1 = min(j0 + a.rows, ny + ng);
    const int j = j0 - 1 + wv;
    const bool live = j < j1;  // the waves past a short last strip only reach the barriers

    // Rows j-1 .. j+1 (top wave: j+2) of column c (in range: ng >= 2), read
    // together with the control block from the buffer the host expects to be the
    // input (StepArgs::in_hint), so that no load waits for another: on a
    // latency-bound small grid that is one memory round trip less. Another buffer
    // (steps that the host does not see: a caller's own graph replayed) is read again below.
    // Every load at the head of the kernel is unconditional (the waves past a short
    // last strip read the top row's), so that none waits in a branch.
    double wm[4], w0[4], w1[4], w2[4] = {0.0, 0.0, 0.0, 0.0};
    const bool top = j == j1 - 1;
    const int jl = min(j, j1 - 1);
    auto load_rows = [&](const double* U) {
        const double* r = U + L.at(0, jl - 1);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            wm[k] = ld_here(r + k * PL + cl);
            w0[k] = ld_here(r + k * PL + L.pitch + cl);
            w1[k] = ld_here(r + k * PL + 2 * L.pitch + cl);
        }
        if (top) {
#pragma unroll
            for (int k = 0; k < 4; k++) w2[k] = ld_here(r + k * PL + 3 * L.pitch + cl);
        }
    };
    const CtlLoads cl_now = ctl_now(ctl);
    load_rows(a.in_hint ? a.buf[1] : a.buf[0]);
    const uint8_t tc = __hip_atomic_load(a.type + L.at(cl, jl), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    int cur;
    double dt;
    if (a.df) {
        const DfHead h = df_head(a, bx == 0 && by == 0);
        if (h.done) return;
        cur = h.cur;
        dt = h.dt;
    } else {
        const CtlNow now = ctl_value(cl_now);
        if (now.done) {
            if (bx == 0 && by == 0 && threadIdx.x == 0) ctl->ran = 0;
            return;
        }
        cur = now.cur ^ (stage == 3 ? 1 : 0);  // the input buffer
        dt = now.dt;
        if (bx == 0 && by == 0 && threadIdx.x == 0) {
            ctl->ran = 1;
            ctl->out = cur ^ 1;
        }
    }
    const double* __restrict__ Ui = cur ? a.buf[1] : a.buf[0];
    double* __restrict__ Uo = cur ? a.buf[0] : a.buf[1];
    GasT<T> g;
    g.gam = (T)a.gam; g.gm1 = (T)a.gm1; g.gp1 = (T)a.gp1; g.c1 = (T)a.c1;
    g.r_gam = Rcp<T>{(T)a.gam, (T)a.r_gam};
    g.r_gm1 = Rcp<T>{(T)a.gm1, (T)a.r_gm1};
    g.r_dx = Rcp<T>{(T)a.dx, (T)a.r_dx};
    g.r_dy = Rcp<T>{(T)a.dy, (T)a.r_dy};
    const T dtc = (T)dt;
    const Rcp<double> r_dx{a.dx, a.r_dx}, r_dy{a.dy, a.r_dy}, r_gm1{a.gm1, a.r_gm1};
    const double dtdx = dt * a.r_dx, dtdy = dt * a.r_dy;  // mixed form only

    extern __shared__ double lds[];
    double* xb = lds + wv * 256;                                             // this wave's x exchange
    double* hb = lds + (a.rows + 1) * 256;                                   // every wave's lower-face states
    T* gb = (T*)(hb + (a.rows + 1) * 256);                                   // and y fluxes
    __shared__ double sp[ROWPAR_MAX_ROWS + 1][5];

    // reference Global_Boundary corners (Test/Sod/Global_Boudary.cpp:62-75), as in step_strip
    if (a.edge_fused == 1 && bx == 0 && by == 0 && wv == 0 && lane < 4 * ng * ng) {
        int side = lane / (2 * ng * ng);
        int rem = lane % (2 * ng * ng);
        int ri = rem / ng, cc = rem % ng;
        int row = ri < ng ? ri : ny + ri;
        int col = side == 0 ? cc : nx + ng + cc;
        int scol = side == 0 ? ng : nx + ng - 1;
        long long o = L.at(col, row);
        for (int k = 0; k < 4; k++) {
            double v = a.corner_from_input ? Ui[L.at(scol, row) + k * PL] : a.corner[(side * 2 * ng + ri) * 4 + k];
            Uo[o + k * PL] = v;
        }
    }

    if (cur != a.in_hint) load_rows(Ui);
    const bool upd = live && j >= j0 && lane >= 2 && lane < STRIP_W + 2 && c < nx + ng;
    double uo[4] = {0.0, 0.0, 0.0, 0.0};  // RK2's U^n
    if (stage >= 2 && upd) {
#pragma unroll
        for (int k = 0; k < 4; k++) uo[k] = Uo[L.at(c, j) + k * PL];
    }
    double ylo[4], yhi[4];
    if (live) {
        cell_states<SCH, LIM, T, true>(wm, w0, w1, ylo, yhi, quirks);
#pragma unroll
        for (int k = 0; k < 4; k++) hb[(wv * 4 + k) * 64 + lane] = yhi[k];
        if (top) {  // the state of row j + 1, which no wave of the block holds
            double lo_unused[4];
            cell_states<SCH, LIM, T, true>(w0, w1, w2, lo_unused, yhi, quirks);
        }
    }
    const bool xrow = live && (j >= j0 || (quirks && RS != RS_SW));
    const int ln = min(lane + 1, 63), lp = max(lane - 1, 0);
    T F[4] = {0, 0, 0, 0};
    if (xrow) {
        double xm[4], xp[4], xlo[4], xhi[4], xr[4];
#pragma unroll
        for (int k = 0; k < 4; k++) xb[k * 64 + lane] = w0[k];
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < 4; k++) {
            xm[k] = xb[k * 64 + lp];
            xp[k] = xb[k * 64 + ln];
        }
        cell_states<SCH, LIM, T, true>(xm, w0, xp, xlo, xhi, quirks);
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < 4; k++) xb[k * 64 + lane] = xhi[k];
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < 4; k++) xr[k] = xb[k * 64 + ln];
        xface<SCH, RS>(g, a.gm1, dtc, quirks, [&](int k) { return w0[k]; }, [&](int k) { return xp[k]; }, xlo, xr, F);
    }
    __syncthreads();
    T G[4] = {0, 0, 0, 0};
    if (live) {
        if (!top) {
#pragma unroll
            for (int k = 0; k < 4; k++) yhi[k] = hb[((wv + 1) * 4 + k) * 64 + lane];
        }
        yface<SCH, RS>(g, a.gm1, dtc, quirks, [&](int k) { return w0[k]; }, [&](int k) { return w1[k]; }, ylo, yhi,
                       [&](int k) { return F[k]; }, G);
    }
    wave_lds_order();
    T* fb = (T*)xb;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        fb[k * 64 + lane] = F[k];
        gb[(wv * 4 + k) * 64 + lane] = G[k];
    }
    __syncthreads();
    double amax = 0.0, umax = 0.0, vmax = 0.0, msum = 0.0;
    int bad = 0;
    if (upd)
        update_cell<SCH, RS, LIM, T, CUT>(a, L, c, j, tc, w0, uo, F, G, fb + lane - 1, gb + (wv - 1) * 256 + lane, dt,
                                          quirks, r_dx, r_dy, r_gm1, dtdx, dtdy, Uo, stage, amax, umax, vmax, msum,
                                          bad);
    // one partial record per block: each wave's, then the waves in order
    amax = wave_max(amax);
    umax = wave_max(umax);
    vmax = wave_max(vmax);
    msum = wave_sum(msum);
    bad = __any(bad);
    if (lane == 0) {
        sp[wv][0] = amax; sp[wv][1] = umax; sp[wv][2] = vmax; sp[wv][3] = msum; sp[wv][4] = bad ? 1.0 : 0.0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
        double A = sp[0][0], U = sp[0][1], V = sp[0][2], m = sp[0][3], b = sp[0][4];
        for (int q = 1; q < nw; q++) {
            A = (A < sp[q][0]) ? sp[q][0] : A;
            U = (U < sp[q][1]) ? sp[q][1] : U;
            V = (V < sp[q][2]) ? sp[q][2] : V;
            m = m + sp[q][3];
            b = (b < sp[q][4]) ? sp[q][4] : b;
        }
        double* part = a.df ? a.df_part + (long long)a.df_k * DF_MAX_REC * PART_STRIDE : a.mass_part;
        double* r = part + PART_STRIDE * (long long)(by * a.nbx + bx);
        r[0] = A; r[1] = U; r[2] = V; r[3] = m; r[4] = b;
    }
}

template <int SCH, int RS, int LIM, typename T, bool CUT>
__global__ __launch_bounds__(64 * (ROWPAR_MAX_ROWS + 1)) void k_step_rowpar(StepArgs a) {
    step_rowpar<SCH, RS, LIM, T, CUT>(a, blockIdx.x, blockIdx.y, a.stage);
}

// Compiled in nine objects, one per scheme and Riemann solver (STEP_SCHEME,
// STEP_RIEMANN), so that a solve loads its own kernels only (a process's first steps on
// a small grid: 4.5 ms with all of them in one object).
template <int SCH, int RS> hipError_t go_rowpar_l(int lim, int prec, const StepArgs& a, hipStream_t s);
template <int SCH, int RS> const void* rowpar_kernel_l();

#ifdef STEP_SCHEME
template <int SCH, int RS, int LIM>
static hipError_t go_rowpar(int prec, const StepArgs& a, hipStream_t s) {
    const dim3 grid(a.nbx, a.nby), block(64 * (a.rows + 1));
    const int l64 = rowpar_lds(a.rows, sizeof(double)), l32 = rowpar_lds(a.rows, sizeof(float));
    if (a.cut) {
        if (prec == 1) hipLaunchKernelGGL((k_step_rowpar<SCH, RS, LIM, float, true>), grid, block, l32, s, a);
        else hipLaunchKernelGGL((k_step_rowpar<SCH, RS, LIM, double, true>), grid, block, l64, s, a);
    } else {
        if (prec == 1) hipLaunchKernelGGL((k_step_rowpar<SCH, RS, LIM, float, false>), grid, block, l32, s, a);
        else hipLaunchKernelGGL((k_step_rowpar<SCH, RS, LIM, double, false>), grid, block, l64, s, a);
    }
    return hipGetLastError();
}
template <int SCH, int RS>
hipError_t go_rowpar_l(int lim, int prec, const StepArgs& a, hipStream_t s) {
    if (lim == LIM_MINMOD) return go_rowpar<SCH, RS, LIM_MINMOD>(prec, a, s);
    if (lim == LIM_VANLEER) return go_rowpar<SCH, RS, LIM_VANLEER>(prec, a, s);
    return go_rowpar<SCH, RS, LIM_VANALBADA>(prec, a, s);
}
template <int SCH, int RS> const void* rowpar_kernel_l() {
    return (const void*)k_step_rowpar<SCH, RS, LIM_MINMOD, double, false>;
}
template hipError_t go_rowpar_l<STEP_SCHEME, STEP_RIEMANN>(int, int, const StepArgs&, hipStream_t);
template const void* rowpar_kernel_l<STEP_SCHEME, STEP_RIEMANN>();

#else  // ------------------------------------------- the flush and the dispatch

// The end of a deferred-finish batch: the finish of its last kernel (parity
// k), if that kernel ran its step, published to the control block as the
// finish kernel leaves it (ran = whether that step ran).
__global__ __launch_bounds__(64) void k_df_flush(StepArgs a, int k) {
    Ctl* ctl = a.ctl;
    const DfHead h = ctl->df[k];
    double A, Um, Vm, m;
    int bad;
    df_reduce(a.df_part + (long long)k * DF_MAX_REC * PART_STRIDE, a.nbx * a.nby, A, Um, Vm, m, bad);
    if (threadIdx.x != 0) return;
    const DfHead n = h.pending ? df_advance(a, h, A, Um, Vm, m, bad, true) : h;
    ctl->dt = n.dt;
    ctl->now_t = n.now_t;
    ctl->iter = n.iter;
    ctl->done = n.done;
    ctl->cur = n.cur;
    ctl->mass_now = n.mass;
    ctl->ran = h.pending;
}

template <int SCH>
static hipError_t go_rowpar_r(int rs, int lim, int prec, const StepArgs& a, hipStream_t s) {
    if (rs == RS_SW) return go_rowpar_l<SCH, RS_SW>(lim, prec, a, s);
    if (rs == RS_PVRS) return go_rowpar_l<SCH, RS_PVRS>(lim, prec, a, s);
    return go_rowpar_l<SCH, RS_HLL>(lim, prec, a, s);
}

hipError_t launch_df_flush(const StepArgs& a, int k, hipStream_t s) {
    if (!a.df_ok || a.nbx * a.nby > DF_MAX_REC || (k != 0 && k != 1)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_df_flush, dim3(1), dim3(64), 0, s, a, k);
    return hipGetLastError();
}

hipError_t launch_step_rowpar(int scheme, int rs, int lim, int prec, const StepArgs& a, hipStream_t s) {
    if (scheme == SCH_LAX || a.rows < 1 || a.rows > ROWPAR_MAX_ROWS) return hipErrorInvalidValue;
    if (a.df && (!a.df_ok || a.nbx * a.nby > DF_MAX_REC || a.stage != 0 || !a.df_part)) return hipErrorInvalidValue;
    if (scheme == SCH_MHM) return go_rowpar_r<SCH_MHM>(rs, lim, prec, a, s);
    if (scheme == SCH_GODUNOV) return go_rowpar_r<SCH_GODUNOV>(rs, lim, prec, a, s);
    return go_rowpar_r<SCH_MUSCL>(rs, lim, prec, a, s);
}

template <int SCH> static const void* rowpar_kernel_r(int rs) {
    if (rs == RS_SW) return rowpar_kernel_l<SCH, RS_SW>();
    if (rs == RS_PVRS) return rowpar_kernel_l<SCH, RS_PVRS>();
    return rowpar_kernel_l<SCH, RS_HLL>();
}
const void* rowpar_kernel(int scheme, int rs) {
    if (scheme == SCH_MHM) return rowpar_kernel_r<SCH_MHM>(rs);
    if (scheme == SCH_GODUNOV) return rowpar_kernel_r<SCH_GODUNOV>(rs);
    return rowpar_kernel_r<SCH_MUSCL>(rs);
}

#endif  // STEP_SCHEME

}  // namespace ibtfo
