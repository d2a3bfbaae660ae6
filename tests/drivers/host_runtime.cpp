// The library's host code (contexts, graphs, tiles, the batch engine) on the CPU:
// linked with ibtfo_capi.cpp and ibtfo_batch.cpp, this file stands in for the HIP
// runtime (memory is host memory, a stream runs what it is given at once or, while it
// captures, records it) and for the kernels (their bookkeeping in the control block,
// no flow). One check per run, named by the first argument; exit status 0 if it holds.
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../../ibtfo_amd/csrc/ibtfo_ctx.h"
#include "../../ibtfo_amd/csrc/ibtfo_geom.h"

using namespace ibtfo;

// ------------------------------------------------------------------ the runtime
struct ihipStream_t { bool capturing = false; std::vector<std::function<void()>> ops; };
struct ihipGraph { std::vector<std::function<void()>> ops; };
struct hipGraphExec { std::vector<std::function<void()>> ops; };
struct ihipEvent_t { double at = 0; };

namespace fake {
long fail_alloc_over = -1;   // allocations of more bytes than this fail (-1: none)
double clock_ms = 0;         // advanced by the step kernels
int ghosts = 0;              // ghosts a geometry finds
int geometries = 0;          // geometry runs
int launches = 0, wrong_hints = 0;
int captures = 0, first_record = -1, last_record = -1;  // captures so far; at the first and last event
int batch_rows = 0;          // strip height of the batch's last solve stepped
int lds_limit = 0, lds_refused = 0;  // the mask kernel's LDS attribute; launches above it
std::function<void()> after_attribute;
double (*step_ms)(const StepArgs&) = nullptr;

void run(hipStream_t s, std::function<void()> f) {
    if (s->capturing) s->ops.push_back(f);
    else f();
}
}  // namespace fake

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (fake::fail_alloc_over >= 0 && (long)n > fake::fail_alloc_over) return hipErrorOutOfMemory;
    *p = calloc(1, n + 1);
    return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { *p = calloc(1, n + 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    if (k == hipMemcpyDeviceToDevice && n > (1u << 20)) return hipSuccess;  // states, which hold no flow here
    fake::run(st, [=] { memmove(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    fake::run(st, [=] { memset(d, v, n); });
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { *s = new ihipStream_t(); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    s->capturing = true;
    fake::captures++;
    s->ops.clear();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    s->capturing = false;
    *g = new ihipGraph{std::move(s->ops)};
    s->ops.clear();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    *e = new hipGraphExec{g->ops};
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (auto& f : e->ops) f();
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { *e = new ihipEvent_t(); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    e->at = fake::clock_ms;
    if (fake::first_record < 0) fake::first_record = fake::captures;
    fake::last_record = fake::captures;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { *ms = (float)(b->at - a->at); return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int v) {
    fake::lds_limit = v;
    auto f = std::move(fake::after_attribute);
    fake::after_attribute = nullptr;
    if (f) f();
    return hipSuccess;
}
}

// ------------------------------------------------------------------ the kernels
static void finish(const FinishArgs& f, int advance) {
    Ctl* c = f.ctl;
    if (!c || c->done) return;
    if (advance == 2) { c->cur ^= 1; return; }
    c->iter++;
    c->now_t += c->dt;
    c->done = !(c->now_t < f.t_end && c->iter < f.max_iter);
    if (!f.keep_cur) c->cur ^= 1;
}
static void step(const StepArgs& a, int stage) {
    Ctl* c = a.ctl;
    c->ran = !c->done;
    if (c->done) return;
    c->out = c->cur ^ 1 ^ (stage == 3 ? 1 : 0);
}
namespace ibtfo {
hipError_t launch_step(int, int, int, int, const StepArgs& a, hipStream_t s) {
    fake::run(s, [a] {
        int cur = a.ctl->cur ^ (a.stage == 3 ? 1 : 0);
        if (a.df) {  // the head of a deferred-finish batch
            DfHead h{};
            if (a.df == 1) { h.iter = a.ctl->iter; h.done = a.ctl->done; h.cur = a.ctl->cur; h.now_t = a.ctl->now_t; }
            else {
                h = a.ctl->df[a.df_k ^ 1];
                if (h.pending) { h.iter++; h.cur ^= 1; h.done = h.iter >= a.max_iter; }
            }
            h.pending = !h.done;
            a.ctl->df[a.df_k] = h;
            cur = h.cur;
        } else step(a, a.stage);
        fake::launches++;
        fake::wrong_hints += a.in_hint != cur;
        if (fake::step_ms) fake::clock_ms += fake::step_ms(a);
    });
    return hipSuccess;
}
hipError_t load_step(int, int, int, int, int) { return hipSuccess; }
hipError_t launch_df_flush(const StepArgs& a, int k, hipStream_t s) {
    fake::run(s, [a, k] {
        DfHead h = a.ctl->df[k];
        a.ctl->ran = h.pending;
        if (h.pending) { h.iter++; h.cur ^= 1; h.done = h.iter >= a.max_iter; }
        a.ctl->iter = h.iter; a.ctl->done = h.done; a.ctl->cur = h.cur;
    });
    return hipSuccess;
}
hipError_t launch_finish(const FinishArgs& f, hipStream_t s) {
    fake::run(s, [f] { finish(f, f.advance); });
    return hipSuccess;
}
hipError_t launch_post(const FinishArgs& f, const FillArgs*, const EdgeArgs*, hipStream_t s) { return launch_finish(f, s); }
hipError_t launch_reduce(const ReduceArgs& a, hipStream_t s) {
    fake::run(s, [a] {
        a.ctl->dt = 1e-6;
        if (a.reset) { a.ctl->iter = 0; a.ctl->now_t = 0; a.ctl->done = a.max_iter <= 0; a.ctl->ran = 0; }
    });
    return hipSuccess;
}
hipError_t launch_uniform_state(double*, double*, double*, long long, const double*, Ctl* c, hipStream_t s) {
    fake::run(s, [c] { c->cur = 0; c->ran = 0; });
    return hipSuccess;
}
hipError_t launch_fill(const FillArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_scatter(const FillArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_edge(const EdgeArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_edge_ref(const EdgeArgs&, const double*, int, hipStream_t) { return hipSuccess; }
hipError_t launch_merge(const MergeArgs&, hipStream_t) { return hipSuccess; }
// the batch's kernels over its slots
hipError_t launch_step_batch(int, int, int, int, const StepArgs* t, const int2* map, int n, int stage, hipStream_t s) {
    fake::run(s, [=] {
        for (int b = 0; b < n; b++)
            if (map[b].x >= 0 && map[b].y == 0) {
                step(t[map[b].x], stage);
                fake::batch_rows = t[map[b].x].rows;
            }
    });
    return hipSuccess;
}
hipError_t launch_post_batch(const FinishArgs* f, int ns, int advance, const FillArgs*, const int2*, int, const EdgeArgs*,
                             const int2*, int, hipStream_t s) {
    fake::run(s, [=] {
        for (int q = 0; q < ns; q++)
            if (f[q].ctl) finish(f[q], advance);
    });
    return hipSuccess;
}
hipError_t launch_gather(const FinishArgs* f, int ns, SlotStatus* out, hipStream_t s) {
    fake::run(s, [=] {
        for (int q = 0; q < ns; q++) {
            SlotStatus st{};
            if (const Ctl* c = f[q].ctl) { st.iter = c->iter; st.done = c->done; st.now_t = c->now_t; st.dt = c->dt; }
            out[q] = st;
        }
    });
    return hipSuccess;
}
hipError_t launch_persist(int, int, int, int, const PersistArgs&, int, hipStream_t) { return hipErrorInvalidValue; }
int persist_blocks(int, int, int, int) { return 0; }
hipError_t geom_run(GeomArgs& g, hipStream_t) {
    fake::geometries++;
    memset(g.type, 0, g.L.plane);
    return hipSuccess;
}
hipError_t geom_ghosts(GeomArgs& g, hipStream_t) { *g.count = (unsigned)fake::ghosts; return hipSuccess; }
hipError_t cut_run(GeomArgs&, hipStream_t) { return hipSuccess; }
hipError_t cut_records(GeomArgs&, hipStream_t) { return hipSuccess; }
hipError_t mask_run(MaskArgs& m, bool lds, hipStream_t) {
    if (lds && (int)mask_lds_bytes(m.W, m.M) > fake::lds_limit) fake::lds_refused++;
    return hipSuccess;
}
const void* mask_rows_kernel() { return nullptr; }
int png_read_file(const char*, std::vector<unsigned char>&, int*, int*) { return IBTFO_E_IO; }
int write_vtk(const ::ibtfo_config*, int, double, const double*, const double*, const char*) { return IBTFO_E_IO; }
int host_initialize(int, const double*, int, int, int, int, double, const double*, const double*, const unsigned char*,
                    double*) { return IBTFO_E_ARG; }
}  // namespace ibtfo

// ------------------------------------------------------------------ the checks
static int failures = 0;
#define CHECK(c) do { if (!(c)) { failures++; printf("%s:%d: %s\n", __FILE__, __LINE__, #c); } } while (0)

static ibtfo_config config(int nx, int ny, int boundary, int edge) {
    ibtfo_config c;
    memset(&c, 0, sizeof c);
    c.N_x = nx; c.N_y = ny; c.num_ghost_cell = 2;
    c.hi_x = 1.0; c.hi_y = (double)ny / nx;
    c.Psy_time = 1e30; c.max_iter = 1 << 30;
    c.CFL_number = 0.5; c.gamma = 1.4;
    c.scheme = IBTFO_MUSCL; c.riemann = IBTFO_HLL; c.limiter = IBTFO_MINMOD;
    c.boundary = boundary; c.time = IBTFO_SINGLESTEP; c.edge = edge; c.precision = IBTFO_FP64;
    const double flow[4] = {1.4, 3.0, 0.0, 1.0};
    memcpy(c.edge_state, flow, sizeof flow);
    return c;
}
static const double UNIFORM[4] = {1.4, 3.0, 0.0, 1.0};
static ibtfo_ctx* solve(const ibtfo_config& c) {
    ibtfo_ctx* x = nullptr;
    CHECK(ibtfo_create(&c, &x) == IBTFO_OK);
    CHECK(ibtfo_geometry(x, IBTFO_LS_NONE, nullptr, 0, nullptr) == IBTFO_OK);
    CHECK(ibtfo_initialize(x, IBTFO_INIT_UNIFORM, UNIFORM, 4) == IBTFO_OK);
    CHECK(ibtfo_prepare(x, 1) == IBTFO_OK);
    return x;
}

// A geometry that fails after its types were written leaves a solve without one:
// nothing runs on the new types with an empty ghost list.
static void geometry_failure() {
    fake::ghosts = 0;
    ibtfo_ctx* x = solve(config(96, 64, IBTFO_IDW_GFM, IBTFO_EDGE_INFLOW));
    fake::ghosts = 5000;
    fake::fail_alloc_over = 1000;
    CHECK(ibtfo_geometry(x, IBTFO_LS_NONE, nullptr, 0, nullptr) == IBTFO_E_NOMEM);
    fake::fail_alloc_over = -1;
    double v;
    CHECK(ibtfo_prepare(x, 1) == IBTFO_E_STATE);
    CHECK(ibtfo_boundary(x) == IBTFO_E_STATE);
    CHECK(ibtfo_compute_dt(x, &v) == IBTFO_E_STATE);
    CHECK(ibtfo_step(x, 1) == IBTFO_E_STATE);
    CHECK(ibtfo_geometry(x, IBTFO_LS_NONE, nullptr, 0, nullptr) == IBTFO_OK);
    CHECK(ibtfo_num_ghosts(x) == 5000);
    CHECK(ibtfo_prepare(x, 1) == IBTFO_OK);
    CHECK(ibtfo_step(x, 1) == IBTFO_OK);
    ibtfo_destroy(x);
}

// Two threads with masks of different widths: the narrow one's call falls between the
// wide one's attribute and its launch.
static void mask_attribute() {
    ibtfo_ctx* a = solve(config(64, 32, IBTFO_IDW_GFM, IBTFO_EDGE_INFLOW));
    ibtfo_ctx* b = solve(config(64, 32, IBTFO_IDW_GFM, IBTFO_EDGE_INFLOW));
    const std::vector<unsigned char> wide(4 * 6000 * 8, 255), narrow(4 * 8 * 8, 255);
    fake::after_attribute = [&] { CHECK(ibtfo_geometry_mask(b, narrow.data(), 8, 8) == IBTFO_OK); };
    CHECK(ibtfo_geometry_mask(a, wide.data(), 6000, 8) == IBTFO_OK);
    CHECK(fake::lds_limit > 0 && fake::lds_refused == 0);
    ibtfo_destroy(a);
    ibtfo_destroy(b);
}

// Replays after an odd number of single steps, and replays of an odd number of steps:
// every step kernel is told the buffer that it then finds current.
static void graph_start() {
    for (int nx : {96, 1200})  // one kernel per step; a finish kernel between
        for (int time : {IBTFO_SINGLESTEP, IBTFO_RK2}) {
            ibtfo_config c = config(nx, nx / 2, IBTFO_REGULAR, IBTFO_EDGE_REFERENCE);
            c.time = time;
            ibtfo_ctx* x = solve(c);
            fake::launches = fake::wrong_hints = 0;
            CHECK(ibtfo_step_graph(x, 0, 50) == IBTFO_OK && fake::launches == 0);
            int steps = 0;
            for (int n : {75, 75, 50, 1, 100, 125}) {
                CHECK(ibtfo_step_graph(x, n, 50) == IBTFO_OK);
                steps += n;
            }
            for (int n : {28, 7, 1, 70}) {
                CHECK(ibtfo_step_graph(x, n, 7) == IBTFO_OK);
                steps += n;
            }
            int it = 0;
            CHECK(ibtfo_status(x, &it, nullptr, nullptr) == IBTFO_OK && it == steps);
            CHECK(fake::launches == steps * (time == IBTFO_RK2 ? 2 : 1) && fake::wrong_hints == 0);
            // a timed run from either buffer: nothing is captured between its events
            for (int odd : {0, 1}) {
                CHECK(ibtfo_step_graph(x, 0, 20 + odd * 2) == IBTFO_OK && ibtfo_step(x, odd) == IBTFO_OK);
                fake::first_record = -1;
                double ms = 0;
                CHECK(ibtfo_time_steps(x, 100, &ms, nullptr) == IBTFO_OK);
                CHECK(fake::first_record >= 0 && fake::first_record == fake::last_record);
            }
            ibtfo_destroy(x);
        }
}

// The autotuner's probes and the steps after it, for an even and an odd probe: the state
// put back is the one that the next probe is told.
static double every_step_alike(const StepArgs&) { return 1.0; }
static void autotune_start() {
    fake::step_ms = every_step_alike;
    for (int probe : {3, 4}) {
        ibtfo_ctx* x = solve(config(1200, 600, IBTFO_IDW_GFM, IBTFO_EDGE_INFLOW));
        CHECK(ibtfo_step(x, 5) == IBTFO_OK);
        fake::launches = fake::wrong_hints = 0;
        CHECK(ibtfo_autotune(x, probe, nullptr, nullptr) == IBTFO_OK);
        CHECK(ibtfo_step(x, 4) == IBTFO_OK);
        CHECK(fake::launches > 20 * probe && fake::wrong_hints == 0);
        int it = 0;
        CHECK(ibtfo_status(x, &it, nullptr, nullptr) == IBTFO_OK && it == 9);
        ibtfo_destroy(x);
    }
}

// The autotuner keeps a tile that is faster than every shape of its list, where that is
// the default tile (10 rows) or the one in force.
static int best_rows = 0;
static double one_tile_best(const StepArgs& a) { return a.rows == best_rows && !a.rowpar ? 1.0 : 2.0; }
static void autotune_own_tile() {
    fake::step_ms = one_tile_best;
    for (int in_force : {0, 11}) {
        ibtfo_ctx* x = solve(config(4096, 2048, IBTFO_REGULAR, IBTFO_EDGE_REFERENCE));
        int rows = 0, par = 1;
        CHECK(ibtfo_set_rows(x, in_force) == IBTFO_OK && ibtfo_tile(x, &best_rows, nullptr, nullptr) == IBTFO_OK);
        CHECK(best_rows == (in_force ? in_force : 10));
        for (int again = 0; again < 2; again++) {
            CHECK(ibtfo_autotune(x, 2, &rows, nullptr) == IBTFO_OK && rows == best_rows);
            CHECK(ibtfo_tile_ex(x, &rows, nullptr, nullptr, &par) == IBTFO_OK && rows == best_rows && !par);
            if (!in_force) CHECK(ibtfo_set_rows(x, 48) == IBTFO_OK);  // the default, found from another tile
        }
        ibtfo_destroy(x);
    }
}

static ibtfo_batch_config batch_config(int rows, int blocks, int slots) {
    ibtfo_batch_config k;
    ibtfo_batch_config_default(&k);
    k.boundary = IBTFO_IDW_GFM;
    k.quirks = 0;
    k.hbm_budget = 1ll << 30;
    k.max_slots = slots;
    k.max_step_blocks = blocks;
    k.max_ghost_blocks = k.max_ring_blocks = 4096;
    k.rows = rows;
    k.chunk = 4;
    return k;
}
static int submit(ibtfo_batch* b, int nx, int ny, int steps) {
    ibtfo_request r;
    memset(&r, 0, sizeof r);
    r.cfg = config(nx, ny, IBTFO_IDW_GFM, IBTFO_EDGE_INFLOW);
    r.cfg.max_iter = steps;
    r.ls_kind = IBTFO_LS_NONE;
    r.init_kind = IBTFO_INIT_UNIFORM;
    r.init_nprm = 4;
    r.init_prm = UNIFORM;
    r.arrival = -1;
    return ibtfo_batch_submit(b, &r, nullptr);
}
static int drain(ibtfo_batch* b) {
    int active = 1, queued = 1, finished = 0;
    for (int k = 0; k < 1000 && (active || queued); k++) CHECK(ibtfo_batch_progress(b, &active, &queued, &finished) == IBTFO_OK);
    return finished;
}

// rows = 0: 8-row strips from three rounds of the chip's waves on, where the solve fits.
static void batch_open_rows() {
    struct { int rows, blocks, want; } cases[] = {{0, 8192, 16}, {0, 12287, 16}, {0, 12288, 8}, {0, 65536, 8}, {4, 8192, 4},
                                                  {16, 65536, 16}};
    for (auto& c : cases) {
        ibtfo_batch_config k = batch_config(c.rows, c.blocks, 4);
        ibtfo_batch* b = nullptr;
        CHECK(ibtfo_batch_create(&k, &b) == IBTFO_OK);
        CHECK(submit(b, 128, 64, 6) == IBTFO_OK);
        CHECK(drain(b) == 1 && fake::batch_rows == c.want);
        ibtfo_batch_destroy(b);
    }
}

// Requests that wait for step blocks (96x64: 2 strips x 4) or ring blocks (1312 cells: 3)
// are built once each, in the order of their arrival.
static void batch_waiting() {
    for (int ring : {0, 1}) {
        ibtfo_batch_config k = batch_config(16, ring ? 4096 : 20, 8);
        if (ring) k.max_ring_blocks = 7;
        ibtfo_batch* b = nullptr;
        CHECK(ibtfo_batch_create(&k, &b) == IBTFO_OK);
        fake::geometries = 0;
        for (int q = 0; q < 5; q++) CHECK(submit(b, 96, 64, 40 + q) == IBTFO_OK);
        int active = 0, queued = 0;
        CHECK(ibtfo_batch_progress(b, &active, &queued, nullptr) == IBTFO_OK && active == 2 && queued == 3);
        CHECK(ibtfo_batch_progress(b, &active, &queued, nullptr) == IBTFO_OK && active == 2 && queued == 3);
        CHECK(fake::geometries == 2);
        CHECK(drain(b) == 5 && fake::geometries == 5);
        long long t = 0, last = 0;
        while (ibtfo_batch_poll(b, &t) == 1) {
            ibtfo_result r;
            CHECK(ibtfo_batch_result(b, t, &r, nullptr) == IBTFO_OK && r.status == IBTFO_OK && r.iter == 39 + t && t > last);
            last = t;
        }
        CHECK(last == 5);
        // a grid that no context takes is still retired with its error
        CHECK(submit(b, 3, 64, 4) == IBTFO_OK && drain(b) == 6);
        ibtfo_result r;
        CHECK(ibtfo_batch_poll(b, &t) == 1 && ibtfo_batch_result(b, t, &r, nullptr) == IBTFO_OK && r.status == IBTFO_E_ARG);
        ibtfo_batch_destroy(b);
    }
}

// The persistent kernel's waves on a SIMD, for every register count (of 512, by eights):
// however the first of them lie, among other waves that end later, the next has room.
static bool stuck(int free, int gaps, int size) { return free <= gaps * (size - 1); }
static void persistent_grid() {
    for (int size = 1; size <= 64; size++) {
        const int fit = std::min(64 / size, 8), waves = persist_per_cu(4 * fit) / 4;
        CHECK(waves >= 1 && waves <= fit);
        for (int placed = 0; placed < waves; placed++) CHECK(!stuck(64 - placed * size, placed + 1, size));
    }
    CHECK(persist_per_cu(3) == 3 && persist_per_cu(1) == 1);  // kernels that other limits hold below one per SIMD
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> checks = {{"geometry_failure", geometry_failure},
                                                         {"mask_attribute", mask_attribute},
                                                         {"graph_start", graph_start},
                                                         {"autotune_start", autotune_start},
                                                         {"autotune_own_tile", autotune_own_tile},
                                                         {"batch_open_rows", batch_open_rows},
                                                         {"batch_waiting", batch_waiting},
                                                         {"persistent_grid", persistent_grid}};
    const auto it = argc > 1 ? checks.find(argv[1]) : checks.end();
    if (it == checks.end()) {
        for (auto& c : checks) printf("%s\n", c.first.c_str());
        return 2;
    }
    it->second();
    printf("%s: %s\n", argv[1], failures ? "FAILED" : "ok");
    return failures ? 1 : 0;
}
