// host_api.cpp -- fq_api.cpp on the CPU: device memory is host memory, copies
// happen at once, and the launchers look at their arguments instead of launching.
// So what the host side hands to the kernels can be checked without a GPU:
//
//   plans   every cost plan that a launch reads, when it is launched, is a plan of the
//           graph as it then is (build_plan's bytes), and lies in live memory.
//   capture a run on a captured stream neither allocates nor waits, and the phase tables
//           that its launches read stay where they are while the state lives.
//   reopen  a slab's step whose plans cannot be made after its graph changed, called
//           again: the slot's open layer takes the change once.
//   cover   the plans of fq_run and of the gradient: per layer one RX on each qubit, after
//           the layer's phase and before the next one's, on passes that have an instance.
//   newplan a captured run whose plans are not there yet: eager runs before and between
//           the replays make their own.
//   dropped the same, after a call that drops all cached plans (64 smaller than its own).
//   nomem   a run where no device memory for all its phase tables is left.
//   deep    host memory that a run or a gradient of many layers takes.
//   passes  the launches of a slab's request, and what fq_slab_passes says.
//   copies  the copies to the device in a step that slots enter.
//   factors the factors that the passes of a slab's request multiply in.
//
// Each run prints "checked <n> wrong <m>"; tests/test_host_api.py has the programs.
#include <hip/hip_runtime.h>
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) (&x)

#include "fq_api.cpp"

#include <functional>
#include <sys/mman.h>

// ---- device memory and streams --------------------------------------------------

static std::map<char *, size_t> g_live;   // device and pinned allocations
static std::vector<char *> g_freed;       // (kept, poisoned: a late read is seen, not undefined)

static bool live(const void *p, size_t n)
{
    auto it = g_live.upper_bound((char *)p);
    if (it == g_live.begin())
        return false;
    --it;
    return (char *)p >= it->first && (char *)p + n <= it->first + it->second;
}

static hipError_t take(void **p, size_t n)
{
    // (a state's pages are never touched)
    void *m = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED)
        return hipErrorOutOfMemory;
    g_live[(char *)m] = n;
    *p = m;
    return hipSuccess;
}

static hipError_t give(void *p)
{
    auto it = g_live.find((char *)p);
    if (it == g_live.end())
        return p ? hipErrorInvalidValue : hipSuccess;
    if (it->second <= (size_t)64 << 20)
        memset(p, 0xff, it->second);
    g_live.erase(it);
    return hipSuccess;
}

static size_t g_largest = SIZE_MAX;   // device allocation that succeeds

// While a stream is captured, allocations and waits are refused, and what is queued
// happens when the graph is replayed.
static bool g_capturing = false;
static std::vector<std::function<void()>> g_nodes;
static void now(std::function<void()> f)
{
    if (g_capturing)
        g_nodes.push_back(f);
    else
        f();
}
static hipError_t refuse(hipError_t e) { return g_capturing ? hipErrorStreamCaptureUnsupported : e; }

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    return g_capturing ? refuse(hipSuccess) : n > g_largest ? hipErrorOutOfMemory : take(p, n);
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return g_capturing ? refuse(hipSuccess) : take(p, n); }
hipError_t hipFree(void *p) { return g_capturing ? refuse(hipSuccess) : give(p); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c)
{
    *c = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { return give(p); }
static int g_copies = 0;
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    ++g_copies;
    now([=] { memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
static hipError_t handle(void **h)
{
    static size_t n = 0;
    *h = (void *)(16 * ++n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle((void **)s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return refuse(hipSuccess); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return refuse(hipSuccess); }
hipError_t hipEventCreate(hipEvent_t *e) { return handle((void **)e); }
static int g_events_left = -1;   // events that can still be made (-1: any number)
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    if (g_events_left == 0)
        return hipErrorOutOfMemory;
    g_events_left -= g_events_left > 0;
    return handle((void **)e);
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetSymbolAddress(void **p, const void *s)
{
    *p = (void *)s;
    return hipSuccess;
}
}

// ---- plans ------------------------------------------------------------------------

static fq_graph *g_graph = nullptr;        // the graph of the program
static std::vector<Geom> g_geoms;          // the geometries its launches may use
static long g_checked = 0, g_wrong = 0;

template <typename T> static bool same(const PlanBlob &pb, size_t o, const T *at, size_t n)
{
    return n == 0 || (live(at, n * sizeof(T)) && memcmp(at, pb.bytes.data() + o, n * sizeof(T)) == 0);
}

// Whether p holds the plan of the graph for a geometry with these widths.
static bool plan_ok(const PlanDev &p, int Q, int nthr, int nh)
{
    for (const Geom &g : g_geoms) {
        if (g.Q != Q || g.nthr != nthr || g.nh != nh)
            continue;
        PlanBlob pb;
        build_plan(g_graph, g, pb);
        const int nnz = ((const int *)(pb.bytes.data() + pb.o_off))[Q];
        // (the scalars, which the caller holds, tell geometries of equal widths apart)
        if (pb.dev.n_hh == p.n_hh && pb.dev.wtot == p.wtot && memcmp(pb.dev.rr, p.rr, sizeof(p.rr)) == 0 &&
            same(pb, pb.o_cH, p.cH, Q) && same(pb, pb.o_om, p.omega, nh) && same(pb, pb.o_off, p.csr_off, Q + 1) &&
            same(pb, pb.o_ch, p.csr_h, nnz) && same(pb, pb.o_cw, p.csr_w, nnz) && same(pb, pb.o_hw, p.hh_w, p.n_hh) &&
            same(pb, pb.o_hu, p.hh_u, p.n_hh) && same(pb, pb.o_hv, p.hh_v, p.n_hh) &&
            same(pb, pb.o_thr, p.thr, (size_t)(1 + g.a_log) << nthr))
            return true;
    }
    return false;
}

static void check(const PlanDev &p, int Q, int nthr, int nh)
{
    now([=] {
        ++g_checked;
        if (!plan_ok(p, Q, nthr, nh))
            ++g_wrong;
    });
}

// Phase tables that captured launches read (and write).
static std::vector<const void *> g_captured;
static void note(const void *tab)
{
    if (g_capturing && tab)
        g_captured.push_back(tab);
}

// ---- launchers ----------------------------------------------------------------------

namespace fq {
int tile_max_q(int dtype) { return dtype == 0 ? 13 : 14; }
size_t tile_lds_bytes(int, int) { return 0; }
int mix_a_log(int dtype, int Q)
{
    if (dtype == 0)
        return Q >= 10 && Q <= 13 ? 4 : Q == 9 ? 3 : 0;
    return Q == 13 || Q == 14 ? 5 : Q >= 10 && Q <= 12 ? 4 : 0;
}
bool mix_lane_bit(int Q, int A, int k)
{
    const int b = Q - A - k * A - 1;
    return k > 0 && (b == 4 || b == 3 || b == 1 || b == 0);
}
int pair_a_log(int dtype, int Q)
{
    if (dtype == 0)
        return Q >= 9 && Q <= 12 ? 3 : 0;
    return Q >= 10 && Q <= 13 ? 4 : 0;
}
bool pair_lane_bit(int Q, int A, int k)
{
    const int b = Q - A - k * A - 1;
    return k > 0 && (b == 3 || b == 1 || b == 0);
}
size_t phase_table_entries(const TileArgs &a, int a_log)
{
    return (size_t)run_tiles(a) * (size_t)(a.Q + 1) + ((size_t)(1 + a_log) << a.nthr) + FQ_MAX_REGS;
}
hipError_t launch_phase_table(const TileArgs &a, int, double2 *, double *, hipStream_t)
{
    check(a.plan, a.Q, a.nthr, a.nh);
    return hipSuccess;
}
hipError_t launch_phase_tables(const TableJobs &m, int njobs, size_t, double2 *, double *, hipStream_t)
{
    for (int j = 0; j < njobs; ++j) {
        const TableGeo &g = m.geo[m.job[j].geo];
        check(g.plan, g.Q, g.nthr, g.nh);
    }
    return hipSuccess;
}
hipError_t launch_slab_phase_table(const TileArgs &a, int, const SlotParams *slots, const SlotPlans *plans, int nslots,
                                   double2 *, size_t, hipStream_t)
{
    for (int k = 0; k < nslots; ++k)
        if (slots[k].active)
            check(plans[k].cost[0], a.Q, a.nthr, a.nh);
    return hipSuccess;
}
hipError_t launch_slab_tables(const SlabGeos &g, const SlabJob *jobs, int njobs, size_t, const SlotPlans *plans,
                              double2 *, hipStream_t)
{
    for (int j = 0; j < njobs; ++j) {
        const TableGeo &t = g.geo[jobs[j].geo];
        check(plans[jobs[j].slot].cost[jobs[j].geo], t.Q, t.nthr, t.nh);
    }
    return hipSuccess;
}
hipError_t launch_slab_expect(int, int a_log, const void *, const TileArgs &a, const SlotPlans *plans, const int *fin,
                              int nfin, int slot_shift, double *, double *, hipStream_t)
{
    for (int i = 0; i < nfin; ++i)
        check(plans[fin[i]].expect, a.Q, a.Q - a_log, g_graph->N - a.Q);
    (void)slot_shift;
    return hipSuccess;
}
hipError_t launch_expect(int, int, const void *, const TileArgs &a, double *, double *, hipStream_t)
{
    check(a.plan, a.Q, a.nthr, a.nh);
    return hipSuccess;
}
hipError_t launch_cut_mul(int, int, const void *, void *, const TileArgs &a, double *, hipStream_t)
{
    check(a.plan, a.Q, a.nthr, a.nh);
    return hipSuccess;
}
static int g_boundaries = 0;   // boundary passes on single states
static int g_passes = 0;       // tile passes
static double g_factor[2] = {1.0, 0.0};   // product of the factors in the cost phases
static int g_common = 0;       // factors common to all amplitudes, multiplied in before the stores
hipError_t launch_mix(int, int, bool, int kind, int, void *, const MixArgs &a, const double2 *tab, hipStream_t)
{
    note(tab);
    ++g_passes;
    g_boundaries += kind == MIX_BOUNDARY && !a.slots;
    const int ns = a.slots ? a.nslots : 1;
    for (int i = 0; i < ns && a.tile0 == 0; ++i) {
        if (kind == MIX_PLAIN) {
            g_common += a.apply_scale != 0;
            continue;
        }
        const double x = a.slots ? a.slots[i].scale_re : a.scale_re, y = a.slots ? a.slots[i].scale_im : a.scale_im;
        const double re = g_factor[0] * x - g_factor[1] * y;
        g_factor[1] = g_factor[0] * y + g_factor[1] * x;
        g_factor[0] = re;
    }
    return hipSuccess;
}
hipError_t launch_tile(int, int, bool, bool, bool, void *, const TileArgs &, const double2 *, hipStream_t)
{
    ++g_passes;
    return hipSuccess;
}
hipError_t launch_tile_pre(int, int, void *, const TileArgs &, const double2 *, hipStream_t)
{
    ++g_passes;
    return hipSuccess;
}
hipError_t launch_tile_mirror(int, int, bool, void *, const TileArgs &, hipStream_t)
{
    ++g_passes;
    return hipSuccess;
}
hipError_t launch_solo(int, int, void *, const SoloArgs &, const double2 *tab, hipStream_t)
{
    note(tab);
    return hipSuccess;
}
hipError_t launch_pair_pass(int, int, bool, int, bool, void *, void *, const PairArgs &, const double2 *, const double *,
                            double *, hipStream_t) { return hipSuccess; }
hipError_t launch_pair_sums(const double *, uint64_t, int, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_pair(int, int, bool, bool, bool, void *, void *, const TileArgs &, const double2 *, const double *,
                       double *, unsigned *grid, hipStream_t)
{
    *grid = 1;
    return hipSuccess;
}
hipError_t launch_finalize(const double *, uint64_t, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_swap_small(int, void *, const SwapRuns &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_swap(int, void *, const SwapArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_topk(int, const void *, int, int, double *, uint64_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_gather(int, const void *, const uint64_t *, size_t, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_fill_zero_one(int, void *, int, hipStream_t) { return hipSuccess; }
hipError_t launch_stream(void *, size_t, int, float *, hipStream_t) { return hipSuccess; }
hipError_t launch_slab_pass(int, int, bool, bool, void *, const TileArgs &, const SlotParams *, int, hipStream_t)
{
    ++g_passes;
    return hipSuccess;
}
}  // namespace fq

// ---- programs -----------------------------------------------------------------------

static void ok(int rc)
{
    if (rc) {
        fprintf(stderr, "failed (%d): %s\n", rc, fq_last_error());
        exit(1);
    }
}

static void add_plan_geoms(int N, const LayerPlan &lp, int A)
{
    for (const FusedPass &p : lp.ps)
        for (int K = 0; K <= 3; ++K)
            g_geoms.push_back(layout_geom(N, p.tile, A, K));
}

static fq_graph *dense_graph(int N)
{
    fq_graph *g = nullptr;
    ok(fq_graph_create(N, &g));
    for (int i = 0; i < N; ++i)
        for (int j = i + 1; j < N; ++j)
            ok(fq_graph_add_edge(g, i, j, 0.25 + 0.01 * i + 0.001 * j));
    g_graph = g;
    return g;
}

// Every geometry that the calls on N qubits use.
static void all_geoms(int N, int dtype)
{
    for (int z2 = 0; z2 < 2; ++z2) {
        const LayerPlan lp = exec_plan(N, dtype, z2 != 0, 1);
        add_plan_geoms(N, lp, mix_a_log(dtype, (int)lp.ps[0].tile.size()));
        const int Q = std::min(12, N - z2);
        g_geoms.push_back(make_geom(N, low_tile(Q), std::min(4, Q)));
        const int Qs = std::min(tile_max_q(dtype), N - z2);
        g_geoms.push_back(make_geom(N, low_tile(Qs), tile_a_log(dtype, Qs)));
    }
    const LayerPlan lp = pair_plan(N, dtype);
    if (!lp.ps.empty())
        add_plan_geoms(N, lp, pair_a_log(dtype, (int)lp.ps[0].tile.size()));
    if (N >= solo_min(dtype) && N <= solo_max(dtype))
        for (int K = 0; K <= 2; K += 2)
            g_geoms.push_back(layout_geom(N, low_tile(N), mix_a_log(dtype, N), K));
}

// plans <call> N dtype P small: `small` cost plans of other weights (of <C>, the
// smallest there are), then the call on new weights, four times.
static int plans(const std::string &call, int N, int dtype, int P, int small)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    std::vector<double> gm(P, 0.3), bt(P, 0.2), gg(P), gb(P);
    int step = 0;
    auto change = [&] { ok(fq_graph_add_edge(g, 0, N - 1, 1.0 + ++step)); };
    for (int i = 0; i < small; ++i) {
        change();
        double e;
        ok(fq_expect_cut(st, g, &e, nullptr));
    }
    fq_slab *sb = nullptr;
    if (call == "slab" || call == "slab_z2")
        ok(fq_slab_create_sched(N, 2, dtype, call == "slab" ? FQ_SCHED_FUSED : FQ_SCHED_Z2, &sb));
    for (int rep = 0; rep < 4; ++rep) {
        change();
        if (sb) {
            for (int k = 0; k < 2; ++k)
                ok(fq_slab_assign(sb, k, g, P, gm.data(), bt.data()));
            for (int p = 0; p < P; ++p)
                ok(fq_slab_step(sb, nullptr));
            int n = 0;
            ok(fq_slab_collect(sb, nullptr, nullptr, nullptr, &n));
        } else if (call == "backward") {
            double e;
            ok(fq_backward(st, g, P, gm.data(), bt.data(), &e, gg.data(), gb.data()));
        } else {
            ok(fq_run(st, g, P, gm.data(), bt.data(), call == "z2" ? FQ_SCHED_Z2 : FQ_SCHED_FUSED));
        }
    }
    // the cache stays bounded: the plans of a call beyond its limit at most
    printf("cached %zu\n", g->plans.size());
    if (sb)
        ok(fq_slab_destroy(sb));
    ok(fq_state_destroy(st));
    return 0;
}

// capture N dtype schedule P0 P1 P2: a run of P0 layers, one of P1 captured, one of P2,
// a cost layer and a gradient.
static int capture(int N, int dtype, int sched, int P0, int P1, int P2)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    const int most = std::max({P0, P1, P2});
    std::vector<double> gm(most, 0.3), bt(most, 0.2), gg(most), gb(most);
    auto run = [&](int P) { ok(fq_run(st, g, P, gm.data(), bt.data(), sched)); };
    run(P0);
    g_capturing = true;
    run(P1);
    g_capturing = false;
    run(P2);
    double e;
    ok(fq_backward(st, g, P2, gm.data(), bt.data(), &e, gg.data(), gb.data()));
    ok(fq_cost_layer(st, g, 0.3, 1));
    for (const void *p : g_captured) {
        ++g_checked;
        g_wrong += !live(p, sizeof(double2));
    }
    const size_t before = g_live.size();
    ok(fq_state_destroy(st));
    // (the stream and its page stay with the library)
    printf("freed %d\n", (int)(before - g_live.size()));
    size_t lost = 0;
    for (const void *p : g_captured)
        lost += live(p, 1);
    printf("kept %zu\n", lost);
    return 0;
}

// reopen N dtype schedule
static int reopen(int N, int dtype, int sched)
{
    fq_graph *g = dense_graph(N);
    fq_slab *sb = nullptr;
    ok(fq_slab_create_sched(N, 2, dtype, sched, &sb));
    std::vector<double> gm(4, 0.3), bt(4, 0.2);
    ok(fq_slab_assign(sb, 0, g, 4, gm.data(), bt.data()));
    ok(fq_slab_step(sb, nullptr));
    ok(fq_graph_add_edge(g, 0, 1, 2.0));
    g_boundaries = 0;
    g_events_left = 1;   // (the phase of the difference has one plan)
    printf("failed %d\n", (int)(fq_slab_step(sb, nullptr) != FQ_OK));
    g_events_left = -1;
    printf("reopened %d\n", g_boundaries);
    const bool own = !sb->packed;   // the step itself then runs such a pass
    ok(fq_slab_step(sb, nullptr));
    printf("again %d\n", g_boundaries - own);
    ok(fq_slab_destroy(sb));
    return 0;
}

// Plan lp of an N-qubit state and its launches for P layers; a_log, lane_bit: of its kernels.
static void cover_plan(int N, const LayerPlan &lp, bool z2, int P, int (*a_log)(int, int), bool (*lane_bit)(int, int, int),
                       int dtype)
{
    auto need = [&](bool good, const char *what) {
        ++g_checked;
        if (!good) {
            ++g_wrong;
            fprintf(stderr, "N=%d dtype=%d z2=%d P=%d: %s\n", N, dtype, z2, P, what);
        }
    };
    const int m = (int)lp.ps.size(), Q = (int)lp.ps[0].tile.size(), A = a_log(dtype, Q);
    std::vector<int> gated(N, 0);
    for (int i = 0; i < m; ++i) {
        const FusedPass &fp = lp.ps[i];
        need((int)fp.tile.size() == Q, "tiles of one width");
        need(std::set<int>(fp.tile.begin(), fp.tile.end()).size() == fp.tile.size(), "distinct positions");
        for (int q : fp.tile)
            need(q >= 0 && q < N, "a position of the state");
        for (int q : fp.gates) {
            gated[q]++;
            need(std::count(fp.tile.begin(), fp.tile.end(), q) == 1, "a gated qubit in the tile");
        }
        if (z2) {
            const bool top = std::count(fp.tile.begin(), fp.tile.end(), N - 1) > 0;
            need(top == (i + 1 == m) && (!top || fp.tile.back() == N - 1), "the top qubit on the last register bit");
        }
        if (A == 0) {
            need(geom_runs(make_geom(N, fp.tile, tile_a_log(dtype, Q))) <= FQ_MAX_RUNS, "bit runs");
            continue;
        }
        MixArgs a;
        int K = 0;
        bool lane = false;
        ok(pass_shape(N, fp.tile, fp.gates, A, lane_bit, !z2 ? Z2_OFF : i + 1 == m ? Z2_MIRROR : Z2_LOWER, a, K, lane));
        need(K == 0 || Q - A > (K - 1) * A, "an instance with as many exchanges");
        int rx = lane;
        for (uint32_t w = a.gates_w; w; w &= w - 1)
            ++rx;
        need(rx == (int)fp.gates.size(), "every gated qubit in a layout");
    }
    for (int q = 0; q < N; ++q)
        need(gated[q] == 1, "one RX on each qubit");
    std::vector<Step> seq;
    for (int p = 0; p < P; ++p)
        layer_steps(lp, p, P, seq);
    std::vector<int> rx(N, -1);   // the last layer whose RX a qubit has had
    int phase = -1;               // the last layer whose phase has run
    for (const Step &s : seq) {
        auto apply = [&](int layer) {
            need(phase == layer, "RX after its layer's phase");
            for (int q : lp.ps[s.pass].gates) {
                need(rx[q] == layer - 1, "RX in order");
                rx[q] = layer;
            }
        };
        if (s.kind == STEP_BOUNDARY)
            apply(s.layer);
        if (s.kind != STEP_PLAIN) {
            ++phase;
            need(std::count(rx.begin(), rx.end(), phase - 1) == N, "the phase after the layer before");
        }
        apply(s.kind == STEP_BOUNDARY ? s.layer + 1 : s.layer);
    }
    need(std::count(rx.begin(), rx.end(), P - 1) == N, "all layers");
    need(!z2 || (seq.back().kind == STEP_PLAIN && seq.back().pass + 1 == m) || a_log == pair_a_log,
         "the mirror pass last");
    for (size_t k = 0, n; k < seq.size(); k += n) {
        n = chunk_group(lp, seq, k);
        int cost = 0;
        for (size_t i = k; i < k + n && n > 1; ++i) {
            cost += seq[i].kind != STEP_PLAIN;
            for (int q : lp.ps[seq[i].pass].tile)
                need(q < lp.chunk && lp.chunk < N - z2, "a pass within a chunk");
        }
        need(cost <= 1, "one phase table a chunk");
    }
}

// newplan N dtype schedule P
static int newplan(int N, int dtype, int sched, int P)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    const std::vector<double> gm(P, 0.3), bt(P, 0.2);
    auto run = [&] { ok(fq_run(st, g, P, gm.data(), bt.data(), sched)); };
    run();
    ok(fq_graph_add_edge(g, 0, 1, 3.0));
    g_capturing = true;
    run();
    g_capturing = false;
    for (int rep = 0; rep < 2; ++rep) {
        run();
        for (auto &f : g_nodes)
            f();
    }
    printf("nodes %zu\n", g_nodes.size());
    ok(fq_state_destroy(st));
    return 0;
}

// dropped N dtype P: <C> plans alone are cached when the run is captured
static int dropped(int N, int dtype, int P)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    const std::vector<double> gm(P, 0.3), bt(P, 0.2);
    auto run = [&] { ok(fq_run(st, g, P, gm.data(), bt.data(), FQ_SCHED_FUSED)); };
    double e;
    ok(fq_expect_cut(st, g, &e, nullptr));
    ok(reserve_phases(st, (size_t)1 << 20));   // (room for the tables)
    g_capturing = true;
    run();
    g_capturing = false;
    const std::vector<double> W = g->W;
    const auto nodes = g_nodes;
    for (int i = 1; i < FQ_PLAN_CACHE; ++i) {
        ok(fq_graph_add_edge(g, 0, 1, 3.0 + i));
        ok(fq_expect_cut(st, g, &e, nullptr));
    }
    const uint64_t epoch = g->plan_epoch;
    ok(fq_graph_add_edge(g, 0, 1, 2.0));
    run();
    printf("drops %d\n", (int)(g->plan_epoch - epoch));
    const std::vector<double> W2 = g->W;
    g->W = W;
    for (auto &f : nodes)
        f();
    g->W = W2;
    ok(fq_state_destroy(st));
    ok(fq_graph_destroy(g));
    printf("nodes %zu\n", nodes.size());
    return 0;
}

// nomem N dtype schedule P KiB: the largest allocation that succeeds once the state is made
static int nomem(int N, int dtype, int sched, int P, int kib)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    const std::vector<double> gm(P, 0.3), bt(P, 0.2);
    g_largest = (size_t)kib << 10;
    ok(fq_run(st, g, P, gm.data(), bt.data(), sched));
    g_largest = SIZE_MAX;
    ok(fq_state_destroy(st));
    return 0;
}

// deep <call> N dtype P: the growth of resident memory
static int deep(const std::string &call, int N, int dtype, int P)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_state *st = nullptr;
    ok(fq_state_create(N, 0, 0, std::min(N, 10), dtype, &st));
    const std::vector<double> gm(P, 0.3), bt(P, 0.2);
    std::vector<double> gg(P), gb(P);
    auto run = [&](int p) {
        double e;
        if (call == "backward")
            ok(fq_backward(st, g, p, gm.data(), bt.data(), &e, gg.data(), gb.data()));
        else
            ok(fq_run(st, g, p, gm.data(), bt.data(), call == "z2" ? FQ_SCHED_Z2 : FQ_SCHED_FUSED));
    };
    auto kib = [] {   // (ru_maxrss would be the parent's where that is larger)
        long k = 0;
        FILE *f = fopen("/proc/self/status", "r");
        for (char line[256]; f && fgets(line, sizeof(line), f);)
            sscanf(line, "VmHWM: %ld", &k);
        fclose(f);
        return k;
    };
    run(256);   // (scratch as large as it gets)
    const long before = kib();
    run(P);
    printf("bytes_per_layer %ld\n", (kib() - before) * 1024 / P);
    ok(fq_state_destroy(st));
    return 0;
}

// cover N0 N1: states of N0 to N1 qubits
static int cover(int N0, int N1)
{
    for (int N = N0; N <= N1; ++N)
        for (int dtype = 0; dtype < 2; ++dtype)
            for (int P = 1; P <= 4; ++P) {
                for (int z2 = 0; z2 < (N >= 3 ? 2 : 1); ++z2)
                    cover_plan(N, exec_plan(N, dtype, z2 != 0, P), z2 != 0, P, mix_a_log, mix_lane_bit, dtype);
                const LayerPlan lp = pair_plan(N, dtype);
                if (!lp.ps.empty())
                    cover_plan(N, lp, true, P, pair_a_log, pair_lane_bit, dtype);
            }
    return 0;
}

// copies N dtype K: slots 0, 3, 6 .. of K enter, then the others; every slot's result
// comes from its own graph's plans
static int copies(int N, int dtype, int K)
{
    fq_graph *g = dense_graph(N);
    all_geoms(N, dtype);
    fq_slab *sb = nullptr;
    ok(fq_slab_create_sched(N, K, dtype, FQ_SCHED_Z2, &sb));
    const std::vector<double> gm(3, 0.3), bt(3, 0.2);
    int most = 0;
    for (int rest = 0; rest < 2; ++rest) {
        for (int k = 0; k < K; ++k)
            if ((k % 3 != 0) == (rest != 0))
                ok(fq_slab_assign(sb, k, g, 3, gm.data(), bt.data()));
        g_copies = 0;
        ok(fq_slab_step(sb, nullptr));
        most = std::max(most, g_copies);
    }
    for (int p = 0; p < 3; ++p)
        ok(fq_slab_step(sb, nullptr));
    ok(fq_slab_destroy(sb));
    printf("copies %d\n", most);
    return 0;
}

// factors <call> N dtype P: the product of all factors is that of RX(beta_p) on N qubits each
static int factors(const std::string &call, int N, int dtype, int P)
{
    fq_graph *g = dense_graph(N);
    std::vector<double> gm(P, 0.3), bt(P);
    for (int p = 0; p < P; ++p)
        bt[p] = 0.3 + 0.7 * p;   // (both branches of the butterfly)
    fq_slab *sb = nullptr;
    ok(fq_slab_create_sched(N, 1, dtype, call == "slab" ? FQ_SCHED_FUSED : FQ_SCHED_Z2, &sb));
    ok(fq_slab_assign(sb, 0, g, P, gm.data(), bt.data()));
    for (int p = 0; p < P; ++p)
        ok(fq_slab_step(sb, nullptr));
    ok(fq_slab_destroy(sb));
    double t, re = 1.0, im = 0.0;
    for (int p = 0; p < P; ++p) {
        double sr, si;
        rx_tform(bt[p], dtype, true, &t, &sr, &si);
        for (int q = 0; q < N; ++q) {
            const double x = re * sr - im * si;
            im = re * si + im * sr;
            re = x;
        }
    }
    printf("common %d off %d\n", g_common, (int)!(std::hypot(g_factor[0] - re, g_factor[1] - im) <= 1e-12 * std::hypot(re, im)));
    return 0;
}

// passes N dtype schedule P
static int passes(int N, int dtype, int sched, int P)
{
    fq_graph *g = dense_graph(N);
    fq_slab *sb = nullptr;
    ok(fq_slab_create_sched(N, 2, dtype, sched, &sb));
    const std::vector<double> gm(P, 0.3), bt(P, 0.2);
    ok(fq_slab_assign(sb, 1, g, P, gm.data(), bt.data()));
    for (int p = 0; p < P; ++p)
        ok(fq_slab_step(sb, nullptr));
    int told = 0;
    ok(fq_slab_passes(N, dtype, sched, P, &told));
    printf("launched %d told %d\n", g_passes, told);
    ok(fq_slab_destroy(sb));
    return 0;
}

int main(int argc, char **argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    auto num = [&](int i) { return i < argc ? atoi(argv[i]) : 0; };
    int rc = 2;
    if (what == "plans" && argc == 7)
        rc = plans(argv[2], num(3), num(4), num(5), num(6));
    if (what == "capture" && argc == 8)
        rc = capture(num(2), num(3), num(4), num(5), num(6), num(7));
    if (what == "newplan" && argc == 6)
        rc = newplan(num(2), num(3), num(4), num(5));
    if (what == "dropped" && argc == 5)
        rc = dropped(num(2), num(3), num(4));
    if (what == "nomem" && argc == 7)
        rc = nomem(num(2), num(3), num(4), num(5), num(6));
    if (what == "deep" && argc == 6)
        rc = deep(argv[2], num(3), num(4), num(5));
    if (what == "cover" && argc == 4)
        rc = cover(num(2), num(3));
    if (what == "copies" && argc == 5)
        rc = copies(num(2), num(3), num(4));
    if (what == "factors" && argc == 6)
        rc = factors(argv[2], num(3), num(4), num(5));
    if (what == "passes" && argc == 6)
        rc = passes(num(2), num(3), num(4), num(5));
    if (what == "reopen" && argc == 5)
        rc = reopen(num(2), num(3), num(4));
    printf("checked %ld wrong %ld\n", g_checked, g_wrong);
    return rc;
}
