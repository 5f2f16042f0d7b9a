// fq_api.cpp -- host side of libforqaoa: handles, validation, cost plans, the
// layer schedules and the C ABI declared in include/forqaoa.h.
#include "forqaoa.h"
#include "fq_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

using namespace fq;

// ---- errors ------------------------------------------------------------------

static thread_local char g_err[512] = "";

static int set_err(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define FQ_HIP(call)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess)                                                               \
            return set_err(FQ_ERR_DEVICE, "%s failed: %s", #call, hipGetErrorString(e_));   \
    } while (0)

extern "C" const char *fq_last_error(void) { return g_err; }

// ---- HBM budget (states and slabs) ----------------------------------------------

#include <mutex>
static std::mutex g_budget_mu;
static size_t g_budget = SIZE_MAX;
static size_t g_in_use = 0;

static bool budget_take(size_t bytes)
{
    std::lock_guard<std::mutex> lk(g_budget_mu);
    if (g_in_use + bytes > g_budget || g_in_use + bytes < g_in_use)
        return false;
    g_in_use += bytes;
    return true;
}

static void budget_give(size_t bytes)
{
    std::lock_guard<std::mutex> lk(g_budget_mu);
    g_in_use = bytes > g_in_use ? 0 : g_in_use - bytes;
}

extern "C" int fq_set_memory_budget(size_t bytes)
{
    std::lock_guard<std::mutex> lk(g_budget_mu);
    g_budget = bytes ? bytes : SIZE_MAX;
    return FQ_OK;
}

extern "C" int fq_memory_in_use(size_t *bytes)
{
    if (!bytes)
        return set_err(FQ_ERR_ARG, "null output pointer");
    std::lock_guard<std::mutex> lk(g_budget_mu);
    *bytes = g_in_use;
    return FQ_OK;
}
extern "C" int fq_version(void) { return 100; }

// ---- RX coefficients ---------------------------------------------------------------

void fq::rx_coeffs(double beta, int dtype, double *c, double *s)
{
    double sn, cs;
    sincos(beta / 2, &sn, &cs);
    if (dtype != FQ_C64) {
        *c = cs;
        *s = sn;
        return;
    }
    // Search FP32 pairs within 3 ulps of the rounded |cos|, |sin| for the
    // smallest |c^2 + s^2 - 1| + |angle error| (both exact or nearly so in FP64:
    // a product of two FP32 values is exact).  Working on magnitudes and
    // restoring the signs afterwards makes RX(-beta) the exact inverse-transpose
    // partner of RX(beta), as the adjoint's uncompute needs.
    const double ac = std::fabs(cs), as = std::fabs(sn);
    const double half = std::atan2(as, ac);
    const float c0 = (float)ac, s0 = (float)as;
    float cb = c0, sb = s0;
    double best = HUGE_VAL;
    for (int i = -3; i <= 3; ++i) {
        float ci = c0;
        for (int k = 0; k < std::abs(i); ++k)
            ci = std::nextafterf(ci, i < 0 ? 0.0f : 2.0f);
        if (ci < 0.0f || ci > 1.0f)
            continue;
        for (int j = -3; j <= 3; ++j) {
            float sj = s0;
            for (int k = 0; k < std::abs(j); ++k)
                sj = std::nextafterf(sj, j < 0 ? 0.0f : 2.0f);
            if (sj < 0.0f || sj > 1.0f)
                continue;
            const double dn = (double)ci * ci + (double)sj * sj - 1.0;
            const double da = std::atan2((double)sj, (double)ci) - half;
            const double score = std::fabs(dn) + std::fabs(da);
            if (score < best) {
                best = score;
                cb = ci;
                sb = sj;
            }
        }
    }
    *c = std::copysign((double)cb, cs);
    *s = std::copysign((double)sb, sn);
}

void fq::rx_tform(double beta, int dtype, bool flip, double *t, double *sigma_re, double *sigma_im)
{
    double sn, cs;
    sincos(beta / 2, &sn, &cs);
    const bool f = flip && std::fabs(sn) > std::fabs(cs);
    double tt = f ? -cs / sn : sn / cs;
    if (dtype == FQ_C64)
        tt = (double)(float)tt;
    *t = tt;
    const double mag = 1.0 / std::sqrt(1.0 + tt * tt);
    *sigma_re = f ? 0.0 : std::copysign(mag, cs);
    *sigma_im = f ? -std::copysign(mag, sn) : 0.0;
}

// RX(beta) as applied with rx_coeffs is sqrt(c^2 + s^2) times a unitary, a
// global factor per gate.  A P-layer evaluation gives every qubit one RX per
// layer, so its state is prod_p (c_p^2 + s_p^2)^(N/2) times the state of a
// unitary circuit; scaling the launch-control amplitude by the inverse removes
// that factor exactly (1 for complex128, where c^2 + s^2 - 1 is ~1e-16).
static double rx_norm_scale(int N, int P, const double *betas, int dtype)
{
    if (dtype != FQ_C64)
        return 1.0;
    double sc = 1.0;
    for (int p = 0; p < P; ++p) {
        double c, s;
        rx_coeffs(betas[p], dtype, &c, &s);
        sc *= std::pow(c * c + s * s, -0.5 * N);
    }
    return sc;
}

// ---- streams the library created -----------------------------------------------
//
// States and slabs run on streams the library creates (a state may be moved to
// a caller's stream instead).  A cached cost plan that is replaced must first
// be released by every stream it was handed to; the library can order that on
// the device only for its own live streams (a destroyed one finished its work
// when it was destroyed), so it keeps a registry of them.

static std::mutex g_streams_mu;
static std::set<hipStream_t> g_own_streams;

static void own_stream(hipStream_t s, bool live)
{
    std::lock_guard<std::mutex> lk(g_streams_mu);
    if (live)
        g_own_streams.insert(s);
    else
        g_own_streams.erase(s);
}

static bool is_own_stream(hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_streams_mu);
    return g_own_streams.count(s) != 0;
}

// A state's stream and a page of pinned host memory that its kernels write results
// to.  Both outlive it: up to FQ_LANES idle ones are kept for the next states
// (making a stream takes 60 to 130 us; a state was made in 78 to 143 us, and now in 8
// to 16).  A result that the kernels write themselves needs no copy behind them:
// <C> at N=16 27 -> 18.5 us.
#define FQ_LANES 16
#define FQ_LANE_DOUBLES 512
struct Lane {
    hipStream_t stream = nullptr;
    double *host = nullptr;
    bool shared = false;   // host is one of g_pages
    int device = -1;
};
static std::mutex g_lanes_mu;
static std::vector<Lane> g_lanes;
static std::vector<double *> g_pages;   // free ones of the first FQ_LANES, allocated together
static bool g_pages_made = false;

static bool lane_take(Lane &l)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return false;
    {
        std::lock_guard<std::mutex> lk(g_lanes_mu);
        for (size_t i = 0; i < g_lanes.size(); ++i)
            if (g_lanes[i].device == dev) {
                l = g_lanes[i];
                g_lanes.erase(g_lanes.begin() + i);
                return true;
            }
    }
    l.device = dev;
    if (hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking) != hipSuccess)
        return false;
    {
        std::lock_guard<std::mutex> lk(g_lanes_mu);
        double *m = nullptr;
        if (!g_pages_made &&
            hipHostMalloc(&m, sizeof(double) * FQ_LANE_DOUBLES * FQ_LANES, hipHostMallocPortable) == hipSuccess) {
            g_pages_made = true;
            for (int i = 0; i < FQ_LANES; ++i)
                g_pages.push_back(m + (size_t)FQ_LANE_DOUBLES * i);
        }
        if (!g_pages.empty()) {
            l.host = g_pages.back();
            l.shared = true;
            g_pages.pop_back();
            return true;
        }
    }
    if (hipHostMalloc(&l.host, sizeof(double) * FQ_LANE_DOUBLES, hipHostMallocDefault) != hipSuccess) {
        hipStreamDestroy(l.stream);
        l.stream = nullptr;
        return false;
    }
    return true;
}

// (its work is done)
static void lane_give(const Lane &l)
{
    {
        std::lock_guard<std::mutex> lk(g_lanes_mu);
        if (g_lanes.size() < FQ_LANES) {
            g_lanes.push_back(l);
            return;
        }
        if (l.shared)
            g_pages.push_back(l.host);
    }
    hipStreamDestroy(l.stream);
    if (!l.shared)
        hipHostFree(l.host);
}

// ---- handles -------------------------------------------------------------------

struct PlanEntry {
    char *dmem = nullptr;         // in a block of the graph, as staging
    size_t cap = 0;               // bytes of both
    PlanDev dev{};
    char *staging = nullptr;      // pinned copy of the blob (asynchronous upload)
    hipEvent_t ready = nullptr;   // upload done
    hipStream_t stream = nullptr; // stream the upload was queued on
    std::vector<hipStream_t> users; // streams the plan was handed to
    bool foreign = false;         // handed to a stream the library did not create
    uint64_t last_use = 0;        // fq_graph::use_clock at the last lookup
};

// Memory of a graph's plans: device and pinned memory in blocks (a pinned
// allocation for each plan took 30 us and more, and a slab's graph has five plans).
#define FQ_PLAN_BLOCK ((size_t)64 << 10)
struct PlanBlock {
    char *dmem = nullptr, *staging = nullptr;
    size_t used = 0, size = 0;
    bool captured = false;   // holds a plan that a captured graph uploads and reads
};

// Plans cached per graph; beyond this the least recently used plan's buffers
// are reused for the next one, unless it is held (PlanHold).
#define FQ_PLAN_CACHE 64

struct fq_graph {
    int N = 0;
    std::vector<double> W;  // N*N, W[min*N+max], current labels
    // key: tile geometry + the bytes of W, so a hit is an exact content match
    std::map<std::string, PlanEntry> plans;
    std::vector<PlanBlock> blocks;
    uint64_t version = 1;       // bumped by every change of W
    uint64_t plan_epoch = 0;    // bumped when a cached plan is dropped or reused
    uint64_t use_clock = 0;
    int holds = 0;              // PlanHold's alive
    uint64_t held_from = 0;     // use_clock when the first of them was made
};

// While one is alive, plans of the graph that get_plan hands out stay as they are: for
// a caller that looks up several plans before it launches what reads the first.
struct PlanHold {
    fq_graph *g;
    explicit PlanHold(fq_graph *graph) : g(graph)
    {
        if (g->holds++ == 0)
            g->held_from = g->use_clock;
    }
    PlanHold(PlanHold &&o) noexcept : g(o.g) { o.g = nullptr; }
    PlanHold(const PlanHold &) = delete;
    PlanHold &operator=(const PlanHold &) = delete;
    ~PlanHold()
    {
        if (g)
            --g->holds;
    }
};

// Drops all cached plans of a graph (all: also the memory of captured graphs' plans);
// the caller has synchronized the device (hipFree waits for the whole device anyway).
static void plans_free(fq_graph *G, bool all)
{
    for (auto &kv : G->plans)
        if (kv.second.ready)
            hipEventDestroy(kv.second.ready);
    G->plans.clear();
    std::vector<PlanBlock> kept;
    for (PlanBlock &b : G->blocks) {
        if (b.captured && !all) {
            kept.push_back(b);
            continue;
        }
        hipFree(b.dmem);
        hipHostFree(b.staging);
    }
    G->blocks.swap(kept);
}

// cap bytes of both memories for a plan, from the last block or a new one.
static bool plan_memory(fq_graph *G, size_t cap, PlanEntry &e)
{
    if (G->blocks.empty() || G->blocks.back().size - G->blocks.back().used < cap) {
        PlanBlock b;
        b.size = std::max(cap, FQ_PLAN_BLOCK);
        if (hipMalloc(&b.dmem, b.size) != hipSuccess)
            return false;
        if (hipHostMalloc(&b.staging, b.size, hipHostMallocDefault) != hipSuccess) {
            hipFree(b.dmem);
            return false;
        }
        G->blocks.push_back(b);
    }
    PlanBlock &b = G->blocks.back();
    e.dmem = b.dmem + b.used;
    e.staging = b.staging + b.used;
    e.cap = cap;
    b.used += cap;
    return true;
}

struct TimingRec {
    int kind;
    hipEvent_t e0, e1;
    double bytes;
    int count;   // passes in it
};

struct fq_state {
    int N = 0, D = 0, B = 0, C = 0, dtype = 0;
    size_t elem = 16, bytes = 0;
    void *sv = nullptr;
    Lane lane;
    hipStream_t stream = nullptr;   // the lane's, or a caller's
    // chunked runs (run_chunks): two streams forked from and joined to `stream`
    hipStream_t side[2] = {nullptr, nullptr};
    hipEvent_t forked = nullptr, joined[2] = {nullptr, nullptr};
    int qmap[FQ_MAXN];
    double init_amp = 0;
    // product of the RX factors of tile passes that left theirs to a later
    // pass (run_layer); 1 between entry points
    double pending_re = 1.0, pending_im = 0.0;
    // inside fq_run: every RX applies one angle to all qubits of an
    // X^(x)N-symmetric state, so rx_tform may drop its X (see rx_tform)
    bool in_run = false;
    bool slot = false;         // a slab's slot (pass_factor)
    double *d_part = nullptr;  // expect partials
    size_t part_cap = 0;
    double *d_cand_p = nullptr;
    uint64_t *d_cand_i = nullptr;
    int cand_blocks = 0;
    double2 *d_phase = nullptr;  // per-launch cost phase factors
    size_t phase_cap = 0;        // bytes
    std::vector<double2 *> old_phase;   // smaller ones before it (reserve_phases)
    void *aux = nullptr;         // adjoint state (lambda), allocated on first use
    double *d_grad = nullptr;    // adjoint per-pass sums
    size_t grad_cap = 0;
    double *d_pair = nullptr;    // partial sums of the pair passes
    size_t pair_cap = 0;
    bool timing = false;
    std::vector<TimingRec> pending;
    std::vector<hipEvent_t> pool;
    double t_ms[FQ_K_COUNT] = {0};
    int64_t t_cnt[FQ_K_COUNT] = {0};
    double t_bytes[FQ_K_COUNT] = {0};
};

static void free_phases(fq_state *st)
{
    for (double2 *p : st->old_phase)
        hipFree(p);
    st->old_phase.clear();
    hipFree(st->d_phase);
    st->d_phase = nullptr;
    st->phase_cap = 0;
}

// ---- timing ------------------------------------------------------------------

static hipEvent_t pool_get(fq_state *st)
{
    if (!st->pool.empty()) {
        hipEvent_t e = st->pool.back();
        st->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess)
        return nullptr;
    return e;
}

static int timing_collect(fq_state *st)
{
    size_t done = 0;
    int rc = FQ_OK;
    for (; done < st->pending.size(); ++done) {
        const TimingRec &r = st->pending[done];
        hipError_t e = hipEventSynchronize(r.e1);
        float ms = 0;
        if (e == hipSuccess)
            e = hipEventElapsedTime(&ms, r.e0, r.e1);
        if (e != hipSuccess) {
            rc = set_err(FQ_ERR_DEVICE, "timing event failed: %s", hipGetErrorString(e));
            break;
        }
        st->t_ms[r.kind] += ms;
        st->t_cnt[r.kind] += r.count;
        st->t_bytes[r.kind] += r.bytes;
        st->pool.push_back(r.e0);
        st->pool.push_back(r.e1);
    }
    // collected records leave the list (a failed one stays for a later call)
    st->pending.erase(st->pending.begin(), st->pending.begin() + (std::ptrdiff_t)done);
    return rc;
}

// Wrap one launch (or the launches of `count` passes) with events when timing is on.
template <typename F>
static int timed(fq_state *st, int kind, double bytes, F &&launch, int count = 1)
{
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (st->timing) {
        if (st->pending.size() > 4096) {
            int rc = timing_collect(st);
            if (rc)
                return rc;
        }
        e0 = pool_get(st);
        e1 = pool_get(st);
        if (!e0 || !e1 || hipEventRecord(e0, st->stream) != hipSuccess) {
            if (e0)
                st->pool.push_back(e0);
            if (e1)
                st->pool.push_back(e1);
            return set_err(FQ_ERR_DEVICE, "timing event unavailable");
        }
    }
    hipError_t e = launch();
    if (e == hipSuccess && st->timing)
        e = hipEventRecord(e1, st->stream);
    if (e != hipSuccess) {
        if (st->timing) {
            st->pool.push_back(e0);
            st->pool.push_back(e1);
        }
        return set_err(FQ_ERR_DEVICE, "kernel launch failed: %s", hipGetErrorString(e));
    }
    if (st->timing)
        st->pending.push_back({kind, e0, e1, bytes, count});
    return FQ_OK;
}

// ---- geometry ------------------------------------------------------------------

struct Geom {
    int N, Q, a_log, nthr, nh;
    uint8_t tpos[16];
    uint8_t hpos[FQ_MAXN];
};

// tile: positions in order (thread bits first, the last a_log are register bits)
static Geom make_geom(int N, const std::vector<int> &tile, int a_log)
{
    Geom g{};
    g.N = N;
    g.Q = (int)tile.size();
    g.a_log = a_log;
    g.nthr = g.Q - a_log;
    g.nh = N - g.Q;
    bool in_tile[FQ_MAXN] = {false};
    for (int i = 0; i < g.Q; ++i) {
        g.tpos[i] = (uint8_t)tile[i];
        in_tile[tile[i]] = true;
    }
    int h = 0;
    for (int p = 0; p < N; ++p)
        if (!in_tile[p])
            g.hpos[h++] = (uint8_t)p;
    return g;
}

// Group consecutive index bits that land on consecutive positions; returns
// the number of runs (may exceed FQ_MAX_RUNS: then r is not usable).
static int make_runs(const uint8_t *pos, int n, BitRuns &r)
{
    int cnt = 0;
    r.n = 0;
    for (int i = 0; i < n;) {
        int j = i + 1;
        while (j < n && pos[j] == pos[j - 1] + 1)
            ++j;
        if (cnt < FQ_MAX_RUNS)
            r.run[cnt] = (uint32_t)i | ((uint32_t)(j - i) << 8) | ((uint32_t)pos[i] << 16);
        cnt++;
        i = j;
    }
    r.n = cnt < FQ_MAX_RUNS ? cnt : FQ_MAX_RUNS;
    return cnt;
}

static int geom_runs(const Geom &g)
{
    BitRuns r;
    return std::max(make_runs(g.hpos, g.nh, r), make_runs(g.tpos, g.nthr, r));
}

// Tile order of the persistent passes (tile_at): 2, one contiguous range of
// tiles per work-group (measured fastest on MI355X for the contiguous and
// the strided passes); FQ_TILE_ORDER (environment, read per call) selects
// another.
static uint32_t tile_order()
{
    const char *e = getenv("FQ_TILE_ORDER");
    return (uint32_t)(e ? std::max(0, std::min(3, atoi(e))) : 2);
}

static void geom_to_args(const Geom &g, TileArgs &a)
{
    memset(&a, 0, sizeof(a));
    a.scale_re = 1.0;
    a.order = tile_order();
    a.N = g.N;
    a.Q = g.Q;
    a.nthr = g.nthr;
    a.nh = g.nh;
    make_runs(g.hpos, g.nh, a.hruns);
    make_runs(g.tpos, g.nthr, a.truns);
    a.rpos_w = 0;
    for (int r = 0; r < g.a_log; ++r) {
        a.rpos[r] = g.tpos[g.nthr + r];
        a.rpos_w |= (uint32_t)g.tpos[g.nthr + r] << (6 * r);
    }
}

static std::string geom_key(const Geom &g)
{
    std::string k;
    k.push_back((char)g.N);
    k.push_back((char)g.Q);
    k.push_back((char)g.a_log);
    k.append(reinterpret_cast<const char *>(g.tpos), g.Q);
    return k;
}

// RX groups: gate bits among the thread bits, a_log per LDS phase.
static int set_gates(TileArgs &a, const Geom &g, uint32_t gate_mask)
{
    a.gate_mask = gate_mask;
    // gated thread bits, lowest first
    std::vector<int> pend;
    for (int i = 0; i < g.nthr; ++i)
        if ((gate_mask >> i) & 1u)
            pend.push_back(i);
    a.ngroups = 0;
    a.grp_mask_w = 0;
    a.grp_gates_w = 0;
    size_t pos = 0;
    while (pos < pend.size()) {
        if (a.ngroups >= FQ_MAX_GROUPS)
            return set_err(FQ_ERR_ARG, "too many LDS phases");
        std::vector<int> bits;
        for (int r = 0; r < g.a_log && pos < pend.size(); ++r)
            bits.push_back(pend[pos++]);
        const int real = (int)bits.size();
        // fill the phase with tile bits that receive no gate in it, from the
        // top (register bits first)
        for (int i = g.Q - 1; (int)bits.size() < g.a_log && i >= 0; --i)
            if (std::find(bits.begin(), bits.end(), i) == bits.end())
                bits.push_back(i);
        std::vector<int> sorted = bits;
        std::sort(sorted.begin(), sorted.end());
        uint16_t gm = 0;
        uint8_t gg = 0;
        for (int r = 0; r < g.a_log; ++r) {
            gm |= (uint16_t)(1u << sorted[r]);
            for (int q = 0; q < real; ++q)
                if (bits[q] == sorted[r])
                    gg |= (uint8_t)(1u << r);
        }
        a.grp_mask[a.ngroups] = gm;
        a.grp_gates[a.ngroups] = gg;
        if (a.ngroups < 4)
            a.grp_mask_w |= (uint64_t)gm << (16 * a.ngroups);
        a.grp_gates_w |= (uint32_t)(gg & 0x1f) << (5 * a.ngroups);
        a.ngroups++;
    }
    return FQ_OK;
}

// ---- cost plans ------------------------------------------------------------------

static size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

// The cut plan of graph G for tile geometry g as one blob (doubles first,
// then ints, each array 16-byte aligned); dev receives the plan's scalars
// (place_plan fills in the arrays' device addresses).
struct PlanBlob {
    std::vector<char> bytes;
    PlanDev dev{};
    size_t o_cH = 0, o_om = 0, o_cw = 0, o_hw = 0, o_thr = 0, o_off = 0, o_ch = 0, o_hu = 0, o_hv = 0;
};

static void build_plan(const fq_graph *G, const Geom &g, PlanBlob &pb)
{
    const int N = G->N;
    int ti[FQ_MAXN], hi[FQ_MAXN];
    for (int p = 0; p < N; ++p)
        ti[p] = hi[p] = -1;
    for (int i = 0; i < g.Q; ++i)
        ti[g.tpos[i]] = i;
    for (int h = 0; h < g.nh; ++h)
        hi[g.hpos[h]] = h;

    std::vector<std::vector<std::pair<int, double>>> csr(g.Q);
    std::vector<double> cH(g.Q, 0.0), omega(std::max(g.nh, 1), 0.0);
    std::vector<int> hh_u, hh_v;
    std::vector<double> hh_w;
    struct TE {
        int a, b;
        double w;
    };
    std::vector<TE> te;
    double wtot = 0;
    for (int i = 0; i < N; ++i)
        for (int j = i + 1; j < N; ++j) {
            const double w = G->W[(size_t)i * N + j];
            if (w == 0)
                continue;
            wtot += w;
            if (ti[i] < 0 && ti[j] < 0) {
                hh_u.push_back(hi[i]);
                hh_v.push_back(hi[j]);
                hh_w.push_back(w);
            } else if (ti[i] >= 0 && ti[j] < 0) {
                csr[ti[i]].push_back({hi[j], w});
                cH[ti[i]] += w;
                omega[hi[j]] += w;
            } else if (ti[i] < 0 && ti[j] >= 0) {
                csr[ti[j]].push_back({hi[i], w});
                cH[ti[j]] += w;
                omega[hi[i]] += w;
            } else {
                te.push_back({ti[i], ti[j], w});
            }
        }
    const int nthr = g.nthr, A = 1 << g.a_log, T = 1 << nthr;
    std::vector<double> thr((size_t)(1 + g.a_log) * T, 0.0);
    for (int t = 0; t < T; ++t) {
        double base = 0;
        for (const TE &e : te) {
            const bool at = e.a < nthr, bt = e.b < nthr;
            if (at && bt) {
                base += e.w * (double)(((t >> e.a) ^ (t >> e.b)) & 1);
            } else if (at != bt) {
                const int th = at ? e.a : e.b;
                const int r = (at ? e.b : e.a) - nthr;
                const int z = (t >> th) & 1;
                base += e.w * z;
                thr[(size_t)(1 + r) * T + t] += e.w * (1 - 2 * z);
            }
        }
        thr[t] = base;
    }
    PlanDev &dev = pb.dev;
    for (int j = 0; j < FQ_MAX_REGS; ++j)
        dev.rr[j] = 0;
    for (int j = 0; j < A; ++j) {
        double v = 0;
        for (const TE &e : te)
            if (e.a >= nthr && e.b >= nthr)
                v += e.w * (double)(((j >> (e.a - nthr)) ^ (j >> (e.b - nthr))) & 1);
        dev.rr[j] = v;
    }
    dev.wtot = wtot;
    dev.n_hh = (int)hh_w.size();

    std::vector<int> off(g.Q + 1, 0);
    std::vector<int> ch;
    std::vector<double> cw;
    for (int i = 0; i < g.Q; ++i) {
        off[i] = (int)ch.size();
        for (auto &pr : csr[i]) {
            ch.push_back(pr.first);
            cw.push_back(pr.second);
        }
    }
    off[g.Q] = (int)ch.size();

    // blob layout
    pb.o_cH = 0;
    pb.o_om = align16(pb.o_cH + sizeof(double) * g.Q);
    pb.o_cw = align16(pb.o_om + sizeof(double) * omega.size());
    pb.o_hw = align16(pb.o_cw + sizeof(double) * std::max<size_t>(cw.size(), 1));
    pb.o_thr = align16(pb.o_hw + sizeof(double) * std::max<size_t>(hh_w.size(), 1));
    pb.o_off = align16(pb.o_thr + sizeof(double) * thr.size());
    pb.o_ch = align16(pb.o_off + sizeof(int) * off.size());
    pb.o_hu = align16(pb.o_ch + sizeof(int) * std::max<size_t>(ch.size(), 1));
    pb.o_hv = align16(pb.o_hu + sizeof(int) * std::max<size_t>(hh_u.size(), 1));
    const size_t total = align16(pb.o_hv + sizeof(int) * std::max<size_t>(hh_v.size(), 1));
    pb.bytes.assign(total, 0);
    auto put = [&](size_t o, const void *src, size_t n) {
        if (n)
            memcpy(pb.bytes.data() + o, src, n);
    };
    put(pb.o_cH, cH.data(), sizeof(double) * g.Q);
    put(pb.o_om, omega.data(), sizeof(double) * omega.size());
    put(pb.o_cw, cw.data(), sizeof(double) * cw.size());
    put(pb.o_hw, hh_w.data(), sizeof(double) * hh_w.size());
    put(pb.o_thr, thr.data(), sizeof(double) * thr.size());
    put(pb.o_off, off.data(), sizeof(int) * off.size());
    put(pb.o_ch, ch.data(), sizeof(int) * ch.size());
    put(pb.o_hu, hh_u.data(), sizeof(int) * hh_u.size());
    put(pb.o_hv, hh_v.data(), sizeof(int) * hh_v.size());
}

// The plan of a blob that lives at base (device memory).
static PlanDev place_plan(const PlanBlob &pb, char *base)
{
    PlanDev dev = pb.dev;
    dev.cH = (const double *)(base + pb.o_cH);
    dev.omega = (const double *)(base + pb.o_om);
    dev.csr_w = (const double *)(base + pb.o_cw);
    dev.hh_w = (const double *)(base + pb.o_hw);
    dev.thr = (const double *)(base + pb.o_thr);
    dev.csr_off = (const int *)(base + pb.o_off);
    dev.csr_h = (const int *)(base + pb.o_ch);
    dev.hh_u = (const int *)(base + pb.o_hu);
    dev.hh_v = (const int *)(base + pb.o_hv);
    return dev;
}

// Whether work queued on the stream is being captured into a graph.
static bool is_capturing(hipStream_t stream)
{
    hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &c) == hipSuccess && c != hipStreamCaptureStatusNone;
}

// Device cut plan of graph G for tile geometry g, cached per (geometry, W
// content).  A new plan is uploaded asynchronously on `stream`; a cached plan
// whose upload was queued on another stream makes `stream` wait for it.
// With FQ_PLAN_CACHE plans cached, the least recently used one whose buffers
// are large enough is replaced: `stream` first waits (on the device, through
// an event) for the work queued so far on every stream that plan was handed
// to, so no launch still reading it sees the new contents, and the host
// blocks on nothing but that plan's own earlier upload.  A held plan is not
// replaced; if all that are large enough are held, the cache grows by the new one
// (at most by the plans of one holder: they are the next one's to replace).
// A new plan on a captured stream is uploaded by the captured graph, on each replay,
// from memory of its own that stays with G: it is not cached, since no call outside
// that graph can know when it is there.
// entry, if not null, receives the plan's entry, which lives until the graph's
// plan_epoch changes.
static int get_plan(fq_graph *G, const Geom &g, PlanDev *out, hipStream_t stream, PlanEntry **entry = nullptr)
{
    std::string key = geom_key(g);
    key.append(reinterpret_cast<const char *>(G->W.data()), G->W.size() * sizeof(double));
    auto note_user = [&](PlanEntry &e) {
        e.last_use = ++G->use_clock;
        if (std::find(e.users.begin(), e.users.end(), stream) == e.users.end()) {
            e.users.push_back(stream);
            e.foreign |= !is_own_stream(stream);
        }
    };
    auto it = G->plans.find(key);
    if (it != G->plans.end()) {
        PlanEntry &e = it->second;
        note_user(e);
        if (e.ready && e.stream != stream) {
            const hipError_t q = hipEventQuery(e.ready);
            if (q == hipErrorNotReady) {
                hipGetLastError();
                FQ_HIP(hipStreamWaitEvent(stream, e.ready, 0));
            } else if (q != hipSuccess) {
                return set_err(FQ_ERR_DEVICE, "plan upload failed: %s", hipGetErrorString(q));
            }
        }
        *out = e.dev;
        if (entry)
            *entry = &e;
        return FQ_OK;
    }
    PlanBlob pb;
    build_plan(G, g, pb);
    const size_t total = pb.bytes.size();
    PlanEntry pe;
    if (is_capturing(stream)) {
        if (!plan_memory(G, align16(total), pe)) {
            hipGetLastError();
            return set_err(FQ_ERR_OOM, "no memory for a new plan under capture: the same call before it makes it");
        }
        G->blocks.back().captured = true;
        memcpy(pe.staging, pb.bytes.data(), total);
        FQ_HIP(hipMemcpyAsync(pe.dmem, pe.staging, total, hipMemcpyHostToDevice, stream));
        *out = place_plan(pb, pe.dmem);
        if (entry)
            *entry = nullptr;
        return FQ_OK;
    }
    bool reused = false;
    if (G->plans.size() >= FQ_PLAN_CACHE) {
        auto victim = G->plans.end();
        bool held = false;
        for (auto v = G->plans.begin(); v != G->plans.end(); ++v) {
            if (G->holds > 0 && v->second.last_use > G->held_from) {
                held = true;
                continue;
            }
            if (v->second.cap >= total && (victim == G->plans.end() || v->second.last_use < victim->second.last_use))
                victim = v;
        }
        if (victim == G->plans.end() && !held) {
            // every cached plan is smaller than this one: drop them all (rare;
            // hipFree waits for the device in any case)
            FQ_HIP(hipDeviceSynchronize());
            plans_free(G, false);
            G->plan_epoch++;
        } else if (victim != G->plans.end()) {
            pe = victim->second;
            G->plans.erase(victim);
            reused = true;
            // the host rewrites staging: its previous upload must be done
            FQ_HIP(hipEventSynchronize(pe.ready));
            if (pe.foreign) {
                // a caller's stream may still read it and cannot be tracked
                FQ_HIP(hipDeviceSynchronize());
            } else {
                for (hipStream_t u : pe.users) {
                    if (u == stream || !is_own_stream(u))
                        continue;
                    FQ_HIP(hipEventRecord(pe.ready, u));
                    FQ_HIP(hipStreamWaitEvent(stream, pe.ready, 0));
                }
            }
            pe.users.clear();
            pe.foreign = false;
            G->plan_epoch++;
        }
    }
    if (!reused) {
        size_t cap = 4096;
        while (cap < total)
            cap *= 2;
        if (hipEventCreateWithFlags(&pe.ready, hipEventDisableTiming) != hipSuccess || !plan_memory(G, cap, pe)) {
            hipGetLastError();
            if (pe.ready)
                hipEventDestroy(pe.ready);
            return set_err(FQ_ERR_OOM, "plan allocation of %zu bytes failed", cap);
        }
    }
    memcpy(pe.staging, pb.bytes.data(), total);
    pe.stream = stream;
    if (hipMemcpyAsync(pe.dmem, pe.staging, total, hipMemcpyHostToDevice, stream) != hipSuccess ||
        hipEventRecord(pe.ready, stream) != hipSuccess) {
        hipGetLastError();
        hipStreamSynchronize(stream);
        hipEventDestroy(pe.ready);   // (its memory stays with the graph)
        return set_err(FQ_ERR_DEVICE, "plan upload failed");
    }
    const PlanDev dev = place_plan(pb, (char *)pe.dmem);
    pe.dev = dev;
    pe.users.clear();
    pe.foreign = false;
    PlanEntry &ne = G->plans[key];
    ne = pe;
    note_user(ne);
    *out = dev;
    if (entry)
        *entry = &ne;
    return FQ_OK;
}

// ---- state --------------------------------------------------------------------------

static int check_state(const fq_state *st)
{
    if (!st)
        return set_err(FQ_ERR_ARG, "null state");
    return FQ_OK;
}

// Register bits per thread of a general tile pass.
static int tile_a_log(int dtype, int Q)
{
    const int want = dtype == FQ_C128 ? 3 : 4;
    return std::max(1, std::min(want, Q));
}

extern "C" int fq_state_create(int N, int D, int B, int C, int dtype, fq_state **out)
{
    if (!out)
        return set_err(FQ_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (dtype != FQ_C128 && dtype != FQ_C64)
        return set_err(FQ_ERR_ARG, "dtype must be FQ_C128 or FQ_C64");
    if (N < 1 || N > 36)
        return set_err(FQ_ERR_ARG, "N=%d out of range [1, 36]", N);
    if (D < 0 || D > N)
        return set_err(FQ_ERR_ARG, "D=%d out of range", D);
    if (D > 0)
        return set_err(FQ_ERR_UNSUPPORTED,
                       "D=%d: multi-device state-vector transposition needs 2^D GPUs; this build "
                       "runs on one GPU (D=0)", D);
    if (B < 0 || B > N - D)
        return set_err(FQ_ERR_ARG, "B=%d must satisfy 0 <= B <= N-D=%d", B, N - D);
    if (C < 1 || C > tile_max_q(dtype))
        return set_err(FQ_ERR_ARG, "C=%d out of range [1, %d] for this dtype (2^C tile in LDS)", C,
                       tile_max_q(dtype));
    fq_state *st = new fq_state();
    st->N = N;
    st->D = D;
    st->B = B;
    st->C = C;
    st->dtype = dtype;
    st->elem = dtype == FQ_C128 ? 16 : 8;
    st->bytes = ((size_t)1 << N) * st->elem;
    for (int p = 0; p < FQ_MAXN; ++p)
        st->qmap[p] = p;
    st->init_amp = pow(1. / sqrt(2.), N);
    if (!budget_take(st->bytes)) {
        delete st;
        return set_err(FQ_ERR_BUDGET, "state of %zu bytes exceeds the memory budget",
                       ((size_t)1 << N) * (dtype == FQ_C128 ? 16 : 8));
    }
    if (hipMalloc(&st->sv, st->bytes) != hipSuccess) {
        hipGetLastError();
        budget_give(((size_t)1 << N) * (dtype == FQ_C128 ? 16 : 8));
        delete st;
        return set_err(FQ_ERR_OOM, "state allocation of %zu bytes failed", ((size_t)1 << N) * (dtype == FQ_C128 ? 16 : 8));
    }
    const int Qr = std::min(12, N);
    st->part_cap = (size_t)1 << (N - Qr);
    st->cand_blocks = (int)std::min<uint64_t>(1024, std::max<uint64_t>(1, ((uint64_t)1 << N) / 4096));
    bool ok = hipMalloc(&st->d_part, sizeof(double) * 2 * st->part_cap) == hipSuccess &&
              hipMalloc(&st->d_cand_p, sizeof(double) * FQ_TOPK_MAX * st->cand_blocks) == hipSuccess &&
              hipMalloc(&st->d_cand_i, sizeof(uint64_t) * FQ_TOPK_MAX * st->cand_blocks) == hipSuccess &&
              lane_take(st->lane);
    if (!ok) {
        hipGetLastError();
        fq_state_destroy(st);
        return set_err(FQ_ERR_OOM, "scratch allocation failed");
    }
    own_stream(st->lane.stream, true);
    st->stream = st->lane.stream;
    *out = st;
    return FQ_OK;
}

extern "C" int fq_state_destroy(fq_state *st)
{
    if (!st)
        return FQ_OK;
    if (st->stream)
        hipStreamSynchronize(st->stream);
    for (auto &r : st->pending) {
        hipEventDestroy(r.e0);
        hipEventDestroy(r.e1);
    }
    for (auto e : st->pool)
        hipEventDestroy(e);
    if (st->sv)
        budget_give(st->bytes);
    hipFree(st->sv);
    hipFree(st->d_part);
    hipFree(st->d_cand_p);
    hipFree(st->d_cand_i);
    free_phases(st);
    if (st->aux)
        budget_give(st->bytes);
    hipFree(st->aux);
    hipFree(st->d_grad);
    hipFree(st->d_pair);
    for (int i = 0; i < 2; ++i) {
        if (st->side[i])
            hipStreamDestroy(st->side[i]);
        if (st->joined[i])
            hipEventDestroy(st->joined[i]);
    }
    if (st->forked)
        hipEventDestroy(st->forked);
    if (st->lane.stream) {
        hipStreamSynchronize(st->lane.stream);   // (a state on a caller's stream)
        own_stream(st->lane.stream, false);
        lane_give(st->lane);
    }
    delete st;
    return FQ_OK;
}

extern "C" int fq_state_info(const fq_state *st, int *N, int *C, int *dtype, size_t *bytes)
{
    if (int rc = check_state(st))
        return rc;
    if (N)
        *N = st->N;
    if (C)
        *C = st->C;
    if (dtype)
        *dtype = st->dtype;
    if (bytes)
        *bytes = st->bytes;
    return FQ_OK;
}

extern "C" int fq_state_device_ptr(const fq_state *st, void **dptr)
{
    if (int rc = check_state(st))
        return rc;
    if (!dptr)
        return set_err(FQ_ERR_ARG, "null output pointer");
    *dptr = st->sv;
    return FQ_OK;
}

extern "C" int fq_state_set_stream(fq_state *st, void *hip_stream)
{
    if (int rc = check_state(st))
        return rc;
    FQ_HIP(hipStreamSynchronize(st->stream));
    st->stream = hip_stream ? (hipStream_t)hip_stream : st->lane.stream;
    return FQ_OK;
}

extern "C" int fq_state_init_zero(fq_state *st)
{
    if (int rc = check_state(st))
        return rc;
    for (int p = 0; p < FQ_MAXN; ++p)
        st->qmap[p] = p;
    return timed(st, FQ_K_COST, (double)st->bytes,
                 [&] { return launch_fill_zero_one(st->dtype, st->sv, st->N, st->stream); });
}

extern "C" int fq_init_h(fq_state *st)
{
    if (int rc = check_state(st))
        return rc;
    st->init_amp = pow(1. / sqrt(2.), st->N);
    return FQ_OK;
}

// ---- graph ------------------------------------------------------------------------

extern "C" int fq_graph_create(int N, fq_graph **out)
{
    if (!out)
        return set_err(FQ_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (N < 1 || N > FQ_MAXN)
        return set_err(FQ_ERR_ARG, "N=%d out of range", N);
    fq_graph *g = new fq_graph();
    g->N = N;
    g->W.assign((size_t)N * N, 0.0);
    *out = g;
    return FQ_OK;
}

extern "C" int fq_graph_add_edge(fq_graph *g, int u, int v, double w)
{
    if (!g)
        return set_err(FQ_ERR_ARG, "null graph");
    if (u < 0 || v < 0 || u >= g->N || v >= g->N)
        return set_err(FQ_ERR_ARG, "edge (%d,%d) out of range for N=%d", u, v, g->N);
    if (u == v)
        return set_err(FQ_ERR_ARG, "self-loop (%d,%d) is not an edge of the cut", u, v);
    if (!std::isfinite(w))
        return set_err(FQ_ERR_ARG, "edge weight must be finite");
    if (u > v)
        std::swap(u, v);
    g->W[(size_t)u * g->N + v] = w;
    g->version++;
    return FQ_OK;
}

extern "C" int fq_graph_destroy(fq_graph *g)
{
    if (!g)
        return FQ_OK;
    if (!g->blocks.empty()) {
        hipDeviceSynchronize();
        plans_free(g, true);
    }
    delete g;
    return FQ_OK;
}

extern "C" int fq_graph_weights(const fq_graph *g, double *W)
{
    if (!g || !W)
        return set_err(FQ_ERR_ARG, "null argument");
    memcpy(W, g->W.data(), sizeof(double) * g->W.size());
    return FQ_OK;
}

// mapping_after_swap_conti (src/swap.cu:27-50): exchange labels out+t, in+t.
extern "C" int fq_graph_relabel(fq_graph *g, int swap_out, int swap_in, int num_swap)
{
    if (!g)
        return set_err(FQ_ERR_ARG, "null graph");
    const int N = g->N;
    if (num_swap < 0 || swap_out < 0 || swap_out + num_swap > swap_in || swap_in + num_swap > N)
        return set_err(FQ_ERR_ARG, "relabel blocks [%d,+%d) [%d,+%d) invalid for N=%d", swap_out,
                       num_swap, swap_in, num_swap, N);
    double *W = g->W.data();
    for (int t = 0; t < num_swap; ++t) {
        const int a = swap_out + t, b = swap_in + t;
        for (int i = 0; i < N; ++i) {
            if (i == a || i == b)
                continue;
            double &wa = i < a ? W[(size_t)i * N + a] : W[(size_t)a * N + i];
            double &wb = i < b ? W[(size_t)i * N + b] : W[(size_t)b * N + i];
            std::swap(wa, wb);
        }
    }
    g->version++;
    return FQ_OK;
}

// ---- gate ops -------------------------------------------------------------------------

static int graph_matches(const fq_state *st, const fq_graph *g)
{
    if (!g)
        return set_err(FQ_ERR_ARG, "null graph");
    if (g->N != st->N)
        return set_err(FQ_ERR_ARG, "graph has N=%d but the state has N=%d", g->N, st->N);
    return FQ_OK;
}

static std::vector<int> low_tile(int Q)
{
    std::vector<int> t(Q);
    for (int i = 0; i < Q; ++i)
        t[i] = i;
    return t;
}

// Cost-phase launch arguments: angle and launch-control amplitude.
static void set_cost(TileArgs &a, double gamma, double init_amp)
{
    // a.scale (the pass's real RX factor, 1 without gates) is set by the caller
    a.gamma = gamma;
    a.init_amp = init_amp;
    a.has_rr = 0;
    for (int j = 0; j < FQ_MAX_REGS; ++j)
        if (a.plan.rr[j] != 0)
            a.has_rr = 1;
}

// Phase tables of one run made by one launch: up to this size together.  At
// N=22 complex128 five of them are 1.3 MB; where a pass takes some hundred us
// or more, its table's launch is under 2% of it.
#define FQ_TABLES_BYTES ((size_t)8 << 20)

// A first buffer holds the tables of any depth where they stay below this: from 2 MiB
// on an allocation takes 7 us instead of 0.7, and its free the same.
#define FQ_TABLES_FIRST (((size_t)2 << 20) - 4096)

// Phase-table buffer of at least `need` bytes (`want` where it is made).  A smaller one
// before it stays with the state: launches in flight and captured graphs read it.  Up to
// FQ_TABLES_BYTES each is at least twice the one before; larger ones differ only by the
// kind of call (run, cost layer, gradient).
static int reserve_phases(fq_state *st, size_t need, size_t want = 0)
{
    if (need <= st->phase_cap)
        return FQ_OK;
    const size_t twice = 2 * st->phase_cap <= FQ_TABLES_BYTES ? 2 * st->phase_cap : 0;
    size_t cap = std::max({need, want, twice});
    void *m = nullptr;
    if (hipMalloc(&m, cap) != hipSuccess && (cap == need || hipMalloc(&m, cap = need) != hipSuccess)) {
        hipGetLastError();
        return set_err(FQ_ERR_OOM, "phase table allocation of %zu bytes failed", cap);
    }
    if (st->d_phase)
        st->old_phase.push_back(st->d_phase);
    st->d_phase = (double2 *)m;
    st->phase_cap = cap;
    return FQ_OK;
}

// Phase table of one cost launch into d_phase; with cut, the table of cut
// coefficients follows it in the same buffer (*cut points there).
static int prepare_phases(fq_state *st, TileArgs &a, int a_log, double **cut = nullptr)
{
    const size_t n = phase_table_entries(a, a_log);
    if (int rc = reserve_phases(st, n * sizeof(double2) + (cut ? n * sizeof(double) : 0)))
        return rc;
    double *c = cut ? reinterpret_cast<double *>(st->d_phase + n) : nullptr;
    FQ_HIP(launch_phase_table(a, a_log, st->d_phase, c, st->stream));
    if (cut)
        *cut = c;
    return FQ_OK;
}

// Cost phase alone: 256 threads x 16 amplitudes per work-group, no LDS.
static int cost_pass(fq_state *st, fq_graph *g, double gamma, bool first)
{
    const int Q = std::min(12, st->N);
    const int a_log = std::max(1, std::min(4, Q));
    Geom geom = make_geom(st->N, low_tile(Q), a_log);
    TileArgs a;
    geom_to_args(geom, a);
    if (int rc = get_plan(g, geom, &a.plan, st->stream))
        return rc;
    set_cost(a, gamma, st->init_amp);
    if (int rc = prepare_phases(st, a, a_log))
        return rc;
    const double bytes = (first ? 1.0 : 2.0) * (double)st->bytes;
    return timed(st, FQ_K_COST, bytes, [&] {
        return launch_tile(st->dtype, a_log, true, first, false, st->sv, a, st->d_phase, st->stream);
    });
}

// Half-state (Z2) modes of a tile pass: tiles with z_{N-1} = 0 only, or the
// mirror pass whose top register bit is qubit N-1 (Z2_EXPAND: and that
// writes the full state's upper half, after the last layer).
enum { Z2_OFF = 0, Z2_LOWER = 1, Z2_MIRROR = 2, Z2_EXPAND = 3 };

// Launch arguments of one tile pass of an N-qubit state: tile positions
// (thread bits first), RX gate positions and the half-state mode.
static int pass_args(int N, int dtype, const std::vector<int> &tile, const std::vector<int> &gates, bool cost,
                     int z2, TileArgs &a, Geom &geom, int a_log = 0)
{
    const int Q = (int)tile.size();
    if (a_log == 0)
        a_log = tile_a_log(dtype, Q);
    geom = make_geom(N, tile, a_log);
    if (geom_runs(geom) > FQ_MAX_RUNS)
        return set_err(FQ_ERR_ARG, "internal: tile geometry needs more than %d bit runs", FQ_MAX_RUNS);
    geom_to_args(geom, a);
    uint32_t gm = 0;
    for (int p : gates) {
        int ti = -1;
        for (int i = 0; i < Q; ++i)
            if (tile[i] == p)
                ti = i;
        if (ti < 0)
            return set_err(FQ_ERR_ARG, "internal: gate %d not in tile", p);
        gm |= 1u << ti;
    }
    if (int rc = set_gates(a, geom, gm))
        return rc;
    if (z2 != Z2_OFF) {
        // the lower half is the tiles whose top index bit (qubit N-1) is 0;
        // a mirror pass pairs tile tau with ~tau instead
        const bool ok = z2 == Z2_LOWER ? geom.nh >= 1 && geom.hpos[geom.nh - 1] == N - 1
                                       : geom.nh >= 1 && tile.back() == N - 1 && !cost;
        if (!ok)
            return set_err(FQ_ERR_ARG, "internal: tile does not fit the half-state pass");
        a.ntiles_run = 1ull << (geom.nh - 1);
        if (z2 >= Z2_MIRROR)
            for (int i = 0; i + 1 < Q; ++i)
                a.mirror_pm += 1ull << tile[i];
    }
    return FQ_OK;
}

// The factor of a tile pass: sigma^(#gates) of each RX set (rx_tform: *t the
// butterfly coefficient) times what earlier passes left pending.  It goes
// into the cost phase, or is applied before the stores (apply), or stays
// pending for a later pass of the same fq_run (cost or not defer: it does not).
struct PassFactor {
    double t = 0, pre_t = 0, re = 1.0, im = 0.0;
    bool apply = false;
};

// (*re, *im) times sigma^n of RX(beta) on amplitudes of st; *t as in rx_tform.
static void absorb_rx(const fq_state *st, double beta, size_t n, double *t, double *re, double *im)
{
    double gr, gi;
    rx_tform(beta, st->dtype, st->in_run, t, &gr, &gi);
    for (size_t k = 0; k < n; ++k) {
        const double nr = *re * gr - *im * gi;
        *im = *re * gi + *im * gr;
        *re = nr;
    }
}

// later: RX(beta) on that many qubits follows this cost pass in plain passes whose factor
// goes into it (FACTOR_TAKEN, of a plain pass: it has gone into the cost pass before it).
// A slab's slots do the last layer so: a factor rounded to FP32 and multiplied in before the
// last stores is the same for all amplitudes, and took <C> of complex64 slots off by up to
// 1.2e-7 (rms of 400 requests, N=12 and 17: 8e-8 and 6e-8; the general kernel, whose RX has
// no such factor, 5.3e-8 and 4.7e-8; now 4.9e-8 and 3.6e-8); in the cost phase every thread
// rounds another product.
#define FACTOR_TAKEN ((size_t)-1)
static PassFactor pass_factor(fq_state *st, size_t ngates, double beta, const double *pre_beta, bool cost, bool defer,
                              size_t later = 0)
{
    PassFactor f;
    double sr = st->pending_re, si = st->pending_im;
    const bool taken = later == FACTOR_TAKEN;
    absorb_rx(st, beta, taken ? 0 : ngates + later, &f.t, &sr, &si);
    if (pre_beta)
        absorb_rx(st, *pre_beta, ngates, &f.pre_t, &sr, &si);
    if (taken)
        return f;
    const bool keep = !cost && defer;
    if (!keep) {
        f.re = sr;
        f.im = si;
        f.apply = !cost;
    }
    st->pending_re = keep ? sr : 1.0;
    st->pending_im = keep ? si : 0.0;
    return f;
}

// The memory-side cache: 256 MiB.
#define FQ_CACHE_LOG 28
#define FQ_CACHE_BYTES ((size_t)1 << FQ_CACHE_LOG)

// States whose plans deal the qubits out instead of splitting them (exec_plan).
#define FQ_DEALT_BYTES ((size_t)64 << 30)

static int carriers_for(int dtype);

// A tile pass on the compile-time kernel (fq_mix.h), ready to launch over
// all its tiles or a range of them.
struct MixPass {
    MixArgs a;
    int K = 0, kind = 0, mir = 0;
    bool lane = false;  // RX on one more thread bit by lane operations
    bool cost = false;
    double bytes = 0;   // read and written by the whole pass
    TileArgs tab;       // cost pass: geometry, plan and angle of its phase table
    size_t entries = 0; // and its size
    const double2 *ptab = nullptr;  // where it is (mix_table, mix_tables)
    const double *ctab = nullptr;   // (pair passes) the table of exponents
};

// First register bit of layout l of a tile pass with K exchanges (MixLay).
static int layout_start(int nthr, int A, int K, int l)
{
    return l == 0 ? nthr : std::max(0, nthr - A * (K - l + 1));
}

// The tile as the last layout of K exchanges holds it: thread bits = the tile
// bits outside its register bits, in increasing order.
static Geom layout_geom(int N, const std::vector<int> &tile, int A, int K)
{
    const int Q = (int)tile.size(), start = layout_start(Q - A, A, K, K);
    std::vector<int> t2;
    for (int i = 0; i < Q; ++i)
        if (i < start || i >= start + A)
            t2.push_back(tile[i]);
    for (int r = 0; r < A; ++r)
        t2.push_back(tile[start + r]);
    return make_geom(N, t2, A);
}

// Geometry of a pass on compile-time phases (2^A registers a thread) into a; K
// exchanges, lane: RX on one more thread bit by lane operations (lane_bit: whether
// there is an instance of that).
static int pass_shape(int N, const std::vector<int> &tile, const std::vector<int> &gates, int A,
                      bool (*lane_bit)(int, int, int), int z2, MixArgs &a, int &K, bool &lane)
{
    const int Q = (int)tile.size(), nthr = Q - A;
    const Geom geom = make_geom(N, tile, A);
    memset(&a, 0, sizeof(a));
    a.N = N;
    a.Q = Q;
    a.nh = geom.nh;
    if (make_runs(geom.hpos, geom.nh, a.hruns) > FQ_MAX_RUNS)
        return set_err(FQ_ERR_ARG, "internal: tile geometry needs more than %d bit runs", FQ_MAX_RUNS);
    uint32_t gm = 0;
    for (int p : gates) {
        const auto it = std::find(tile.begin(), tile.end(), p);
        if (it == tile.end())
            return set_err(FQ_ERR_ARG, "internal: gate %d not in tile", p);
        gm |= 1u << (it - tile.begin());
    }
    // exchanges: as many as it takes from the top thread bit down to the
    // lowest gated one, one fewer if only the bit below them is left and RX on
    // it can run on lanes
    int low = nthr;
    for (int i = nthr - 1; i >= 0; --i)
        if ((gm >> i) & 1u)
            low = i;
    K = (nthr - low + A - 1) / A;
    lane = K > 1 && low == nthr - (K - 1) * A - 1 && lane_bit(Q, A, K - 1);
    if (lane)
        --K;
    for (int i = 0; i < Q; ++i)
        a.tpos[i] = geom.tpos[i];
    uint32_t left = lane ? gm & ~(1u << low) : gm;
    for (int l = 0; l <= K; ++l) {
        const int start = layout_start(nthr, A, K, l);
        const uint32_t m = (left >> start) & ((1u << A) - 1u);
        a.gates_w |= m << (A * l);
        left &= ~(m << start);
    }
    for (int r = 0; r < A; ++r) {
        a.rpos0_w |= (uint32_t)geom.tpos[nthr + r] << (6 * r);
        a.rposk_w |= (uint32_t)geom.tpos[layout_start(nthr, A, K, K) + r] << (6 * r);
    }
    a.ntiles = 1ull << geom.nh;
    if (z2 != Z2_OFF) {
        // the lower half is the tiles whose top index bit (qubit N-1) is 0; a
        // mirror pass pairs tile tau with ~tau instead
        const bool ok = geom.nh >= 1 && (z2 == Z2_LOWER ? geom.hpos[geom.nh - 1] == N - 1 : tile.back() == N - 1);
        if (!ok)
            return set_err(FQ_ERR_ARG, "internal: tile does not fit the half-state pass");
        a.ntiles = 1ull << (geom.nh - 1);
        if (z2 >= Z2_MIRROR)
            for (int i = 0; i + 1 < Q; ++i)
                a.mirror_pm += 1ull << tile[i];
    }
    a.ntab = a.ntiles;
    return FQ_OK;
}

// The factors of a prepared pass and its angle: what differs between the layers.
static void mix_factors(fq_state *st, size_t ngates, double beta, double gamma, const double *pre_beta, bool defer,
                        MixPass &mp, size_t later = 0)
{
    MixArgs &a = mp.a;
    const PassFactor f = pass_factor(st, ngates, beta, pre_beta, mp.cost, defer, later);
    a.t = f.t;
    a.pre_t = f.pre_t;
    a.tf = (float)f.t;   // exact for complex64 (rx_tform rounds t to FP32)
    a.pre_tf = (float)f.pre_t;
    a.scale_re = f.re;
    a.scale_im = f.im;
    a.apply_scale = f.apply;
    mp.tab.gamma = gamma;
}

// A pass without its factors (mix_factors); arguments as tile_pass.  The mirror pass
// may be a boundary pass too: the phase of a mirror element is that of the N-qubit
// index it stands for (Cut(b) = Cut(~b)).
static int mix_prepare(fq_state *st, const std::vector<int> &tile, const std::vector<int> &gates, fq_graph *g, bool cost,
                       bool first, int z2, bool boundary, MixPass &mp)
{
    const int N = st->N, A = mix_a_log(st->dtype, (int)tile.size());
    MixArgs &a = mp.a;
    if (int rc = pass_shape(N, tile, gates, A, mix_lane_bit, z2, a, mp.K, mp.lane))
        return rc;
    if (z2 >= Z2_MIRROR && cost && !first && !boundary)
        return set_err(FQ_ERR_ARG, "internal: the mirror pass is no cost pass of its own");
    if (cost) {
        // phase table of the layout the cost phase runs in: layout 0, or for a
        // boundary pass the last one
        TileArgs &ca = mp.tab;
        const Geom cgeom = layout_geom(N, tile, A, boundary ? mp.K : 0);
        geom_to_args(cgeom, ca);
        ca.ntiles_run = a.ntiles;
        if (int rc = get_plan(g, cgeom, &ca.plan, st->stream))
            return rc;
        set_cost(ca, 0.0, st->init_amp);
        mp.entries = phase_table_entries(ca, A);
        a.has_rr = ca.has_rr;
        a.init_amp = st->init_amp;
    }
    // runs of 128 B from HBM: neighbouring tiles, which share DRAM pages, on one XCD.
    // Per layer on MI355X, N=34 complex64 fused 125 -> 104 ms (8 ranges of tiles
    // instead of 64: 102), N=33 complex128 122 -> 101; RX on the top 10 qubits at
    // N=34 113 -> 71 (8 ranges 113); no difference at N=30 complex128.
    // From 64 GiB on, where the plans deal the qubits out (exec_plan), every pass:
    // N=33 complex64 half state 34.8 -> 31.8 ms per layer (33.9 by the general kernel's
    // order, one range of tiles for each of its work-groups), N=32 complex128 34.0 ->
    // 31.2 (32.7), N=34 complex64 fused 111 -> 107.
    int carried = 0;
    while (carried < (int)tile.size() && tile[carried] == carried)
        ++carried;
    // Not below 2 GiB: RX on the top 10 qubits of 512 MiB (N=26 complex64) 317 us, in
    // order 241; 1 GiB 467 and 442; 2 GiB 944 and 997; 4 GiB 1,885 and 2,068.
    a.by_xcd = (carried <= carriers_for(st->dtype) || st->bytes >= FQ_DEALT_BYTES) && a.ntiles >= 2048 &&
               st->bytes >= 8 * FQ_CACHE_BYTES;
    // complex64 of 2 GiB only with the top qubits in the tile (RX on qubits 10..19 of N=28
    // 1,078 us, in order 863, by the general kernel 908; N=29 1,630 and 1,721).
    if (st->dtype == FQ_C64 && st->bytes == 8 * FQ_CACHE_BYTES && *std::max_element(tile.begin(), tile.end()) != N - 1)
        a.by_xcd = 0;
    mp.cost = cost;
    mp.kind = boundary ? MIX_BOUNDARY : first ? MIX_FIRST : cost ? MIX_COST : MIX_PLAIN;
    mp.mir = z2 == Z2_MIRROR ? 1 : z2 == Z2_EXPAND ? 2 : 0;
    // a half-state pass reads and writes half the state; the expanding one
    // writes the whole state
    mp.bytes = (double)st->bytes * (z2 == Z2_OFF ? (first ? 1.0 : 2.0) : z2 == Z2_EXPAND ? 1.5 : first ? 0.5 : 1.0);
    return FQ_OK;
}

// The phase table of one pass, at the start of the state's buffer.
static int mix_table(fq_state *st, MixPass &mp)
{
    if (!mp.cost)
        return FQ_OK;
    if (int rc = prepare_phases(st, mp.tab, mix_a_log(st->dtype, mp.a.Q)))
        return rc;
    mp.ptab = st->d_phase;
    return FQ_OK;
}

// The phase tables of several passes in one launch where they are small and
// of few geometries (*done), with cuts also the table of exponents of each
// geometry; `done` false: each pass needs its own launch.
template <typename Pass>
static int mix_tables(fq_state *st, std::vector<Pass> &mps, bool *done, bool cuts = false)
{
    *done = false;
    TableJobs m;
    size_t total = 0, most = 0, ncut = 0;
    int nj = 0, ng = 0;
    for (const Pass &mp : mps) {
        if (!mp.cost)
            continue;
        if (nj == FQ_TABLE_JOBS)
            return FQ_OK;
        TableGeo g;
        memset(&g, 0, sizeof(g));
        g.Q = mp.tab.Q;
        g.nthr = mp.tab.nthr;
        g.nh = mp.tab.nh;
        g.a_log = mp.tab.Q - mp.tab.nthr;
        g.ntiles = mp.tab.ntiles_run;
        g.plan = mp.tab.plan;
        int k = 0;
        bool fresh = false;
        while (k < ng && memcmp(&m.geo[k], &g, sizeof(g)) != 0)
            ++k;
        if (k == ng) {
            if (ng == FQ_TABLE_GEOS)
                return FQ_OK;
            m.cut_offset[ng] = (uint32_t)ncut;
            ncut += cuts ? mp.entries : 0;
            m.geo[ng++] = g;
            fresh = true;
        }
        m.job[nj++] = {mp.tab.gamma, (uint16_t)k, (uint16_t)(cuts && fresh), (uint32_t)total};
        total += mp.entries;
        most = std::max(most, mp.entries);
        if (total * sizeof(double2) > FQ_TABLES_BYTES)
            return FQ_OK;
    }
    if (nj < 2)
        return FQ_OK;
    const size_t need = total * sizeof(double2) + ncut * sizeof(double);
    // a table for each pass where there is no memory, or a captured stream cannot get any
    if (need > st->phase_cap && is_capturing(st->stream))
        return FQ_OK;
    if (reserve_phases(st, need, std::min(FQ_TABLE_JOBS * most * sizeof(double2) + ncut * sizeof(double), FQ_TABLES_FIRST)))
        return FQ_OK;
    double *cut = cuts ? (double *)(st->d_phase + total) : nullptr;
    FQ_HIP(launch_phase_tables(m, nj, most, st->d_phase, cut, st->stream));
    nj = 0;
    for (Pass &mp : mps)
        if (mp.cost) {
            mp.ptab = st->d_phase + m.job[nj].offset;
            mp.ctab = cuts ? cut + m.cut_offset[m.job[nj].geo] : nullptr;
            ++nj;
        }
    *done = true;
    return FQ_OK;
}

static int mix_pass(fq_state *st, const std::vector<int> &tile, const std::vector<int> &gates, double beta,
                    fq_graph *g, double gamma, bool cost, bool first, int kind, int z2, const double *pre_beta,
                    bool defer)
{
    MixPass mp;
    if (int rc = mix_prepare(st, tile, gates, g, cost, first, z2, pre_beta != nullptr, mp))
        return rc;
    mix_factors(st, gates.size(), beta, gamma, pre_beta, defer, mp);
    if (int rc = mix_table(st, mp))
        return rc;
    return timed(st, kind, mp.bytes, [&] {
        return launch_mix(st->dtype, mp.K, mp.lane, mp.kind, mp.mir, st->sv, mp.a, mp.ptab, st->stream);
    });
}

// One tile pass with RX on gate positions (and optionally the cost phase).
// pre_beta (with cost, not first, not a mirror pass): RX(*pre_beta) on the
// same positions before the cost phase -- the pass that ends one layer and
// opens the next.  The kernel applies each RX as the one-FMA butterfly of
// rx_tform, i.e. sigma^-1 RX per gate; the pass's factor sigma^(#gates) (times
// sigma_pre^(#gates)) and any factor earlier passes left pending go into the
// cost phase of a cost pass; a pass without it multiplies them in before its
// stores, unless defer is set: then they stay pending for the next pass of the
// same fq_run (a layer's RX factors grow the amplitudes by at most 2^(N/2)
// before a cost pass absorbs them).
static int tile_pass(fq_state *st, const std::vector<int> &tile, const std::vector<int> &gates,
                     double beta, fq_graph *g, double gamma, bool cost, bool first, int kind,
                     int z2 = Z2_OFF, const double *pre_beta = nullptr, bool defer = false)
{
    if (pre_beta && (!cost || first))
        return set_err(FQ_ERR_ARG, "internal: a layer-boundary pass needs the cost phase of a later layer");
    if (mix_a_log(st->dtype, (int)tile.size()) > 0)
        return mix_pass(st, tile, gates, beta, g, gamma, cost, first, kind, z2, pre_beta, defer);
    if (pre_beta && z2 >= Z2_MIRROR)
        return set_err(FQ_ERR_ARG, "internal: no mirror boundary pass at this tile width");
    TileArgs a;
    Geom geom;
    if (int rc = pass_args(st->N, st->dtype, tile, gates, cost, z2, a, geom))
        return rc;
    const int a_log = geom.a_log;
    // the pass's factor: sigma^(#gates) per RX set, times what is pending
    double sr = st->pending_re, si = st->pending_im;
    auto absorb = [&](double b, double *t) {
        double gr, gi;
        rx_tform(b, st->dtype, st->in_run, t, &gr, &gi);
        for (size_t k = 0; k < gates.size(); ++k) {
            const double nr = sr * gr - si * gi;
            si = sr * gi + si * gr;
            sr = nr;
        }
    };
    absorb(beta, &a.rx_t);
    if (pre_beta)
        absorb(*pre_beta, &a.pre_t);
    a.rx_tf = (float)a.rx_t;   // exact for complex64 (rx_tform rounds t to FP32)
    a.pre_tf = (float)a.pre_t;
    if (cost || !defer) {
        a.scale_re = sr;
        a.scale_im = si;
        a.apply_scale = !cost;
        st->pending_re = 1.0;
        st->pending_im = 0.0;
    } else {
        st->pending_re = sr;
        st->pending_im = si;
    }
    if (cost) {
        // the complex64 boundary pass applies the cost phase in its last LDS
        // phase's layout: thread bits = the tile bits outside that phase,
        // register bits = the phase's bits (both in increasing order), so its
        // phase table comes from the plan of that ordering of the same tile
        TileArgs ca = a;
        Geom cgeom = geom;
        if (pre_beta && st->dtype == FQ_C64 && a.ngroups > 0) {
            const unsigned gm = a.grp_mask[a.ngroups - 1];
            std::vector<int> t2;
            for (int i = 0; i < geom.Q; ++i)
                if (!((gm >> i) & 1u))
                    t2.push_back(geom.tpos[i]);
            for (int i = 0; i < geom.Q; ++i)
                if ((gm >> i) & 1u)
                    t2.push_back(geom.tpos[i]);
            cgeom = make_geom(st->N, t2, a_log);
        }
        if (int rc = get_plan(g, cgeom, &ca.plan, st->stream))
            return rc;
        set_cost(ca, gamma, st->init_amp);
        if (int rc = prepare_phases(st, ca, a_log))
            return rc;
        a.plan = ca.plan;
        a.gamma = ca.gamma;
        a.init_amp = ca.init_amp;
        a.has_rr = ca.has_rr;
    }
    // a half-state pass reads and writes half the state; the expanding one
    // writes the whole state
    const double bytes = (double)st->bytes * (z2 == Z2_OFF ? (first ? 1.0 : 2.0) : z2 == Z2_EXPAND ? 1.5 : 1.0);
    return timed(st, kind, bytes, [&] {
        if (z2 >= Z2_MIRROR)
            return launch_tile_mirror(st->dtype, a_log, z2 == Z2_EXPAND, st->sv, a, st->stream);
        if (pre_beta)
            return launch_tile_pre(st->dtype, a_log, st->sv, a, st->d_phase, st->stream);
        return launch_tile(st->dtype, a_log, cost, first, true, st->sv, a, cost ? st->d_phase : nullptr,
                           st->stream);
    });
}

static int carriers_for(int dtype) { return dtype == FQ_C128 ? 3 : 4; }

// Tile width of the fused and strided passes: the LDS limit by default;
// FQ_TILE_Q (environment, read per call) may lower it (smaller tiles: two
// work-groups per CU).
static int pass_tile_q(int dtype)
{
    const char *e = getenv("FQ_TILE_Q");
    const int env_q = e ? atoi(e) : 0;
    const int mx = tile_max_q(dtype);
    return env_q > 0 && env_q < mx ? env_q : mx;
}

// One tile pass of a fused layer: its tile positions and RX targets.
struct FusedPass {
    std::vector<int> tile, gates;
};

// Qubits per block when the strided passes' new qubits are dealt out (see
// cover_passes): 2 by default; FQ_PASS_BLOCK (environment, read per call)
// selects another, 0 for contiguous blocks.
static int pass_block()
{
    const char *e = getenv("FQ_PASS_BLOCK");
    return e ? std::max(0, atoi(e)) : 2;
}

// Whether the carried low qubits' RX moves out of the cost pass (see
// cover_passes): on by default; FQ_CARRIER_GATES=0 (environment, read per
// call) keeps every low qubit's RX in pass 0.
static bool carrier_gates()
{
    const char *e = getenv("FQ_CARRIER_GATES");
    return e ? atoi(e) != 0 : true;
}

// The tile passes of one fused layer, covering every qubit once.  Pass 0 is
// the low Qmax qubits (cost phase and their RX); the other qubits go to the
// fewest passes that fit, each tile being the lowest qubits as carriers
// (runs of at least 128 contiguous bytes) plus the pass's new qubits.  The new qubits are dealt to the
// passes in blocks, from the top qubit down and from the last pass down, so
// the last pass holds qubit N-1 (the half-state mirror pass needs it) and
// every strided pass mixes middle and high index bits.  On MI355X this
// spreads a pass's accesses over the DRAM better than one contiguous block
// of qubits per pass (N=30 complex128: strided passes 8.0 and 7.2 ms -> 6.8
// and 7.0 ms; N=34 complex64: 65 and 98 ms -> 57 and 81 ms).  A pass that
// would need more bit runs than the tile kernel takes gets larger blocks.
// carriers: lowest qubits that every strided pass carries (0: carriers_for).
static std::vector<FusedPass> cover_passes(int N, int Qmax, int dtype, int boundary = -1, int carriers = 0)
{
    std::vector<FusedPass> ps;
    Qmax = std::min(Qmax, N);
    FusedPass p1;
    p1.tile = low_tile(Qmax);
    p1.gates = p1.tile;
    ps.push_back(p1);
    const int rest = N - Qmax;
    if (rest <= 0)
        return ps;
    const int cmin = std::min(carriers > 0 ? carriers : carriers_for(dtype), Qmax - 1);
    const int per_max = Qmax - cmin;
    const int npass = (rest + per_max - 1) / per_max;
    std::vector<int> want(npass);
    for (int k = 0; k < npass; ++k)
        want[k] = rest / npass + (k < rest % npass ? 1 : 0);
    for (int blk = pass_block() > 0 ? pass_block() : rest;; ++blk) {
        std::vector<std::vector<int>> news(npass);
        int q = N - 1, k = npass - 1;
        while (q >= Qmax) {
            for (int i = 0; i < blk && q >= Qmax && (int)news[k].size() < want[k]; ++i)
                news[k].push_back(q--);
            k = (k + npass - 1) % npass;
        }
        std::vector<FusedPass> more;
        bool fits = true;
        for (int k2 = 0; k2 < npass; ++k2) {
            std::vector<int> &nw = news[k2];
            std::sort(nw.begin(), nw.end());
            const int c = Qmax - want[k2];
            const int a_log = tile_a_log(dtype, Qmax);
            // lane order: the 64 lanes of a wave are the tile's first six
            // positions; past the carriers they take the pass's lowest new
            // qubits whose byte-address bit is outside [19, hi] (one load
            // instruction whose lanes differ only in bits 19..22 measured up
            // to 1.6x slower), else the highest; never N-1, which stays the
            // top register bit for the half-state mirror pass. hi = 22 for
            // states under 32 GiB; from 32 GiB on hi = 28 (lane bits 23..28
            // measured 2-8% slower per layer at N=31..33 complex128 and N=34
            // complex64, while at N=29 complex128 the window to 28 cost 1.5%)
            const int lanes = std::max(0, std::min(6, Qmax - a_log) - c);
            const int elem_log = dtype == FQ_C128 ? 4 : 3;
            const int win_hi = N + elem_log >= 35 ? 28 : 22;
            std::vector<int> lane_q;
            for (int q : nw)
                if ((int)lane_q.size() < lanes && q != N - 1 && (q + elem_log < 19 || q + elem_log > win_hi))
                    lane_q.push_back(q);
            for (int i = (int)nw.size() - 1; i >= 0 && (int)lane_q.size() < lanes; --i)
                if (nw[i] != N - 1 && std::find(lane_q.begin(), lane_q.end(), nw[i]) == lane_q.end())
                    lane_q.push_back(nw[i]);
            std::sort(lane_q.begin(), lane_q.end());
            FusedPass p;
            for (int i = 0; i < c; ++i)
                p.tile.push_back(i);
            for (int q : lane_q)
                p.tile.push_back(q);
            for (int q : nw)
                if (std::find(lane_q.begin(), lane_q.end(), q) == lane_q.end())
                    p.tile.push_back(q);
            p.gates = nw;
            fits = fits && geom_runs(make_geom(N, p.tile, tile_a_log(dtype, Qmax))) <= FQ_MAX_RUNS;
            more.push_back(p);
        }
        if (fits || blk >= rest) {
            if (carrier_gates()) {
                // RX on a carried low qubit may run in any strided pass that
                // carries it (the RX gates of a layer commute and all follow
                // the cost phase of pass 0): give each to the strided pass
                // with the fewest gates, which takes LDS phases and VALU work
                // off the cost pass
                // -- not to the pass given as boundary (pipelined layers run
                // its RX twice per launch), unless no other pass carries q
                for (int q = 0; q < Qmax; ++q) {
                    int best = -1;
                    for (int pass = 0; pass < 2 && best < 0; ++pass)
                        for (int k2 = 0; k2 < npass; ++k2)
                            if (q < Qmax - want[k2] && (pass == 1 || k2 + 1 != boundary) &&
                                (best < 0 || more[k2].gates.size() < more[best].gates.size()))
                                best = k2;
                    if (best < 0)
                        continue;
                    more[best].gates.push_back(q);
                    ps[0].gates.erase(std::find(ps[0].gates.begin(), ps[0].gates.end(), q));
                }
            }
            ps.insert(ps.end(), more.begin(), more.end());
            return ps;
        }
    }
}

// Split arbitrary RX targets into tile passes (targets below C: one chunk pass).
static int rx_targets_once(fq_state *st, std::vector<int> targets, double beta);

static int rx_targets(fq_state *st, std::vector<int> targets, double beta)
{
    if (!st->in_run) {
        // outside fq_run the butterfly keeps its X, so |t| = |tan(beta/2)|:
        // beyond 2.5 (an amplitude growth above 2.7 per gate before the pass's
        // factor is applied) RX(beta) runs as two passes of RX(beta/2)
        double sn, cs;
        sincos(beta / 2, &sn, &cs);
        if (std::fabs(sn) > 2.5 * std::fabs(cs)) {
            if (int rc = rx_targets_once(st, targets, beta / 2))
                return rc;
            return rx_targets_once(st, targets, beta / 2);
        }
    }
    return rx_targets_once(st, targets, beta);
}

// Tile width of an RX pass with n targets outside the low chunk (FQ_MAXQ: the full one).
// Few targets in full tiles took longer than in the general kernel, whose work-groups
// walk ranges of tiles: MI355X, complex64 N=28, 1 target in the middle and 5 at the top,
// general kernel 892 and 877 us, 2^14 901 and 919, 2^12 778 and 792; complex128 N=28, 1
// and 5 at the top, general kernel 1,605 and 1,755, 2^13 1,765 and 1,685, 2^11 1,589 and
// 1,632.  Which width is best turns on the addresses in flight at a time, and differs
// once the state exceeds the memory-side cache (N=24, 4 and 5 at the top, complex128:
// general 94 and 95, 2^13 98 and 101, 2^11 97 and 109, 2^10 90 and 92): taken where it
// was faster for targets in the middle and at the top, from 32 MiB to 8 GiB.
static int rx_width(const fq_state *st, int n)
{
    if (st->bytes < (size_t)32 << 20)
        return FQ_MAXQ;
    const bool large = st->bytes > FQ_CACHE_BYTES;
    if (n == 6 && st->bytes >= FQ_CACHE_BYTES)
        return st->dtype == FQ_C64 ? 13 : 12;
    if (st->dtype == FQ_C64)
        return n <= 2 ? 12 : n == 3 ? 10 : n == 5 ? 11 + large : FQ_MAXQ;
    return n == 4 ? 10 : n == 5 ? 10 + large : !large || n > 3 ? FQ_MAXQ : n == 1 ? 11 : 12;
}

static int rx_targets_once(fq_state *st, std::vector<int> targets, double beta)
{
    const int N = st->N;
    const int Ceff = std::min(st->C, N);
    std::sort(targets.begin(), targets.end());
    if (targets.empty())
        return FQ_OK;
    if (targets.back() < Ceff) {
        // complex64: no wider than it takes, but 2^11 amplitudes (a work-group per 2^10 is
        // one wave: N=28, RX on 10 qubits 935 us, the general kernel 872, 2^11 788, 2^12
        // 790; N=23 36, 35.5, 34.7, 34.4; 1 qubit of a chunk of 13, N=16 2^13 20.3 us,
        // general 19.9, 2^11 16.7); chunks below 10 qubits only beyond the memory-side
        // cache.  complex128, whose 2^9 is as many bytes: N=28 1,638, 2^11 1,650
        int Q = Ceff;
        if (st->dtype == FQ_C64 && (Ceff >= 10 || st->bytes > FQ_CACHE_BYTES))
            Q = std::min(N, std::max(targets.back() + 1, 11));
        return tile_pass(st, low_tile(Q), targets, beta, nullptr, 0, false, false, FQ_K_RX);
    }
    const int Qfull = std::min(pass_tile_q(st->dtype), N);
    const int per = std::max(1, Qfull - std::min(carriers_for(st->dtype), Qfull - 1));
    size_t pos = 0;
    while (pos < targets.size()) {
        std::vector<int> chunk;
        while (pos < targets.size() && (int)chunk.size() < per)
            chunk.push_back(targets[pos++]);
        std::vector<int> tile;
        const int Qmax = std::min(Qfull, rx_width(st, (int)chunk.size()));
        for (;;) {
            // the chunk's targets plus the lowest other qubits as carriers
            tile = chunk;
            for (int p = 0; (int)tile.size() < Qmax && p < N; ++p)
                if (std::find(chunk.begin(), chunk.end(), p) == chunk.end())
                    tile.push_back(p);
            std::sort(tile.begin(), tile.end());
            const int a_log = tile_a_log(st->dtype, (int)tile.size());
            if (chunk.size() == 1 || geom_runs(make_geom(N, tile, a_log)) <= FQ_MAX_RUNS)
                break;
            chunk.pop_back();  // scattered targets: fewer per pass
            --pos;
        }
        if (int rc = tile_pass(st, tile, chunk, beta, nullptr, 0, false, false, FQ_K_RX))
            return rc;
    }
    return FQ_OK;
}

extern "C" int fq_cost_layer(fq_state *st, fq_graph *g, double gamma, int is_first)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = graph_matches(st, g))
        return rc;
    if (!std::isfinite(gamma))
        return set_err(FQ_ERR_ARG, "gamma must be finite");
    return cost_pass(st, g, gamma, is_first != 0);
}

extern "C" int fq_multi_rx(fq_state *st, const int *targets, int gate_size, double beta)
{
    if (int rc = check_state(st))
        return rc;
    if (gate_size < 0 || (gate_size > 0 && !targets))
        return set_err(FQ_ERR_ARG, "bad target list");
    if (!std::isfinite(beta))
        return set_err(FQ_ERR_ARG, "beta must be finite");
    std::vector<int> t(targets, targets + gate_size);
    std::vector<bool> seen(st->N, false);
    for (int q : t) {
        if (q < 0 || q >= st->N)
            return set_err(FQ_ERR_ARG, "target %d out of range for N=%d", q, st->N);
        if (seen[q])
            return set_err(FQ_ERR_ARG, "target %d listed twice", q);
        seen[q] = true;
    }
    return rx_targets(st, t, beta);
}

// Qubit p changes places with qubit partner[p] (partner[partner[p]] == p).
static int exchange_qubits(fq_state *st, const uint8_t *partner)
{
    const int N = st->N;
    int moved = 0, least = N;   // pairs; the lowest upper qubit of one
    SwapRuns pairs;
    pairs.n = 0;
    for (int p = 0; p < N; ++p)
        if (partner[p] > p) {
            moved++;
            least = std::min(least, (int)partner[p]);
            if (p > 0 && partner[p - 1] == partner[p] - 1 && partner[p - 1] > p - 1)
                pairs.run[pairs.n - 1] += 1u << 8;
            else
                pairs.run[pairs.n++] = (uint32_t)p | 1u << 8 | (uint32_t)partner[p] << 16;
        }
    // an amplitude stays where the bits of each pair are equal
    const double bytes = 2.0 * (double)st->bytes * (1.0 - std::ldexp(1.0, -moved));
    if (st->bytes <= FQ_SWAP_SMALL)
        return timed(st, FQ_K_SWAP, bytes, [&] { return launch_swap_small(st->dtype, st->sv, pairs, N, st->stream); });
    SwapArgs a;
    memset(&a, 0, sizeof(a));
    // the tile takes qubits from the lowest up, each with its partner: 2^10
    // complex128 and 2^12 complex64 amplitudes, two of them 32 and 64 KiB
    // (complex64 N=27 13 qubits with 2^10 and 2^12: 462 and 450 us; below N=24, too
    // few units for the chip: N=20 8 qubits 7.2 and 8.5)
    const int most = st->dtype == FQ_C128 || N < 24 ? 10 : 12;
    bool in[FQ_MAXN] = {false};
    for (int p = 0; p < N; ++p) {
        const int n = partner[p] == p ? 1 : 2;
        if (!in[p] && a.tb + n <= most) {
            in[p] = in[partner[p]] = true;
            a.tb += n;
        }
    }
    std::vector<int> lower, upper, rest;
    int t = 0, bit[FQ_MAXN];
    for (int p = 0; p < N; ++p) {
        bit[p] = t;
        if (in[p]) {
            a.tpos[t++] = (uint8_t)p;
        } else if (partner[p] > p) {
            lower.push_back(p);
            upper.push_back(partner[p]);
        } else if (partner[p] == p) {
            rest.push_back(p);
        }
    }
    for (int i = 0; i < t; ++i)
        a.partner[i] = (uint8_t)bit[partner[a.tpos[i]]];
    auto runs = [](const std::vector<int> &pos, SwapRuns &r) {
        for (size_t i = 0, j; i < pos.size(); i = j) {
            for (j = i + 1; j < pos.size() && pos[j] == pos[j - 1] + 1; ++j)
                ;
            r.run[r.n++] = (uint32_t)i | ((uint32_t)(j - i) << 8) | ((uint32_t)pos[i] << 16);
        }
    };
    runs(lower, a.lower);
    runs(upper, a.upper);
    runs(rest, a.rest);
    a.nr = (int)rest.size();
    a.npairs = (1ull << lower.size()) * ((1ull << lower.size()) + 1) / 2;
    a.rest_fast = a.nr > 0 && rest[0] < least;
    a.large = st->bytes > FQ_CACHE_BYTES;
    return timed(st, FQ_K_SWAP, bytes, [&] { return launch_swap(st->dtype, st->sv, a, st->stream); });
}

extern "C" int fq_swap_conti(fq_state *st, int swap_out, int swap_in, int num_swap)
{
    if (int rc = check_state(st))
        return rc;
    const int N = st->N, k = num_swap;
    if (k < 0 || swap_out < 0 || swap_out + k > swap_in || swap_in + k > N)
        return set_err(FQ_ERR_ARG, "swap blocks [%d,+%d) [%d,+%d) invalid for N=%d", swap_out, k,
                       swap_in, k, N);
    if (k == 0)
        return FQ_OK;
    uint8_t partner[FQ_MAXN];
    for (int p = 0; p < N; ++p)
        partner[p] = (uint8_t)p;
    for (int i = 0; i < k; ++i) {
        partner[swap_out + i] = (uint8_t)(swap_in + i);
        partner[swap_in + i] = (uint8_t)(swap_out + i);
    }
    if (int rc = exchange_qubits(st, partner))
        return rc;
    for (int i = 0; i < k; ++i)
        std::swap(st->qmap[swap_out + i], st->qmap[swap_in + i]);
    return FQ_OK;
}

// ---- schedules -----------------------------------------------------------------------


// Whether the layers of the fused and half-state schedules are pipelined
// (run_layers): by default (measured on MI355X, N=30 fused: complex128
// 50.0 -> 65.0 layers/s, complex64 94 -> 110); FQ_LAYER_PIPE=0 (environment,
// read per call) runs them in layer order.
static bool layer_pipe()
{
    const char *e = getenv("FQ_LAYER_PIPE");
    return e ? atoi(e) != 0 : true;
}

// The passes of one layer of the fused (z2 false) or half-state schedule and,
// when the layers are pipelined, the pass besides pass 0 that ends every
// other layer (end1 < 0: layer order).  end1 is the last pass of the fused
// schedule and pass 1 of the half-state one (its last pass is the mirror
// pass, which has no cost phase); the carried low qubits' RX goes to the
// other passes.  Measured at N=30 complex128 against ends {0, 1} with the
// carried RX on the fewest-gate pass: fused 62.5 -> 65.0 layers/s,
// half state 120.9 -> 123.8.
struct LayerPlan {
    std::vector<FusedPass> ps;
    int end1;
    int open0 = 0;   // pipelined: the pass that opens layer 0 (0 or end1)
    bool split = false;  // exec_plan's split of the qubits (layers end on passes 0 and 2)
    int chunk = 0;   // log2 amplitudes of a chunk (exec_plan; 0: passes run over the whole state)
};

static LayerPlan layer_plan(int N, int dtype, bool z2)
{
    const int Qmax = z2 ? std::min(pass_tile_q(dtype), N - 1) : pass_tile_q(dtype);
    // one carrier fewer (64 B runs) where that covers the qubits in two passes:
    // per layer at N=24 complex128 182 -> 149 us, N=25 complex64 198 -> 161 us
    // (states of 256 MiB, which the memory-side cache holds)
    const int fewer = carriers_for(dtype) - 1;
    const bool two = !z2 && N - Qmax == Qmax - fewer;
    LayerPlan lp{cover_passes(N, Qmax, dtype, -1, two ? fewer : 0), -1, 0, false, 0};
    const int m = (int)lp.ps.size();
    if (layer_pipe() && m >= (z2 ? 3 : 2)) {
        lp.end1 = z2 ? 1 : m - 1;
        if (m >= 3)
            lp.ps = cover_passes(N, Qmax, dtype, lp.end1);
    }
    return lp;
}

// Chunked runs: log2 bytes of a chunk (0: off); FQ_CHUNK (environment, read
// per call).  128 MiB by default, half of the memory-side cache, since two
// chunks are in flight (run_layers).  Measured on MI355X per layer, N=30
// complex128 fused: no chunks 14.59 ms; one stream with chunks of 64, 128, 256
// and 512 MiB 15.9, 15.2, 14.2 and 15.2 ms; two streams with 64, 128 and
// 256 MiB 13.3, 12.8 and 14.5 ms.
static int chunk_log()
{
    const char *e = getenv("FQ_CHUNK");
    return e ? atoi(e) : 27;
}

// Two passes of width Q: the low Q qubits, and the others over the lowest 2Q - N
// (whose RX stays in pass 0).
static std::vector<FusedPass> split_two(int N, int Q)
{
    FusedPass p0, p1;
    p0.tile = low_tile(Q);
    p0.gates = p0.tile;
    p1.tile = low_tile(2 * Q - N);
    for (int q = Q; q < N; ++q) {
        p1.tile.push_back(q);
        p1.gates.push_back(q);
    }
    return {p0, p1};
}

// Three passes of width Q (exec_plan): qubits above pass 0 that pass 1 takes (0:
// they do not fit three passes).
static int split_low(int N, int Q, int dtype, int least)
{
    const int rest = N - Q, most = Q - carriers_for(dtype);
    const int n1 = std::max(least, rest - most);
    return n1 <= most && n1 < rest ? n1 : 0;
}

// (lane_bit: whether RX can run on the thread bit below k exchanges' reach)
static std::vector<FusedPass> split_three(int N, int Q, int n1, int A, bool (*lane_bit)(int, int, int))
{
    const int c1 = Q - n1, c2 = Q - (N - Q - n1);   // carried low qubits
    // exchanges of a pass whose lowest gated tile bit is `low`; a lane bit counts 0.4
    auto cost = [&](int low) {
        const int nthr = Q - A, K = low < nthr ? (nthr - low + A - 1) / A : 0;
        return K > 1 && low == nthr - (K - 1) * A - 1 && lane_bit(Q, A, K - 1) ? K - 0.6 : (double)K;
    };
    // the carried qubits' RX goes to pass 1, which is no boundary pass; of the
    // other low ones pass 2 takes those below x that save more exchanges in
    // pass 0 than they cost in pass 2
    int x = c1;
    for (int y = c1 + 1; y <= std::min(c2, Q - A); ++y)
        if (cost(y) + cost(c1) < cost(x) + cost(x > c1 ? c1 : c2))
            x = y;
    FusedPass p0, p1, p2;
    p0.tile = low_tile(Q);
    p1.tile = low_tile(c1);
    p2.tile = low_tile(c2);
    for (int q = Q; q < N; ++q) {
        FusedPass &p = q < Q + n1 ? p1 : p2;
        p.tile.push_back(q);
        p.gates.push_back(q);
    }
    for (int q = 0; q < Q; ++q)
        (q < c1 ? p1 : q < x ? p2 : p0).gates.push_back(q);
    return {p0, p1, p2};
}

// The plan fq_run uses for P layers: layer_plan's, except that a plan of three
// passes splits the qubits otherwise: pass 1 takes the 9 qubits right above
// pass 0's and pass 2 the top ones, and layers end alternately on passes 0 and
// 2, also on the half state (whose pass 2 is the mirror pass), so that pass 2 has
// few gates, all in reach of one exchange.  Where the stored state is larger
// than the memory-side cache (256 MiB), the launches between two uses of pass 2
// (pass 1, the boundary pass 0, pass 1), which stay within the low `chunk`
// qubits, run chunk by chunk, and a chunk crosses the HBM once for the three of
// them: per layer at N=30 complex128 fused 14.47 -> 12.71 ms, N=32 complex64
// 30.5 -> 27.8, half state N=30 complex64 3.88 -> 3.58.  9 qubits: per layer at N=30 complex128 fused 14.41, 12.72,
// 12.80 and 13.07 ms with 7, 8, 9 and 10; N=32 complex64 30.6, 30.6, 27.9 and
// 29.0; half state N=30 complex128 7.62, 6.79, 6.66 and 6.88.  Where the plan
// of tuning knobs is asked for, layer_plan's passes run as they are.
static LayerPlan exec_plan(int N, int dtype, bool z2, int P)
{
    LayerPlan lp = layer_plan(N, dtype, z2);
    for (const char *k : {"FQ_TILE_Q", "FQ_PASS_BLOCK", "FQ_CARRIER_GATES", "FQ_LAYER_PIPE"})
        if (getenv(k))
            return lp;
    const int elem_log = dtype == FQ_C128 ? 4 : 3, Ns = z2 ? N - 1 : N;
    if (lp.ps.size() <= 2 && (!z2 || N < 24)) {
        // Two passes of the narrowest tiles that cover N with 128 B runs: a
        // full-width tile leaves most CUs of a small state idle (16 tiles at
        // N=17) and takes a pass's whole latency for its 128 KiB.  Per layer,
        // with one phase-table launch a run (mix_tables), full-width tiles and
        // a launch per table before: N=14 complex128 17.6 -> 6.1 us, N=18 22.3
        // -> 10.2, N=20 30.6 -> 16.7; half state N=20 complex64 31.1 -> 10.8
        // (also one pass per layer instead of two), and against one tile of full
        // width: N=13 complex128 8.7 -> 4.5, N=14 complex64 13.0 -> 5.7.
        const int Q = std::min(tile_max_q(dtype),
                               std::max(dtype == FQ_C128 ? 9 : 10, (N + carriers_for(dtype) + 1) / 2));
        if (Q >= N)
            return lp;
        lp.ps = split_two(N, Q);
        lp.end1 = 1;
        lp.split = true;
        lp.open0 = z2 && P % 2 == 0 ? 1 : 0;
        return lp;
    }
    if (lp.ps.size() != 3)
        return lp;
    const int Q = tile_max_q(dtype);
    const int n1 = split_low(N, Q, dtype, 9);
    // A pass 2 that carries no more than 128 B runs (complex64 from N=33, complex128
    // from N=32) has 1,024 of them, each in another region of 2^22 amplitudes or
    // more: such a boundary pass took 113 ms at N=34 complex64 (58 with the qubits
    // dealt out as layer_plan does).  Per layer there, split 136 ms, dealt out 102;
    // N=33 56.3 and 54.3.
    if (n1 == 0 || N - Q - n1 == Q - carriers_for(dtype))
        return lp;
    lp.ps = split_three(N, Q, n1, mix_a_log(dtype, Q), mix_lane_bit);
    lp.end1 = 2;
    lp.split = true;
    const int chunk = chunk_log() - elem_log;
    if (Ns + elem_log > FQ_CACHE_LOG && chunk >= Q + n1 && chunk < Ns)
        lp.chunk = chunk;
    // the last layer must end on the mirror pass, which writes the full state
    lp.open0 = z2 && P % 2 == 0 ? 2 : 0;
    return lp;
}

// One pass of a run: pass index, kind, layer.
enum { STEP_FIRST = 0, STEP_COST = 1, STEP_PLAIN = 2, STEP_BOUNDARY = 3 };
struct Step {
    int pass, kind, layer;
};

// The passes of layer p of P in launch order.  In layer order, layer p runs
// passes 0..m-1 with its cost phase in pass 0.  Pipelined: the cost phase is
// diagonal, so it can run in any pass; the pass that ends layer p applies
// RX(beta_p), the phase of gamma_{p+1} and RX(beta_{p+1}) on its qubits, which
// opens layer p+1.  Layers end alternately on two passes (end1 and pass 0), so
// every layer after the first runs m-1 passes: 1 + P(m-1) passes in all
// instead of Pm.  Every RX of a layer still follows its cost phase and precedes
// the next one, and RX gates on distinct qubits commute.  Layer p expects
// layers 0..p-1 to have run with the same plan.
static void layer_steps(const LayerPlan &lp, int p, int P, std::vector<Step> &out)
{
    const int m = (int)lp.ps.size();
    const bool last = p + 1 == P;
    if (lp.end1 < 0) {
        for (int i = 0; i < m; ++i)
            out.push_back({i, i > 0 ? STEP_PLAIN : p == 0 ? STEP_FIRST : STEP_COST, p});
        return;
    }
    const int open = p % 2 == 0 ? lp.open0 : lp.open0 == 0 ? lp.end1 : 0;
    const int e = open == 0 ? lp.end1 : 0;   // the pass that ends layer p
    if (p == 0)
        out.push_back({open, STEP_FIRST, p});
    // (a half-state plan that ends on pass 1 has the mirror pass among the
    // middle ones, and it comes last in the last layer)
    if (last && !lp.split)
        out.push_back({e, STEP_PLAIN, p});
    for (int i = 1; i < m; ++i)
        if (i != lp.end1)
            out.push_back({i, STEP_PLAIN, p});
    if (last && lp.split)
        out.push_back({e, STEP_PLAIN, p});
    if (!last)
        out.push_back({e, STEP_BOUNDARY, p});
}

// n passes chunk by chunk (2^nlog chunks), alternate chunks on two streams of
// the state: while one chunk's first pass reads from the HBM, the other's later
// passes run from the cache.  launch(i, c, stream) queues chunk c of pass i.
// Every pass has its phase table before the streams fork.
template <typename F>
static int run_chunks(fq_state *st, int kind, size_t n, double bytes, int nlog, F &&launch)
{
    for (int i = 0; i < 2; ++i) {
        if (!st->side[i])
            FQ_HIP(hipStreamCreateWithFlags(&st->side[i], hipStreamNonBlocking));
        if (!st->joined[i])
            FQ_HIP(hipEventCreateWithFlags(&st->joined[i], hipEventDisableTiming));
    }
    if (!st->forked)
        FQ_HIP(hipEventCreateWithFlags(&st->forked, hipEventDisableTiming));
    return timed(st, kind, bytes, [&] {
        hipError_t e = hipEventRecord(st->forked, st->stream);
        for (int i = 0; i < 2 && e == hipSuccess; ++i)
            e = hipStreamWaitEvent(st->side[i], st->forked, 0);
        for (uint64_t c = 0; c < 1ull << nlog && e == hipSuccess; ++c)
            for (size_t i = 0; i < n && e == hipSuccess; ++i)
                e = launch(i, c, st->side[c & 1]);
        // joined also after a failed launch: what was queued precedes the
        // stream's later work
        for (int i = 0; i < 2; ++i) {
            hipError_t j = hipEventRecord(st->joined[i], st->side[i]);
            if (j == hipSuccess)
                j = hipStreamWaitEvent(st->stream, st->joined[i], 0);
            e = e == hipSuccess ? j : e;
        }
        return e;
    }, (int)n);
}

// Tiles of chunk c of 2^nlog.
static MixArgs chunk_args(const MixArgs &whole, uint64_t c, int nlog)
{
    MixArgs a = whole;
    a.ntiles >>= nlog;
    a.tile0 = c * a.ntiles;
    a.by_xcd = 0;   // (cached)
    return a;
}

// Number of steps from seq[k] on that run chunk by chunk together: a run of
// passes that stay within one chunk, with at most one cost phase among them (one
// phase table); 1: a single pass over the whole state.
static size_t chunk_group(const LayerPlan &lp, const std::vector<Step> &seq, size_t k)
{
    auto local = [&](const Step &s) {
        const std::vector<int> &t = lp.ps[s.pass].tile;
        return lp.chunk > 0 && *std::max_element(t.begin(), t.end()) < lp.chunk;
    };
    size_t n = 1;
    if (local(seq[k])) {
        bool c = seq[k].kind != STEP_PLAIN;
        for (; k + n < seq.size() && local(seq[k + n]) && !(c && seq[k + n].kind != STEP_PLAIN); ++n)
            c = c || seq[k + n].kind != STEP_PLAIN;
    }
    return n;
}

// End of the steps from seq[k] on that are prepared together: whole groups
// (chunk_group) with at most FQ_TABLE_JOBS cost passes, so that a deep run needs no more
// host memory than one of that many layers.
static size_t window_end(const LayerPlan &lp, const std::vector<Step> &seq, size_t k)
{
    int jobs = 0;
    for (size_t n; k < seq.size(); k += n) {
        n = chunk_group(lp, seq, k);
        for (size_t i = k; i < k + n; ++i)
            jobs += seq[i].kind != STEP_PLAIN;
        if (jobs > FQ_TABLE_JOBS)
            break;
    }
    return k;
}

// Layers [p0, p1) of P.  expand: the last layer's mirror pass also writes the
// upper half of the full state.
static int run_layers(fq_state *st, fq_graph *g, const LayerPlan &lp, int p0, int p1, int P, const double *gammas,
                      const double *betas, bool z2, bool expand)
{
    const PlanHold hold(g);   // the passes' plans, until their tables are queued
    const std::vector<FusedPass> &ps = lp.ps;
    const int m = (int)ps.size();
    std::vector<Step> seq;
    for (int p = p0; p < p1; ++p)
        layer_steps(lp, p, P, seq);
    auto cost = [](const Step &s) { return s.kind != STEP_PLAIN; };
    // every pass on the compile-time kernel (the pass widths of tuning knobs
    // may have none): prepared first, and small phase tables made at once
    const bool mix = mix_a_log(st->dtype, (int)ps[0].tile.size()) > 0;
    // the passes of a layer repeat: prepared once, with each layer's factors
    struct Prepared {
        int pass, kind, mode;
        MixPass mp;
    };
    std::vector<Prepared> made;
    std::vector<MixPass> mps;
    for (size_t k0 = 0; k0 < seq.size();) {
        const size_t k1 = mix ? window_end(lp, seq, k0) : seq.size();
        mps.clear();
        for (size_t k = k0; k < k1; ++k) {
            const Step &s = seq[k];
            const FusedPass &fp = ps[s.pass];
            const bool last = s.layer + 1 == P && k + 1 == seq.size();
            const int mode = !z2 ? (int)Z2_OFF
                             : s.pass + 1 < m ? (int)Z2_LOWER
                                              : s.layer + 1 == P && s.kind == STEP_PLAIN && expand ? (int)Z2_EXPAND
                                                                                                    : (int)Z2_MIRROR;
            const bool bd = s.kind == STEP_BOUNDARY;
            const int L = bd ? s.layer + 1 : s.layer;
            const double gamma = cost(s) ? gammas[L] : 0.0;
            const double *pre = bd ? &betas[s.layer] : nullptr;
            // plain passes leave their RX factor to the next cost pass, except
            // the run's very last pass, which leaves the state exact (a slot's: in its
            // last layer's cost pass)
            if (!mix) {
                if (int rc = tile_pass(st, fp.tile, fp.gates, betas[L], g, gamma, cost(s), s.kind == STEP_FIRST,
                                       FQ_K_FUSED, mode, pre, !last))
                    return rc;
                continue;
            }
            size_t i = 0;
            while (i < made.size() && !(made[i].pass == s.pass && made[i].kind == s.kind && made[i].mode == mode))
                ++i;
            if (i == made.size()) {
                made.push_back({s.pass, s.kind, mode, {}});
                if (int rc = mix_prepare(st, fp.tile, fp.gates, g, cost(s), s.kind == STEP_FIRST, mode, bd, made[i].mp))
                    return rc;
            }
            mps.push_back(made[i].mp);
            const size_t later = !st->slot || L + 1 < P ? 0 : cost(s) ? st->N - fp.gates.size() : FACTOR_TAKEN;
            mix_factors(st, fp.gates.size(), betas[L], gamma, pre, !last, mps.back(), later);
        }
        bool tables = false;
        if (int rc = mix_tables(st, mps, &tables))
            return rc;
        for (size_t k = k0; mix && k < k1;) {
            const size_t n = chunk_group(lp, seq, k);
            MixPass *const group = &mps[k - k0];
            int rc = FQ_OK;
            for (size_t i = 0; i < n && !tables && rc == FQ_OK; ++i)
                rc = mix_table(st, group[i]);
            if (rc == FQ_OK && n > 1) {
                const int nlog = (z2 ? st->N - 1 : st->N) - lp.chunk;
                double bytes = 0;
                for (size_t i = 0; i < n; ++i)
                    bytes += group[i].bytes;
                rc = run_chunks(st, FQ_K_FUSED, n, bytes, nlog, [&](size_t i, uint64_t c, hipStream_t stream) {
                    const MixPass &mp = group[i];
                    return launch_mix(st->dtype, mp.K, mp.lane, mp.kind, mp.mir, st->sv, chunk_args(mp.a, c, nlog),
                                      mp.ptab, stream);
                });
            } else if (rc == FQ_OK) {
                const MixPass &mp = group[0];
                rc = timed(st, FQ_K_FUSED, mp.bytes, [&] {
                    return launch_mix(st->dtype, mp.K, mp.lane, mp.kind, mp.mir, st->sv, mp.a, mp.ptab, st->stream);
                });
            }
            if (rc)
                return rc;
            k += n;
        }
        k0 = k1;
    }
    return FQ_OK;
}

// P layers of a state that is one tile (k_solo), FQ_SOLO_LAYERS a launch, and one
// launch for their phase tables.  done false: not such a state, or a plan of tuning
// knobs is asked for.
static int solo_run(fq_state *st, fq_graph *g, int P, const double *gammas, const double *betas, bool *done)
{
    const int N = st->N;
    *done = false;
    if (N < solo_min(st->dtype) || N > solo_max(st->dtype))
        return FQ_OK;
    for (const char *k : {"FQ_TILE_Q", "FQ_PASS_BLOCK", "FQ_CARRIER_GATES", "FQ_LAYER_PIPE"})
        if (getenv(k))
            return FQ_OK;
    *done = true;
    const PlanHold hold(g);
    const std::vector<int> tile = low_tile(N);
    const int A = mix_a_log(st->dtype, N);
    // odd layers go down the layouts and take their cost phase in the last one
    TileArgs tab[2];
    int ntab = 0, most = FQ_SOLO_LAYERS;
    for (int p0 = 0, n; p0 < P; p0 += n) {
        n = std::min(most, P - p0);
        std::vector<MixPass> mps(n);
        SoloArgs a;
        memset(&a, 0, sizeof(a));
        a.P = n;
        a.first = p0 == 0;
        a.init_amp = st->init_amp;
        for (int i = 0; i < std::min(n, 2); ++i) {
            if (i == ntab) {
                const Geom geom = layout_geom(N, tile, A, i ? 2 : 0);
                geom_to_args(geom, tab[i]);
                tab[i].ntiles_run = 1;
                if (int rc = get_plan(g, geom, &tab[i].plan, st->stream))
                    return rc;
                set_cost(tab[i], 0.0, st->init_amp);
                ++ntab;
            }
            a.has_rr |= tab[i].has_rr;
        }
        MixArgs shape;
        int K = 0;
        bool lane = false;
        if (int rc = pass_shape(N, tile, tile, A, mix_lane_bit, Z2_OFF, shape, K, lane))
            return rc;
        if (K != 2 || lane)
            return set_err(FQ_ERR_ARG, "internal: a state of %d qubits takes %d exchanges", N, K);
        a.gates_w = shape.gates_w;
        for (int i = 0; i < n; ++i) {
            MixPass &mp = mps[i];
            const PassFactor f = pass_factor(st, N, betas[p0 + i], nullptr, true, false);
            a.t[i] = f.t;
            a.scale_re[i] = f.re;
            a.scale_im[i] = f.im;
            mp.cost = true;
            mp.tab = tab[i & 1];
            mp.tab.gamma = gammas[p0 + i];
            mp.entries = phase_table_entries(mp.tab, A);
        }
        bool tables = false;
        if (int rc = mix_tables(st, mps, &tables))
            return rc;
        if (!tables && n > 1) {   // no memory for them: a layer each, in the room of one table
            most = 1;
            n = 0;
            continue;
        }
        if (!tables)
            if (int rc = prepare_phases(st, mps[0].tab, A))
                return rc;
        for (int i = 0; i < n; ++i)
            a.table[i] = tables ? (uint32_t)(mps[i].ptab - st->d_phase) : 0;
        const double bytes = (a.first ? 1.0 : 2.0) * (double)st->bytes;
        if (int rc = timed(st, FQ_K_FUSED, bytes, [&] { return launch_solo(st->dtype, N, st->sv, a, st->d_phase, st->stream); }))
            return rc;
    }
    return FQ_OK;
}

// FQ_SCHED_REFERENCE without its single steps: every layer applies RX(beta) to
// each qubit once, wherever the transpositions have moved it, so the P layers are
// those of the fused schedule in the labels of the start, followed by the
// product of all transpositions.  That permutation of the qubits is a product of
// two exchanges of disjoint pairs, each one pass over the state: a cycle
// (c_0 .. c_{n-1}) is c_i <-> c_{-i}, then c_i <-> c_{1-i}.  N=28 P=3 complex128
// C=12 with <C> on MI355X: 30.8 -> 12.6 ms (every step was a pass over the state,
// bound by HBM: 6 a layer).
static int reference_run(fq_state *st, fq_graph *g, const std::vector<int> &sizes, int P, const double *gammas,
                         const double *betas)
{
    const int N = st->N;
    if (P == 0)
        return FQ_OK;
    bool done = false;
    if (int rc = solo_run(st, g, P, gammas, betas, &done))
        return rc;
    if (!done)
        if (int rc = run_layers(st, g, exec_plan(N, st->dtype, false, P), 0, P, P, gammas, betas, false, true))
            return rc;
    int at[FQ_MAXN], to[FQ_MAXN], qmap[FQ_MAXN];   // position -> the position its qubit came from, and back
    for (int p = 0; p < N; ++p)
        at[p] = p;
    for (int p = 0; p < P; ++p)
        for (size_t i = 0, in = 0; i + 1 < sizes.size(); ++i) {
            in += sizes[i];
            for (int t = 0; t < sizes[i + 1]; ++t)
                std::swap(at[t], at[in + t]);
        }
    uint8_t first[FQ_MAXN], second[FQ_MAXN];
    bool seen[FQ_MAXN] = {false}, any[2] = {false, false};
    for (int p = 0; p < N; ++p) {
        to[at[p]] = p;
        qmap[p] = st->qmap[at[p]];
    }
    for (int p = 0; p < N; ++p) {
        std::vector<int> c;
        for (int q = p; !seen[q]; q = to[q]) {
            seen[q] = true;
            c.push_back(q);
        }
        const int n = (int)c.size();
        for (int i = 0; i < n; ++i) {
            first[c[i]] = (uint8_t)c[(n - i) % n];
            second[c[i]] = (uint8_t)c[(n + 1 - i) % n];
            any[0] |= first[c[i]] != c[i];
            any[1] |= second[c[i]] != c[i];
        }
    }
    if (any[0])
        if (int rc = exchange_qubits(st, first))
            return rc;
    if (any[1])
        if (int rc = exchange_qubits(st, second))
            return rc;
    std::copy(qmap, qmap + N, st->qmap);
    for (int p = 0; p < P; ++p)
        for (size_t i = 0, in = 0; i + 1 < sizes.size(); ++i) {
            in += sizes[i];
            if (int rc = fq_graph_relabel(g, 0, (int)in, sizes[i + 1]))
                return rc;
        }
    return FQ_OK;
}

extern "C" int fq_run(fq_state *st, fq_graph *g, int P, const double *gammas, const double *betas,
                      int schedule)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = graph_matches(st, g))
        return rc;
    if (P < 0 || (P > 0 && (!gammas || !betas)))
        return set_err(FQ_ERR_ARG, "bad layer count or angle arrays");
    for (int p = 0; p < P; ++p)
        if (!std::isfinite(gammas[p]) || !std::isfinite(betas[p]))
            return set_err(FQ_ERR_ARG, "angles must be finite");
    const int N = st->N;
    st->pending_re = 1.0;
    st->pending_im = 0.0;
    struct InRun {
        fq_state *st;
        ~InRun() { st->in_run = false; }
    } in_run_guard{st};
    st->in_run = true;
    if (schedule == FQ_SCHED_REFERENCE) {
        // src/Weighted.cpp:97-137
        std::vector<int> sizes;
        for (int i = 0; i < N; i += st->C)
            sizes.push_back(std::min(st->C, N - i));
        // (with class timing on, launch by launch, so that each class is timed)
        if (!st->timing)
            return reference_run(st, g, sizes, P, gammas, betas);
        for (int p = 0; p < P; ++p) {
            if (int rc = cost_pass(st, g, gammas[p], p == 0))
                return rc;
            int swap_in = 0;
            for (size_t i = 0; i < sizes.size(); ++i) {
                std::vector<int> t(sizes[i]);
                for (int q = 0; q < sizes[i]; ++q)
                    t[q] = q;
                if (int rc = rx_targets(st, t, betas[p]))
                    return rc;
                if (i + 1 < sizes.size()) {
                    swap_in += sizes[i];
                    if (int rc = fq_swap_conti(st, 0, swap_in, sizes[i + 1]))
                        return rc;
                    if (int rc = fq_graph_relabel(g, 0, swap_in, sizes[i + 1]))
                        return rc;
                }
            }
        }
        return FQ_OK;
    }
    if (schedule == FQ_SCHED_Z2) {
        // Cut(b) = Cut(~b), RX^{(x)N} commutes with X^{(x)N} and |+> is
        // X^{(x)N}-invariant, so psi(b) = psi(~b): the layers run on the
        // half z_{N-1} = 0 and the other half is written once at the end.
        if (N < 3)
            return set_err(FQ_ERR_ARG, "the half-state schedule needs N >= 3");
        bool done = false;   // (a small state as a whole: the same amplitudes)
        const int rc = solo_run(st, g, P, gammas, betas, &done);
        if (rc || done)
            return rc;
        return run_layers(st, g, exec_plan(N, st->dtype, true, P), 0, P, P, gammas, betas, true, true);
    }
    if (schedule != FQ_SCHED_FUSED)
        return set_err(FQ_ERR_ARG, "unknown schedule %d", schedule);
    bool done = false;
    const int rc = solo_run(st, g, P, gammas, betas, &done);
    if (rc || done)
        return rc;
    return run_layers(st, g, exec_plan(N, st->dtype, false, P), 0, P, P, gammas, betas, false, true);
}

extern "C" int fq_layer_passes(int N, int dtype, int schedule, int max_pass, int *npass, int *tile_q,
                               int *tiles, uint64_t *gates)
{
    if (N < 1 || N > 36 || (dtype != FQ_C128 && dtype != FQ_C64) || !npass || !tile_q || !tiles || !gates)
        return set_err(FQ_ERR_ARG, "bad N, dtype or null output");
    std::vector<FusedPass> ps;
    if (schedule == FQ_SCHED_FUSED || (schedule == FQ_SCHED_Z2 && N >= 3))
        ps = layer_plan(N, dtype, schedule == FQ_SCHED_Z2).ps;
    else
        return set_err(FQ_ERR_ARG, "schedule must be FQ_SCHED_FUSED or FQ_SCHED_Z2 (N >= 3)");
    if ((int)ps.size() > max_pass)
        return set_err(FQ_ERR_ARG, "%zu passes do not fit max_pass=%d", ps.size(), max_pass);
    *npass = (int)ps.size();
    *tile_q = (int)ps[0].tile.size();
    for (size_t p = 0; p < ps.size(); ++p) {
        for (int i = 0; i < 16; ++i)
            tiles[p * 16 + i] = i < (int)ps[p].tile.size() ? ps[p].tile[i] : -1;
        uint64_t m = 0;
        for (int q : ps[p].gates)
            m |= 1ull << q;
        gates[p] = m;
    }
    return FQ_OK;
}

// ---- observables -------------------------------------------------------------------------

extern "C" int fq_expect_cut(fq_state *st, fq_graph *g, double *expect, double *norm2)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = graph_matches(st, g))
        return rc;
    if (!expect)
        return set_err(FQ_ERR_ARG, "null output pointer");
    const int Q = std::min(12, st->N);
    const int a_log = std::max(1, std::min(4, Q));
    Geom geom = make_geom(st->N, low_tile(Q), a_log);
    TileArgs a;
    geom_to_args(geom, a);
    if (int rc = get_plan(g, geom, &a.plan, st->stream))
        return rc;
    // up to 256 tiles (N=20, what the lane's page holds) each writes its sums there, and
    // they are added up here in k_finalize's order, without its launch: <C> at N=16 16.8 us
    // instead of 18.7, N=20 17.8 instead of 19.1; after a run of 4 layers, N=16, 55 instead of
    // 69, since a wait of more than about 40 us takes 10 us longer
    double *const h = st->lane.host;
    const bool direct = 2 * run_tiles(a) <= FQ_LANE_DOUBLES;
    int rc = timed(st, FQ_K_REDUCE, (double)st->bytes, [&] {
        return launch_expect(st->dtype, a_log, st->sv, a, direct ? h : st->d_part, h, st->stream);
    });
    if (rc)
        return rc;
    FQ_HIP(hipStreamSynchronize(st->stream));
    for (uint64_t w = direct ? run_tiles(a) / 2 : 0; w > 0; w /= 2)
        for (uint64_t i = 0; i < 2 * w; ++i)
            h[i] += h[i + 2 * w];
    *expect = h[0];
    if (norm2)
        *norm2 = h[1];
    return FQ_OK;
}

// ---- allocation-free <C> ----------------------------------------------------------------
//
// fq_expect_cut_static runs the kernels of fq_expect_cut with their scratch
// (per-tile partial sums, the cut plan, the two-double result) in `scratch`,
// a fixed device array of this library, instead of memory it allocates: for
// callers that cannot allocate device memory (code under HIP graph capture,
// serving loops).  Each GPU holds its own copy until the process ends; every
// call on one GPU uses that copy, so calls that overlap on one GPU race.

#define FQ_STATIC_MAX_N 30
#define FQ_STATIC_TILE_Q 12
// 2 doubles per 2^12-amplitude tile at the largest N (4 MiB), the cut plan
// of a 12-qubit tile (under 16 KiB at N=30 on a complete graph), the result
#define FQ_STATIC_PART_BYTES ((size_t)16 << (FQ_STATIC_MAX_N - FQ_STATIC_TILE_Q))
#define FQ_STATIC_PLAN_BYTES ((size_t)64 << 10)
#define FQ_STATIC_BYTES (FQ_STATIC_PART_BYTES + FQ_STATIC_PLAN_BYTES + 256)

static __device__ __align__(256) unsigned char scratch[FQ_STATIC_BYTES];

static std::mutex g_scratch_mu;
static std::vector<unsigned char *> g_scratch_ptr;  // device address of scratch, per device

// Device address of this GPU's scratch: hipGetSymbolAddress once per device,
// with that device current.
static int scratch_address(unsigned char **out)
{
    int dev = 0;
    FQ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= dev)
        g_scratch_ptr.resize(dev + 1, nullptr);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_err(FQ_ERR_DEVICE, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = (unsigned char *)p;
    }
    *out = g_scratch_ptr[dev];
    return FQ_OK;
}

extern "C" int fq_expect_cut_static(fq_state *st, fq_graph *g, double *expect, double *norm2)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = graph_matches(st, g))
        return rc;
    if (!expect)
        return set_err(FQ_ERR_ARG, "null output pointer");
    if (st->N > FQ_STATIC_MAX_N)
        return set_err(FQ_ERR_ARG, "N=%d exceeds the static scratch of fq_expect_cut_static (N <= %d)", st->N,
                       FQ_STATIC_MAX_N);
    unsigned char *base = nullptr;
    if (int rc = scratch_address(&base))
        return rc;
    double *part = (double *)base;
    char *plan_mem = (char *)(base + FQ_STATIC_PART_BYTES);
    double *out2 = (double *)(base + FQ_STATIC_PART_BYTES + FQ_STATIC_PLAN_BYTES);
    const int Q = std::min(FQ_STATIC_TILE_Q, st->N);
    const int a_log = std::max(1, std::min(4, Q));
    Geom geom = make_geom(st->N, low_tile(Q), a_log);
    TileArgs a;
    geom_to_args(geom, a);
    PlanBlob pb;
    build_plan(g, geom, pb);
    if (pb.bytes.size() > FQ_STATIC_PLAN_BYTES)
        return set_err(FQ_ERR_ARG, "cut plan of %zu bytes exceeds the static scratch (%zu)", pb.bytes.size(),
                       (size_t)FQ_STATIC_PLAN_BYTES);
    a.plan = place_plan(pb, plan_mem);
    // the previous call on this stream may still read the plan: stream order
    // keeps this upload behind it
    FQ_HIP(hipMemcpyAsync(plan_mem, pb.bytes.data(), pb.bytes.size(), hipMemcpyHostToDevice, st->stream));
    FQ_HIP(launch_expect(st->dtype, a_log, st->sv, a, part, out2, st->stream));
    double h[2];
    FQ_HIP(hipMemcpyAsync(h, out2, sizeof(h), hipMemcpyDeviceToHost, st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    *expect = h[0];
    if (norm2)
        *norm2 = h[1];
    return FQ_OK;
}

// ---- adjoint gradient ------------------------------------------------------------------

static int ensure_aux(fq_state *st, size_t grad_slots)
{
    if (!st->aux) {
        if (!budget_take(st->bytes))
            return set_err(FQ_ERR_BUDGET, "adjoint state of %zu bytes exceeds the memory budget", st->bytes);
        if (hipMalloc(&st->aux, st->bytes) != hipSuccess) {
            hipGetLastError();
            st->aux = nullptr;
            budget_give(st->bytes);
            return set_err(FQ_ERR_OOM, "adjoint state allocation of %zu bytes failed", st->bytes);
        }
    }
    if (grad_slots > st->grad_cap) {
        FQ_HIP(hipStreamSynchronize(st->stream));
        hipFree(st->d_grad);
        st->d_grad = nullptr;
        st->grad_cap = 0;
        if (hipMalloc(&st->d_grad, sizeof(double) * 2 * grad_slots) != hipSuccess)
            return set_err(FQ_ERR_OOM, "gradient scratch allocation failed");
        st->grad_cap = grad_slots;
    }
    return FQ_OK;
}

// lambda = Cut psi_P (on the half state from N = 3 on); sum |psi|^2 Cut and
// sum |psi|^2 into out.
static int cut_lambda(fq_state *st, fq_graph *g, double *out)
{
    const int N = st->N, Q = std::min(12, N >= 3 ? N - 1 : N);
    const int a_log = std::max(1, std::min(4, Q));
    Geom geom = make_geom(N, low_tile(Q), a_log);
    TileArgs a;
    geom_to_args(geom, a);
    if (N >= 3)
        a.ntiles_run = 1ull << (geom.nh - 1);   // qubit N-1 is the top hidden bit
    if (int rc = get_plan(g, geom, &a.plan, st->stream))
        return rc;
    FQ_HIP(launch_cut_mul(st->dtype, a_log, st->sv, st->aux, a, st->d_part, st->stream));
    FQ_HIP(launch_finalize(st->d_part, run_tiles(a), out, st->stream));
    return FQ_OK;
}

// Partial sums of the pair passes (doubles).
static int ensure_pair_scratch(fq_state *st, size_t part)
{
    if (part > st->pair_cap) {
        FQ_HIP(hipStreamSynchronize(st->stream));
        hipFree(st->d_pair);
        st->d_pair = nullptr;
        st->pair_cap = 0;
        if (hipMalloc(&st->d_pair, sizeof(double) * part) != hipSuccess)
            return set_err(FQ_ERR_OOM, "gradient scratch allocation failed");
        st->pair_cap = part;
    }
    return FQ_OK;
}

// One pair pass of the walk back on compile-time phases (fq_pair.hip).
struct PairPass {
    PairArgs a;
    int K = 0, kind = 0;
    bool lane = false, mir = false, cost = false;
    TileArgs tab;
    size_t entries = 0;
    const double2 *ptab = nullptr;
    const double *ctab = nullptr;
};

// The passes of the pair walk back over an N-qubit half state: two of the
// narrowest tiles, or three of full width, as exec_plan's; no passes where they do
// not fit (very small and very large states) or a tuning knob is set.  Chunks hold
// both states.
static LayerPlan pair_plan(int N, int dtype)
{
    LayerPlan lp{{}, -1, 0, false, 0};
    for (const char *k : {"FQ_TILE_Q", "FQ_PASS_BLOCK", "FQ_CARRIER_GATES", "FQ_LAYER_PIPE"})
        if (getenv(k))
            return lp;
    const int Qmin = dtype == FQ_C128 ? 9 : 10, Qmax = dtype == FQ_C128 ? 12 : 13;
    const int Q2 = std::max(Qmin, (N + carriers_for(dtype) + 1) / 2);
    if (Q2 >= N)
        return lp;
    lp.split = true;
    if (Q2 <= Qmax) {
        lp.ps = split_two(N, Q2);
        lp.end1 = 1;
        return lp;
    }
    const int n1 = split_low(N, Qmax, dtype, 8);
    if (n1 == 0)
        return lp;
    lp.ps = split_three(N, Qmax, n1, pair_a_log(dtype, Qmax), pair_lane_bit);
    lp.end1 = 2;
    const int elem_log = dtype == FQ_C128 ? 4 : 3, chunk = chunk_log() - 1 - elem_log;
    if (N + elem_log > FQ_CACHE_LOG && chunk >= Qmax + n1 && chunk < N - 1)
        lp.chunk = chunk;
    return lp;
}

// The walk back over plan lp: <C> and the gradient sums of psi_P and lambda (both
// on the half state, cut_lambda), not yet doubled.  out: the passes' sums after
// those of <C>, in the lane's page or d_grad.  Every RX is the
// butterfly of rx_tform on both states, which grows them by (1 + t^2)^(1/2) a gate:
// mag2 follows the inverse of what <lambda|psi> has taken on, each sum gets its
// value as a weight, and each cost pass scales it back to 1.
static int pair_walk(fq_state *st, fq_graph *g, const LayerPlan &lp, int P, const double *gammas, const double *betas,
                     double *out, double *expect, double *grad_gammas, double *grad_betas)
{
    const PlanHold hold(g);
    const int N = st->N, m = (int)lp.ps.size(), Q = (int)lp.ps[0].tile.size(), A = pair_a_log(st->dtype, Q);
    std::vector<Step> seq;
    for (int p = 0; p < P; ++p)
        layer_steps(lp, p, P, seq);
    std::reverse(seq.begin(), seq.end());
    // partial sums of as many passes as fit 16 MiB at once
    const uint64_t tiles = 1ull << (N - 1 - Q);
    const size_t per = 3 * (size_t)tiles, batch = std::max<size_t>(1, std::min(seq.size(), ((size_t)2 << 20) / per));
    if (int rc = ensure_pair_scratch(st, batch * per))
        return rc;
    const double bytes = 2.0 * (double)st->bytes;   // two half states read and written
    std::vector<double> weight(seq.size());   // of each pass's sums (the states' magnitude before it)
    // the passes of a layer repeat: prepared once, with each layer's angles
    struct Prepared {
        int pass, kind;
        PairPass q;
    };
    std::vector<Prepared> made;
    std::vector<PairPass> pp;
    double mag2 = 1.0;
    for (size_t k0 = 0; k0 < seq.size();) {
        const size_t k1 = std::min(window_end(lp, seq, k0), k0 + batch);
        pp.clear();
        for (size_t k = k0; k < k1; ++k) {
            const Step &s = seq[k];
            const bool bd = s.kind == STEP_BOUNDARY;
            size_t i = 0;
            while (i < made.size() && (made[i].pass != s.pass || made[i].kind != s.kind))
                ++i;
            if (i == made.size()) {
                made.push_back({s.pass, s.kind, {}});
                PairPass &q = made[i].q;
                MixArgs &a = q.a.m;
                memset(&q.a, 0, sizeof(q.a));
                q.kind = bd ? PAIR_BOUNDARY : s.kind == STEP_PLAIN ? PAIR_PLAIN : PAIR_COST;
                q.mir = s.pass + 1 == m;
                q.cost = q.kind != PAIR_PLAIN;
                if (int rc = pass_shape(N, lp.ps[s.pass].tile, lp.ps[s.pass].gates, A, pair_lane_bit,
                                        q.mir ? Z2_MIRROR : Z2_LOWER, a, q.K, q.lane))
                    return rc;
                if (q.cost) {
                    const Geom geom = layout_geom(N, lp.ps[s.pass].tile, A, q.K);
                    geom_to_args(geom, q.tab);
                    q.tab.ntiles_run = a.ntiles;
                    if (int rc = get_plan(g, geom, &q.tab.plan, st->stream))
                        return rc;
                    q.entries = phase_table_entries(q.tab, A);
                }
            }
            pp.push_back(made[i].q);
            PairPass &q = pp.back();
            MixArgs &a = q.a.m;
            double sr, si, t1, t0;
            const int later = bd ? s.layer + 1 : s.layer;
            rx_tform(-betas[later], st->dtype, true, &t1, &sr, &si);
            rx_tform(-betas[s.layer], st->dtype, true, &t0, &sr, &si);
            a.pre_t = t1;
            a.t = bd ? t0 : t1;
            a.pre_tf = (float)a.pre_t;   // exact for complex64
            a.tf = (float)a.t;
            weight[k] = mag2;
            double w = 1.0;
            auto gate = [&](bool on, double t, double &slot) {
                slot = on ? w : 0.0;
                w *= on ? 1.0 / (1.0 + t * t) : 1.0;
            };
            gate(q.lane, t1, q.a.up[PAIR_LANE]);
            for (int i = 0; i < A * (q.K + 1); ++i)
                gate((a.gates_w >> i) & 1u, t1, q.a.up[i]);
            if (q.cost) {
                q.a.phase = w;
                a.scale_re = std::sqrt(mag2 * w);
                w /= a.scale_re * a.scale_re;
                set_cost(q.tab, -gammas[later], st->init_amp);
            }
            if (bd) {
                for (int l = q.K; l >= 0; --l)
                    for (int r = 0; r < A; ++r)
                        gate((a.gates_w >> (A * l + r)) & 1u, t0, q.a.down[A * l + r]);
                gate(q.lane, t0, q.a.down[PAIR_LANE]);
            }
            mag2 *= w;
        }
        bool tables = false;
        if (int rc = mix_tables(st, pp, &tables, true))
            return rc;
        auto launch = [&](size_t k, const MixArgs &a, hipStream_t stream) {
            const PairPass &q = pp[k - k0];
            PairArgs pa = q.a;
            pa.m = a;
            return launch_pair_pass(st->dtype, q.K, q.lane, q.kind, q.mir, st->sv, st->aux, pa, q.ptab, q.ctab,
                                    st->d_pair + per * (k - k0), stream);
        };
        for (size_t k = k0; k < k1;) {
            const size_t n = std::min(chunk_group(lp, seq, k), k1 - k);   // (its sums fit)
            for (size_t i = k - k0; i < k - k0 + n && !tables; ++i)
                if (pp[i].cost) {
                    double *ctab = nullptr;
                    if (int rc = prepare_phases(st, pp[i].tab, A, &ctab))
                        return rc;
                    pp[i].ptab = st->d_phase;
                    pp[i].ctab = ctab;
                }
            int rc;
            if (n > 1) {
                const int nlog = N - 1 - lp.chunk;
                rc = run_chunks(st, FQ_K_ADJOINT, n, bytes * (double)n, nlog, [&](size_t i, uint64_t c, hipStream_t stream) {
                    return launch(k + i, chunk_args(pp[k - k0 + i].a.m, c, nlog), stream);
                });
            } else {
                rc = timed(st, FQ_K_ADJOINT, bytes, [&] { return launch(k, pp[k - k0].a.m, st->stream); });
            }
            if (rc)
                return rc;
            k += n;
        }
        FQ_HIP(launch_pair_sums(st->d_pair, tiles, (int)(k1 - k0), out + 2 + 3 * k0, st->stream));
        k0 = k1;
    }
    std::vector<double> sums(2 + 3 * seq.size());
    if (out == st->d_grad)
        FQ_HIP(hipMemcpyAsync(sums.data(), out, sizeof(double) * sums.size(), hipMemcpyDeviceToHost, st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    if (out != st->d_grad)
        std::copy(out, out + sums.size(), sums.begin());
    *expect = sums[0];
    const double *h = sums.data() + 2;
    for (int k = 0; k < P; ++k)
        grad_gammas[k] = grad_betas[k] = 0.0;
    for (size_t k = 0; k < seq.size(); ++k) {
        const bool bd = seq[k].kind == STEP_BOUNDARY;
        const int later = bd ? seq[k].layer + 1 : seq[k].layer;
        grad_betas[later] += weight[k] * h[3 * k];
        if (seq[k].kind != STEP_PLAIN)
            grad_gammas[later] = -weight[k] * h[3 * k + 1];
        if (bd)
            grad_betas[seq[k].layer] += weight[k] * h[3 * k + 2];
    }
    return FQ_OK;
}

// Reverse-uncompute gradient of <C> (fq_adjoint.hip, fq_pair.hip).  The state must hold
// psi_P of fq_run(FUSED or Z2) with the same graph and angles (identity qubit
// map); it is consumed (for N >= 3 its lower half is walked back to |+>^N and
// its upper half is left as it was).
extern "C" int fq_backward(fq_state *st, fq_graph *g, int P, const double *gammas,
                           const double *betas, double *expect, double *grad_gammas,
                           double *grad_betas)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = graph_matches(st, g))
        return rc;
    if (P < 1 || !gammas || !betas || !grad_gammas || !grad_betas)
        return set_err(FQ_ERR_ARG, "bad layer count or null arrays");
    for (int p = 0; p < st->N; ++p)
        if (st->qmap[p] != p)
            return set_err(FQ_ERR_ARG, "fq_backward needs the identity qubit map (fused schedule)");
    const int N = st->N;
    // Half states: psi_P and lambda = Cut psi_P satisfy x(b) = x(~b) (Cut(b) =
    // Cut(~b)), and so do both states walked back through U^+ M^+, so for
    // N >= 3 every pass runs on the half z_{N-1} = 0 (the last one as the
    // mirror pass) and every sum counts each element for itself and its
    // complement: the sums are doubled.  The state's upper half is left
    // stale (the state is consumed).
    const bool z2 = N >= 3;
    const double mult = z2 ? 2.0 : 1.0;
    if (const LayerPlan lp = pair_plan(N, st->dtype); !lp.ps.empty()) {
        // the sums of <C>, then of 1 + P (m - 1) passes: in the lane's page, or
        // copied from device memory where they do not fit
        const size_t nsums = 2 + 3 * (1 + (size_t)P * (lp.ps.size() - 1));
        if (int rc = ensure_aux(st, (nsums + 1) / 2))
            return rc;
        double *out = nsums <= FQ_LANE_DOUBLES ? st->lane.host : st->d_grad;
        if (int rc = cut_lambda(st, g, out))
            return rc;
        double e = 0;
        if (int rc = pair_walk(st, g, lp, P, gammas, betas, out, &e, grad_gammas, grad_betas))
            return rc;
        for (int k = 0; k < P; ++k) {
            grad_gammas[k] *= mult;
            grad_betas[k] *= mult;
        }
        if (expect)
            *expect = mult * e;
        return FQ_OK;
    }
    // 2^12-amplitude tiles of psi and lambda share the LDS (2 x 68 KiB);
    // 512 threads x 8 amplitudes of each state
    const int Qb = std::min(12, z2 ? N - 1 : N);
    // The passes of a layer and, as in fq_run's pipelined layers, the pass
    // besides pass 0 that ends every other layer (end1 < 0: layer order)
    std::vector<FusedPass> ps = cover_passes(N, Qb, st->dtype);
    const int m = (int)ps.size();
    const bool pipe = layer_pipe() && m >= (z2 ? 3 : 2);
    const int end1 = pipe ? (z2 ? 1 : m - 1) : -1;
    if (pipe && m >= 3)
        ps = cover_passes(N, Qb, st->dtype, end1);
    // The walk back undoes, in reverse order, the launches of a forward run
    // over this plan: kind 1 a cost pass of layer p (phase, then RX(beta_p)
    // on its qubits: undone as RX then phase), kind 2 RX(beta_p) alone, kind
    // 3 a layer-boundary pass (RX(beta_p), phase gamma_{p+1}, RX(beta_{p+1})).
    // The unitary is the same whichever decomposition the forward used.
    struct Launch {
        int pass, kind, p;
    };
    std::vector<Launch> fwd;
    for (int p = 0; p < P; ++p) {
        if (!pipe) {
            for (int i = 0; i < m; ++i)
                fwd.push_back({i, i == 0 ? 1 : 2, p});
            continue;
        }
        const bool last = p + 1 == P;
        const int e = p % 2 == 0 ? end1 : 0;
        if (p == 0)
            fwd.push_back({0, 1, 0});
        if (last)
            fwd.push_back({e, 2, p});
        for (int i = 1; i < m; ++i)
            if (i != end1)
                fwd.push_back({i, 2, p});
        if (!last)
            fwd.push_back({e, 3, p});
    }
    // gradient slots (two doubles each): slot 0 the <C> sums, then per launch
    // one slot (beta sum, gamma sum), a boundary pass a second (beta_p sum)
    size_t nslot = 1;
    for (const Launch &L : fwd)
        nslot += L.kind == 3 ? 2 : 1;
    if (int rc = ensure_aux(st, nslot))
        return rc;

    if (int rc = cut_lambda(st, g, st->d_grad))
        return rc;
    // (launch index in fwd, first slot) of every launch, for the sums below
    std::vector<size_t> slot_of(fwd.size());
    {
        size_t s_next = 1;
        for (size_t n = 0; n < fwd.size(); ++n) {
            slot_of[n] = s_next;
            s_next += fwd[n].kind == 3 ? 2 : 1;
        }
    }
    for (size_t n = fwd.size(); n-- > 0;) {
        const Launch &L = fwd[n];
        const int i = L.pass;
        const bool costbw = L.kind != 2;
        const bool boundary = L.kind == 3;
        const int Q = (int)ps[i].tile.size();
        // 512 threads x 8 amplitudes of each state
        const int a_log = std::max(1, std::min(3, Q));
        const bool mirror = z2 && i + 1 == m;
        Geom geom;
        TileArgs a;
        if (int rc = pass_args(N, st->dtype, ps[i].tile, ps[i].gates, costbw,
                               z2 ? (mirror ? Z2_MIRROR : Z2_LOWER) : Z2_OFF, a, geom, a_log))
            return rc;
        // the RX undone first: beta_{p+1} in a boundary pass, else beta_p
        const int pb = boundary ? L.p + 1 : L.p;
        rx_coeffs(-betas[pb], st->dtype, &a.rx_c, &a.rx_s);
        if (boundary)
            rx_coeffs(-betas[L.p], st->dtype, &a.pre_c, &a.pre_s);
        double *ctab = nullptr;
        if (costbw) {
            if (int rc = get_plan(g, geom, &a.plan, st->stream))
                return rc;
            set_cost(a, -gammas[pb], st->init_amp);
            if (int rc = prepare_phases(st, a, a_log, &ctab))
                return rc;
        }
        if (boundary && 2 * run_tiles(a) > st->part_cap)
            return set_err(FQ_ERR_ARG, "internal: partial-sum buffer too small for a boundary pair pass");
        double *slot = st->d_grad + 2 * slot_of[n];
        int rc = timed(st, FQ_K_ADJOINT, 4.0 * (double)st->bytes / mult, [&] {
            unsigned grid = 0;
            hipError_t e = launch_pair(st->dtype, a_log, costbw, mirror, boundary, st->sv, st->aux, a,
                                       costbw ? st->d_phase : nullptr, ctab, st->d_part, &grid, st->stream);
            if (e != hipSuccess)
                return e;
            e = launch_finalize(st->d_part, grid, slot, st->stream);
            if (e != hipSuccess || !boundary)
                return e;
            return launch_finalize(st->d_part + 2 * (size_t)grid, grid, slot + 2, st->stream);
        });
        if (rc)
            return rc;
    }
    std::vector<double> h(2 * nslot);
    FQ_HIP(hipMemcpyAsync(h.data(), st->d_grad, sizeof(double) * h.size(), hipMemcpyDeviceToHost,
                          st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    if (expect)
        *expect = mult * h[0];
    for (int k = 0; k < P; ++k) {
        grad_betas[k] = 0.0;
        grad_gammas[k] = 0.0;
    }
    for (size_t n = 0; n < fwd.size(); ++n) {
        const Launch &L = fwd[n];
        const size_t s0 = slot_of[n];
        const int pb = L.kind == 3 ? L.p + 1 : L.p;
        grad_betas[pb] += mult * h[2 * s0];
        if (L.kind != 2)
            grad_gammas[pb] = -mult * h[2 * s0 + 1];
        if (L.kind == 3)
            grad_betas[L.p] += mult * h[2 * (s0 + 1)];
    }
    return FQ_OK;
}

static uint64_t to_logical_index(const fq_state *st, uint64_t b)
{
    uint64_t L = 0;
    for (int p = 0; p < st->N; ++p)
        L |= ((b >> p) & 1ull) << st->qmap[p];
    return L;
}

static uint64_t to_physical_index(const fq_state *st, uint64_t L)
{
    uint64_t b = 0;
    for (int p = 0; p < st->N; ++p)
        b |= ((L >> st->qmap[p]) & 1ull) << p;
    return b;
}

extern "C" int fq_topk(fq_state *st, int k, uint64_t *idx, double *prob)
{
    if (int rc = check_state(st))
        return rc;
    if (k < 1 || k > FQ_TOPK_MAX || !idx || !prob)
        return set_err(FQ_ERR_ARG, "k=%d must be in [1, %d] with non-null outputs", k, FQ_TOPK_MAX);
    if ((uint64_t)k > (1ull << st->N))
        return set_err(FQ_ERR_ARG, "k=%d exceeds the number of basis states", k);
    const int nb = st->cand_blocks;
    int rc = timed(st, FQ_K_TOPK, (double)st->bytes, [&] {
        return launch_topk(st->dtype, st->sv, st->N, nb, st->d_cand_p, st->d_cand_i, st->stream);
    });
    if (rc)
        return rc;
    std::vector<double> cp((size_t)nb * FQ_TOPK_MAX);
    std::vector<uint64_t> ci((size_t)nb * FQ_TOPK_MAX);
    FQ_HIP(hipMemcpyAsync(cp.data(), st->d_cand_p, sizeof(double) * cp.size(),
                          hipMemcpyDeviceToHost, st->stream));
    FQ_HIP(hipMemcpyAsync(ci.data(), st->d_cand_i, sizeof(uint64_t) * ci.size(),
                          hipMemcpyDeviceToHost, st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    std::vector<size_t> order(cp.size());
    for (size_t i = 0; i < order.size(); ++i)
        order[i] = i;
    std::partial_sort(order.begin(), order.begin() + k, order.end(), [&](size_t x, size_t y) {
        return cp[x] > cp[y] || (cp[x] == cp[y] && ci[x] < ci[y]);
    });
    for (int i = 0; i < k; ++i) {
        prob[i] = cp[order[i]];
        idx[i] = to_logical_index(st, ci[order[i]]);
    }
    return FQ_OK;
}

extern "C" int fq_qubit_map(const fq_state *st, int *map)
{
    if (int rc = check_state(st))
        return rc;
    if (!map)
        return set_err(FQ_ERR_ARG, "null output pointer");
    for (int p = 0; p < st->N; ++p)
        map[p] = st->qmap[p];
    return FQ_OK;
}

extern "C" int fq_state_copy_out(fq_state *st, void *host, size_t bytes, int logical)
{
    if (int rc = check_state(st))
        return rc;
    if (!host || bytes != st->bytes)
        return set_err(FQ_ERR_ARG, "copy_out needs exactly %zu bytes", st->bytes);
    bool ident = true;
    for (int p = 0; p < st->N; ++p)
        ident = ident && st->qmap[p] == p;
    if (!logical || ident) {
        FQ_HIP(hipMemcpyAsync(host, st->sv, bytes, hipMemcpyDeviceToHost, st->stream));
        FQ_HIP(hipStreamSynchronize(st->stream));
        return FQ_OK;
    }
    std::vector<char> tmp(bytes);
    FQ_HIP(hipMemcpyAsync(tmp.data(), st->sv, bytes, hipMemcpyDeviceToHost, st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    // physical -> logical index, one table lookup per index byte
    const int nbytes_idx = (st->N + 7) / 8;
    std::vector<uint64_t> tab((size_t)nbytes_idx * 256, 0);
    for (int k = 0; k < nbytes_idx; ++k)
        for (int v = 0; v < 256; ++v) {
            uint64_t L = 0;
            for (int i = 0; i < 8 && 8 * k + i < st->N; ++i)
                if ((v >> i) & 1)
                    L |= 1ull << st->qmap[8 * k + i];
            tab[(size_t)k * 256 + v] = L;
        }
    const uint64_t n = 1ull << st->N;
    char *dst = (char *)host;
    for (uint64_t b = 0; b < n; ++b) {
        uint64_t L = 0;
        for (int k = 0; k < nbytes_idx; ++k)
            L |= tab[(size_t)k * 256 + ((b >> (8 * k)) & 255)];
        memcpy(dst + L * st->elem, tmp.data() + b * st->elem, st->elem);
    }
    return FQ_OK;
}

extern "C" int fq_state_copy_in(fq_state *st, const void *host, size_t bytes)
{
    if (int rc = check_state(st))
        return rc;
    if (!host || bytes != st->bytes)
        return set_err(FQ_ERR_ARG, "copy_in needs exactly %zu bytes", st->bytes);
    FQ_HIP(hipMemcpyAsync(st->sv, host, bytes, hipMemcpyHostToDevice, st->stream));
    FQ_HIP(hipStreamSynchronize(st->stream));
    return FQ_OK;
}

extern "C" int fq_state_gather(fq_state *st, const uint64_t *idx, size_t n, double *out, int logical)
{
    if (int rc = check_state(st))
        return rc;
    if (n == 0)
        return FQ_OK;
    if (!idx || !out)
        return set_err(FQ_ERR_ARG, "null argument");
    const uint64_t lim = 1ull << st->N;
    std::vector<uint64_t> phys(n);
    for (size_t i = 0; i < n; ++i) {
        if (idx[i] >= lim)
            return set_err(FQ_ERR_ARG, "index %llu out of range", (unsigned long long)idx[i]);
        phys[i] = logical ? to_physical_index(st, idx[i]) : idx[i];
    }
    uint64_t *d_idx = nullptr;
    double *d_out = nullptr;
    if (hipMalloc(&d_idx, sizeof(uint64_t) * n) != hipSuccess ||
        hipMalloc(&d_out, sizeof(double) * 2 * n) != hipSuccess) {
        hipFree(d_idx);
        return set_err(FQ_ERR_OOM, "gather scratch allocation failed");
    }
    int rc = FQ_OK;
    if (hipMemcpyAsync(d_idx, phys.data(), sizeof(uint64_t) * n, hipMemcpyHostToDevice, st->stream) != hipSuccess ||
        launch_gather(st->dtype, st->sv, d_idx, n, d_out, st->stream) != hipSuccess ||
        hipMemcpyAsync(out, d_out, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, st->stream) != hipSuccess ||
        hipStreamSynchronize(st->stream) != hipSuccess)
        rc = set_err(FQ_ERR_DEVICE, "gather failed");
    hipFree(d_idx);
    hipFree(d_out);
    return rc;
}

extern "C" int fq_state_clone(fq_state *dst, const fq_state *src)
{
    if (int rc = check_state(dst))
        return rc;
    if (int rc = check_state(src))
        return rc;
    if (dst->N != src->N || dst->dtype != src->dtype)
        return set_err(FQ_ERR_ARG, "clone needs equal N and dtype");
    if (dst == src)
        return FQ_OK;
    // the copy runs on dst's stream after src's queued work; src's later work
    // waits for the copy (it must not overwrite src while it is read)
    hipEvent_t ev = nullptr;
    FQ_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    hipError_t e = hipEventRecord(ev, src->stream);
    if (e == hipSuccess)
        e = hipStreamWaitEvent(dst->stream, ev, 0);
    if (e == hipSuccess)
        e = hipMemcpyAsync(dst->sv, src->sv, src->bytes, hipMemcpyDeviceToDevice, dst->stream);
    if (e == hipSuccess)
        e = hipEventRecord(ev, dst->stream);
    if (e == hipSuccess)
        e = hipStreamWaitEvent(src->stream, ev, 0);
    hipEventDestroy(ev);
    if (e != hipSuccess)
        return set_err(FQ_ERR_DEVICE, "clone: %s", hipGetErrorString(e));
    for (int p = 0; p < FQ_MAXN; ++p)
        dst->qmap[p] = src->qmap[p];
    return FQ_OK;
}

extern "C" int fq_sync(fq_state *st)
{
    if (int rc = check_state(st))
        return rc;
    FQ_HIP(hipStreamSynchronize(st->stream));
    return FQ_OK;
}

extern "C" int fq_timing_enable(fq_state *st, int on)
{
    if (int rc = check_state(st))
        return rc;
    st->timing = on != 0;
    return FQ_OK;
}

extern "C" int fq_timing_get(fq_state *st, int kind, double *ms, int64_t *count, double *bytes)
{
    if (int rc = check_state(st))
        return rc;
    if (kind < 0 || kind >= FQ_K_COUNT)
        return set_err(FQ_ERR_ARG, "unknown kernel class %d", kind);
    if (int rc = timing_collect(st))
        return rc;
    if (ms)
        *ms = st->t_ms[kind];
    if (count)
        *count = st->t_cnt[kind];
    if (bytes)
        *bytes = st->t_bytes[kind];
    return FQ_OK;
}

extern "C" int fq_stream_probe(size_t bytes, int reps, double *inplace_gbs, double *read_gbs,
                               double *write_gbs)
{
    if (bytes < ((size_t)1 << 20) || bytes % 8 || reps < 1 || !inplace_gbs || !read_gbs || !write_gbs)
        return set_err(FQ_ERR_ARG, "stream probe needs bytes >= 1 MiB (a multiple of 8), reps >= 1 and outputs");
    if (!budget_take(bytes))
        return set_err(FQ_ERR_BUDGET, "stream probe of %zu bytes exceeds the memory budget", bytes);
    void *buf = nullptr;
    float *sink = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    double out[3] = {0, 0, 0};
    int rc = FQ_OK;
    hipError_t e = hipMalloc(&buf, bytes);
    if (e == hipSuccess)
        e = hipMalloc(&sink, sizeof(float));
    if (e == hipSuccess)
        e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (e == hipSuccess)
        e = hipEventCreate(&e0);
    if (e == hipSuccess)
        e = hipEventCreate(&e1);
    if (e == hipSuccess)
        e = launch_stream(buf, bytes, 2, sink, s);  // first touch
    // modes 0 (in place), 1 (read), 2 (fill): traffic 2, 1, 1 x bytes
    for (int mode = 0; mode < 3 && e == hipSuccess; ++mode) {
        e = hipEventRecord(e0, s);
        for (int r = 0; r < reps && e == hipSuccess; ++r)
            e = launch_stream(buf, bytes, mode, sink, s);
        if (e == hipSuccess)
            e = hipEventRecord(e1, s);
        if (e == hipSuccess)
            e = hipEventSynchronize(e1);
        float ms = 0.0f;
        if (e == hipSuccess)
            e = hipEventElapsedTime(&ms, e0, e1);
        if (e == hipSuccess && ms > 0.0f)
            out[mode] = (mode == 0 ? 2.0 : 1.0) * (double)bytes * reps / (ms * 1e-3) / 1e9;
    }
    if (e != hipSuccess)
        rc = set_err(FQ_ERR_DEVICE, "stream probe: %s", hipGetErrorString(e));
    if (s)
        hipStreamSynchronize(s);
    if (e0)
        hipEventDestroy(e0);
    if (e1)
        hipEventDestroy(e1);
    if (s)
        hipStreamDestroy(s);
    hipFree(sink);
    hipFree(buf);
    budget_give(bytes);
    if (rc)
        return rc;
    *inplace_gbs = out[0];
    *read_gbs = out[1];
    *write_gbs = out[2];
    return FQ_OK;
}

extern "C" int fq_timing_reset(fq_state *st)
{
    if (int rc = check_state(st))
        return rc;
    if (int rc = timing_collect(st))
        return rc;
    for (int k = 0; k < FQ_K_COUNT; ++k) {
        st->t_ms[k] = 0;
        st->t_cnt[k] = 0;
        st->t_bytes[k] = 0;
    }
    return FQ_OK;
}

// ---- packed slabs (continuous batching) ------------------------------------------------

struct SlotHost {
    fq_graph *g = nullptr;
    int P = 0, layer = 0;
    int phase = 0;  // 0 free, 1 active, 2 finished (result pending collection)
    std::vector<double> gammas, betas;
    double amp_scale = 1.0;   // rx_norm_scale of the request
    SlotPlans plans{};        // cost and <C> plans of g, fetched at assignment
    bool fresh = false;       // not yet in device memory
    uint64_t gversion = 0;    // g->version the plans belong to
    uint64_t gepoch = 0;      // g->plan_epoch the plan pointers belong to
    PlanEntry *entries[5] = {nullptr};   // of the plans, while that is the graph's epoch
    std::vector<double> W;    // the weights of the open layer's phase
    int has_rr[4] = {0, 0, 0, 0};
};

// One pass of a packed slab on the compile-time kernel (fq_mix.h): its
// launch arguments without the slots' factors.
struct PackedPass {
    MixArgs a;
    int K = 0;
    bool lane = false, mir = false;
};

// Launch arguments of one slab tile pass (fixed for the slab's lifetime).
struct SlabPass {
    TileArgs args;
    int a_log = 1, slot_shift = 0;
    bool mirror = false;
};

// Layers per step of a new slab of large slots (fq_slab_set_layers_per_step):
// FQ_SLAB_LAYERS (environment, read per slab creation), default 1.
static int slab_layers_default()
{
    const char *e = getenv("FQ_SLAB_LAYERS");
    const int v = e ? atoi(e) : 1;
    return v >= 1 ? v : 1;
}

struct fq_slab {
    int N = 0, K = 0, s = 0, dtype = 0;
    bool z2 = false;  // slots hold the half state z_{N-1} = 0
    size_t elem = 8, slot_bytes = 0, bytes = 0;
    void *sv = nullptr;
    hipStream_t stream = nullptr;
    std::vector<SlotHost> slots;
    // a step's parameters, uploaded together: SlotParams [K], MixSlot [2 K],
    // SlabJob [2 K], finishing slots [K]
    char *d_step = nullptr, *h_step = nullptr;
    SlotPlans *d_plans = nullptr, *h_plans = nullptr;
    double2 *d_tabs = nullptr;
    size_t tab_stride = 0;
    double *d_part = nullptr;
    double *h_res = nullptr;   // results (pinned host memory that the kernels write)
    hipEvent_t done = nullptr;
    bool pending = false;  // a step was enqueued and not yet observed complete
    double init_amp = 0;
    std::vector<FusedPass> passes;
    // launch arguments built once at creation
    TileArgs cost_args{};      // phase tables: pass-1 geometry of the N-qubit state
    Geom cost_geom{}, exp_geom{};
    std::vector<SlabPass> pass_args;
    TileArgs exp_args{};       // <C> over the virtual state
    int exp_alog = 1, exp_shift = 0;
    // packed: every step runs one pass of a two-pass plan on each slot, in one
    // launch for all slots that do the same (fq_slab_step)
    bool packed = false;
    std::vector<PackedPass> pk;
    Geom pk_geom[4];          // cost geometries, 2 * (boundary pass) + pass
    SlabGeos pk_tab{};
    size_t pk_entries = 0;    // of the largest table
    int pk_end = 0;           // pass that ends the next step's layer
    // large slots: each slot runs the single-state tile passes of fq_run
    // (pipelined layers) over its own 2^N (or 2^(N-1)) amplitudes instead of
    // one packed launch; views[k] is slot k seen as a state (its amplitudes,
    // the slab's stream, its own phase-table buffer)
    bool per_slot = false;
    LayerPlan slot_plan;
    std::vector<fq_state *> views;
    int layers_per_step = 1;   // per_slot slabs: layers a step runs per slot
};

// Offsets of the arrays of a step's parameters.
static size_t step_mix(int K) { return sizeof(SlotParams) * (size_t)K; }
static size_t step_jobs(int K) { return step_mix(K) + sizeof(MixSlot) * 2 * (size_t)K; }
static size_t step_fin(int K) { return step_jobs(K) + sizeof(SlabJob) * 2 * (size_t)K; }
static size_t step_bytes(int K) { return step_fin(K) + sizeof(int) * (size_t)K; }

static void slab_free(fq_slab *sb)
{
    if (sb->stream)
        hipStreamSynchronize(sb->stream);
    for (fq_state *v : sb->views) {
        free_phases(v);
        delete v;
    }
    sb->views.clear();
    if (sb->sv)
        budget_give(sb->bytes);
    hipFree(sb->sv);
    hipFree(sb->d_step);
    hipHostFree(sb->h_step);
    hipFree(sb->d_plans);
    hipFree(sb->d_tabs);
    hipFree(sb->d_part);
    if (sb->done)
        hipEventDestroy(sb->done);
    if (sb->stream) {
        own_stream(sb->stream, false);
        hipStreamDestroy(sb->stream);
    }
    delete sb;
}

// Reduction tile width of a slab's <C> (a half-state slab reduces its N-1 stored qubits).
static int slab_qe(const fq_slab *sb) { return std::min(12, sb->z2 ? sb->N - 1 : sb->N); }

// Phase-table arguments of a slab's cost pass: the N-qubit geometry of pass 1
// (a half-state slab uses its lower half of the tiles).
static TileArgs slab_cost_args(const fq_slab *sb, Geom *gout)
{
    const int Q1 = (int)sb->passes[0].tile.size();
    Geom g1 = make_geom(sb->N, sb->passes[0].tile, tile_a_log(sb->dtype, Q1));
    TileArgs a1;
    geom_to_args(g1, a1);
    if (sb->z2)
        a1.ntiles_run = 1ull << (g1.nh - 1);
    if (gout)
        *gout = g1;
    return a1;
}

// Passes and table geometries of a packed slab (two-pass plan lp).
static int slab_build_packed(fq_slab *sb, const LayerPlan &lp)
{
    const int N = sb->N;
    for (int i = 0; i < 2; ++i) {
        const FusedPass &fp = lp.ps[i];
        const int A = mix_a_log(sb->dtype, (int)fp.tile.size());
        PackedPass p;
        p.mir = sb->z2 && i == 1;
        if (int rc = pass_shape(N, fp.tile, fp.gates, A, mix_lane_bit,
                                !sb->z2 ? Z2_OFF : p.mir ? Z2_MIRROR : Z2_LOWER, p.a, p.K, p.lane))
            return rc;
        p.a.init_amp = sb->init_amp;
        sb->pk.push_back(p);
        for (int bd = 0; bd < 2; ++bd) {
            const Geom g = layout_geom(N, fp.tile, A, bd ? p.K : 0);
            sb->pk_geom[2 * bd + i] = g;
            TileArgs ta;
            geom_to_args(g, ta);
            ta.ntiles_run = p.a.ntiles;
            TableGeo &tg = sb->pk_tab.geo[2 * bd + i];
            tg.Q = ta.Q;
            tg.nthr = ta.nthr;
            tg.nh = ta.nh;
            tg.a_log = A;
            tg.ntiles = p.a.ntiles;
            sb->pk_entries = std::max(sb->pk_entries, phase_table_entries(ta, A));
        }
    }
    sb->slot_plan = lp;
    sb->tab_stride = 2 * sb->pk_entries;   // a slot's first layer has two tables
    return FQ_OK;
}

// Tile-pass and <C> launch arguments of a slab (its virtual state: the Ns
// stored qubits, then the slot bits; the mirror pass of a half-state slab
// keeps qubit N-1 as a position above them).
static int slab_build_args(fq_slab *sb)
{
    const int N = sb->N;
    const int Ns = sb->z2 ? N - 1 : N;
    sb->pass_args.clear();
    for (size_t i = 0; i < sb->passes.size(); ++i) {
        const FusedPass &ps = sb->passes[i];
        const int Q = (int)ps.tile.size();
        SlabPass sp;
        sp.a_log = tile_a_log(sb->dtype, Q);
        sp.mirror = sb->z2 && i + 1 == sb->passes.size();
        std::vector<int> tile = ps.tile;
        if (sp.mirror)
            tile.back() = Ns + sb->s;
        Geom gv = make_geom(Ns + sb->s + (sp.mirror ? 1 : 0), tile, sp.a_log);
        if (geom_runs(gv) > FQ_MAX_RUNS)
            return set_err(FQ_ERR_ARG, "internal: slab tile needs too many bit runs");
        geom_to_args(gv, sp.args);
        uint32_t gm = 0;
        for (int q : ps.gates)
            for (int ti = 0; ti < Q; ++ti)
                if (ps.tile[ti] == q)
                    gm |= 1u << ti;
        if (int rc = set_gates(sp.args, gv, gm))
            return rc;
        if (sp.mirror)
            for (int ti = 0; ti + 1 < Q; ++ti)
                sp.args.mirror_pm += 1ull << tile[ti];
        sp.slot_shift = sp.mirror ? N - Q : Ns - Q;
        sb->pass_args.push_back(sp);
    }
    const int Qe = slab_qe(sb);
    sb->exp_alog = std::max(1, std::min(4, Qe));
    sb->exp_geom = make_geom(N, low_tile(Qe), sb->exp_alog);
    geom_to_args(make_geom(Ns + sb->s, low_tile(Qe), sb->exp_alog), sb->exp_args);
    sb->exp_shift = Ns - Qe;
    const LayerPlan lp = exec_plan(N, sb->dtype, sb->z2, 1);
    sb->packed = lp.split && lp.ps.size() == 2 && (int)lp.ps[0].tile.size() < tile_max_q(sb->dtype);
    if (sb->packed)
        return slab_build_packed(sb, lp);
    // passes that fill the device on one slot: one slot after the other (three
    // passes, or tiles of full width, which take no packed launches)
    const int Q1 = (int)sb->passes[0].tile.size();
    sb->per_slot = lp.split || Ns - Q1 >= 10;   // (or 1,024 tiles)
    if (sb->per_slot) {
        sb->slot_plan = lp;
        sb->slot_plan.chunk = 0;   // a step is one layer, launched pass by pass
    }
    return FQ_OK;
}

// Per-slot state views of a slab (after its amplitudes and stream exist); of a
// per-slot slab each with a phase-table buffer, so no step allocates.
static int slab_make_views(fq_slab *sb)
{
    const LayerPlan &lp = sb->slot_plan;
    const int m = (int)lp.ps.size();
    size_t need = 0;   // the tables of the first layer's two cost passes
    for (int i = 0; i < m && sb->per_slot; ++i) {
        if (i != 0 && i != lp.end1)
            continue;
        TileArgs a;
        size_t most = 0;
        if (const int A = mix_a_log(sb->dtype, (int)lp.ps[i].tile.size())) {
            geom_to_args(layout_geom(sb->N, lp.ps[i].tile, A, 0), a);
            a.ntiles_run = sb->z2 ? 1ull << (a.nh - 1) : 0;
            most = phase_table_entries(a, A);
        } else {
            Geom geom;
            const int z2 = !sb->z2 ? Z2_OFF : i + 1 < m ? Z2_LOWER : Z2_MIRROR;
            if (int rc = pass_args(sb->N, sb->dtype, lp.ps[i].tile, lp.ps[i].gates, true, z2, a, geom))
                return rc;
            most = phase_table_entries(a, geom.a_log);
        }
        need += most * sizeof(double2);
    }
    for (int k = 0; k < sb->K; ++k) {
        fq_state *v = new fq_state();
        v->N = sb->N;
        v->dtype = sb->dtype;
        v->elem = sb->elem;
        v->bytes = sb->slot_bytes;
        v->sv = (char *)sb->sv + sb->slot_bytes * (size_t)k;
        v->stream = sb->stream;
        for (int q = 0; q < FQ_MAXN; ++q)
            v->qmap[q] = q;
        v->init_amp = sb->init_amp;
        v->in_run = true;   // a slot runs fq_run's layers on a QAOA state
        v->slot = true;
        sb->views.push_back(v);
        if (need && hipMalloc(&v->d_phase, need) != hipSuccess) {
            hipGetLastError();
            v->d_phase = nullptr;
            return set_err(FQ_ERR_OOM, "slab phase-table allocation failed");
        }
        v->phase_cap = need;
    }
    return FQ_OK;
}

// Cost and <C> plans of a slot's graph (again after the graph changed).
static int slab_slot_plans(fq_slab *sb, SlotHost &h)
{
    const PlanHold hold(h.g);   // (so that none of them replaces another)
    for (int i = 0; i < (sb->packed ? 4 : 1); ++i) {
        if (int rc = get_plan(h.g, sb->packed ? sb->pk_geom[i] : sb->cost_geom, &h.plans.cost[i], sb->stream,
                              &h.entries[i]))
            return rc;
        h.has_rr[i] = 0;
        for (int j = 0; j < FQ_MAX_REGS; ++j)
            if (h.plans.cost[i].rr[j] != 0)
                h.has_rr[i] = 1;
    }
    if (int rc = get_plan(h.g, sb->exp_geom, &h.plans.expect, sb->stream, &h.entries[4]))
        return rc;
    h.fresh = true;
    h.gversion = h.g->version;
    h.gepoch = h.g->plan_epoch;
    h.W = h.g->W;
    return FQ_OK;
}

// Whether a step's last pass also opens the next layer of a slot that goes on.
static bool slab_opens_ahead(const fq_slab *sb)
{
    return (sb->packed || sb->per_slot) && sb->slot_plan.end1 >= 0;
}

// The pass that ended a running slot's last layer (and opened the next one).
static int slab_ended_on(const fq_slab *sb, const SlotHost &h)
{
    return sb->packed ? 1 - sb->pk_end : (h.layer - 1) % 2 == 0 ? sb->slot_plan.end1 : 0;
}

// That pass again on v (the slot, or a copy of it): RX(pre), the phase of gamma with
// weights W, RX(beta).  Waits.
static int slab_again(fq_slab *sb, const SlotHost &h, fq_state *v, const std::vector<double> &W, double pre, double gamma,
                      double beta)
{
    const LayerPlan &lp = sb->slot_plan;
    const int e = slab_ended_on(sb, h);
    const int mode = !sb->z2 ? Z2_OFF : e + 1 < (int)lp.ps.size() ? Z2_LOWER : Z2_MIRROR;
    fq_graph g;   // (plans of its own: none of the slot's graph goes for them)
    g.N = sb->N;
    g.W = W;
    const int rc = tile_pass(v, lp.ps[e].tile, lp.ps[e].gates, beta, &g, gamma, true, false, FQ_K_FUSED, mode, &pre, false);
    const hipError_t done = hipStreamSynchronize(sb->stream);
    plans_free(&g, true);
    return rc == FQ_OK && done != hipSuccess ? set_err(FQ_ERR_DEVICE, "slab: %s", hipGetErrorString(done)) : rc;
}

// A graph that changes while a request runs counts from the next layer on.  That
// layer is open already (with the old weights): RX off, the phase of the difference,
// RX on again.
static int slab_reopen(fq_slab *sb, int slot)
{
    SlotHost &h = sb->slots[slot];
    const int L = h.layer;
    std::vector<double> W = h.g->W;
    bool any = false;
    for (size_t i = 0; i < W.size(); ++i) {
        W[i] -= h.W[i];
        any |= W[i] != 0;
    }
    if (any)
        if (int rc = slab_again(sb, h, sb->views[slot], W, -h.betas[L], h.gammas[L], h.betas[L]))
            return rc;
    h.W = h.g->W;   // (now, not with the new plans: a step that fails on those is called again)
    return FQ_OK;
}

static bool slab_slot_stale(const SlotHost &h)
{
    return h.g->version != h.gversion || h.g->plan_epoch != h.gepoch;
}

// A slab without its launch arguments, memory or stream.
static fq_slab *slab_shape(int N, int nslots, int s, int dtype, bool z2)
{
    fq_slab *sb = new fq_slab();
    sb->N = N;
    sb->K = nslots;
    sb->s = s;
    sb->dtype = dtype;
    sb->z2 = z2;
    sb->elem = dtype == FQ_C128 ? 16 : 8;
    sb->slot_bytes = ((size_t)1 << (z2 ? N - 1 : N)) * sb->elem;
    sb->bytes = sb->slot_bytes * nslots;
    sb->slots.resize(nslots);
    sb->init_amp = pow(1. / sqrt(2.), N);
    sb->passes = cover_passes(N, std::min(tile_max_q(dtype), z2 ? N - 1 : N), dtype);
    return sb;
}

extern "C" int fq_slab_passes(int N, int dtype, int schedule, int P, int *npass)
{
    if (N < 1 || N > 36 || (dtype != FQ_C128 && dtype != FQ_C64) || P < 1 || !npass)
        return set_err(FQ_ERR_ARG, "bad N, dtype or layer count, or null output");
    if (schedule != FQ_SCHED_FUSED && (schedule != FQ_SCHED_Z2 || N < 3))
        return set_err(FQ_ERR_ARG, "slab schedule must be FQ_SCHED_FUSED or FQ_SCHED_Z2 (N >= 3)");
    fq_slab *sb = slab_shape(N, 1, 0, dtype, schedule == FQ_SCHED_Z2);
    const int rc = slab_build_args(sb);
    const int m = (int)(sb->packed || sb->per_slot ? sb->slot_plan.ps : sb->passes).size();
    *npass = slab_opens_ahead(sb) ? 1 + P * (m - 1) : P * m;
    delete sb;
    return rc;
}

extern "C" int fq_slab_create(int N, int nslots, int dtype, fq_slab **out)
{
    return fq_slab_create_sched(N, nslots, dtype, FQ_SCHED_FUSED, out);
}

extern "C" int fq_slab_create_sched(int N, int nslots, int dtype, int schedule, fq_slab **out)
{
    if (!out)
        return set_err(FQ_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (dtype != FQ_C128 && dtype != FQ_C64)
        return set_err(FQ_ERR_ARG, "dtype must be FQ_C128 or FQ_C64");
    if (schedule != FQ_SCHED_FUSED && schedule != FQ_SCHED_Z2)
        return set_err(FQ_ERR_ARG, "slab schedule must be FQ_SCHED_FUSED or FQ_SCHED_Z2");
    if (nslots < 1 || (nslots & (nslots - 1)))
        return set_err(FQ_ERR_ARG, "nslots=%d must be a power of two", nslots);
    int s = 0;
    while ((1 << s) < nslots)
        ++s;
    if (N < 1 || N + s > 36)
        return set_err(FQ_ERR_ARG, "N=%d with %d slots out of range", N, nslots);
    const bool z2 = schedule == FQ_SCHED_Z2;
    if (z2 && N < 3)
        return set_err(FQ_ERR_ARG, "the half-state schedule needs N >= 3");
    fq_slab *sb = slab_shape(N, nslots, s, dtype, z2);
    if (!budget_take(sb->bytes)) {
        delete sb;
        return set_err(FQ_ERR_BUDGET, "slab of %d x 2^%d amplitudes exceeds the memory budget", nslots, N);
    }
    // launch arguments and scratch sizes
    sb->cost_args = slab_cost_args(sb, &sb->cost_geom);
    sb->tab_stride = phase_table_entries(sb->cost_args, sb->cost_geom.a_log);
    const int Qe = slab_qe(sb);
    const size_t etiles = ((size_t)1 << ((z2 ? N - 1 : N) - Qe)) * nslots;
    if (int rc = slab_build_args(sb)) {
        budget_give(sb->bytes);
        delete sb;
        return rc;
    }
    bool ok = hipMalloc(&sb->sv, sb->bytes) == hipSuccess;
    if (!ok) {
        hipGetLastError();
        sb->sv = nullptr;
        budget_give(sb->bytes);
        slab_free(sb);
        return set_err(FQ_ERR_OOM, "slab allocation of %zu bytes failed", (size_t)(((size_t)1 << N) * (dtype == FQ_C128 ? 16 : 8) * nslots));
    }
    // one pinned allocation: a step's parameters, the plans, the results
    const size_t o_plans = (step_bytes(nslots) + 63) & ~(size_t)63, o_res = o_plans + sizeof(SlotPlans) * nslots;
    ok = hipMalloc(&sb->d_step, step_bytes(nslots)) == hipSuccess &&
         hipHostMalloc(&sb->h_step, o_res + sizeof(double) * 2 * nslots, hipHostMallocDefault) == hipSuccess &&
         hipMalloc(&sb->d_plans, sizeof(SlotPlans) * nslots) == hipSuccess &&
         hipMalloc(&sb->d_tabs, sizeof(double2) * sb->tab_stride * nslots) == hipSuccess &&
         hipMalloc(&sb->d_part, sizeof(double) * 2 * etiles) == hipSuccess &&
         hipStreamCreateWithFlags(&sb->stream, hipStreamNonBlocking) == hipSuccess &&
         hipEventCreateWithFlags(&sb->done, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        hipGetLastError();
        slab_free(sb);
        return set_err(FQ_ERR_OOM, "slab scratch allocation failed");
    }
    own_stream(sb->stream, true);
    sb->layers_per_step = slab_layers_default();
    if (sb->per_slot || sb->packed)
        if (int rc = slab_make_views(sb)) {
            slab_free(sb);
            return rc;
        }
    memset(sb->h_step, 0, step_bytes(nslots));
    sb->h_plans = (SlotPlans *)(sb->h_step + o_plans);
    sb->h_res = (double *)(sb->h_step + o_res);
    *out = sb;
    return FQ_OK;
}

extern "C" int fq_slab_destroy(fq_slab *sb)
{
    if (sb)
        slab_free(sb);
    return FQ_OK;
}

extern "C" int fq_slab_info(const fq_slab *sb, int *N, int *nslots, int *free_slots, int *active)
{
    if (!sb)
        return set_err(FQ_ERR_ARG, "null slab");
    int fr = 0, ac = 0;
    for (const SlotHost &h : sb->slots) {
        fr += h.phase == 0;
        ac += h.phase == 1;
    }
    if (N)
        *N = sb->N;
    if (nslots)
        *nslots = sb->K;
    if (free_slots)
        *free_slots = fr;
    if (active)
        *active = ac;
    return FQ_OK;
}

extern "C" int fq_slab_assign(fq_slab *sb, int slot, fq_graph *g, int P, const double *gammas,
                              const double *betas)
{
    if (!sb || !g)
        return set_err(FQ_ERR_ARG, "null slab or graph");
    if (slot < 0 || slot >= sb->K)
        return set_err(FQ_ERR_ARG, "slot %d out of range", slot);
    if (g->N != sb->N)
        return set_err(FQ_ERR_ARG, "graph has N=%d, slab has N=%d", g->N, sb->N);
    if (P < 1 || !gammas || !betas)
        return set_err(FQ_ERR_ARG, "bad layer count or angle arrays");
    for (int p = 0; p < P; ++p)
        if (!std::isfinite(gammas[p]) || !std::isfinite(betas[p]))
            return set_err(FQ_ERR_ARG, "angles must be finite");
    SlotHost &h = sb->slots[slot];
    if (h.phase != 0)
        return set_err(FQ_ERR_ARG, "slot %d is not free", slot);
    h.g = g;
    if (int rc = slab_slot_plans(sb, h)) {
        h.g = nullptr;
        return rc;
    }
    h.P = P;
    h.layer = 0;
    h.phase = 1;
    h.gammas.assign(gammas, gammas + P);
    h.betas.assign(betas, betas + P);
    h.amp_scale = rx_norm_scale(sb->N, P, betas, sb->dtype);
    return FQ_OK;
}

extern "C" int fq_slab_poll(fq_slab *sb, int *busy)
{
    if (!sb || !busy)
        return set_err(FQ_ERR_ARG, "null argument");
    if (!sb->pending) {
        *busy = 0;
        return FQ_OK;
    }
    hipError_t e = hipEventQuery(sb->done);
    if (e == hipErrorNotReady) {
        *busy = 1;
        return FQ_OK;
    }
    if (e != hipSuccess)
        return set_err(FQ_ERR_DEVICE, "slab step failed: %s", hipGetErrorString(e));
    sb->pending = false;
    *busy = 0;
    return FQ_OK;
}

// One layer of every active slot of a packed slab.  The slots go in step: a step
// ends their layers on one of the two passes (pk_end, alternately) with a
// boundary pass, which opens the next layer there, or with a plain one where the
// request is done; a slot that enters first writes its state in the other pass.
// Each of the three is one launch over its slots, and one launch makes all
// phase tables.  48 requests of N=16..26, complex64 half states, on MI355X: 13.3
// -> 10.7 ms (5.2 where fewer of them are of N=26), the device's time 14 -> 7.2 ms
// for the latter: the general kernel ran two full-width passes per layer, one
// work-group per CU.
static int slab_step_packed(fq_slab *sb)
{
    const int K = sb->K, e = sb->pk_end;
    MixSlot *h = (MixSlot *)(sb->h_step + step_mix(K));
    SlabJob *jobs = (SlabJob *)(sb->h_step + step_jobs(K));
    const MixSlot *d = (const MixSlot *)(sb->d_step + step_mix(K));
    int n = 0, nj = 0, at[4] = {0, 0, 0, 0};
    MixArgs args[3];
    enum { FIRST = 0, BOUNDARY = 1, PLAIN = 2 };
    for (int kind = FIRST; kind <= PLAIN; ++kind) {
        const int pass = kind == FIRST ? 1 - e : e;
        const PackedPass &pp = sb->pk[pass];
        args[kind] = pp.a;
        for (int k = 0; k < K; ++k) {
            SlotHost &s = sb->slots[k];
            if (s.phase != 1)
                continue;
            const int L = s.layer;
            const bool last = L + 1 == s.P;
            if (kind == FIRST ? L != 0 : last != (kind == PLAIN))
                continue;
            fq_state *v = sb->views[k];
            if (kind == FIRST) {
                v->pending_re = 1.0;
                v->pending_im = 0.0;
            }
            const int open = kind == BOUNDARY ? L + 1 : L;
            const size_t ng = sb->slot_plan.ps[pass].gates.size();
            const PassFactor f = pass_factor(v, ng, s.betas[open], kind == BOUNDARY ? &s.betas[L] : nullptr, kind != PLAIN,
                                             false, open + 1 < s.P ? 0 : kind == PLAIN ? FACTOR_TAKEN : sb->N - ng);
            MixSlot &m = h[n++];
            m.t = f.t;
            m.pre_t = f.pre_t;
            m.tf = (float)f.t;
            m.pre_tf = (float)f.pre_t;
            m.scale_re = f.re;
            m.scale_im = f.im;
            m.base = (sb->slot_bytes / sb->elem) * (uint64_t)k;
            m.table = 0;
            m.has_rr = 0;
            args[kind].apply_scale = f.apply;
            if (kind != PLAIN) {
                const int geo = 2 * (kind == BOUNDARY) + pass;
                m.table = (uint32_t)(sb->tab_stride * k + sb->pk_entries * (kind == BOUNDARY));
                m.has_rr = s.has_rr[geo];
                jobs[nj++] = {s.gammas[open], (uint32_t)k, (uint32_t)geo, m.table, 0};
            }
        }
        at[kind + 1] = n;
    }
    FQ_HIP(hipMemcpyAsync(sb->d_step, sb->h_step, step_bytes(K), hipMemcpyHostToDevice, sb->stream));
    if (nj > 0)
        FQ_HIP(launch_slab_tables(sb->pk_tab, (const SlabJob *)(sb->d_step + step_jobs(K)), nj, sb->pk_entries, sb->d_plans,
                                  sb->d_tabs, sb->stream));
    for (int kind = FIRST; kind <= PLAIN; ++kind) {
        const int ns = at[kind + 1] - at[kind];
        if (ns == 0)
            continue;
        const PackedPass &pp = sb->pk[kind == FIRST ? 1 - e : e];
        args[kind].slots = d + at[kind];
        args[kind].nslots = ns;
        FQ_HIP(launch_mix(sb->dtype, pp.K, pp.lane, kind == FIRST ? MIX_FIRST : kind == BOUNDARY ? MIX_BOUNDARY : MIX_PLAIN,
                          pp.mir ? 1 : 0, sb->sv, args[kind], sb->d_tabs, sb->stream));
    }
    sb->pk_end = 1 - e;
    return FQ_OK;
}

// The plans of slots [k0, k1) to the device.  Slots that enter together go in one copy,
// with what lies between them (a copy takes 4 us, a slot's plans are 1.7 KB): 4 requests
// on a slab of N=3 complex64 slots 149 us with a copy for each.
static int slab_upload_plans(fq_slab *sb, int k0, int k1)
{
    if (k0 == k1)
        return FQ_OK;
    FQ_HIP(hipMemcpyAsync(sb->d_plans + k0, sb->h_plans + k0, sizeof(SlotPlans) * (size_t)(k1 - k0), hipMemcpyHostToDevice,
                          sb->stream));
    for (int k = k0; k < k1; ++k)
        sb->slots[k].fresh = false;
    return FQ_OK;
}

// Advance every active slot by one layer: one packed launch per tile pass.
// Slots that complete their last layer also get <C> reduced; their results
// are read with fq_slab_collect once fq_slab_poll reports the step done.
extern "C" int fq_slab_step(fq_slab *sb, int *nfinishing)
{
    if (!sb)
        return set_err(FQ_ERR_ARG, "null slab");
    if (sb->pending) {
        FQ_HIP(hipEventSynchronize(sb->done));
        sb->pending = false;
    }
    const int K = sb->K;
    // the slots' plans stay until the step is queued: the passes of large slots look
    // up plans of their own, and <C> comes after them
    std::vector<PlanHold> holds;
    for (const SlotHost &h : sb->slots)
        if (h.phase == 1)
            holds.emplace_back(h.g);
    // refresh plans of changed graphs; a refresh can release a graph's plan
    // cache, so repeat until every active slot's plans are current
    for (bool again = true; again;) {
        again = false;
        for (int k = 0; k < K; ++k) {
            SlotHost &h = sb->slots[k];
            if (h.phase != 1)
                continue;
            if (slab_slot_stale(h)) {
                if (h.layer > 0 && h.g->version != h.gversion && slab_opens_ahead(sb))
                    if (int rc = slab_reopen(sb, k))
                        return rc;
                if (int rc = slab_slot_plans(sb, h))
                    return rc;
                again = true;
            } else {
                for (PlanEntry *e : h.entries)
                    if (e)
                        e->last_use = ++h.g->use_clock;
            }
        }
    }
    // layers of this step per slot (per_slot slabs may run several)
    std::vector<int> nl(K, 0);
    SlotParams *params = (SlotParams *)sb->h_step;
    int *fin = (int *)(sb->h_step + step_fin(K));
    int nact = 0, nfin = 0;
    int fresh0 = 0, fresh1 = 0;   // slots with new plans, not uploaded yet
    for (int k = 0; k < K; ++k) {
        SlotHost &h = sb->slots[k];
        SlotParams &sp = params[k];
        memset(&sp, 0, sizeof(sp));
        if (h.phase != 1)
            continue;
        if (h.fresh) {
            sb->h_plans[k] = h.plans;
            if (fresh1 == 0 || k - fresh1 > 8) {
                if (int rc = slab_upload_plans(sb, fresh0, fresh1))
                    return rc;
                fresh0 = k;
            }
            fresh1 = k + 1;
        }
        nl[k] = sb->per_slot ? std::min(sb->layers_per_step, h.P - h.layer) : 1;
        const int L = h.layer;
        rx_coeffs(h.betas[L], sb->dtype, &sp.rx_c, &sp.rx_s);
        sp.gamma = h.gammas[L];
        // the general kernel applies RX with rx_coeffs (norm factor amp_scale);
        // the others run fq_run's passes, whose RX factors are exact
        sp.init_amp = sb->init_amp * (sb->per_slot || sb->packed ? 1.0 : h.amp_scale);
        sp.active = 1;
        sp.cost_first = L == 0;
        sp.ptab = sb->d_tabs + sb->tab_stride * (size_t)k;
        sp.has_rr = h.has_rr[0];
        ++nact;
        if (L + nl[k] == h.P)
            fin[nfin++] = k;
    }
    if (int rc = slab_upload_plans(sb, fresh0, fresh1))
        return rc;
    if (nfinishing)
        *nfinishing = nfin;
    if (nact == 0)
        return FQ_OK;
    if (sb->packed) {
        if (int rc = slab_step_packed(sb))
            return rc;
    } else {
        FQ_HIP(hipMemcpyAsync(sb->d_step, sb->h_step, step_bytes(K), hipMemcpyHostToDevice, sb->stream));
    }
    if (sb->per_slot) {
        // each slot nl[k] layers of fq_run's pipelined schedule on its own
        // amplitudes (the slots' layers interleaved on the slab's stream)
        const int most = *std::max_element(nl.begin(), nl.end());
        for (int rep = 0; rep < most; ++rep) {
            for (int k = 0; k < K; ++k) {
                if (!params[k].active || rep >= nl[k])
                    continue;
                SlotHost &h = sb->slots[k];
                fq_state *v = sb->views[k];
                const int L = h.layer + rep;
                if (L == 0) {
                    v->pending_re = 1.0;
                    v->pending_im = 0.0;
                }
                if (int rc = run_layers(v, h.g, sb->slot_plan, L, L + 1, h.P, h.gammas.data(), h.betas.data(), sb->z2,
                                        false))
                    return rc;
            }
        }
    } else if (!sb->packed) {
        const SlotParams *d = (const SlotParams *)sb->d_step;
        FQ_HIP(launch_slab_phase_table(sb->cost_args, sb->cost_geom.a_log, d, sb->d_plans, K, sb->d_tabs, sb->tab_stride,
                                       sb->stream));
        for (size_t i = 0; i < sb->pass_args.size(); ++i) {
            const SlabPass &sp = sb->pass_args[i];
            FQ_HIP(launch_slab_pass(sb->dtype, sp.a_log, i == 0, sp.mirror, sb->sv, sp.args, d, sp.slot_shift,
                                    sb->stream));
        }
    }
    if (nfin > 0)
        FQ_HIP(launch_slab_expect(sb->dtype, sb->exp_alog, sb->sv, sb->exp_args, sb->d_plans,
                                  (const int *)(sb->d_step + step_fin(K)), nfin, sb->exp_shift, sb->d_part, sb->h_res,
                                  sb->stream));
    FQ_HIP(hipEventRecord(sb->done, sb->stream));
    sb->pending = true;
    for (int k = 0; k < K; ++k) {
        SlotHost &h = sb->slots[k];
        if (h.phase != 1)
            continue;
        h.layer += nl[k];
        if (h.layer == h.P)
            h.phase = 2;
    }
    return FQ_OK;
}

extern "C" int fq_slab_set_layers_per_step(fq_slab *sb, int layers)
{
    if (!sb)
        return set_err(FQ_ERR_ARG, "null slab");
    if (layers < 1)
        return set_err(FQ_ERR_ARG, "layers per step must be >= 1");
    sb->layers_per_step = layers;
    return FQ_OK;
}

// Results of the slots that finished: slot index, <C>, sum |psi|^2.  Waits
// for the enqueued step, then frees those slots.  n receives the count
// (capacity: the slab's slot count).
extern "C" int fq_slab_collect(fq_slab *sb, int *slots, double *expect, double *norm2, int *n)
{
    if (!sb || !n)
        return set_err(FQ_ERR_ARG, "null argument");
    if (sb->pending) {
        FQ_HIP(hipEventSynchronize(sb->done));
        sb->pending = false;
    }
    int c = 0;
    for (int k = 0; k < sb->K; ++k) {
        SlotHost &h = sb->slots[k];
        if (h.phase != 2)
            continue;
        if (slots)
            slots[c] = k;
        // a half-state slab holds one of the two equal halves
        const double f = sb->z2 ? 2.0 : 1.0;
        if (expect)
            expect[c] = f * sb->h_res[2 * k];
        if (norm2)
            norm2[c] = f * sb->h_res[2 * k + 1];
        ++c;
        h.phase = 0;
        h.g = nullptr;
    }
    *n = c;
    return FQ_OK;
}

// A running slot's amplitudes after the layers it has run, at tmp: its last
// boundary pass has also opened the next layer, which is undone there.
static int slab_close_layer(fq_slab *sb, int slot, void *tmp)
{
    const SlotHost &h = sb->slots[slot];
    fq_state v;
    v.N = sb->N;
    v.dtype = sb->dtype;
    v.elem = sb->elem;
    v.bytes = sb->slot_bytes;
    v.sv = tmp;
    v.stream = sb->stream;
    v.in_run = true;
    for (int q = 0; q < FQ_MAXN; ++q)
        v.qmap[q] = q;
    v.init_amp = sb->init_amp;
    const FusedPass &open = sb->slot_plan.ps[slab_ended_on(sb, h)];
    if (h.layer + 1 == h.P && mix_a_log(sb->dtype, (int)open.tile.size()) > 0) {
        // (the last layer's cost pass took the factor of its plain passes: off again)
        double t, re = 1.0, im = 0.0;
        absorb_rx(&v, h.betas[h.layer], sb->N - open.gates.size(), &t, &re, &im);
        const double m = re * re + im * im;
        v.pending_re = re / m;
        v.pending_im = -im / m;
    }
    const int rc = slab_again(sb, h, &v, h.W, -h.betas[h.layer], -h.gammas[h.layer], 0.0);
    free_phases(&v);
    v.sv = nullptr;
    return rc;
}

// Amplitudes of one slot (identity layout) to host memory.  Waits.
extern "C" int fq_slab_copy_out(fq_slab *sb, int slot, void *host, size_t bytes)
{
    if (!sb || !host)
        return set_err(FQ_ERR_ARG, "null argument");
    const size_t full = ((size_t)1 << sb->N) * sb->elem;
    if (slot < 0 || slot >= sb->K || bytes != full)
        return set_err(FQ_ERR_ARG, "bad slot or size (%zu bytes expected)", full);
    const char *src = (const char *)sb->sv + sb->slot_bytes * (size_t)slot;
    const SlotHost &h = sb->slots[slot];
    void *tmp = nullptr;
    int rc = FQ_OK;
    if (slab_opens_ahead(sb) && h.phase == 1 && h.layer > 0) {
        if (hipMalloc(&tmp, sb->slot_bytes) != hipSuccess) {
            hipGetLastError();
            return set_err(FQ_ERR_OOM, "scratch for a running slot's amplitudes failed");
        }
        if (hipMemcpyAsync(tmp, src, sb->slot_bytes, hipMemcpyDeviceToDevice, sb->stream) == hipSuccess)
            rc = slab_close_layer(sb, slot, tmp);
        else
            rc = set_err(FQ_ERR_DEVICE, "copy of a running slot's amplitudes failed");
    }
    if (rc == FQ_OK && (hipMemcpyAsync(host, tmp ? (const char *)tmp : src, sb->slot_bytes, hipMemcpyDeviceToHost,
                                       sb->stream) != hipSuccess ||
                        hipStreamSynchronize(sb->stream) != hipSuccess))
        rc = set_err(FQ_ERR_DEVICE, "copy of a slot's amplitudes failed");
    hipFree(tmp);
    if (rc)
        return rc;
    sb->pending = false;
    if (sb->z2) {
        // psi(b) = psi(~b): the upper half is the stored half reversed
        const size_t half = (size_t)1 << (sb->N - 1), e = sb->elem;
        char *h = (char *)host;
        for (size_t i = 0; i < half; ++i)
            memcpy(h + (half + i) * e, h + (half - 1 - i) * e, e);
    }
    return FQ_OK;
}
