// fq_mix.h -- gfx950 tile passes of the layer schedules, with the LDS
// phases fixed at compile time.  fq_kernels.hip keeps the general tile pass
// (any tile width, RX on any subset of the tile bits).
//
// A work-group owns a tile of 2^Q amplitudes, 2^A of them per thread in
// registers.  RX on register bits is done in registers; the other gated bits
// come into registers by exchanges of register bits with thread bits through
// LDS.  One exchange moves the real parts and then the imaginary parts, so
// its buffer is half a tile: a full-width tile (128 KiB) takes 70 KiB of LDS
// and two work-groups fit on a CU, one in its butterflies and exchanges while
// the loads and stores of the other are in flight.  (The general pass keeps the
// whole tile in LDS, one work-group per CU.)
//
// What bounds a pass: the memory.  Per complex128 tile a plain pass with two
// exchanges issues 3,400 vector instructions per CU and holds the LDS for
// 4,100 cycles, of the 17,000 cycles the tile takes at 8 TB/s.  Measured on
// MI355X, against the general pass: N=22 complex128 (64 MiB, two passes a layer,
// pipelined to one) 50 -> 40 us per layer, N=24 (256 MiB, in the memory-side
// cache) 216 -> 193 us, a plain pass over QAOA amplitudes 80 us (6.7 TB/s; 65 us
// over zeros: the rate depends on how many bits toggle).
#pragma once

#include "fq_exchange.h"
#include "fq_internal.h"

#include <hip/hip_runtime.h>

namespace fq {

// Layouts 0..K (UP) or K..0: RX on each layout's gated register bits, an
// exchange between neighbours, RX on lane bit LB (>= 0) in layout 0.  X0:
// exchanges done before in this tile.
template <typename Lay, typename T, typename R, int A, int K, int L, int X0, int LB>
__device__ __forceinline__ void mix_up(T (&v)[1 << A], R *lds, const int (&sb)[K + 1], uint32_t gates, R t)
{
    if constexpr (L == 0 && LB >= 0)
        rx_lane<T, R, A, LB>(v, t);
    rx_registers_t<T, R, A>(v, (gates >> (A * L)) & ((1u << A) - 1u), t);
    if constexpr (L < K) {
        mix_exchange<Lay, T, R, A, L, L + 1, ((X0 + L) & 1) != 0>(v, lds, sb[L], sb[L + 1]);
        mix_up<Lay, T, R, A, K, L + 1, X0, LB>(v, lds, sb, gates, t);
    }
}

template <typename Lay, typename T, typename R, int A, int K, int L, int X0, int LB>
__device__ __forceinline__ void mix_down(T (&v)[1 << A], R *lds, const int (&sb)[K + 1], uint32_t gates, R t)
{
    rx_registers_t<T, R, A>(v, (gates >> (A * L)) & ((1u << A) - 1u), t);
    if constexpr (L > 0) {
        mix_exchange<Lay, T, R, A, L, L - 1, ((X0 + K - L) & 1) != 0>(v, lds, sb[L], sb[L - 1]);
        mix_down<Lay, T, R, A, K, L - 1, X0, LB>(v, lds, sb, gates, t);
    } else if constexpr (LB >= 0) {
        rx_lane<T, R, A, LB>(v, t);
    }
}

// v[j] times the product of the factors fr[r] of j's set bits (and f): a tree
// over the register bits, one product per node.
template <typename T, typename R, int A, int RB, bool SET>
__device__ __forceinline__ void mix_phase(T (&v)[1 << A], const R (&fx)[A], const R (&fy)[A], R x, R y, int j)
{
    if constexpr (RB == 0) {
        if (SET) {
            v[j].x = x;
            v[j].y = y;
        } else {
            cmul_by(v[j], x, y);
        }
    } else {
        mix_phase<T, R, A, RB - 1, SET>(v, fx, fy, x, y, j);
        if (RB == 3)
            __builtin_amdgcn_sched_barrier(0);   // depth first: the products of one path live at a time
        mix_phase<T, R, A, RB - 1, SET>(v, fx, fy, x * fx[RB - 1] - y * fy[RB - 1], x * fy[RB - 1] + y * fx[RB - 1],
                                        j | (1 << (RB - 1)));
    }
}

// The cost phase times (sx, sy) on a thread's amplitudes (SET: of a state of ones):
// the tile's row of the table (entry i in lane i, broadcast by readlane), the
// thread's entry f_thr, the thread's register entries and the
// register-register ones.
template <typename T, typename R, int Q, int A, bool SET>
__device__ __forceinline__ void mix_cost(T (&v)[1 << A], double2 f_row, double2 f_thr, const double2 *thr_tab,
                                         const double2 *rr_tab, int has_rr, double sx, double sy, int t)
{
    constexpr int NT = Q - A, N = 1 << A;
    // all loads at once, behind the products of the thread's factor (each of them in
    // its turn took 1 us of a small state's pass: N=20 complex128 14.2 -> 13.9 us, and
    // N=24 139 -> 132)
    double2 f_reg[A];
#pragma unroll
    for (int r = 0; r < A; ++r)
        f_reg[r] = thr_tab[((1 + r) << NT) + t];
    __builtin_amdgcn_sched_barrier(0);
    double x = f_thr.x, y = f_thr.y;
    auto mul = [&](double2 f) {
        const double nx = x * f.x - y * f.y;
        y = x * f.y + y * f.x;
        x = nx;
    };
    mul(lane_bcast(f_row, Q));
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const double2 f = lane_bcast(f_row, i);
        const double nx = x * f.x - y * f.y;
        const double ny = x * f.y + y * f.x;
        const bool on = (t >> i) & 1;
        x = on ? nx : x;
        y = on ? ny : y;
    }
    mul(make_double2(sx, sy));
    const R x0 = (R)x, y0 = (R)y;
    R fx[A], fy[A];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < A; ++r) {
        const double2 f = lane_bcast(f_row, NT + r), g = f_reg[r];
        fx[r] = (R)(g.x * f.x - g.y * f.y);
        fy[r] = (R)(g.x * f.y + g.y * f.x);
        __builtin_amdgcn_sched_barrier(0);
    }
    mix_phase<T, R, A, A, SET>(v, fx, fy, x0, y0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (has_rr) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double2 f = rr_tab[j];
            cmul_by(v[j], (R)f.x, (R)f.y);
        }
    }
}

// Whether the instances of this width take packed launches.
template <typename R> static constexpr bool mix_packs(int Q) { return Q < (sizeof(R) == 4 ? 14 : 13); }

// One work-group per tile: with two of them on a CU the dispatcher's order keeps
// loads and butterflies apart better than persistent groups with a range of
// tiles each (N=30 complex128 13.64 -> 13.37 ms per layer).
//
// One tile pass.  KIND: MIX_PLAIN RX on the gated bits; MIX_FIRST the
// launch-control write (no read) with the cost phase, then RX; MIX_COST the
// cost phase, then RX; MIX_BOUNDARY RX of one layer (pre), the cost phase of
// the next, RX of the next.  MIR (half states): qubit N-1 is the top tile bit
// and its upper half is tile ~tau at complemented offsets; 2 also writes the
// upper half of the full state.  RX is the butterfly of rx_tform; the pass's
// factor goes into the cost phase, or is multiplied in before the stores
// where a.apply_scale is set.
// LG: RX also on the thread bit just below those that the K exchanges reach,
// by lane operations.
template <typename R, int Q, int A, int K, int KIND, int MIR, bool LG>
__global__ void __launch_bounds__(1 << (Q - A), 4)
    k_mix(typename CT<R>::T *__restrict__ sv0, const MixArgs a, const double2 *__restrict__ ptab0)
{
    typedef typename CT<R>::T T;
    typedef MixLay<R, Q, A, K> Lay;
    constexpr int N = 1 << A, NT = Q - A, AH = MIR ? N / 2 : N;
    constexpr int NB = MIR ? A - 1 : A;   // register bits that are address bits
    constexpr bool COST = KIND != MIX_PLAIN;
    constexpr int LB = LG ? Q - A - K * A - 1 : -1;
    constexpr int LS = KIND == MIX_BOUNDARY || MIR ? 0 : K;   // layout of the stores
    extern __shared__ __align__(16) unsigned char fq_smem_m[];
    R *lds = reinterpret_cast<R *>(fq_smem_m);
    const int t = threadIdx.x;
    const uint64_t hmask = (1ull << a.nh) - 1ull;

    // offsets of the thread in the load and the store layout, LDS slots
    uint64_t toff = 0, soff = 0;
    int sb[K + 1];
#pragma unroll
    for (int l = 0; l <= K; ++l)
        sb[l] = 0;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const bool on = (t >> k) & 1;
        toff |= on ? 1ull << a.tpos[k] : 0ull;
        if (LS != 0)
            soff |= on ? 1ull << a.tpos[Lay::p(LS, k)] : 0ull;
#pragma unroll
        for (int l = 0; l <= K; ++l)
            sb[l] += on ? Lay::w(Lay::p(l, k)) : 0;
    }
    // a packed launch's slot has its own amplitudes, factors and phase table
    // (not at full width, which large states run at: there this cost 1.5%)
    typename CT<R>::T *__restrict__ sv = sv0;
    const double2 *__restrict__ ptab = ptab0;
    R rt = sizeof(R) == 4 ? (R)a.tf : (R)a.t;
    R pt = sizeof(R) == 4 ? (R)a.pre_tf : (R)a.pre_t;
    double scale_re = a.scale_re, scale_im = a.scale_im;
    int has_rr = a.has_rr;
    if (mix_packs<R>(Q) && a.slots) {
        const MixSlot &s = a.slots[blockIdx.y];
        sv += s.base;
        ptab += s.table;
        rt = sizeof(R) == 4 ? (R)s.tf : (R)s.t;
        pt = sizeof(R) == 4 ? (R)s.pre_tf : (R)s.pre_t;
        scale_re = s.scale_re;
        scale_im = s.scale_im;
        has_rr = s.has_rr;
    }
    const uint64_t q1 = Q + 1;
    const double2 *thr_tab = COST ? ptab + a.ntab * q1 : nullptr;
    const double2 *rr_tab = COST ? thr_tab + ((size_t)(1 + A) << NT) : nullptr;

    // by_xcd: work-groups go round the 8 XCDs in turn; an XCD takes consecutive
    // tiles from 8 of 64 ranges
    const uint32_t b = blockIdx.x;
    const uint64_t tile = a.tile0 + (a.by_xcd ? (b & 63u) * (gridDim.x >> 6) + (b >> 6) : b);
    const uint64_t base = unpack_runs_uniform(tile, a.hruns);
    // cost phase: the tile's row of the table, entry i in lane i (broadcast by
    // readlane), and the thread's entry, loaded ahead of the amplitudes
    double2 f_row = make_double2(1.0, 0.0), f_thr = make_double2(1.0, 0.0);
    if (COST) {
        f_row = ptab[tile * q1 + (t & 63) % (Q + 1)];
        f_thr = thr_tab[t];
    }
    T v[N];
    if (KIND != MIX_FIRST) {
        uint64_t ro[N];
        reg_offsets<N, NB>(a.rpos0_w, ro);
        const T *p0 = sv + (base + toff);
#pragma unroll
        for (int j = 0; j < AH; ++j)
            v[j] = p0[ro[j]];
        if (MIR) {
            const T *pm = sv + (unpack_runs_uniform(~tile & hmask, a.hruns) + a.mirror_pm - toff);
#pragma unroll
            for (int j = AH; j < N; ++j)
                v[j] = pm[-(int64_t)ro[j - AH]];
        }
    }
    auto cost = [&]() {
        const bool first = KIND == MIX_FIRST;
        mix_cost<T, R, Q, A, KIND == MIX_FIRST>(v, f_row, f_thr, thr_tab, rr_tab, has_rr,
                                                first ? a.init_amp * scale_re : scale_re,
                                                first ? a.init_amp * scale_im : scale_im, t);
    };
    if constexpr (KIND == MIX_FIRST || KIND == MIX_COST)
        cost();
    if constexpr (KIND == MIX_BOUNDARY) {
        mix_up<Lay, T, R, A, K, 0, 0, LB>(v, lds, sb, a.gates_w, pt);
        cost();
        mix_down<Lay, T, R, A, K, K, K, LB>(v, lds, sb, a.gates_w, rt);
    } else {
        mix_up<Lay, T, R, A, K, 0, 0, LB>(v, lds, sb, a.gates_w, rt);
        if constexpr (MIR && K > 0)
            mix_exchange<Lay, T, R, A, K, 0, (K & 1) != 0>(v, lds, sb[K], sb[0]);
    }
    if (!COST && a.apply_scale) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            cmul_by(v[j], (R)scale_re, (R)scale_im);
    }
    uint64_t ro[N];
    reg_offsets<N, NB>(LS == 0 ? a.rpos0_w : a.rposk_w, ro);
    T *const p0 = sv + (base + (LS == 0 ? toff : soff));
#pragma unroll
    for (int j = 0; j < AH; ++j)
        p0[ro[j]] = v[j];
    if (MIR) {
        T *const pm = sv + (unpack_runs_uniform(~tile & hmask, a.hruns) + a.mirror_pm - toff);
#pragma unroll
        for (int j = AH; j < N; ++j)
            pm[-(int64_t)ro[j - AH]] = v[j];
        if (MIR == 2) {
            const uint64_t half = 1ull << (a.N - 1);
#pragma unroll
            for (int j = 0; j < AH; ++j)
                p0[half + ro[j]] = v[j + AH];
#pragma unroll
            for (int j = AH; j < N; ++j)
                pm[half - ro[j - AH]] = v[j - AH];
        }
    }
}

// ---- small states ------------------------------------------------------------

// Layers of a state that is one tile, in one launch of one work-group: the
// amplitudes stay in registers, the layers go through the layouts up and down
// in turn, each with its cost phase where it begins.  A layer takes the latency of
// its table entries and of K exchanges, instead of that of a launch, a load and
// a store besides: per layer on MI355X 4.0 us at N=12 and 2.8 at N=10 complex128
// (a launch each: 7.1 and 5.4), 3.7 and 2.9 complex64 (6.9 and 5.5).  One
// work-group's butterflies set the limit: at N=13 complex64 it took 6.7 us, two
// narrow passes 5.7.
template <typename R, int Q, int A, int K>
__global__ void __launch_bounds__(1 << (Q - A), 1)
    k_solo(typename CT<R>::T *__restrict__ sv, const SoloArgs a, const double2 *__restrict__ ptab)
{
    typedef typename CT<R>::T T;
    typedef MixLay<R, Q, A, K> Lay;
    constexpr int N = 1 << A, NT = Q - A;
    static_assert(K % 2 == 0, "the exchanges of a layer start with the real parts");
    extern __shared__ __align__(16) unsigned char fq_smem_1[];
    R *lds = reinterpret_cast<R *>(fq_smem_1);
    const int t = threadIdx.x;
    int sb[K + 1], soff = 0;
#pragma unroll
    for (int l = 0; l <= K; ++l)
        sb[l] = 0;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const int on = (t >> k) & 1;
        soff |= on << Lay::p(K, k);
#pragma unroll
        for (int l = 0; l <= K; ++l)
            sb[l] += on * Lay::w(Lay::p(l, k));
    }
    T v[N];
    if (a.first) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            v[j].x = (R)a.init_amp;
            v[j].y = 0;
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j)
            v[j] = sv[t + (j << NT)];
    }
    const uint32_t gates = a.gates_w;
    auto cost = [&](int p) {
        const double2 *tab = ptab + a.table[p], *thr = tab + (Q + 1);
        const double2 f_row = tab[(t & 63) % (Q + 1)], f_thr = thr[t];
        mix_cost<T, R, Q, A, false>(v, f_row, f_thr, thr, thr + ((1 + A) << NT), a.has_rr, a.scale_re[p], a.scale_im[p], t);
    };
    bool up = true;
    for (int p = 0; p < a.P; ++p, up = !up) {
        cost(p);
        if (up)
            mix_up<Lay, T, R, A, K, 0, 0, -1>(v, lds, sb, gates, (R)a.t[p]);
        else
            mix_down<Lay, T, R, A, K, K, 0, -1>(v, lds, sb, gates, (R)a.t[p]);
    }
    if (up) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            sv[t + (j << NT)] = v[j];
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j)
            sv[soff + (j << Lay::start(K))] = v[j];
    }
}

template <typename R, int Q, int A>
static hipError_t launch_solo_q(void *sv, const SoloArgs &a, const double2 *ptab, hipStream_t stream)
{
    constexpr int K = 2;
    constexpr size_t lds = sizeof(R) * (size_t)MixLay<R, Q, A, K>::slots();
    static_assert(lds <= 65536, "static limit of dynamic LDS");
    hipLaunchKernelGGL((k_solo<R, Q, A, K>), dim3(1), dim3(1u << (Q - A)), lds, stream,
                       reinterpret_cast<typename CT<R>::T *>(sv), a, ptab);
    return hipGetLastError();
}

// ---- launchers ---------------------------------------------------------------

// Whether RX on the thread bit below the K exchanges' can run on lanes.
template <int Q, int A, int K> static constexpr bool mix_has_lane()
{
    return K > 0 && (Q - A - K * A == 5 || Q - A - K * A == 4 || Q - A - K * A == 2 || Q - A - K * A == 1);
}

template <typename R, int Q, int A, int K, int KIND, int MIR, bool LG>
static hipError_t launch_mix_t(void *sv, const MixArgs &a, const double2 *ptab, hipStream_t stream)
{
    typedef typename CT<R>::T T;
    constexpr unsigned threads = 1u << (Q - A);
    constexpr size_t lds = K > 0 ? sizeof(R) * (size_t)MixLay<R, Q, A, K>::slots() : 0;
    const void *fn = reinterpret_cast<const void *>(&k_mix<R, Q, A, K, KIND, MIR, LG>);
    if (a.slots && !mix_packs<R>(Q))
        return hipErrorInvalidValue;
    if (lds > 65536) {
        if (hipError_t e = allow_large_lds(fn))
            return e;
    }
    hipLaunchKernelGGL((k_mix<R, Q, A, K, KIND, MIR, LG>), dim3((unsigned)a.ntiles, a.slots ? (unsigned)a.nslots : 1u),
                       dim3(threads), lds, stream, reinterpret_cast<T *>(sv), a, ptab);
    return hipGetLastError();
}

template <typename R, int Q, int A, int K, bool LG>
static hipError_t launch_mix_k(int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab, hipStream_t s)
{
    switch (kind * 4 + mir) {
        case MIX_PLAIN * 4 + 0: return launch_mix_t<R, Q, A, K, MIX_PLAIN, 0, LG>(sv, a, ptab, s);
        case MIX_PLAIN * 4 + 1: return launch_mix_t<R, Q, A, K, MIX_PLAIN, 1, LG>(sv, a, ptab, s);
        case MIX_PLAIN * 4 + 2: return launch_mix_t<R, Q, A, K, MIX_PLAIN, 2, LG>(sv, a, ptab, s);
        case MIX_FIRST * 4 + 0: return launch_mix_t<R, Q, A, K, MIX_FIRST, 0, LG>(sv, a, ptab, s);
        case MIX_FIRST * 4 + 1: return launch_mix_t<R, Q, A, K, MIX_FIRST, 1, LG>(sv, a, ptab, s);
        case MIX_COST * 4 + 0: return launch_mix_t<R, Q, A, K, MIX_COST, 0, LG>(sv, a, ptab, s);
        case MIX_BOUNDARY * 4 + 0: return launch_mix_t<R, Q, A, K, MIX_BOUNDARY, 0, LG>(sv, a, ptab, s);
        case MIX_BOUNDARY * 4 + 1: return launch_mix_t<R, Q, A, K, MIX_BOUNDARY, 1, LG>(sv, a, ptab, s);
        default: return hipErrorInvalidValue;
    }
}

template <typename R, int Q, int A, int K>
static hipError_t launch_mix_l(bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                               hipStream_t s)
{
    if (!lane)
        return launch_mix_k<R, Q, A, K, false>(kind, mir, sv, a, ptab, s);
    if constexpr (mix_has_lane<Q, A, K>())
        return launch_mix_k<R, Q, A, K, true>(kind, mir, sv, a, ptab, s);
    return hipErrorInvalidValue;
}

template <typename R, int Q, int A>
static hipError_t launch_mix_q(int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                               hipStream_t s)
{
    switch (k) {
        case 0: return launch_mix_l<R, Q, A, 0>(lane, kind, mir, sv, a, ptab, s);
        case 1: return launch_mix_l<R, Q, A, 1>(lane, kind, mir, sv, a, ptab, s);
        case 2: return launch_mix_l<R, Q, A, 2>(lane, kind, mir, sv, a, ptab, s);
        case 3:
            if constexpr (Q - A > 2 * A)
                return launch_mix_l<R, Q, A, 3>(lane, kind, mir, sv, a, ptab, s);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fq
