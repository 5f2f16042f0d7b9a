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

#include "fq_device.h"
#include "fq_internal.h"

#include <hip/hip_runtime.h>

namespace fq {

// Layouts of a tile pass with K exchanges one way.  Layout 0: register bits
// are the top A tile bits and thread bit k is tile bit k (the global loads:
// lanes hold the lowest tile bits).  Layout l >= 1: register bits
// [start, start + A), start = max(0, nthr - A (K - l + 1)); layout K holds the
// highest thread bits, so its lanes hold the lowest tile bits again and the
// tile can be stored from it.
// W: the LDS slot of tile element e is the sum of W[i] over its set bits i, so
// the thread's and the register's parts add and the latter is an address
// constant.  W[i] is 2^i plus paddings that keep the map injective and put
// the lanes of every layout on distinct banks (32 distinct 8-byte slots per
// half wave in FP64, 64 distinct 4-byte slots per wave in FP32).
// P: tile bit of each thread bit, per layout.
template <typename R, int Q, int A, int K> struct MixGeo;

#define FQ_L(...) {__VA_ARGS__}
#define FQ_GEO(R_, Q_, A_, K_, W_, ...)                                                  \
    template <> struct MixGeo<R_, Q_, A_, K_> {                                          \
        static constexpr int w(int i) { constexpr int W[Q_] = W_; return W[i]; }         \
        static constexpr int p(int l, int k)                                             \
        {                                                                                \
            constexpr int P[K_ + 1][Q_ - A_] = __VA_ARGS__;                              \
            return P[l][k];                                                              \
        }                                                                                \
    };
FQ_GEO(double, 13, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 33, 65, 132, 288, 560, 1124, 2248, 4488),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {0, 1, 2, 3, 4, 9, 10, 11, 12}))
FQ_GEO(double, 13, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 64, 130, 258, 516, 1032, 2064, 4130),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {0, 7, 9, 10, 11, 5, 6, 8, 12}, {0, 1, 2, 3, 4, 9, 10, 11, 12}))
FQ_GEO(double, 13, 4, 3,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 136, 272, 548, 1121, 2216, 4452),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {4, 5, 6, 7, 10, 8, 9, 11, 12}, {0, 5, 6, 7, 8, 9, 10, 11, 12}, {0, 1, 2, 3, 4, 9, 10, 11, 12}))
FQ_GEO(double, 12, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 64, 128, 272, 548, 1092, 2192),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {0, 1, 2, 3, 8, 9, 10, 11}))
FQ_GEO(double, 12, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 136, 272, 548, 1121, 2224),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {4, 5, 6, 7, 10, 8, 9, 11}, {0, 1, 2, 3, 8, 9, 10, 11}))
FQ_GEO(double, 11, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 68, 136, 272, 548, 1090),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {0, 1, 2, 7, 8, 9, 10}))
FQ_GEO(double, 11, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 33, 66, 136, 272, 552, 1092),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {4, 5, 6, 7, 10, 8, 9}, {0, 1, 2, 7, 8, 9, 10}))
FQ_GEO(double, 9, 3, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 72, 144, 288),
       FQ_L({0, 1, 2, 3, 4, 5}, {0, 1, 2, 6, 7, 8}))
FQ_GEO(double, 9, 3, 2,
       FQ_L(1, 2, 4, 8, 16, 33, 68, 136, 290),
       FQ_L({0, 1, 2, 3, 4, 5}, {3, 4, 5, 6, 8, 7}, {0, 1, 2, 6, 7, 8}))
FQ_GEO(double, 10, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 136, 272, 546),
       FQ_L({0, 1, 2, 3, 4, 5}, {0, 1, 6, 7, 8, 9}))
FQ_GEO(double, 10, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 136, 272, 545),
       FQ_L({0, 1, 2, 3, 4, 5}, {4, 5, 6, 7, 9, 8}, {0, 1, 6, 7, 8, 9}))
FQ_GEO(float, 14, 5, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 66, 136, 272, 544, 1104, 2242, 4484, 8912),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {0, 1, 2, 3, 9, 10, 11, 12, 13}))
FQ_GEO(float, 14, 5, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 66, 136, 272, 544, 1104, 2240, 4484, 8961),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {5, 6, 7, 8, 12, 13, 9, 10, 11}, {0, 1, 2, 3, 9, 10, 11, 12, 13}))
FQ_GEO(float, 13, 5, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 66, 132, 264, 528, 1056, 2128, 4256),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {0, 1, 2, 8, 9, 10, 11, 12}))
FQ_GEO(float, 13, 5, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 65, 132, 264, 528, 1056, 2128, 4290),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {5, 6, 7, 8, 9, 12, 10, 11}, {0, 1, 2, 8, 9, 10, 11, 12}))
FQ_GEO(float, 12, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 68, 136, 272, 544, 1092, 2176),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {0, 1, 2, 3, 8, 9, 10, 11}))
FQ_GEO(float, 12, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 68, 136, 272, 544, 1089, 2178),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {4, 5, 6, 7, 10, 11, 8, 9}, {0, 1, 2, 3, 8, 9, 10, 11}))
FQ_GEO(float, 11, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 65, 136, 272, 544, 1096),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {0, 1, 2, 7, 8, 9, 10}))
FQ_GEO(float, 11, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 66, 132, 264, 528, 1089),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {4, 5, 6, 7, 8, 10, 9}, {0, 1, 2, 7, 8, 9, 10}))
FQ_GEO(float, 10, 4, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 68, 136, 272, 544),
       FQ_L({0, 1, 2, 3, 4, 5}, {0, 1, 6, 7, 8, 9}))
FQ_GEO(float, 10, 4, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 65, 132, 264, 528),
       FQ_L({0, 1, 2, 3, 4, 5}, {4, 5, 6, 7, 8, 9}, {0, 1, 6, 7, 8, 9}))
#undef FQ_GEO
#undef FQ_L
// no exchange: all gated bits are register bits
template <typename R, int Q, int A> struct MixGeo<R, Q, A, 0> {
    static constexpr int w(int) { return 0; }
    static constexpr int p(int, int k) { return k; }
};

template <typename R, int Q, int A, int K> struct MixLay : MixGeo<R, Q, A, K> {
    static constexpr int NT = Q - A;
    static constexpr int start(int l) { return NT - A * (K - l + 1) > 0 ? NT - A * (K - l + 1) : 0; }
    // tile bit of register bit r in layout l
    static constexpr int reg(int l, int r) { return l == 0 ? NT + r : start(l) + r; }
    static constexpr int reg_slot(int l, int j)
    {
        int s = 0;
        for (int r = 0; r < A; ++r)
            if ((j >> r) & 1)
                s += MixGeo<R, Q, A, K>::w(reg(l, r));
        return s;
    }
    static constexpr int slots()
    {
        int s = 1;
        for (int i = 0; i < Q; ++i)
            s += MixGeo<R, Q, A, K>::w(i);
        return s;
    }
};

// Registers of a tile from layout L0 to layout L1.  YF: the imaginary parts go
// first.  The first part's slots in layout L0 are free for their own thread to
// write (the previous exchange read that part there, or a barrier precedes).
template <typename Lay, typename T, typename R, int A, int L0, int L1, bool YF>
__device__ __forceinline__ void mix_exchange(T (&v)[1 << A], R *lds, int s0, int s1)
{
    constexpr int N = 1 << A;
#pragma unroll
    for (int j = 0; j < N; ++j)
        lds[s0 + Lay::reg_slot(L0, j)] = YF ? v[j].y : v[j].x;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < N; ++j)
        (YF ? v[j].y : v[j].x) = lds[s1 + Lay::reg_slot(L1, j)];
    lds_barrier();
#pragma unroll
    for (int j = 0; j < N; ++j)
        lds[s0 + Lay::reg_slot(L0, j)] = YF ? v[j].x : v[j].y;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < N; ++j)
        (YF ? v[j].x : v[j].y) = lds[s1 + Lay::reg_slot(L1, j)];
}

// The value of a register in lane ^ 2^B (B = 0, 1, 3: one DPP move per 32 bits).
template <int B> __device__ __forceinline__ int lane_xor(int x)
{
    constexpr int ctrl = B == 0 ? 0xB1 : B == 1 ? 0x4E : 0x128;   // quad_perm 1,0,3,2 / 2,3,0,1 / row_ror:8
    return __builtin_amdgcn_mov_dpp(x, ctrl, 0xf, 0xf, true);
}
template <int B> __device__ __forceinline__ float lane_xor(float x)
{
    return __int_as_float(lane_xor<B>(__float_as_int(x)));
}
template <int B> __device__ __forceinline__ double lane_xor(double x)
{
    return __hiloint2double(lane_xor<B>(__double2hiint(x)), lane_xor<B>(__double2loint(x)));
}

// Exchange of lane bit 4 between two registers (lane_xchg16 for each half).
__device__ __forceinline__ void lane_xchg16(double &a, double &b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// RX on lane bit B without LDS.  Bit 4: a swap with register bit 0, the
// butterfly there, the swap back; bits 0, 1 and 3: the partner lane's values
// (both lanes run the same butterfly).  About 100 instructions per thread for
// 16 FP64 amplitudes, where an exchange through LDS takes 128 LDS accesses
// and three barriers.
template <typename T, typename R, int A, int B>
__device__ __forceinline__ void rx_lane(T (&v)[1 << A], R t)
{
    if constexpr (B == 4) {
#pragma unroll
        for (int j = 0; j < (1 << A); j += 2) {
            lane_xchg16(v[j].x, v[j + 1].x);
            lane_xchg16(v[j].y, v[j + 1].y);
            rx_pair_t<T, R>(v[j], v[j + 1], t);
            lane_xchg16(v[j].x, v[j + 1].x);
            lane_xchg16(v[j].y, v[j + 1].y);
        }
    } else {
#pragma unroll
        for (int j = 0; j < (1 << A); ++j) {
            const R px = lane_xor<B>(v[j].x), py = lane_xor<B>(v[j].y);
            v[j].x = fma(t, py, v[j].x);
            v[j].y = fma(-t, px, v[j].y);
        }
    }
}

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
    k_mix(typename CT<R>::T *__restrict__ sv, const MixArgs a, const double2 *__restrict__ ptab)
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
    const uint64_t q1 = Q + 1;
    const double2 *thr_tab = COST ? ptab + a.ntab * q1 : nullptr;
    const double2 *rr_tab = COST ? thr_tab + ((size_t)(1 + A) << NT) : nullptr;
    const R rt = sizeof(R) == 4 ? (R)a.tf : (R)a.t;
    const R pt = sizeof(R) == 4 ? (R)a.pre_tf : (R)a.pre_t;

    const uint64_t tile = a.tile0 + blockIdx.x;
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
        mul(KIND == MIX_FIRST ? make_double2(a.init_amp * a.scale_re, a.init_amp * a.scale_im)
                              : make_double2(a.scale_re, a.scale_im));
        const R x0 = (R)x, y0 = (R)y;
        R fx[A], fy[A];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < A; ++r) {
            const double2 f = lane_bcast(f_row, NT + r), g = thr_tab[((1 + r) << NT) + t];
            fx[r] = (R)(g.x * f.x - g.y * f.y);
            fy[r] = (R)(g.x * f.y + g.y * f.x);
            __builtin_amdgcn_sched_barrier(0);
        }
        mix_phase<T, R, A, A, KIND == MIX_FIRST>(v, fx, fy, x0, y0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (a.has_rr) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const double2 f = rr_tab[j];
                cmul_by(v[j], (R)f.x, (R)f.y);
            }
        }
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
            cmul_by(v[j], (R)a.scale_re, (R)a.scale_im);
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
    if (lds > 65536) {
        if (hipError_t e = allow_large_lds(fn))
            return e;
    }
    hipLaunchKernelGGL((k_mix<R, Q, A, K, KIND, MIR, LG>), dim3((unsigned)a.ntiles), dim3(threads), lds, stream,
                       reinterpret_cast<T *>(sv), a, ptab);
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
