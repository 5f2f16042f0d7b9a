// fq_exchange.h -- what the tile passes (fq_mix.h) and the pair passes of the
// gradient (fq_pair.hip) share: the layouts of a tile over registers and
// threads, the exchange between two of them through LDS, RX on lane bits.
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
// the lanes of a layout on distinct banks (32 distinct 8-byte slots per
// half wave in FP64, 64 distinct 4-byte slots per wave in FP32).  So it is in
// every layout but four of the narrowest tiles: 20 of 32 slots in layout 2 of
// (double, 9, 3, 2), 36 of 64 in layout 2 of (float, 11, 4, 2), 32 and 33 of 64 in
// layouts 1 and 2 of (float, 10, 4, 2).
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
FQ_GEO(double, 10, 3, 1,
       FQ_L(1, 2, 4, 8, 16, 32, 64, 144, 272, 545),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {0, 1, 2, 3, 7, 8, 9}))
FQ_GEO(double, 10, 3, 2,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 144, 296, 576),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {0, 4, 5, 6, 8, 7, 9}, {0, 1, 2, 3, 7, 8, 9}))
FQ_GEO(double, 10, 3, 3,
       FQ_L(1, 2, 4, 8, 16, 36, 72, 144, 289, 578),
       FQ_L({0, 1, 2, 3, 4, 5, 6}, {3, 4, 5, 8, 9, 6, 7}, {0, 4, 5, 6, 9, 7, 8}, {0, 1, 2, 3, 7, 8, 9}))
FQ_GEO(double, 12, 3, 1,
       FQ_L(1, 2, 4, 8, 16, 34, 66, 132, 264, 544, 1096, 2178),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {0, 1, 2, 3, 4, 5, 9, 10, 11}))
FQ_GEO(double, 12, 3, 2,
       FQ_L(1, 2, 4, 8, 16, 32, 66, 136, 272, 552, 1090, 2184),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {0, 1, 2, 7, 8, 6, 9, 10, 11}, {0, 1, 2, 3, 4, 5, 9, 10, 11}))
FQ_GEO(double, 12, 3, 3,
       FQ_L(1, 2, 4, 8, 16, 32, 68, 132, 264, 528, 1057, 2114),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7, 8}, {3, 4, 6, 10, 11, 5, 7, 8, 9}, {0, 1, 2, 8, 9, 6, 7, 10, 11}, {0, 1, 2, 3, 4, 5, 9, 10, 11}))
FQ_GEO(double, 11, 3, 1,
       FQ_L(1, 2, 4, 8, 16, 34, 66, 132, 272, 546, 1088),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {0, 1, 2, 3, 4, 8, 9, 10}))
FQ_GEO(double, 11, 3, 2,
       FQ_L(1, 2, 4, 8, 16, 34, 68, 136, 290, 560, 1120),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {0, 1, 6, 7, 9, 5, 8, 10}, {0, 1, 2, 3, 4, 8, 9, 10}))
FQ_GEO(double, 11, 3, 3,
       FQ_L(1, 2, 4, 8, 16, 33, 65, 132, 272, 552, 1090),
       FQ_L({0, 1, 2, 3, 4, 5, 6, 7}, {3, 4, 5, 7, 10, 6, 8, 9}, {0, 1, 7, 8, 9, 5, 6, 10}, {0, 1, 2, 3, 4, 8, 9, 10}))
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

}  // namespace fq
