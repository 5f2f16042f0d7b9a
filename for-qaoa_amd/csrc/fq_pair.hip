// fq_pair.hip -- the pair passes of the adjoint gradient on compile-time LDS
// phases: psi and lambda of one tile walked back together.  fq_adjoint.hip has
// the mathematics, lambda = Cut psi, and the general pair pass for states
// smaller than these tiles.
//
// Both states of a tile of 2^Q amplitudes sit in registers (2^A of each per
// thread).  An exchange moves 8-byte items through one buffer: in complex64
// psi's amplitudes and then lambda's, in complex128 the four components in
// turn.  So the buffer is a quarter (complex128) or half of what the general
// pass holds, two work-groups share a CU, and the loads of one overlap the
// butterflies of the other.
//
// What bounds a pass: complex64 its vector instructions (the boundary pass:
// two RX sets on two states, 13 per amplitude pair and gate with the pair
// sums), the others the memory.  Tiles of 2^13 complex64 and 2^12 complex128
// amplitudes: 64 KiB of each state, the widest whose buffer (64 KiB and 32 KiB)
// leaves room for a second work-group.  At N=26 complex64 (512 MiB of half
// states read, and again written, a pass: 200 us at HBM speed): plain 240 us, boundary
// 356 us; the walk back of 8 layers 5.6 -> 4.5 ms against the general passes.
#include "fq_exchange.h"

namespace fq {

// Tables that do not change during a launch, read at uniform addresses: scalar
// loads.
typedef const __attribute__((address_space(4))) double *ConstDoubles;

// A thread's 2^A amplitudes of psi and lambda, by component (arrays of plain
// scalars stay in registers; arrays of the vector types went to scratch here).
template <typename R, int A> struct PairRegs {
    R px[1 << A], py[1 << A], lx[1 << A], ly[1 << A];
};

// 8-byte items of register j: complex64 psi and lambda, complex128 the four components.
template <typename R> struct PairItem;
template <> struct PairItem<float> {
    typedef float2 I;
    static constexpr int NC = 2;
    template <int C, int A> static __device__ __forceinline__ I get(const PairRegs<float, A> &v, int j)
    {
        return C == 0 ? make_float2(v.px[j], v.py[j]) : make_float2(v.lx[j], v.ly[j]);
    }
    template <int C, int A> static __device__ __forceinline__ void set(PairRegs<float, A> &v, int j, I x)
    {
        if constexpr (C == 0) {
            v.px[j] = x.x;
            v.py[j] = x.y;
        } else {
            v.lx[j] = x.x;
            v.ly[j] = x.y;
        }
    }
};
template <> struct PairItem<double> {
    typedef double I;
    static constexpr int NC = 4;
    template <int C, int A> static __device__ __forceinline__ I get(const PairRegs<double, A> &v, int j)
    {
        return C == 0 ? v.px[j] : C == 1 ? v.py[j] : C == 2 ? v.lx[j] : v.ly[j];
    }
    template <int C, int A> static __device__ __forceinline__ void set(PairRegs<double, A> &v, int j, I x)
    {
        if constexpr (C == 0)
            v.px[j] = x;
        else if constexpr (C == 1)
            v.py[j] = x;
        else if constexpr (C == 2)
            v.lx[j] = x;
        else
            v.ly[j] = x;
    }
};

// Component C of both states from layout L0 to L1; then the next one.  BACK:
// the components in descending order, which starts with the one the last
// exchange ended on: its slots in layout L0 are the thread's own.
template <typename Lay, typename R, int A, int L0, int L1, bool BACK, int N = 0>
__device__ __forceinline__ void pair_exchange(PairRegs<R, A> &v, typename PairItem<R>::I *lds, int s0, int s1)
{
    typedef PairItem<R> It;
    constexpr int C = BACK ? It::NC - 1 - N : N;
    if constexpr (N > 0)
        lds_barrier();   // the previous component has been read
#pragma unroll
    for (int j = 0; j < (1 << A); ++j) {
        lds[s0 + Lay::reg_slot(L0, j)] = It::template get<C, A>(v, j);
        if (j % 4 == 3)
            __builtin_amdgcn_sched_barrier(0);   // few register pairs being put together at a time
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < (1 << A); ++j)
        It::template set<C, A>(v, j, lds[s1 + Lay::reg_slot(L1, j)]);
    if constexpr (N + 1 < It::NC)
        pair_exchange<Lay, R, A, L0, L1, BACK, N + 1>(v, lds, s0, s1);
}

// B(t) (rx_pair_t) on one pair of amplitudes.
template <typename R> __device__ __forceinline__ void pair_butterfly(R &x0, R &y0, R &x1, R &y1, R t)
{
    const R a = fma(t, y1, x0), b = fma(-t, x1, y0), c = fma(t, y0, x1), d = fma(-t, x0, y1);
    x0 = a;
    y0 = b;
    x1 = c;
    y1 = d;
}

// RX on the gated register bits of both states and its pair sums,
// Im(conj(l0) p1 + conj(l1) p0) for Im<lambda|X_j|psi>.  RX is the butterfly
// B(t) of rx_tform, which multiplies both states by (1 + t^2)^(1/2) against the
// unitary; w[r] is the inverse of the factor that <lambda|X|psi> has taken when
// bit r's turn comes (PairArgs).  The terms of four pairs are summed in the
// amplitude precision, then in FP64.  An ungated bit runs t = 0 (the identity)
// and has weight 0.
template <typename R, int A>
__device__ __forceinline__ void pair_rx(PairRegs<R, A> &v, uint32_t mask, R t, const double *w, double &acc)
{
#pragma unroll
    for (int r = 0; r < A; ++r) {
        const R tr = ((mask >> r) & 1u) ? t : R(0);
        double sum = 0.0;
        R part = 0;
        int n = 0;
#pragma unroll
        for (int j = 0; j < (1 << A); ++j) {
            if (!((j >> r) & 1)) {
                const int k = j | (1 << r);
                part += (v.lx[j] * v.py[k] - v.ly[j] * v.px[k]) + (v.lx[k] * v.py[j] - v.ly[k] * v.px[j]);
                if (++n % 4 == 0) {
                    sum += (double)part;
                    part = 0;
                }
                pair_butterfly(v.px[j], v.py[j], v.px[k], v.py[k], tr);
                pair_butterfly(v.lx[j], v.ly[j], v.lx[k], v.ly[k], tr);
            }
        }
        acc = fma(sum, w[r], acc);
        asm volatile("" : "+v"(acc));   // added here: sunk to the kernel's end, every bit's sums stay live
        __builtin_amdgcn_sched_barrier(0);   // one bit's terms live at a time
    }
}

// The same on lane bit B: both lanes of a pair count their own term.
template <typename R, int A, int B>
__device__ __forceinline__ void pair_rx_lane(PairRegs<R, A> &v, R t, double w, double &acc)
{
    double sum = 0.0;
    R part = 0;
#pragma unroll
    for (int j = 0; j < (1 << A); ++j) {
        const R px = lane_xor<B>(v.px[j]), py = lane_xor<B>(v.py[j]);
        const R lx = lane_xor<B>(v.lx[j]), ly = lane_xor<B>(v.ly[j]);
        part += v.lx[j] * py - v.ly[j] * px;
        if (j % 8 == 7) {
            sum += (double)part;
            part = 0;
        }
        v.px[j] = fma(t, py, v.px[j]);
        v.py[j] = fma(-t, px, v.py[j]);
        v.lx[j] = fma(t, ly, v.lx[j]);
        v.ly[j] = fma(-t, lx, v.ly[j]);
    }
    acc = fma(sum, w, acc);
    asm volatile("" : "+v"(acc));
}

template <typename Lay, typename R, int A, int K, int L, int X0, int LB>
__device__ __forceinline__ void pair_up(PairRegs<R, A> &v, typename PairItem<R>::I *lds, const int (&sb)[K + 1],
                                        uint32_t gates, R t, const double *w, double &acc)
{
    if constexpr (L == 0 && LB >= 0)
        pair_rx_lane<R, A, LB>(v, t, w[PAIR_LANE], acc);
    pair_rx<R, A>(v, (gates >> (A * L)) & ((1u << A) - 1u), t, w + A * L, acc);
    if constexpr (L < K) {
        pair_exchange<Lay, R, A, L, L + 1, ((X0 + L) & 1) != 0>(v, lds, sb[L], sb[L + 1]);
        pair_up<Lay, R, A, K, L + 1, X0, LB>(v, lds, sb, gates, t, w, acc);
    }
}

template <typename Lay, typename R, int A, int K, int L, int X0, int LB>
__device__ __forceinline__ void pair_down(PairRegs<R, A> &v, typename PairItem<R>::I *lds, const int (&sb)[K + 1],
                                          uint32_t gates, R t, const double *w, double &acc)
{
    pair_rx<R, A>(v, (gates >> (A * L)) & ((1u << A) - 1u), t, w + A * L, acc);
    if constexpr (L > 0) {
        pair_exchange<Lay, R, A, L, L - 1, ((X0 + K - L) & 1) != 0>(v, lds, sb[L], sb[L - 1]);
        pair_down<Lay, R, A, K, L - 1, X0, LB>(v, lds, sb, gates, t, w, acc);
    } else if constexpr (LB >= 0) {
        pair_rx_lane<R, A, LB>(v, t, w[PAIR_LANE], acc);
    }
}

// Phase factor and s/2 of every register's amplitude by a tree over the
// register bits: both states times the factor, the term of Im<lambda|S|phi>
// (S = 2 (s/2)) added up.
template <typename R, int A, int RB>
__device__ __forceinline__ void pair_phase(PairRegs<R, A> &v, const R (&fx)[A], const R (&fy)[A], const double (&cr)[A],
                                           ConstDoubles rr_c, ConstDoubles rr_f, R x, R y, double h,
                                           double &acc, int j)
{
    if constexpr (RB == 0) {
        const R im = v.lx[j] * v.py[j] - v.ly[j] * v.px[j];
        h += rr_c[j];
        const R gx = (R)rr_f[2 * j], gy = (R)rr_f[2 * j + 1];
        const R nx = x * gx - y * gy;
        y = x * gy + y * gx;
        x = nx;
        acc = fma(2.0 * h, (double)im, acc);
        const R px = v.px[j], lx = v.lx[j];
        v.px[j] = px * x - v.py[j] * y;
        v.py[j] = px * y + v.py[j] * x;
        v.lx[j] = lx * x - v.ly[j] * y;
        v.ly[j] = lx * y + v.ly[j] * x;
    } else {
        pair_phase<R, A, RB - 1>(v, fx, fy, cr, rr_c, rr_f, x, y, h, acc, j);
        if (RB == 2)
            __builtin_amdgcn_sched_barrier(0);   // depth first
        pair_phase<R, A, RB - 1>(v, fx, fy, cr, rr_c, rr_f, x * fx[RB - 1] - y * fy[RB - 1],
                                     x * fy[RB - 1] + y * fx[RB - 1], h + cr[RB - 1], acc, j | (1 << (RB - 1)));
    }
}

// One pair pass.  KIND: PAIR_PLAIN undoes RX on the gated bits; PAIR_COST a cost
// pass (RX undone, then the phase); PAIR_BOUNDARY a layer-boundary pass (RX of
// the later layer (pre), the phase, RX of the earlier one).  The phase table is
// built for -gamma, its companion ctab holds the exponents over gamma: s/2 of an
// amplitude is the sum of the entries whose factors make its phase.  MIR: the
// half-state mirror pass, as in k_mix.  partials[3 i ..]: work-group i's sums of
// the first RX set, of the phase and of the second RX set.
template <typename R, int Q, int A, int K, int KIND, bool MIR, bool LG>
__global__ void __launch_bounds__(1 << (Q - A), 4)
    k_pair(typename CT<R>::T *__restrict__ psi, typename CT<R>::T *__restrict__ lam, const PairArgs pa,
           const double2 *__restrict__ ptab, const double *__restrict__ ctab, double *__restrict__ partials)
{
    typedef typename CT<R>::T T;
    typedef typename PairItem<R>::I I;
    typedef MixLay<double, Q, A, K> Lay;   // 8-byte items
    const MixArgs &a = pa.m;
    constexpr int N = 1 << A, NT = Q - A, AH = MIR ? N / 2 : N;
    constexpr int NB = MIR ? A - 1 : A;
    constexpr bool COST = KIND != PAIR_PLAIN;
    constexpr int LB = LG ? Q - A - K * A - 1 : -1;
    constexpr int LS = KIND == PAIR_BOUNDARY || MIR ? 0 : K;   // layout of the stores
    extern __shared__ __align__(16) unsigned char fq_smem_p[];
    __shared__ double s_red[3][(1 << NT) / 64 > 0 ? (1 << NT) / 64 : 1];
    I *lds = reinterpret_cast<I *>(fq_smem_p);
    const int t = threadIdx.x, lane = t & 63;
    const uint64_t hmask = (1ull << a.nh) - 1ull;

    uint64_t toff = 0, soff = 0;
    int sb[K + 1];
#pragma unroll
    for (int i = 0; i <= K; ++i)
        sb[i] = 0;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const bool on = (t >> k) & 1;
        toff |= on ? 1ull << a.tpos[k] : 0ull;
        if (LS != 0)
            soff |= on ? 1ull << a.tpos[Lay::p(LS, k)] : 0ull;
#pragma unroll
        for (int i = 0; i <= K; ++i)
            sb[i] += on ? Lay::w(Lay::p(i, k)) : 0;
    }
    const uint64_t tile = a.tile0 + blockIdx.x, q1 = Q + 1;
    const uint64_t thr0 = a.ntab * q1, rr0 = thr0 + ((uint64_t)(1 + A) << NT);
    const uint64_t base = unpack_runs_uniform(tile, a.hruns);
    PairRegs<R, A> v;
    // element of register j (mirror: its upper half at complemented offsets)
    auto at = [&](const uint64_t (&ro)[N], uint64_t b0, uint64_t bm, int j) -> uint64_t {
        return j < AH ? b0 + ro[j] : bm - ro[j - (MIR ? AH : 0)];
    };
    const uint64_t bm = MIR ? unpack_runs_uniform(~tile & hmask, a.hruns) + a.mirror_pm - toff : 0;
    {
        uint64_t ro[N];
        reg_offsets<N, NB>(a.rpos0_w, ro);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint64_t i = at(ro, base + toff, bm, j);
            const T x = psi[i], y = lam[i];
            v.px[j] = x.x;
            v.py[j] = x.y;
            v.lx[j] = y.x;
            v.ly[j] = y.y;
        }
    }
    double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
    if constexpr (KIND == PAIR_BOUNDARY)
        pair_up<Lay, R, A, K, 0, 0, LB>(v, lds, sb, a.gates_w, sizeof(R) == 4 ? (R)a.pre_tf : (R)a.pre_t, pa.up, acc0);
    else
        pair_up<Lay, R, A, K, 0, 0, LB>(v, lds, sb, a.gates_w, sizeof(R) == 4 ? (R)a.tf : (R)a.t, pa.up, acc0);
    if constexpr (COST) {
        // the tile's rows (entry i in lane i, broadcast by readlane) and the thread's entries
        const double2 f_row = ptab[tile * q1 + lane % (Q + 1)], f_thr = ptab[thr0 + t];
        const double c_row = ctab[tile * q1 + lane % (Q + 1)], c_thr = ctab[thr0 + t];
        double x = f_thr.x, y = f_thr.y, h = c_thr + lane_bcast(c_row, Q);
        auto mul = [&](double2 f) {
            const double nx = x * f.x - y * f.y;
            y = x * f.y + y * f.x;
            x = nx;
        };
        mul(lane_bcast(f_row, Q));
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const double2 f = lane_bcast(f_row, i);
            const double c = lane_bcast(c_row, i);
            const double nx = x * f.x - y * f.y;
            const double ny = x * f.y + y * f.x;
            const bool on = (t >> i) & 1;
            x = on ? nx : x;
            y = on ? ny : y;
            h += on ? c : 0.0;
        }
        // the magnitude the states have taken on goes into the phase
        const R x0 = (R)(x * a.scale_re), y0 = (R)(y * a.scale_re);
        R fx[A], fy[A];
        double cr[A];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < A; ++r) {
            const double2 f = lane_bcast(f_row, NT + r), g = ptab[thr0 + ((1 + r) << NT) + t];
            fx[r] = (R)(g.x * f.x - g.y * f.y);
            fy[r] = (R)(g.x * f.y + g.y * f.x);
            cr[r] = lane_bcast(c_row, NT + r) + ctab[thr0 + ((1 + r) << NT) + t];
            __builtin_amdgcn_sched_barrier(0);
        }
        // (the register-register entries also where they are 1 and 0: with a
        // second branch the compiler hoisted what the two had in common and
        // spilled 1,300 bytes a lane)
        pair_phase<R, A, A>(v, fx, fy, cr, (ConstDoubles)(uintptr_t)(ctab + rr0), (ConstDoubles)(uintptr_t)(ptab + rr0), x0,
                            y0, h, acc1, 0);
        __builtin_amdgcn_sched_barrier(0);
        acc1 *= pa.phase;
        asm volatile("" : "+v"(acc1));
    }
    if constexpr (KIND == PAIR_BOUNDARY)
        pair_down<Lay, R, A, K, K, K, LB>(v, lds, sb, a.gates_w, sizeof(R) == 4 ? (R)a.tf : (R)a.t, pa.down, acc2);
    if constexpr (MIR && KIND != PAIR_BOUNDARY && K > 0)
        pair_exchange<Lay, R, A, K, 0, (K & 1) != 0>(v, lds, sb[K], sb[0]);
    {
        uint64_t ro[N];
        reg_offsets<N, NB>(LS == 0 ? a.rpos0_w : a.rposk_w, ro);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint64_t i = at(ro, base + (LS == 0 ? toff : soff), bm, j);
            T x, y;
            x.x = v.px[j];
            x.y = v.py[j];
            y.x = v.lx[j];
            y.y = v.ly[j];
            psi[i] = x;
            lam[i] = y;
            if (j % 4 == 3)
                __builtin_amdgcn_sched_barrier(0);
        }
    }
    // fixed-order sums: lanes by shuffle, then the waves
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        acc0 += __shfl_xor(acc0, off, 64);
        if (COST)
            acc1 += __shfl_xor(acc1, off, 64);
        if (KIND == PAIR_BOUNDARY)
            acc2 += __shfl_xor(acc2, off, 64);
    }
    if (lane == 0) {
        s_red[0][t >> 6] = acc0;
        s_red[1][t >> 6] = acc1;
        s_red[2][t >> 6] = acc2;
    }
    __syncthreads();
    if (t < 3) {
        double x = 0.0;
        for (int i = 0; i < (1 << NT) / 64; ++i)
            x += s_red[t][i];
        partials[3 * tile + t] = x;
    }
}

// Sums of the passes: work-group s adds up pass s's n triples in a fixed order.
__global__ void __launch_bounds__(256) k_pair_sums(const double *__restrict__ partials, uint64_t n,
                                                   double *__restrict__ out)
{
    __shared__ double s[3][256];
    const double *p = partials + 3 * n * blockIdx.x;
    const int t = threadIdx.x;
    double x[3] = {0.0, 0.0, 0.0};
    for (uint64_t i = t; i < n; i += 256)
        for (int k = 0; k < 3; ++k)
            x[k] += p[3 * i + k];
    for (int k = 0; k < 3; ++k)
        s[k][t] = x[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w)
            for (int k = 0; k < 3; ++k)
                s[k][t] += s[k][t + w];
        __syncthreads();
    }
    if (t < 3)
        out[3 * blockIdx.x + t] = s[t][0];
}

// ---- launchers ---------------------------------------------------------------

template <typename R, int Q, int A, int K, int KIND, bool MIR, bool LG>
static hipError_t launch_pair_k(void *psi, void *lam, const PairArgs &a, const double2 *ptab, const double *ctab,
                                double *partials, hipStream_t stream)
{
    typedef typename CT<R>::T T;
    constexpr size_t lds = K > 0 ? 8 * (size_t)MixLay<double, Q, A, K>::slots() : 0;
    const void *fn = reinterpret_cast<const void *>(&k_pair<R, Q, A, K, KIND, MIR, LG>);
    if (lds > 65536 - 1024) {
        if (hipError_t e = allow_large_lds(fn))
            return e;
    }
    hipLaunchKernelGGL((k_pair<R, Q, A, K, KIND, MIR, LG>), dim3((unsigned)a.m.ntiles), dim3(1u << (Q - A)), lds, stream,
                       reinterpret_cast<T *>(psi), reinterpret_cast<T *>(lam), a, ptab, ctab, partials);
    return hipGetLastError();
}

template <int Q, int A, int K> static constexpr bool pair_has_lane()
{
    return K > 0 && (Q - A - K * A == 4 || Q - A - K * A == 2 || Q - A - K * A == 1);
}

template <typename R, int Q, int A, int K, bool LG>
static hipError_t launch_pair_l(int kind, bool mir, void *psi, void *lam, const PairArgs &a, const double2 *ptab,
                                const double *ctab, double *part, hipStream_t s)
{
    switch (kind * 2 + (mir ? 1 : 0)) {
        case PAIR_PLAIN * 2: return launch_pair_k<R, Q, A, K, PAIR_PLAIN, false, LG>(psi, lam, a, ptab, ctab, part, s);
        case PAIR_PLAIN * 2 + 1: return launch_pair_k<R, Q, A, K, PAIR_PLAIN, true, LG>(psi, lam, a, ptab, ctab, part, s);
        case PAIR_COST * 2: return launch_pair_k<R, Q, A, K, PAIR_COST, false, LG>(psi, lam, a, ptab, ctab, part, s);
        case PAIR_BOUNDARY * 2:
            return launch_pair_k<R, Q, A, K, PAIR_BOUNDARY, false, LG>(psi, lam, a, ptab, ctab, part, s);
        case PAIR_BOUNDARY * 2 + 1:
            return launch_pair_k<R, Q, A, K, PAIR_BOUNDARY, true, LG>(psi, lam, a, ptab, ctab, part, s);
        default: return hipErrorInvalidValue;
    }
}

template <typename R, int Q, int A>
static hipError_t launch_pair_q(int k, bool lane, int kind, bool mir, void *psi, void *lam, const PairArgs &a,
                                const double2 *ptab, const double *ctab, double *part, hipStream_t s)
{
#define FQ_PK(K_)                                                                                   \
    if constexpr (Q - A > (K_ - 1) * A)                                                             \
        if (k == K_) {                                                                              \
            if (!lane)                                                                              \
                return launch_pair_l<R, Q, A, K_, false>(kind, mir, psi, lam, a, ptab, ctab, part, s); \
            if constexpr (pair_has_lane<Q, A, K_>())                                                \
                return launch_pair_l<R, Q, A, K_, true>(kind, mir, psi, lam, a, ptab, ctab, part, s); \
            return hipErrorInvalidValue;                                                            \
        }
    FQ_PK(0)
    FQ_PK(1)
    FQ_PK(2)
    FQ_PK(3)
#undef FQ_PK
    return hipErrorInvalidValue;
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

hipError_t launch_pair_pass(int dtype, int k, bool lane, int kind, bool mir, void *psi, void *lam, const PairArgs &a,
                            const double2 *ptab, const double *ctab, double *partials, hipStream_t stream)
{
#define FQ_PQ(R, Q, A) \
    case Q: return launch_pair_q<R, Q, A>(k, lane, kind, mir, psi, lam, a, ptab, ctab, partials, stream);
    if (dtype == 0) {
        switch (a.m.Q) {
            FQ_PQ(double, 12, 3)
            FQ_PQ(double, 11, 3)
            FQ_PQ(double, 10, 3)
            FQ_PQ(double, 9, 3)
            default: return hipErrorInvalidValue;
        }
    }
    switch (a.m.Q) {
        FQ_PQ(float, 13, 4)
        FQ_PQ(float, 12, 4)
        FQ_PQ(float, 11, 4)
        FQ_PQ(float, 10, 4)
        default: return hipErrorInvalidValue;
    }
#undef FQ_PQ
}

hipError_t launch_pair_sums(const double *partials, uint64_t n, int passes, double *out, hipStream_t stream)
{
    hipLaunchKernelGGL(k_pair_sums, dim3((unsigned)passes), dim3(256), 0, stream, partials, n, out);
    return hipGetLastError();
}

}  // namespace fq
