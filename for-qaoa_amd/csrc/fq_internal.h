// fq_internal.h -- structures shared by the gfx950 kernels and the host side of
// libforqaoa.  Not part of the public ABI (include/forqaoa.h is).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstddef>

#define FQ_MAXN 40         // qubits (2^40 complex64 = 8 TiB: the HBM limit bites first)
#define FQ_MAXQ 14         // tile qubits held in LDS (2^14 complex64 = 128 KiB)
#define FQ_MAX_GROUPS 5    // LDS re-mapping phases per tile pass
#define FQ_MAX_RUNS 8      // bit runs of a scattered index
#define FQ_TOPK_MAX 16
#define FQ_MAX_REG_LOG 5   // register bits per thread of a tile pass
#define FQ_MAX_REGS (1 << FQ_MAX_REG_LOG)

namespace fq {

// Device view of a cost plan: the Max-Cut quadratic form split for one tile
// geometry.  For a tile (2^Q amplitudes whose index bits at tile positions
// vary) with the other N-Q "high" bits fixed by the tile index:
//   Cut(z) = K(zH) + sum_{tile bit i} c_i(zH) z_i + Cut_tile(z_tile)
//   c_i(zH) = cH[i] - 2 sum_{(h,w) in csr(i)} w zH_h
//   K(zH)  = sum_{hh edges} w [zH_u != zH_v] + sum_h omega[h] zH_h
// The tile bits split into nthr thread bits and A_LOG register bits; the
// thread-dependent, tile-independent part comes from per-thread tables
//   thr[t]                   = edges inside the thread bits + register-thread
//                              edges' constant parts
//   thr[(1+r)*2^nthr + t]    = d_r(t) (coefficient of register bit r)
// and the register-register edges from rr[j] (j = register index).
struct PlanDev {
    const double *cH;      // [Q]
    const int *csr_off;    // [Q+1]
    const int *csr_h;      // [nnz] high-bit index
    const double *csr_w;   // [nnz]
    const int *hh_u;       // [n_hh] high-bit index
    const int *hh_v;       // [n_hh]
    const double *hh_w;    // [n_hh]
    const double *omega;   // [nh]
    const double *thr;     // [(1 + A_LOG) << nthr]
    int n_hh;
    int pad_;
    double wtot;           // sum of all weights
    double rr[FQ_MAX_REGS];  // register-register cut contributions
};

// Index bits [src, src+len) go to physical positions [dst, dst+len); one run
// packed per word as src | len << 8 | dst << 16.
struct BitRuns {
    int n;
    uint32_t run[FQ_MAX_RUNS];
};

// One tile pass: load 2^Q amplitudes per work-group (tile bits tpos[], high
// bits hpos[]), optionally apply the cost phase, RX on the gate bits, store.
struct TileArgs {
    int N, Q, nthr, nh;
    BitRuns hruns;           // tile index -> high positions
    BitRuns truns;           // thread index -> positions of the thread bits
    uint8_t rpos[8];         // positions of the register bits
    uint32_t rpos_w;         // the same packed, 6 bits each (rpos[r] at bit 6r)
    uint64_t ntiles_run;     // tiles processed (0: all 2^nh)
    uint64_t mirror_pm;      // mirror pass: sum of 2^p over the real tile positions
    uint32_t order;          // tile order of the persistent loop (tile_at)
    uint32_t gate_mask;      // over tile bits
    int ngroups;
    uint16_t grp_mask[FQ_MAX_GROUPS];  // tile-bit mask of each LDS phase (A_LOG bits)
    uint8_t grp_gates[FQ_MAX_GROUPS];  // register bits of that phase that receive RX
    uint64_t grp_mask_w;     // grp_mask[0..3], 16 bits each (read with a shift, not an index)
    uint32_t grp_gates_w;    // grp_gates[0..4], 5 bits each
    double rx_c, rx_s;       // cos(beta/2), sin(beta/2) (host-computed, src/rx.cu:121)
    double pre_c, pre_s;     // layer-boundary pass: RX of the previous layer, applied first
    // k_tile applies RX up to a factor as the butterfly [[1, -it], [-it, 1]]
    // (rx_tform), one FMA per output component
    double rx_t, pre_t;
    float rx_tf, pre_tf;     // the same in FP32 (scalar operands of the complex64 butterflies)
    double scale_re, scale_im;  // factor of the pass: folded into the cost phase,
    int apply_scale;            // or (apply_scale) multiplied in before the stores
    double gamma, init_amp;  // cost phase angle, launch-control amplitude
    int has_rr;              // any register-register edge in the plan
    PlanDev plan;
};

// One pass of the compile-time tile kernel (fq_mix.h).
enum { MIX_PLAIN = 0, MIX_FIRST = 1, MIX_COST = 2, MIX_BOUNDARY = 3 };
// The same of a pair pass of the gradient (fq_pair.hip).
enum { PAIR_PLAIN = 0, PAIR_COST = 1, PAIR_BOUNDARY = 2 };
// One slot of a packed launch: its first amplitude, its factors (as in MixArgs)
// and its phase table's first entry.
struct MixSlot {
    double t, pre_t;
    double scale_re, scale_im;
    float tf, pre_tf;
    uint64_t base;
    uint32_t table;
    int has_rr;
};
struct MixArgs {
    int N, Q, nh;
    int has_rr;              // any register-register edge in the plan
    BitRuns hruns;           // tile index -> high positions
    uint8_t tpos[16];        // position of each tile bit (thread bits, then register bits)
    uint32_t rpos0_w;        // positions of the register bits of layout 0, 6 bits each
    uint32_t rposk_w;        // and of the last layout
    uint32_t gates_w;        // gated register bits of layout l at bit A l
    uint64_t tile0, ntiles;  // tiles [tile0, tile0 + ntiles) of this launch
    uint64_t ntab;           // tiles of the whole pass (rows of its phase table)
    uint64_t mirror_pm;      // mirror pass: sum of 2^p over the real tile positions
    double t, pre_t;         // rx_tform coefficients of this layer and of the one before
    float tf, pre_tf;
    double scale_re, scale_im;  // factor of the pass: in the cost phase, or before the
    int apply_scale;            // stores (apply_scale)
    double init_amp;
    int by_xcd;              // tile order (a multiple of 64 tiles)
    const MixSlot *slots;    // packed launch (blockIdx.y: the slot), else null
    int nslots;
};
// Layers of a small state (k_solo): per layer the place of its phase table, its
// factors as above.
#define FQ_SOLO_LAYERS 64
struct SoloArgs {
    int P, first, has_rr;
    uint32_t gates_w;
    double init_amp;
    uint32_t table[FQ_SOLO_LAYERS];
    double t[FQ_SOLO_LAYERS], scale_re[FQ_SOLO_LAYERS], scale_im[FQ_SOLO_LAYERS];
};
// One pair pass: t, pre_t and the real scale as above (a boundary pass undoes
// RX(pre) first), and the weights of its sums: the inverse of the factor that
// <lambda|X|psi> has taken in this pass when the sum is formed, for register bit r
// of layout l at A l + r (0: not gated), the lane bit at PAIR_LANE, the phase.
#define PAIR_LANE 16
struct PairArgs {
    MixArgs m;
    double up[PAIR_LANE + 1], down[PAIR_LANE + 1], phase;
};

// Tiles a launch processes (a Z2-reduced state runs the lower half only).
__host__ __device__ inline uint64_t run_tiles(const TileArgs &a)
{
    return a.ntiles_run ? a.ntiles_run : (1ull << a.nh);
}

// The phase tables of the cost passes of one run (k_phase_tables): the distinct
// geometries, and per pass its geometry, angle and place.
#define FQ_TABLE_GEOS 3
#define FQ_TABLE_JOBS 64
struct TableGeo {
    int Q, nthr, nh, a_log;
    uint64_t ntiles;
    PlanDev plan;
};
struct TableJob {
    double gamma;
    uint16_t geo, cut;       // cut: this job also writes the geometry's exponents
    uint32_t offset;         // entries
};
struct TableJobs {
    TableGeo geo[FQ_TABLE_GEOS];
    uint32_t cut_offset[FQ_TABLE_GEOS];  // place of each geometry's exponents
    TableJob job[FQ_TABLE_JOBS];
};

// Device plans of a slot's graph: the cost passes' geometries (the general
// kernel uses the first; the packed passes 2 * (boundary pass) + pass), <C>.
struct SlotPlans {
    PlanDev cost[4];
    PlanDev expect;
};
// Per-slot parameters of a step of the general kernel, in device memory.
struct SlotParams {
    double rx_c, rx_s;       // RX(beta) of the slot's current layer
    double gamma;            // cost angle of the slot's current layer
    double init_amp;         // (1/sqrt 2)^N
    int active;              // the slot runs this step
    int cost_first;          // layer 0: launch-control write, no read
    int has_rr;
    const double2 *ptab;     // the slot's phase table for this step
};
// Phase tables of a packed step: the geometries (plan unused) and, per table,
// angle, slot, geometry and first entry.
struct SlabGeos {
    TableGeo geo[4];
};
struct SlabJob {
    double gamma;
    uint32_t slot, geo, offset, pad;
};

#define FQ_SWAP_BITS 12     // qubits of an exchange tile: 2^12 complex64, 2^10 complex128

// As BitRuns, for any set of positions.
struct SwapRuns {
    int n;
    uint32_t run[FQ_MAXN / 2];
};

// Exchange of pairs of qubits (k_exchange).
struct SwapArgs {
    int tb;                          // tile qubits
    int rest_fast;                   // consecutive units step the rest index first
    int nr;                          // bits of the rest index
    int large;                       // the state exceeds the memory-side cache
    uint8_t tpos[FQ_SWAP_BITS];      // tile bit -> position (ascending)
    uint8_t partner[FQ_SWAP_BITS];   // tile bit -> the tile bit it changes places with (itself if none)
    SwapRuns lower, upper, rest;     // positions of the pairs outside the tile, and of the others
    uint64_t npairs;                 // X <= Y
};

// Resident work-groups per CU of kernel fn at this block size and dynamic
// LDS (at least 1), cached per (fn, threads, lds): the runtime query costs
// tens of microseconds and the persistent launchers ask on every launch.
int occupancy_per_cu(const void *fn, int threads, size_t lds);
// Lets kernel fn take up to 159 KiB of dynamic LDS (set once per kernel).
hipError_t allow_large_lds(const void *fn);
// Compute units of the current device (cached).
int device_cu_count();

// Launchers (fq_kernels.hip).  All enqueue on `stream` and return the HIP
// launch status.
hipError_t launch_tile(int dtype, int a_log, bool cost, bool first, bool gates, void *sv,
                       const TileArgs &a, const double2 *phase_tab, hipStream_t stream);
// Layer-boundary pass: RX(pre) on the pass's qubits, cost phase, RX(rx).
hipError_t launch_tile_pre(int dtype, int a_log, void *sv, const TileArgs &a, const double2 *ptab,
                           hipStream_t stream);
// Tile passes of fq_mix.h.  mix_a_log: register bits per thread of its
// instance for tiles of 2^Q amplitudes (0: none).  k: exchanges one way (they
// reach the tile bits from Q - (k + 1) A up), lane: RX also on the bit below
// those, where mix_lane_bit says there is such an instance; kind MIX_*, mir:
// 0, the half-state mirror pass (1; 2 writes the full state's upper half too).
int mix_a_log(int dtype, int Q);
bool mix_lane_bit(int Q, int A, int k);
hipError_t launch_mix(int dtype, int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                      hipStream_t stream);
// Mirror pass of a Z2-reduced state: the top register bit of the virtual tile
// selects the complementary tile (complemented element offsets) and RX on it
// is the butterfly of the global spin flip.  expand: also write the upper
// half of the full state.
hipError_t launch_tile_mirror(int dtype, int a_log, bool expand, void *sv, const TileArgs &a,
                              hipStream_t stream);
// Phase factors of a cost-phase launch into tab (size phase_table_entries);
// with cut not null, their exponents over gamma into cut (same size).
hipError_t launch_phase_table(const TileArgs &a, int a_log, double2 *tab, double *cut,
                              hipStream_t stream);
size_t phase_table_entries(const TileArgs &a, int a_log);
// njobs tables of at most `entries` entries each; cut not null: the exponents of
// the geometries too
hipError_t launch_phase_tables(const TableJobs &m, int njobs, size_t entries, double2 *tab, double *cut,
                               hipStream_t stream);
hipError_t launch_swap(int dtype, void *sv, const SwapArgs &a, hipStream_t stream);
// Runs of pairs: the lower position, their number, the upper position (bits 0, 8, 16).
// States up to 1 MiB: a call that waits takes 12.2 to 14.2 us instead of 13.4 to 14.5 (N=4
// to 16 complex128, the lower half with the upper one); at 2 MiB 15.2 instead of 14.5, at
// 16 MiB 27 instead of 18, since one side of a pair is read in single amplitudes.
#define FQ_SWAP_SMALL ((size_t)1 << 20)
hipError_t launch_swap_small(int dtype, void *sv, const SwapRuns &pairs, int N, hipStream_t stream);
// partials == out2: the sums of each tile, without the second launch of one work-group that
// adds them up.  (The last work-group adding up instead, by a fence and an atomic of each,
// took N=16 18.4 us instead of 18.5, N=20 22.9 instead of 19.4, N=22 46 instead of 28.5, and
// N=3, whose work-group is one thread, 135 instead of 15.)
hipError_t launch_expect(int dtype, int a_log, const void *sv, const TileArgs &a, double *partials,
                         double *out2, hipStream_t stream);
hipError_t launch_topk(int dtype, const void *sv, int N, int nblocks, double *cand_p,
                       uint64_t *cand_i, hipStream_t stream);
hipError_t launch_gather(int dtype, const void *sv, const uint64_t *idx, size_t n, double *out,
                         hipStream_t stream);
hipError_t launch_fill_zero_one(int dtype, void *sv, int N, hipStream_t stream);
// streaming probe over bytes (a multiple of 8): mode 0 in-place scale,
// 1 read-only, 2 fill; sink: one float
hipError_t launch_stream(void *p, size_t bytes, int mode, float *sink, hipStream_t stream);
hipError_t launch_finalize(const double *partials, uint64_t n, double *out2, hipStream_t stream);
// adjoint (fq_adjoint.hip)
// grid receives the number of work-groups (= partial sum pairs written).
// With costbw, ptab and ctab are the phase and cut tables of one
// launch_phase_table call.
// mirror: the half-state mirror pass (qubit N-1 the top register bit).
// boundary (with costbw): after the conjugate phase, RX with a.pre_c, a.pre_s
// on the same gate bits; its sums go to partials[2 * (*grid) ...], the
// work-group's second pair of partial sums.
hipError_t launch_pair(int dtype, int a_log, bool costbw, bool mirror, bool boundary, void *psi, void *lam,
                       const TileArgs &a, const double2 *ptab, const double *ctab, double *partials,
                       unsigned *grid, hipStream_t stream);
hipError_t launch_cut_mul(int dtype, int a_log, const void *psi, void *lam, const TileArgs &a,
                          double *partials, hipStream_t stream);
size_t pair_lds_bytes(int dtype, int Q);
// Qubits of a state that k_solo takes: [solo_min, solo_max].
inline int solo_min(int dtype) { return dtype == 0 ? 9 : 10; }
inline int solo_max(int) { return 12; }
hipError_t launch_solo(int dtype, int N, void *sv, const SoloArgs &a, const double2 *ptab, hipStream_t stream);
// Pair passes of fq_pair.hip; arguments as launch_mix (register bits per thread
// pair_a_log, 0: no instance for this tile width).  partials: three sums per tile.
int pair_a_log(int dtype, int Q);
bool pair_lane_bit(int Q, int A, int k);
hipError_t launch_pair_pass(int dtype, int k, bool lane, int kind, bool mir, void *psi, void *lam, const PairArgs &a,
                            const double2 *ptab, const double *ctab, double *partials, hipStream_t stream);
// out[3 s ..] = the sums of pass s's n triples (partials + 3 n s)
hipError_t launch_pair_sums(const double *partials, uint64_t n, int passes, double *out, hipStream_t stream);
// packed slabs (fq_serve.hip)
hipError_t launch_slab_phase_table(const TileArgs &local, int a_log, const SlotParams *slots, const SlotPlans *plans,
                                   int nslots, double2 *tabs, size_t stride, hipStream_t stream);
hipError_t launch_slab_tables(const SlabGeos &g, const SlabJob *jobs, int njobs, size_t entries, const SlotPlans *plans,
                              double2 *tabs, hipStream_t stream);
hipError_t launch_slab_pass(int dtype, int a_log, bool cost, bool mirror, void *sv, const TileArgs &a,
                            const SlotParams *slots, int slot_shift, hipStream_t stream);
// <C> and sum |psi|^2 of the nfin slots fin[] into out[2 slot]
hipError_t launch_slab_expect(int dtype, int a_log, const void *sv, const TileArgs &a, const SlotPlans *plans,
                              const int *fin, int nfin, int slot_shift, double *partials, double *out,
                              hipStream_t stream);
int tile_max_q(int dtype);
size_t tile_lds_bytes(int dtype, int Q);

// RX(beta) coefficients c = cos(beta/2), s = sin(beta/2) (src/rx.cu:121) as
// the kernels of amplitude type dtype apply them.  FQ_C128: the FP64 values.
// FQ_C64: an FP32 pair (returned as doubles, exact when cast back) chosen so
// that c^2 + s^2 = 1 as nearly as FP32 allows.  Rounding cos and sin to FP32
// independently leaves c^2 + s^2 - 1 up to ~1e-7, and RX scales the norm of
// the state by exactly c^2 + s^2, so that error compounds over every qubit
// and layer into a drift of N*P*(c^2 + s^2 - 1) in <C>.
void rx_coeffs(double beta, int dtype, double *c, double *s);
// RX(beta) as sigma * B(t), B(t) = [[1, -it], [-it, 1]] with t rounded to the
// amplitude type of dtype and sigma (FP64, from the rounded t) making
// sigma * B(t) exactly unitary: RX of an angle within one rounding of beta.
// t = tan(beta/2), sigma = cos(beta/2)-like, real.  With flip and
// |sin(beta/2)| > |cos(beta/2)| instead RX(beta) = -i sin(beta/2) X B(t') with
// t' = tan((beta - pi)/2) = -cot(beta/2): the X is dropped and sigma is
// -i/sqrt(1 + t'^2) (signed).  Dropping X is exact only where the caller
// applies RX(beta) to every qubit of an X^(x)N-symmetric state (a QAOA layer:
// the dropped X's form X^(x)N, which commutes with every layer and leaves the
// state unchanged).  |t| <= 1 with flip; without it |t| = |tan(beta/2)|.
void rx_tform(double beta, int dtype, bool flip, double *t, double *sigma_re, double *sigma_im);

}  // namespace fq
