// fq_mix_c64.hip -- complex64 instances of the tile passes in fq_mix.h, and the
// choice between the two types.
#include "fq_mix.h"

namespace fq {

hipError_t launch_mix_c128(int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                           hipStream_t stream);

static hipError_t launch_mix_c64(int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                                 hipStream_t stream)
{
    switch (a.Q) {
        case 14: return launch_mix_q<float, 14, 5>(k, lane, kind, mir, sv, a, ptab, stream);
        case 13: return launch_mix_q<float, 13, 5>(k, lane, kind, mir, sv, a, ptab, stream);
        case 12: return launch_mix_q<float, 12, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 11: return launch_mix_q<float, 11, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 10: return launch_mix_q<float, 10, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_mix(int dtype, int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                      hipStream_t stream)
{
    return dtype == 0 ? launch_mix_c128(k, lane, kind, mir, sv, a, ptab, stream)
                      : launch_mix_c64(k, lane, kind, mir, sv, a, ptab, stream);
}

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

hipError_t launch_solo_c128(int N, void *sv, const SoloArgs &a, const double2 *ptab, hipStream_t stream);

hipError_t launch_solo(int dtype, int N, void *sv, const SoloArgs &a, const double2 *ptab, hipStream_t stream)
{
    if (dtype == 0)
        return launch_solo_c128(N, sv, a, ptab, stream);
    switch (N) {
        case 12: return launch_solo_q<float, 12, 4>(sv, a, ptab, stream);
        case 11: return launch_solo_q<float, 11, 4>(sv, a, ptab, stream);
        case 10: return launch_solo_q<float, 10, 4>(sv, a, ptab, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fq
