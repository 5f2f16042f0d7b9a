// fq_mix_c128.hip -- complex128 instances of the tile passes in fq_mix.h.
#include "fq_mix.h"

namespace fq {

hipError_t launch_mix_c128(int k, bool lane, int kind, int mir, void *sv, const MixArgs &a, const double2 *ptab,
                           hipStream_t stream)
{
    switch (a.Q) {
        case 13: return launch_mix_q<double, 13, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 12: return launch_mix_q<double, 12, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 11: return launch_mix_q<double, 11, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 10: return launch_mix_q<double, 10, 4>(k, lane, kind, mir, sv, a, ptab, stream);
        case 9: return launch_mix_q<double, 9, 3>(k, lane, kind, mir, sv, a, ptab, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_solo_c128(int N, void *sv, const SoloArgs &a, const double2 *ptab, hipStream_t stream)
{
    switch (N) {
        case 12: return launch_solo_q<double, 12, 4>(sv, a, ptab, stream);
        case 11: return launch_solo_q<double, 11, 4>(sv, a, ptab, stream);
        case 10: return launch_solo_q<double, 10, 4>(sv, a, ptab, stream);
        case 9: return launch_solo_q<double, 9, 3>(sv, a, ptab, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fq
