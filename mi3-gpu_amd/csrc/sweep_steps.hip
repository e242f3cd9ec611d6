// Instantiation and launch of the step-staged sweep (q <= 8).
#include "k_potts.hip"
#include "launch.h"

namespace mi3 {

namespace {
template <int KW, int S, int NW, int NPC>
hipError_t run_shape(const SweepArgs& a, hipStream_t st, uint32_t stage_kb) {
    auto kern = k_sweep_steps<KW, S, NW, NPC>;
    const uint32_t rowb = a.nchunk * NPC * 1024;
    const uint32_t nst = stage_kb * 1024 > rowb ? stage_kb * 1024 / rowb : 1;
    const size_t lds = 2ull * nst * rowb;
    if (lds > 163840 || a.nwalk % (2 * S * NW)) return hipErrorInvalidValue;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(a.nwalk / (2 * S * NW)), dim3(64 * NW), lds, st, a.Ju, a.seq,
                       a.pos, a.ld, a.L, a.q, a.nchunk, a.nsteps, a.k0, a.k1, a.step0,
                       a.walker_base, a.nbeta, nst);
    return hipGetLastError();
}

// Shape (slots x waves) by how many walkers a CU gets (us a step, three contexts
// at once / one alone):
//   up to 64 (32 for q > 4): 4 x 4, 32 walkers a work-group: L=93 q=4, 16384 walkers
//              0.54 / 1.0, 0.54 / 1.2 for 8 x 8, 1.2 / 3.7 chunk-staged; at q=8
//              0.97 / 1.5, so 8 x 8 there (0.67 / 1.5)
//   up to 128: 8 x 8: 32768 walkers 0.81 / 1.3, 0.96 / 2.1 for 16 x 8
//   beyond:    16 x 8 for up to two state words: 65536 walkers 1.43 / 2.3, 1.64 / 2.1
//              for 8 x 8; 2^18 alone 5.6 at L=93 and 13.4 at L=232, against 7.2 and
//              16.1 chunk-staged; 8 slots for longer chains (22.8 against 24.8 at
//              L=300)
// Two work-groups of 8 waves share a CU while their stages fit beside each
// other; longer rows take 16 waves.
template <int KW, int NPC>
hipError_t run_kw(const SweepArgs& a, hipStream_t st) {
    const bool wide = 4ull * a.nchunk * NPC * 1024 > 163840;
    if (a.nwalk <= (NPC == 2 ? 64 : 32) * a.ncu) return run_shape<KW, 4, 4, NPC>(a, st, 16);
    if constexpr (KW <= 2) {
        if (a.nwalk > 128 * a.ncu)
            return wide ? run_shape<KW, 16, 16, NPC>(a, st, 64) : run_shape<KW, 16, 8, NPC>(a, st, 32);
    }
    return wide ? run_shape<KW, 8, 16, NPC>(a, st, 64) : run_shape<KW, 8, 8, NPC>(a, st, 32);
}
}  // namespace

hipError_t launch_sweep_steps(const SweepArgs& a, hipStream_t st) {
    const uint32_t kw = state_words(a.L), kb = steps_slot_kb(a.q, a.nchunk);
#define MI3_SCASE(KW_, NPC_) \
    if (kw == KW_ && kb == NPC_) return run_kw<KW_, NPC_>(a, st);
    MI3_SCASE(1, 2) MI3_SCASE(2, 2) MI3_SCASE(3, 2) MI3_SCASE(4, 2)
    MI3_SCASE(5, 2) MI3_SCASE(6, 2) MI3_SCASE(7, 2) MI3_SCASE(8, 2)
    MI3_SCASE(1, 8) MI3_SCASE(2, 8)
#undef MI3_SCASE
    return hipErrorInvalidValue;
}

}  // namespace mi3
