// Instantiation and launch of the unstaged sweep (few walkers).
#include "k_potts.hip"
#include "launch.h"

#include <utility>

namespace mi3 {

namespace {
template <int NC>
hipError_t run_nc(const SweepArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((k_sweep_direct<NC, 1>), dim3(a.nwalk / 2), dim3(64), 0, st, a.Ju,
                       a.seq, a.pos, a.ld, a.L, a.q, chunk_floats(a.q) * 4, a.nsteps, a.k0, a.k1,
                       a.step0, a.walker_base, a.nbeta);
    return hipGetLastError();
}

template <int... I>
hipError_t run_any(const SweepArgs& a, hipStream_t st, std::integer_sequence<int, I...>) {
    hipError_t e = hipErrorInvalidValue;
    ((a.nchunk == (uint32_t)(I + 1) ? (void)(e = run_nc<I + 1>(a, st)) : (void)0), ...);
    return e;
}

template <int KW, int S>
hipError_t batch_kw(const BatchModel* models, const BatchTile* tiles, uint32_t ntiles,
                    uint32_t wpb, hipStream_t st) {
    const uint32_t waves = ntiles * (wpb / (2 * S));
    const uint32_t per = (waves + 7) / 8;
    hipLaunchKernelGGL((k_sweep_batch_direct<KW, S>), dim3(8 * per), dim3(64), 0, st, models, tiles,
                       wpb / (2 * S), waves, per);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_sweep_direct(const SweepArgs& a, hipStream_t st) {
    return run_any(a, st, std::make_integer_sequence<int, MAX_L / CH>{});
}

// Walkers of a half-wave in a batch: one while the card has idle CUs for them
// (a step of 512 or 2048 walkers takes 1.2 and 2.0 us at L=232 q=21, against
// 2.6 us with four), four beyond (4096 walkers: 3.4 us against 4.0); the narrow
// rows of q <= 8 favour one throughout (0.56 against 0.79 us at L=93 q=4, 4096
// walkers).
hipError_t launch_sweep_batch_direct(uint32_t kw, uint32_t q, uint32_t wpb, uint32_t nwalk,
                                     uint32_t ncu, const BatchModel* models,
                                     const BatchTile* tiles, uint32_t ntiles, hipStream_t st) {
    if (ntiles == 0) return hipSuccess;
    const bool one = q <= 8 || nwalk <= 8 * ncu;
#define MI3_DCASE(KW_)                                                          \
    if (kw == KW_) return one ? batch_kw<KW_, 1>(models, tiles, ntiles, wpb, st) \
                              : batch_kw<KW_, 4>(models, tiles, ntiles, wpb, st);
    MI3_DCASE(1) MI3_DCASE(2) MI3_DCASE(3) MI3_DCASE(4)
    MI3_DCASE(5) MI3_DCASE(6) MI3_DCASE(7) MI3_DCASE(8)
#undef MI3_DCASE
    return hipErrorInvalidValue;
}

}  // namespace mi3
