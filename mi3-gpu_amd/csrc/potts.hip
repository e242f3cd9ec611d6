// Launch rule of the sweep; instantiation and launch of the energy kernels and
// of the staging probe.
#include "k_potts.hip"
#include "launch.h"

namespace mi3 {

namespace {
template <typename F>
hipError_t set_lds(F kernel, size_t bytes) {
    static_assert(sizeof(F) > 0, "");
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

}  // namespace

// Form of the sweep.  A tile asked for by size (128 or 256 walkers) runs
// chunk-staged; the default goes by what fills the card:
//   few walkers per CU: no staging at all (direct_walkers);
//   q <= 8 with rows of up to 64 KB: several steps' rows staged at once;
//   otherwise chunk by chunk.
hipError_t launch_sweep(const SweepArgs& a, hipStream_t st) {
    if (a.nwalk % SWEEP_WALKERS_PER_BLOCK || a.q > MAX_Q || a.L > MAX_L || a.L < 2 || a.ncu == 0)
        return hipErrorInvalidValue;
    if (a.wpb == 0 || a.wpb >= 512) {
        if (a.nwalk <= direct_walkers(a.q, a.ncu)) return launch_sweep_direct(a, st);
        if (steps_slot_kb(a.q, a.nchunk)) return launch_sweep_steps(a, st);
    }
    switch (state_words(a.L)) {
        case 1: return launch_sweep_chunks<1>(a, st);
        case 2: return launch_sweep_chunks<2>(a, st);
        case 3: return launch_sweep_chunks<3>(a, st);
        case 4: return launch_sweep_chunks<4>(a, st);
        case 5: return launch_sweep_chunks<5>(a, st);
        case 6: return launch_sweep_chunks<6>(a, st);
        case 7: return launch_sweep_chunks<7>(a, st);
        case 8: return launch_sweep_chunks<8>(a, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_sweep_batch(uint32_t kw, uint32_t pf, uint32_t wpb, const BatchModel* models,
                              const BatchTile* tiles, uint32_t ntiles, uint32_t* counter,
                              uint32_t grid, hipStream_t st) {
    if (grid == 0 || ntiles == 0) return hipSuccess;
    switch (kw) {
        case 1: return launch_sweep_batch_chunks<1>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 2: return launch_sweep_batch_chunks<2>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 3: return launch_sweep_batch_chunks<3>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 4: return launch_sweep_batch_chunks<4>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 5: return launch_sweep_batch_chunks<5>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 6: return launch_sweep_batch_chunks<6>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 7: return launch_sweep_batch_chunks<7>(pf, wpb, models, tiles, ntiles, counter, grid, st);
        case 8: return launch_sweep_batch_chunks<8>(pf, wpb, models, tiles, ntiles, counter, grid, st);
    }
    return hipErrorInvalidValue;
}

namespace {
template <int PF, int INF>
hipError_t stage_probe_pf(const SweepArgs& a, hipStream_t st) {
    constexpr int NW = 16;
    auto kern = k_stage_probe<PF, NW, INF>;
    size_t lds = 2ull * chunk_floats(a.q) * sizeof(float);
    hipError_t e = set_lds(kern, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(a.nwalk / 512), dim3(64 * NW), lds, st, a.Ju, a.pos, a.L,
                       a.nchunk, a.nsteps);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_stage_probe(const SweepArgs& a, int inflight, hipStream_t st) {
    if (a.nwalk % 512 || a.q > MAX_Q || a.L > MAX_L || a.L < 2) return hipErrorInvalidValue;
    const uint32_t pf = pf_class(a.q);
#define MI3_PCASE(PF_)                                                             \
    if (pf == PF_) return inflight == 2 ? stage_probe_pf<PF_, 2>(a, st)             \
                                        : stage_probe_pf<PF_, 1>(a, st);
    MI3_PCASE(1) MI3_PCASE(4) MI3_PCASE(7) MI3_PCASE(10)
#undef MI3_PCASE
    return hipErrorInvalidValue;
}

// Form of the energies, as of the sweep: unstaged for few sequences, the rows
// of a stage at once for q <= 8, otherwise chunk by chunk.
hipError_t launch_energies(const EnergyArgs& a, hipStream_t st) {
    if (a.q > MAX_Q || a.L > MAX_L || a.L < 2 || a.ncu == 0) return hipErrorInvalidValue;
    if (a.nseq == 0) return hipSuccess;
    if (a.nseq <= direct_sequences(a.q, a.ncu)) return launch_energies_direct(a, st);
    if (steps_slot_kb(a.q, a.nchunk)) return launch_energies_rows(a, st);
    switch (state_words(a.L)) {
        case 1: return launch_energies_chunks<1>(a, st);
        case 2: return launch_energies_chunks<2>(a, st);
        case 3: return launch_energies_chunks<3>(a, st);
        case 4: return launch_energies_chunks<4>(a, st);
        case 5: return launch_energies_chunks<5>(a, st);
        case 6: return launch_energies_chunks<6>(a, st);
        case 7: return launch_energies_chunks<7>(a, st);
        case 8: return launch_energies_chunks<8>(a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mi3
