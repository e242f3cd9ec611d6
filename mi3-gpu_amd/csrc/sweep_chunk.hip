// Instantiation and launch of the chunk-staged sweep for MI3_KW state words
// (the build compiles this file once for each).
#include "k_potts.hip"
#include "launch.h"

namespace mi3 {

namespace {
template <typename F>
hipError_t set_lds(F kernel, size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Launch shapes (walker slots per half-wave S, waves NW): W = 2*S*NW walkers
// per work-group.  16 waves of at most 128 registers (4 waves per SIMD) hide
// the gathers' latency better than 8 waves of 256, wherever the state fits:
// measured on MI355X at L=120/232/300/450, q=21 and q=4.
template <int KW, int PF, int S, int NW>
hipError_t sweep_kws(const SweepArgs& a, hipStream_t st) {
    constexpr uint32_t W = 2 * S * NW;
    auto kern = k_sweep<KW, S, NW, PF>;
    size_t lds = 2ull * chunk_floats(a.q) * sizeof(float);
    hipError_t e = set_lds(kern, lds);
    if (e != hipSuccess) return e;
    if (a.nwalk % W) return hipErrorInvalidValue;
    dim3 grid(a.nwalk / W);
    hipLaunchKernelGGL(kern, grid, dim3(64 * NW), lds, st, a.Ju, a.seq, a.pos, a.ld, a.L, a.q,
                       a.nchunk, a.nsteps, a.k0, a.k1, a.step0, a.walker_base, a.nbeta);
    return hipGetLastError();
}

template <int KW, int PF>
struct SweepDisp {
    static hipError_t run(const SweepArgs& a, hipStream_t st) {
        // 128 and 256 walkers as the caller asked; at the default by the rule
        // (a step of 128, 256 or 512 walkers: 7.0, 7.2 and 8.2 us at L=232 q=21, 2.7,
        // 2.9 and 3.8 us at L=93)
        const uint32_t w =
            (a.wpb == 128 || a.wpb == 256) ? a.wpb : chunk_tile(a.nwalk, 512, a.ncu);
        if constexpr (KW >= 5) {
            // five to eight state words: 8 slots at most fit in 128 registers
            if (w <= 128) return sweep_kws<KW, PF, 4, 16>(a, st);
            return sweep_kws<KW, PF, 8, 16>(a, st);
        } else {
            if (w <= 128) return sweep_kws<KW, PF, 8, 8>(a, st);
            if (w <= 256) return sweep_kws<KW, PF, 8, 16>(a, st);
            // four state words do not fit 16 slots in 128 registers; the
            // spills still pay for q > 8, not for the small chunks of q <= 8 (which
            // come here in tiles of 512 for three words and four alone)
            if constexpr (KW != 3 && PF == 1)
                return sweep_kws<KW, PF, 8, 16>(a, st);
            else
                return sweep_kws<KW, PF, 16, 16>(a, st);
        }
    }
};

template <int KW, int PF, int S, int NW>
hipError_t batch_kws(const BatchModel* models, const BatchTile* tiles, uint32_t ntiles,
                     uint32_t* counter, uint32_t grid, hipStream_t st) {
    auto kern = k_sweep_batch<KW, S, NW, PF>;
    size_t lds = 2ull * PF * POTTS_THREADS * 4 * sizeof(float);  // two padded chunks
    hipError_t e = set_lds(kern, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW), lds, st, models, tiles, ntiles, counter);
    return hipGetLastError();
}

template <int KW, int PF>
hipError_t batch_kw(uint32_t wpb, const BatchModel* models, const BatchTile* tiles,
                    uint32_t ntiles, uint32_t* counter, uint32_t grid, hipStream_t st) {
    if constexpr (KW >= 5) {
        if (wpb == 128) return batch_kws<KW, PF, 4, 16>(models, tiles, ntiles, counter, grid, st);
        if (wpb == 256) return batch_kws<KW, PF, 8, 16>(models, tiles, ntiles, counter, grid, st);
        return hipErrorInvalidValue;
    } else {
        if (wpb == 128) return batch_kws<KW, PF, 8, 8>(models, tiles, ntiles, counter, grid, st);
        if (wpb == 256) return batch_kws<KW, PF, 8, 16>(models, tiles, ntiles, counter, grid, st);
        if (wpb == 512) return batch_kws<KW, PF, 16, 16>(models, tiles, ntiles, counter, grid, st);
        return hipErrorInvalidValue;
    }
}
}  // namespace

template <>
hipError_t launch_sweep_chunks<MI3_KW>(const SweepArgs& a, hipStream_t st) {
    switch (pf_class(a.q)) {
        case 1: return SweepDisp<MI3_KW, 1>::run(a, st);
        case 4: return SweepDisp<MI3_KW, 4>::run(a, st);
        case 7: return SweepDisp<MI3_KW, 7>::run(a, st);
        case 10: return SweepDisp<MI3_KW, 10>::run(a, st);
    }
    return hipErrorInvalidValue;
}

template <>
hipError_t launch_sweep_batch_chunks<MI3_KW>(uint32_t pf, uint32_t wpb, const BatchModel* models,
                                             const BatchTile* tiles, uint32_t ntiles,
                                             uint32_t* counter, uint32_t grid, hipStream_t st) {
    switch (pf) {
        case 1: return batch_kw<MI3_KW, 1>(wpb, models, tiles, ntiles, counter, grid, st);
        case 4: return batch_kw<MI3_KW, 4>(wpb, models, tiles, ntiles, counter, grid, st);
        case 7: return batch_kw<MI3_KW, 7>(wpb, models, tiles, ntiles, counter, grid, st);
        case 10: return batch_kw<MI3_KW, 10>(wpb, models, tiles, ntiles, counter, grid, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mi3
