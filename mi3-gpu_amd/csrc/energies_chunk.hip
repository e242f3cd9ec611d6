// Instantiation and launch of the chunk-staged energies for MI3_KW state words
// (the build compiles this file once for each).
#include "k_potts.hip"
#include "launch.h"

namespace mi3 {

namespace {
template <int KW, int PF, int S, int NW>
hipError_t run_shape(const EnergyArgs& a, hipStream_t st) {
    constexpr uint32_t W = 2 * S * NW;
    // with four state words (L = 385..512), the 57 KB chunks of q = 17..21
    // stream through the overlapping four-slot ring (all 160 KB of LDS):
    // 7.10 against 7.94 ms at L=400, 10.7 against 11.8 ms at L=500.  The
    // others are double-buffered (the ring took 6% longer at L=300 and 1% at
    // L=232)
    constexpr bool OVL = PF == 7 && KW == 4 && NW == 16;
    auto kern = k_energies<KW, S, NW, PF, OVL>;
    const size_t lds = OVL ? (size_t)OverlapRing::BYTES : 2ull * chunk_floats(a.q) * sizeof(float);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((a.nseq + W - 1) / W), dim3(64 * NW), lds, st, a.Ju, a.seq, a.E,
                       a.ld, a.nseq, a.L, a.q, a.nchunk);
    return hipGetLastError();
}

// Sequences per work-group (2 x slots x waves): every staged chunk is read once
// per sequence, so a full card takes as many as registers hold (512; 256 beyond
// four state words; 2^18 sequences: 2.09 ms at L=232 q=21, 3.9 with 256, 7.7 with
// 128).
template <int KW, int PF>
hipError_t run_pf(const EnergyArgs& a, hipStream_t st) {
    const uint32_t w = chunk_tile(a.nseq, KW <= 4 ? 512 : 256, a.ncu);
    if constexpr (KW <= 4) {
        if (w == 512) return run_shape<KW, PF, 16, 16>(a, st);
        if (w == 256) return run_shape<KW, PF, 8, 16>(a, st);
        return run_shape<KW, PF, 8, 8>(a, st);
    } else {
        if (w == 256) return run_shape<KW, PF, 8, 16>(a, st);
        return run_shape<KW, PF, 4, 16>(a, st);
    }
}
}  // namespace

template <>
hipError_t launch_energies_chunks<MI3_KW>(const EnergyArgs& a, hipStream_t st) {
    // (up to 8 letters and two state words always take staged rows)
    if constexpr (MI3_KW > 2)
        if (pf_class(a.q) == 1) return run_pf<MI3_KW, 1>(a, st);
    switch (pf_class(a.q)) {
        case 4: return run_pf<MI3_KW, 4>(a, st);
        case 7: return run_pf<MI3_KW, 7>(a, st);
        case 10: return run_pf<MI3_KW, 10>(a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mi3
