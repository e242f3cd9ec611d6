// Instantiation and launch of the energies that stage whole rows (q <= 8) and
// of the unstaged ones (few sequences).
#include "k_potts.hip"
#include "launch.h"

#include <utility>

namespace mi3 {

namespace {
template <int KW, int S, int NW, int NPC>
hipError_t run_shape(const EnergyArgs& a, hipStream_t st, uint32_t stage_kb) {
    constexpr uint32_t W = 2 * S * NW;
    auto kern = k_energies_rows<KW, S, NW, NPC>;
    const uint32_t rowb = a.nchunk * NPC * 1024;
    const uint32_t nrow = stage_kb * 1024 > rowb ? stage_kb * 1024 / rowb : 1;
    const size_t lds = 2ull * nrow * rowb;
    if (lds > 163840) return hipErrorInvalidValue;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((a.nseq + W - 1) / W), dim3(64 * NW), lds, st, a.Ju, a.seq, a.E,
                       a.ld, a.nseq, a.L, a.q, a.nchunk, nrow);
    return hipGetLastError();
}

// Shape (slots x waves) by how many sequences a CU gets, as the sweep's (us,
// three contexts at once / one alone, q=4):
//   up to 32:  4 x 4: 8192 sequences of L=93 19 / 48, 23 / 57 for 8 x 8; 8 x 8 where a
//              row takes so much LDS that one work-group fills it (16384 sequences
//              of L=232 q=8 alone: 405 against 833)
//   up to 128: 8 x 8: 16384 sequences of L=93 24 / 57, 26 / 55 for 4 x 4; 32768 35 / 58,
//              36 / 86 for 16 x 8
//   up to 256 in rows of up to 32 KB of 8 KB chunks: 8 x 16: 46000 sequences of L=93 q=8
//              58 / 104, 58 / 114 for 16 x 8 (56 / 103 chunk-staged); 65536 75 / 106, 61 /
//              115 (75 / 109); L=128 q=7 116 / 159, 111 / 178 (114 / 168).  Longer rows 16 x 8
//              (65536 of L=150 q=8 168 / 274, 240 / 242 for 8 x 16)
//   beyond:    16 x 8 for up to two state words (65536 sequences of L=93 56 / 87, 69 / 80
//              for 8 x 8; 2^18 alone 276, of L=232 1253; chunk-staged 327 and 1649),
//              16 x 16 for wide rows (L=232 q=8: 1464 against 2249 alone); 8 x 16 for
//              longer chains (2^17 sequences of L=300: 1075, 1136 for 8 x 8)
template <int KW, int NPC>
hipError_t run_kw(const EnergyArgs& a, hipStream_t st) {
    const bool wide = 4ull * a.nchunk * NPC * 1024 > 163840;
    if (a.nseq <= 32 * a.ncu && !wide) return run_shape<KW, 4, 4, NPC>(a, st, 16);
    if (a.nseq <= 128 * a.ncu) return run_shape<KW, 8, 8, NPC>(a, st, 32);
    if constexpr (KW == 1 && NPC == 8)
        if (a.nseq <= 256 * a.ncu && a.nchunk <= 4) return run_shape<KW, 8, 16, NPC>(a, st, 32);
    if constexpr (KW <= 2)
        return wide ? run_shape<KW, 16, 16, NPC>(a, st, 64) : run_shape<KW, 16, 8, NPC>(a, st, 32);
    else
        return run_shape<KW, 8, 16, NPC>(a, st, 32);
}

template <int NC>
hipError_t run_nc(const EnergyArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(k_energies_direct<NC>, dim3((a.nseq + 1) / 2), dim3(64), 0, st, a.Ju, a.seq,
                       a.E, a.ld, a.nseq, a.L, a.q, chunk_floats(a.q) * 4);
    return hipGetLastError();
}

template <int... I>
hipError_t run_any(const EnergyArgs& a, hipStream_t st, std::integer_sequence<int, I...>) {
    hipError_t e = hipErrorInvalidValue;
    ((a.nchunk == (uint32_t)(I + 1) ? (void)(e = run_nc<I + 1>(a, st)) : (void)0), ...);
    return e;
}
}  // namespace

hipError_t launch_energies_rows(const EnergyArgs& a, hipStream_t st) {
    const uint32_t kw = state_words(a.L), kb = steps_slot_kb(a.q, a.nchunk);
#define MI3_SCASE(KW_, NPC_) \
    if (kw == KW_ && kb == NPC_) return run_kw<KW_, NPC_>(a, st);
    MI3_SCASE(1, 2) MI3_SCASE(2, 2) MI3_SCASE(3, 2) MI3_SCASE(4, 2)
    MI3_SCASE(5, 2) MI3_SCASE(6, 2) MI3_SCASE(7, 2) MI3_SCASE(8, 2)
    MI3_SCASE(1, 8) MI3_SCASE(2, 8)
#undef MI3_SCASE
    return hipErrorInvalidValue;
}

hipError_t launch_energies_direct(const EnergyArgs& a, hipStream_t st) {
    return run_any(a, st, std::make_integer_sequence<int, MAX_L / CH>{});
}

}  // namespace mi3
