// Host-side launchers shared between translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi3 {

struct SweepArgs {
    const float* Ju;  // chunked layout, chunk stride chunk_floats(q)
    uint8_t* seq;
    const uint32_t* pos;
    uint32_t ld, nwalk, L, q, nchunk, nsteps, k0, k1, walker_base;
    uint64_t step0;
    float nbeta;
    uint32_t wpb;  // walkers per work-group: 128, 256, or 512 / 0 (the library's choice)
    uint32_t ncu;  // compute units of the device
};

struct EnergyArgs {
    const float* Ju;
    const uint8_t* seq;
    float* E;
    uint32_t ld, nseq, L, q, nchunk;
    uint32_t ncu;  // compute units of the device
};

// The walker count must be a multiple of 512.
constexpr uint32_t SWEEP_WALKERS_PER_BLOCK = 512;

// Largest q / L the register-resident kernels are instantiated for.
constexpr uint32_t MAX_Q = 25;
constexpr uint32_t MAX_L = 1024;

// Threads per work-group of the sweep / energy kernels.
constexpr uint32_t POTTS_THREADS = 512;

// float4 loads per thread to stage one chunk of q*q*32 floats; the chunked
// coupling layout pads every chunk to POTTS_THREADS * pf_class(q) float4 so
// that staging needs no bounds checks.
__host__ __device__ inline uint32_t pf_class(uint32_t q) {
    uint32_t need = (q * q * 32 / 4 + POTTS_THREADS - 1) / POTTS_THREADS;
    if (need <= 1) return 1;
    if (need <= 4) return 4;
    if (need <= 7) return 7;
    return 10;
}

// Floats per (padded) chunk.
__host__ __device__ inline uint32_t chunk_floats(uint32_t q) { return pf_class(q) * POTTS_THREADS * 4; }

// The chunked couplings of an L-site model are addressed with 32-bit byte
// offsets (buffer resources): true when they fit.
inline bool chunked_fits(uint32_t L, uint32_t q) {
    const uint64_t nchunk = (L + 31) / 32;
    return (uint64_t)L * nchunk * chunk_floats(q) * 4 < (1ull << 32);
}

// One model of a batch, as the persistent sweep reads it (device memory).
struct BatchModel {
    const float* Ju;        // chunked couplings
    uint8_t* seq;           // site-major walkers, L rows of ld bytes
    const uint32_t* pos;    // site list of this launch
    const uint64_t* step;   // global step counter (even)
    uint32_t ld, L, q, nchunk, nsteps, k0, k1, walker_base;
    float nbeta;
    uint32_t pad_;
};

// A work-group tile of a batch: walkers [block*W, (block+1)*W) of `model`.
struct BatchTile {
    uint32_t model, block;
};

// Largest walker count that is swept without staging (sweep_direct).  Alone on
// the card it is the fastest form up to some 32 walkers a CU, but its time
// grows with the walkers from the start, and with the work of other streams
// beside it, where a staged tile leaves their CUs alone; the line lies where
// three contexts sweeping at once lose nothing either (us a step and context,
// three at once / one alone, unstaged against the staged form taken instead:
// L=93 q=21, 2048 walkers 0.95 / 0.77 against 0.95 / 2.7, 4096 1.9 / 1.3 against
// 0.95 / 2.7; L=232 q=21, 1024 walkers 2.1 / 1.2 against 2.5 / 7.0; L=93 q=4, 2048
// walkers 0.22 / 0.50 against 0.32 / 0.85, 4096 0.41 / 0.55 against 0.32 / 0.85).
inline uint32_t direct_walkers(uint32_t q, uint32_t ncu) { return (q <= 8 ? 12 : 6) * ncu; }

// Largest sequence count whose energies are taken without staging, by the same
// measure (us, three contexts at once / one alone: L=232 q=21, 1024 sequences 83 /
// 133, 2048 200-330 / 165 against 324 / 960, 4096 770 / 266 against 321 / 950; L=93
// q=4, 4096 sequences 13 / 18 against 18 / 48, 8192 27 / 32 against 19 / 48).
inline uint32_t direct_sequences(uint32_t q, uint32_t ncu) { return (q <= 8 ? 16 : 8) * ncu; }

// Sites that the energies of many sequences take together as one of q^k letters
// (1: none): a gather then adds k*k couplings, and the energies are bound by their
// gathers and what each takes to address.  Reduced alphabets only: the folded one has
// to stay within MAX_Q letters, and for q = 2 three sites (8 letters, whole rows
// staged) take as long as four at half the cost of their table.  The table is formed
// anew when the couplings change (15 us at L=93 q=4 against 8 without folding), so
// few sequences and short chains are left as they are.  us, unfolded / folded, table
// included: L=93 q=4, 2^18 sequences 247 / 160, 2^17 132 / 87, 2^16 90 / 85, 2^14
// 61 / 69; L=232 q=4, 2^18 1245 / 518, 2^16 454 / 270; L=93 q=2, 2^18 242 / 78; L=93
// q=5, 2^18 262 / 222; L=17 q=4, 2^18 35 / 32.  The error against 64 bits is about
// half (fewer additions).
inline uint32_t fold_width(uint32_t q) { return q == 2 ? 3 : q <= 5 ? 2 : 1; }
inline uint32_t fold_sites(uint32_t q, uint32_t L, uint32_t nseq, uint32_t ncu) {
    return L >= 32 && nseq > 256 * ncu ? fold_width(q) : 1;
}

// Walkers (or sequences) per work-group of the chunk-staged kernels, `most` or
// less: half as many take 0.7-0.97 of the time, on twice the CUs, so tiles are
// halved only while they occupy at most a quarter of the card.
inline uint32_t chunk_tile(uint32_t n, uint32_t most, uint32_t ncu) {
    uint32_t w = most;
    while (w > 128 && (n + w / 2 - 1) / (w / 2) <= ncu / 4) w /= 2;
    return w;
}

// LDS per chunk in the step-staged sweep, in KB (2 for q <= 4, 8 for q <= 8),
// or 0 where a row of couplings does not fit 64 KB and the form does not
// apply.
inline uint32_t steps_slot_kb(uint32_t q, uint32_t nchunk) {
    const uint32_t kb = q <= 4 ? 2 : 8;
    return q <= 8 && nchunk * kb <= 64 ? kb : 0;
}

// Returns a hipError_t; grid/LDS sizing done inside.
hipError_t launch_sweep_direct(const SweepArgs& a, hipStream_t st);
hipError_t launch_sweep_steps(const SweepArgs& a, hipStream_t st);
template <int KW>
hipError_t launch_sweep_chunks(const SweepArgs& a, hipStream_t st);
hipError_t launch_sweep(const SweepArgs& a, hipStream_t st);
hipError_t launch_energies_direct(const EnergyArgs& a, hipStream_t st);
hipError_t launch_energies_rows(const EnergyArgs& a, hipStream_t st);
template <int KW>
hipError_t launch_energies_chunks(const EnergyArgs& a, hipStream_t st);
hipError_t launch_energies(const EnergyArgs& a, hipStream_t st);

// The sweep's coupling-row staging alone (k_stage_probe) for the sites of
// a.pos, one work-group per 512 walkers; inflight 1 or 2 chunk copies.
hipError_t launch_stage_probe(const SweepArgs& a, int inflight, hipStream_t st);

// State words per lane (4 residues each) for L sites: ceil(L / 128).
inline uint32_t state_words(uint32_t L) { return (L + 127) / 128; }

// Persistent sweep over `ntiles` tiles of models that share state_words(L)
// == kw and pf_class(q) == pf, with `wpb` walkers per tile (128, 256 or 512),
// on `grid` work-groups.  `counter` (one u32) must be zero at launch.
hipError_t launch_sweep_batch(uint32_t kw, uint32_t pf, uint32_t wpb, const BatchModel* models,
                              const BatchTile* tiles, uint32_t ntiles, uint32_t* counter,
                              uint32_t grid, hipStream_t st);

template <int KW>
hipError_t launch_sweep_batch_chunks(uint32_t pf, uint32_t wpb, const BatchModel* models,
                                     const BatchTile* tiles, uint32_t ntiles, uint32_t* counter,
                                     uint32_t grid, hipStream_t st);

// The same without staging, for classes of few walkers (`nwalk` in all; q the
// smallest alphabet of the class).
hipError_t launch_sweep_batch_direct(uint32_t kw, uint32_t q, uint32_t wpb, uint32_t nwalk,
                                     uint32_t ncu, const BatchModel* models,
                                     const BatchTile* tiles, uint32_t ntiles, hipStream_t st);

// Chunked symmetric coupling layout from packed couplings (k_unpack_chunked).
hipError_t launch_unpack_chunked(const float* J, float* out, uint32_t L, uint32_t q,
                                 uint32_t nchunk, hipStream_t st);

#define MI3_DECL_KW(KW)                                                                       \
    template <>                                                                               \
    hipError_t launch_energies_chunks<KW>(const EnergyArgs& a, hipStream_t st);                \
    template <>                                                                               \
    hipError_t launch_sweep_chunks<KW>(const SweepArgs& a, hipStream_t st);                    \
    template <>                                                                               \
    hipError_t launch_sweep_batch_chunks<KW>(uint32_t pf, uint32_t wpb, const BatchModel* models, \
                                             const BatchTile* tiles, uint32_t ntiles,         \
                                             uint32_t* counter, uint32_t grid, hipStream_t st);
MI3_DECL_KW(1) MI3_DECL_KW(2) MI3_DECL_KW(3) MI3_DECL_KW(4)
MI3_DECL_KW(5) MI3_DECL_KW(6) MI3_DECL_KW(7) MI3_DECL_KW(8)
#undef MI3_DECL_KW

}  // namespace mi3
