// Metropolis sweep and batch Potts energies for gfx950.
//
// Both kernels use one work distribution:
//   * a walker (or sequence) is owned by a half-wave: lane j (0..31) holds the
//     residues of sites m = j + 32k, k = 0..4*KW-1, packed 4 per u32 register,
//     for S walkers ("slots"); a wave therefore owns 2*S walkers and a
//     work-group of NWAVES waves owns W = 2*S*NWAVES walkers for the whole
//     launch (the walker state never leaves registers between site updates);
//   * couplings for one site i are streamed through LDS in chunks of 32
//     neighbour sites, laid out [a*q + c][32] so that the 32 lanes of a
//     half-wave (32 distinct neighbour sites) gather from 32 distinct banks
//     whatever residues their walkers hold;
//   * chunks are double-buffered in LDS: the next chunk is copied from global
//     memory straight into LDS (buffer_load ... lds) while the current one is
//     gathered, one barrier per chunk.
//
// Chunked coupling layout (built by k_unpack_chunked in k_misc.hip):
//   Ju[i][c][a*q + b][jl] = J_{i,m}(a, b),  m = 32c + jl,
// symmetric (both i<m and i>m filled), zero for m == i and m >= L.
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace mi3 {

// Native 4-float vector (HIP's float4 is a union-based struct, which keeps
// arrays of it out of registers).
typedef float f4v __attribute__((ext_vector_type(4)));

// w[idx] for a wave-uniform idx, as a select chain over registers.  The
// empty asm keeps the compiler from turning the chain back into a dynamic
// index (which would move the state array to scratch memory).
template <int KW>
__device__ __forceinline__ uint32_t select_word(const uint32_t (&w)[KW], uint32_t idx) {
    uint32_t r = w[0];
#pragma unroll
    for (int k = 1; k < KW; k++) {
        uint32_t t = w[k];
        asm volatile("" : "+v"(t));
        r = (idx == (uint32_t)k) ? t : r;
    }
    return r;
}

// Word k of a walker's packed state.  Static indices address registers
// directly; for KW >= 3 the (unrolled) index goes through the opaque select
// chain so the state array stays in registers.
template <int KW>
__device__ __forceinline__ uint32_t state_word(const uint32_t (&w)[KW], uint32_t k) {
    if constexpr (KW <= 2)
        return (KW == 1 || k == 0) ? w[0] : w[KW - 1];
    else
        return select_word<KW>(w, k);
}

constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x / 2); }

// Sweep gather schedule: slots per group and groups of reads in flight
// (8 and 1, 8 and 2, 4 and 2, 4 and 3, 16 and 1 time alike at L=232 q=21).
constexpr int SWEEP_G = 8;
constexpr int SWEEP_P = 1;

// Value of v in the partner lane of a reduction level below 16, within a
// row of 16 lanes, by DPP: m=8 row_ror:8 (lane ^ 8), m=4 row_half_mirror
// (lane ^ 7: the pair differs in bit 2, and in bits 0-1, which the later
// levels sum over anyway), m=2 and m=1 quad permutations (lane ^ 2, ^ 1).
__device__ __forceinline__ float dpp_partner(float v, int m) {
    const int x = __float_as_int(v);
    switch (m) {
        case 8: return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false));
        case 4: return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, false));
        case 2: return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false));
        default: return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false));
    }
}

// Reduce S per-lane partial sums over the 32 lanes of each half-wave at once
// (butterfly with operand exchange): afterwards lane j holds the full sum of
// slot j >> (5 - log2 S).  The first level pairs lanes j and j + 16: one
// v_permlane16_swap exchanges the odd 16-lane rows of v[s] with the even
// rows of v[s + h], so one add leaves rows 0 and 2 with slot s and rows 1
// and 3 with slot s + h, with no selects.  Each later level adds the partner
// lane's value to both slots of a pair (DPP inside the add) and keeps one of
// them by the lane's bit m.  No LDS, and no inline asm: the wait states that
// a DPP read needs after its source is written are inserted by the compiler
// only behind instructions it knows.
template <int S>
__device__ __forceinline__ float transposed_sum(float (&v)[S], uint32_t lane) {
    int n = S;
    if (n > 1) {
        const int h = n / 2;
#pragma unroll
        for (int s = 0; s < S / 2; s++) {
            if (s < h) {
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[s]),
                                                                __float_as_uint(v[s + h]), false,
                                                                false);
                v[s] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
            }
        }
        n = h;
    } else {
        // one slot: lane j ^ 16 through ds_swizzle
        v[0] += swz_xor<16>(v[0]);
    }
#pragma unroll
    for (int l = 1; l < 5; l++) {
        const int m = 16 >> l;
        if (n > 1) {
            const int h = n / 2;
#pragma unroll
            for (int s = 0; s < S / 2; s++) {
                if (s < h) {
                    const float x = v[s] + dpp_partner(v[s], m);
                    const float y = v[s + h] + dpp_partner(v[s + h], m);
                    v[s] = (lane & m) ? y : x;
                }
            }
            n = h;
        } else {
            v[0] += dpp_partner(v[0], m);
        }
    }
    return v[0];
}

// Buffer resource for raw buffer loads (gfx9 dword3 = 0x00020000): 32-bit
// offsets, so staging addresses need no 64-bit arithmetic.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                             0x00020000);
}

// Copy one padded chunk (PF * NT float4) from global memory straight into
// LDS with buffer_load ... lds: lane l of wave w moves float4 number
// k*NT + 64*w + l; the hardware writes the 64 float4 of a wave contiguously
// at the wave-uniform LDS address.  No registers hold the data in flight;
// completion is awaited with s_waitcnt vmcnt(0) before the next barrier.
typedef __attribute__((address_space(3))) void lds_void;

template <int PF, int NT>
__device__ __forceinline__ void chunk_dma(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff,
                                          char* lds_buf, int wave) {
#pragma unroll
    for (int k = 0; k < PF; k++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            r, (lds_void*)(lds_buf + (k * NT + wave * 64) * 16), 16, voff, soff + k * NT * 16, 0,
            0);
}

// s_waitcnt vmcnt(0) (expcnt, lgkmcnt left at their maxima): every
// vector-memory operation of this wave, including LDS DMA, has completed.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// s_waitcnt vmcnt(N): at most N vector-memory operations of this wave are
// still in flight (gfx9 encoding: vmcnt bits 3:0 and 15:14).  Loads complete
// in issue order, so all but the youngest N have landed.
template <int N>
__device__ __forceinline__ void wait_vmem_upto() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Work-group barrier that leaves LDS DMA in flight.  __syncthreads() waits
// for vmcnt(0) (its workgroup release fence covers LDS DMA writes), which
// drains every copy issued ahead; here only this wave's LDS and scalar loads
// are awaited (lgkmcnt(0) as a builtin, so that the compiler's own wait
// tracking sees them complete), then s_barrier, whose memory clobber keeps
// memory accesses on their side.
__device__ __forceinline__ void barrier_copies_in_flight() {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_barrier" ::: "memory");
}

// ---------------------------------------------------------------------------
// Chunk ring with overlapping slots, for the 57,344-byte padded chunks of
// q = 17..21 (7 float4 per thread of 512 staging threads).  Two such chunks
// fill 112 KB of the 160 KB of LDS, and three do not fit, so a plain ring can
// only double-buffer: the copy of chunk n+1 starts when chunk n-1 has been
// read and must land within the gathers of chunk n.  Here four slots
// X0..X3 (chunk n in X[n mod 4]) overlap in pairs two apart, X0/X2 and
// X1/X3, by 32 KB:
//   X0 = [0, 56K)   X2 = [24K, 80K)   X1 = [80K, 136K)   X3 = [104K, 160K)
// (K = 1024 bytes); slots one apart are disjoint.  A chunk's copy is split
// into its part outside the partner slot (24 KB, "early") and its part
// inside it (32 KB, "late"):
//   * early(n+2) is issued at the start of chunk n: it overlaps none of the
//     slots of chunks n and n+1;
//   * late(n+1) is issued at the start of chunk n: it overlaps only the slot
//     of chunk n-1, which every wave finished reading before the barrier
//     that started chunk n.
// So a chunk's copy has two chunks' time for 24 KB and one for 32 KB
// (double buffering gives one for all 56 KB), and LDS reads never meet a
// copy in flight.  The energy kernel streams the q = 17..21 chunks of its
// four-state-word shape this way (for fewer state words, and in the sweep,
// which is bound by VALU issue and LDS traffic, the ring was slower).  Per chunk each of the 8 staging waves issues 4 late then
// 3 early one-KB copies; at the end of chunk n only early(n+2), the 3
// youngest, may still be in flight (vmcnt 3), and the barrier that follows
// must not wait for it (barrier_copies_in_flight).
struct OverlapRing {
    static constexpr uint32_t PIECE = 1024;   // one wave's copy: 64 x 16 bytes
    static constexpr uint32_t CHB = 57344;    // padded chunk: 56 pieces
    static constexpr int EARLY_OPS = 3, LATE_OPS = 4;  // per staging wave
    static constexpr uint32_t BYTES = 163840;
    // slot base (0, 80K, 24K, 104K for r = 0..3), first piece of the late
    // part (the upper 32 pieces of X0 and X1, the lower 32 of X2 and X3) and
    // of the early part, as arithmetic on r (scalar, no branches)
    __device__ static uint32_t base(uint32_t r) { return (r & 1u) * 81920u + (r >> 1) * 24576u; }
    __device__ static uint32_t late_first(uint32_t r) { return 24u - (r >> 1) * 24u; }
    __device__ static uint32_t early_first(uint32_t r) { return (r >> 1) * 32u; }

    // copy `nops` pieces starting at piece `first` of the chunk at byte
    // offset `off` of the chunked layout into ring slot r; wave w < 8 moves
    // pieces first + 8*o + w
    template <int NOPS>
    __device__ static void copy(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t off,
                                char* lds, uint32_t r, uint32_t first, int wave) {
        char* dst = lds + base(r) + (first + wave) * PIECE;
        const uint32_t src = off + first * PIECE;
#pragma unroll
        for (int o = 0; o < NOPS; o++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(dst + o * 8 * PIECE), 16, voff,
                                                     src + o * 8 * PIECE, 0, 0);
    }
};
static_assert(OverlapRing::CHB == 7 * 512 * 16, "padded chunk of the PF = 7 class");
static_assert(OverlapRing::BYTES == 106496 + OverlapRing::CHB, "slots fill the LDS");

// 128 * byte e of w (e a compile-time constant after unrolling) in one
// VALU op: a shift with an SDWA byte select on its source.  Left to itself
// the compiler makes byte 0 a shift and a mask.
__device__ __forceinline__ uint32_t byte_x128(uint32_t w, int e) {
    uint32_t r;
    switch (e) {
        case 0:
            asm("v_lshlrev_b32_sdwa %0, 7, %1 dst_sel:DWORD dst_unused:UNUSED_PAD "
                "src0_sel:DWORD src1_sel:BYTE_0" : "=v"(r) : "v"(w));
            break;
        case 1:
            asm("v_lshlrev_b32_sdwa %0, 7, %1 dst_sel:DWORD dst_unused:UNUSED_PAD "
                "src0_sel:DWORD src1_sel:BYTE_1" : "=v"(r) : "v"(w));
            break;
        case 2:
            asm("v_lshlrev_b32_sdwa %0, 7, %1 dst_sel:DWORD dst_unused:UNUSED_PAD "
                "src0_sel:DWORD src1_sel:BYTE_2" : "=v"(r) : "v"(w));
            break;
        default:
            asm("v_lshlrev_b32_sdwa %0, 7, %1 dst_sel:DWORD dst_unused:UNUSED_PAD "
                "src0_sel:DWORD src1_sel:BYTE_3" : "=v"(r) : "v"(w));
            break;
    }
    return r;
}

// ---------------------------------------------------------------------------
// Metropolis sweep: nsteps single-site updates per walker.
//
// Step t of the launch is global step g = step0 + t (step0 even).  All
// walkers update the same site pos_list[t].  Walker w proposes residue
// b = mulhi(x, q) and accepts iff exp(-beta*dE) > (y >> 8) * 2^-24, where
// (x, y) are words (0,1) or (2,3) of Philox(key, (g>>1, w, TAG_WALK)) for
// even or odd g.  dE = sum_{m != pos} J_{pos,m}(b, s_m) - J_{pos,m}(a, s_m).
// Restates metropolis/DeltaEnergy (mcmc.cl:360-458) with counter-based
// streams in place of MWC64X.
//
// Per step: lane j draws the random numbers of walker slot j >> SH; every
// lane then needs, for every slot, the walker's current residue a (held by
// the lane owning site pos) and proposal b, gathers J(a, s_m) and J(b, s_m)
// for its sites chunk by chunk, and one transposed butterfly leaves each lane
// with the dE of its own slot; it decides, and the owner lane of pos takes the
// accepted residues.  Three forms share this step and differ in where the
// gathers read (all give the same sums in the same order, bit for bit):
//   sweep_block    chunks staged in LDS one at a time, one barrier per chunk:
//                  rows of couplings too large to hold (q > 8, long chains)
//   sweep_steps    the whole rows of several steps staged at once, one
//                  barrier per stage: small alphabets
//   sweep_direct   no staging, one wave per work-group gathering from L2:
//                  too few walkers to pay for a staged row

// Value of v in lane e of each row of 16 lanes (DPP row_newbcast).
#define MI3_RB_CASE(E) \
    case E:            \
        return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + E, 0xF, 0xF, false);
__device__ __forceinline__ uint32_t row_bcast(uint32_t v, int e) {
    switch (e) {
        MI3_RB_CASE(0) MI3_RB_CASE(1) MI3_RB_CASE(2) MI3_RB_CASE(3) MI3_RB_CASE(4)
        MI3_RB_CASE(5) MI3_RB_CASE(6) MI3_RB_CASE(7) MI3_RB_CASE(8) MI3_RB_CASE(9)
        MI3_RB_CASE(10) MI3_RB_CASE(11) MI3_RB_CASE(12) MI3_RB_CASE(13) MI3_RB_CASE(14)
        default: return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x15F, 0xF, 0xF, false);
    }
}
#undef MI3_RB_CASE

// Byte permute as asm, for stores to the state word that holds a site: the
// compiler merges branches on that word, if they hold plain instructions, into
// one access with a variable index, which moves the state to scratch memory
// (L=301 q=4 unstaged: 11 us a step against 0.8).
__device__ __forceinline__ uint32_t perm_apart(uint32_t hi, uint32_t lo, uint32_t sel) {
    uint32_t r;
    asm("v_perm_b32 %0, %1, %2, %3" : "=v"(r) : "v"(hi), "v"(lo), "v"(sel));
    return r;
}

// The walkers of a wave and what a step does with them around its gathers.
// QB: q <= 16, so that a residue times q fits a byte and four are multiplied at
// once; bytes are cut to four bits as they are loaded, so that one that is no
// residue does not reach its neighbours (cut at each step: 1% of a sweep).
template <int KW, int S, bool QB>
struct Walkers {
    static constexpr int SH = 5 - ilog2(S);  // lane j reduces and decides slot j >> SH
    // lanes of a quad that decide the same slot: each draws another pair of steps
    static constexpr int R = S == 16 ? 2 : 4;
    static_assert((1 << ilog2(S)) == S && S <= 16, "S must be a power of two <= 16");

    static constexpr uint32_t LETTER = QB ? 0x0f0f0f0fu : ~0u;
    static constexpr int NP = (S + 3) / 4;   // residues of a site, four slots to a word

    uint32_t st[S][KW];       // residues of sites j + 32k, four to a word
    // this step's current residues, byte s % 4 of word s / 4, kept for its end;
    // fetched again there where the state leaves no registers for them
    static constexpr bool KEEP = KW * S <= 48;
    uint32_t kept[KEEP ? NP : 1];
    uint32_t Xe, Xo;          // this lane's draws (steps 2h, 2h+1 of its own pair)
    int remap;                // bpermute address: row lane e <- the lane deciding slot e

    // A lane's S walkers are neighbours in a row of the sequence buffer: where
    // rows are aligned for it, one S-byte load per site fetches all of them (the
    // byte loads, S times as many, took a fifth of the energies' time at L=93
    // q=4), and byte permutes turn four sites' loads into S words.
    static constexpr bool WIDE = S >= 4;
    __device__ static __forceinline__ bool rows_aligned(const uint8_t* seq, uint32_t ldseq) {
        return (((uint32_t)(uintptr_t)seq | ldseq) & (S - 1)) == 0;
    }
    // 4 x 4 bytes transposed: word i holds byte i of a, b, c, d (and back)
    __device__ static __forceinline__ void transpose4(uint32_t& a, uint32_t& b, uint32_t& c,
                                                      uint32_t& d) {
        const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u);
        const uint32_t ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
        const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u);
        const uint32_t cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
        a = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
        b = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
        c = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
        d = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
    }

    // (walkers from `end` on read as residue 0)
    __device__ __forceinline__ void load(const uint8_t* seq, uint32_t ldseq, uint32_t L,
                                         uint32_t wfirst, uint32_t lane,
                                         uint32_t end = 0xffffffffu) {
        const uint32_t j = lane & 31;
        remap = (int)((((lane & 15) << SH) & 31) | (lane & 32)) * 4;
        Xe = Xo = 0;
        if constexpr (WIDE) {
            if (rows_aligned(seq, ldseq)) {
                typedef uint32_t wv __attribute__((ext_vector_type(S / 4)));
#pragma unroll
                for (int i = 0; i < KW; i++) {
                    uint32_t v[4][S / 4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t m = j + CH * (4 * i + e);
                        wv x = (wv)0u;
                        if (m < L && wfirst < end)
                            x = *reinterpret_cast<const wv*>(seq + (size_t)m * ldseq + wfirst);
#pragma unroll
                        for (int d = 0; d < S / 4; d++) v[e][d] = x[d];
                    }
#pragma unroll
                    for (int d = 0; d < S / 4; d++) {
                        transpose4(v[0][d], v[1][d], v[2][d], v[3][d]);
#pragma unroll
                        for (int g = 0; g < 4; g++)
                            st[4 * d + g][i] = wfirst + 4 * d + g < end ? v[g][d] & LETTER : 0u;
                    }
                }
                return;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
            const bool valid = wfirst + s < end;
#pragma unroll
            for (int i = 0; i < KW; i++) {
                uint32_t word = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t m = j + CH * (4 * i + e);
                    uint32_t v = (valid && m < L) ? seq[(size_t)m * ldseq + wfirst + s] : 0u;
                    word |= v << (8 * e);
                }
                st[s][i] = word & LETTER;
            }
            asm volatile("" ::: "memory");
        }
    }

    __device__ __forceinline__ void store(uint8_t* seq, uint32_t ldseq, uint32_t L,
                                          uint32_t wfirst, uint32_t lane) const {
        const uint32_t j = lane & 31;
        if constexpr (WIDE) {
            if (rows_aligned(seq, ldseq)) {
                typedef uint32_t wv __attribute__((ext_vector_type(S / 4)));
#pragma unroll
                for (int i = 0; i < KW; i++) {
                    uint32_t v[4][S / 4];
#pragma unroll
                    for (int d = 0; d < S / 4; d++) {
#pragma unroll
                        for (int g = 0; g < 4; g++) v[g][d] = st[4 * d + g][i];
                        transpose4(v[0][d], v[1][d], v[2][d], v[3][d]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t m = j + CH * (4 * i + e);
                        wv x;
#pragma unroll
                        for (int d = 0; d < S / 4; d++) x[d] = v[e][d];
                        if (m < L) *reinterpret_cast<wv*>(seq + (size_t)m * ldseq + wfirst) = x;
                    }
                }
                return;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
#pragma unroll
            for (int i = 0; i < KW; i++) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t m = j + CH * (4 * i + e);
                    if (m < L) seq[(size_t)m * ldseq + wfirst + s] = (uint8_t)(st[s][i] >> (8 * e));
                }
            }
        }
    }

    // Draw of step t of the launch (step0 even).  The lanes deciding one slot
    // share the work: lane i of R draws the steps 2(h + i), 2(h + i) + 1 every
    // R pairs of steps, and a quad permutation hands each out.
    __device__ __forceinline__ uint32_t draws(uint32_t t, uint64_t step0, uint32_t walker,
                                              uint32_t lane, uint32_t q, uint32_t k0,
                                              uint32_t k1) {
        const uint32_t i = (t >> 1) & (R - 1);
        if ((t & 1) == 0 && i == 0) {
            const uint64_t h = ((step0 + t) >> 1) + (lane & (R - 1));
            uint4 r = philox4x32_10(make_uint4((uint32_t)h, (uint32_t)(h >> 32), walker, TAG_WALK),
                                    k0, k1);
            Xe = ((r.y >> 8) << 8) | mulhi_range(r.x, q);
            Xo = ((r.w >> 8) << 8) | mulhi_range(r.z, q);
        }
        const int x = (int)((t & 1) ? Xo : Xe);
        int p;
        if constexpr (R == 2) {
            if (i == 0) p = __builtin_amdgcn_mov_dpp(x, 0xA0, 0xF, 0xF, false);    // quad 0,0,2,2
            else p = __builtin_amdgcn_mov_dpp(x, 0xF5, 0xF, 0xF, false);           // quad 1,1,3,3
        } else {
            if (i == 0) p = __builtin_amdgcn_mov_dpp(x, 0x00, 0xF, 0xF, false);
            else if (i == 1) p = __builtin_amdgcn_mov_dpp(x, 0x55, 0xF, 0xF, false);
            else if (i == 2) p = __builtin_amdgcn_mov_dpp(x, 0xAA, 0xF, 0xF, false);
            else p = __builtin_amdgcn_mov_dpp(x, 0xFF, 0xF, 0xF, false);
        }
        return (uint32_t)p;
    }

    // Current residues of every slot at site pos, in every lane: four slots to
    // a word, so one ds_bpermute from the owner lane serves four.
    __device__ __forceinline__ void residues(uint32_t pos, uint32_t lane,
                                             uint32_t (&apk)[NP]) const {
        const uint32_t kp = pos >> 5, owner = pos & 31;
        const uint32_t wd = kp >> 2, e0 = kp & 3;
        const int own_addr = (int)((owner + (lane & 32)) * 4);
#pragma unroll
        for (int g = 0; g < NP; g++) {
            uint32_t w[S < 4 ? S : 4];
#pragma unroll
            for (int e = 0; e < (S < 4 ? S : 4); e++) w[e] = select_word<KW>(st[4 * g + e], wd);
            uint32_t p;
            if constexpr (S == 1)
                p = __builtin_amdgcn_ubfe(w[0], e0 * 8, 8);
            else
                p = __builtin_amdgcn_perm(w[1], w[0], 0x0c0c0400u + e0 * 0x00000101u);
            if constexpr (S >= 4)
                p |= __builtin_amdgcn_perm(w[3], w[2], 0x04000c0cu + e0 * 0x01010000u);
            apk[g] = p;
        }
#pragma unroll
        for (int g = 0; g < NP; g++)
            apk[g] = (uint32_t)__builtin_amdgcn_ds_bpermute(own_addr, (int)apk[g]);
    }

    // Row addresses of every slot: baseA, baseB = (a, b) * q * 128 + origin
    // (origin: this lane's column, plus where the couplings of the site
    // start).  The proposals move to row lane s once, and each slot's is
    // broadcast by DPP inside the add.  (A ds_bpermute takes the LDS 2.5 times
    // as long as a gather; before, every slot took one, and two swizzles.)
    __device__ __forceinline__ void bases(uint32_t pos, uint32_t lane, uint32_t bmine, uint32_t q,
                                          uint32_t origin, uint32_t (&baseA)[S],
                                          uint32_t (&baseB)[S]) {
        // (opaque, so that the compiler does not turn the adds of disjoint bit
        // ranges below into ors, which do not fuse with the products)
        uint32_t org = origin;
        asm("" : "+v"(org));
        const uint32_t bl = (uint32_t)__builtin_amdgcn_ds_bpermute(remap, (int)bmine);
        uint32_t apk[NP];
        residues(pos, lane, apk);
        if constexpr (KEEP) {
#pragma unroll
            for (int g = 0; g < NP; g++) kept[g] = apk[g];
        }
        const uint32_t brow = __umul24(bl, q * (CH * 4));
#pragma unroll
        for (int s = 0; s < S; s++) baseB[s] = row_bcast(brow, s) + org;
#pragma unroll
        for (int g = 0; g < NP; g++) {
            const uint32_t aq = QB ? apk[g] * q : apk[g];
#pragma unroll
            for (int s = 4 * g; s < 4 * g + 4 && s < S; s++)
                baseA[s] = QB ? byte_x128(aq, s & 3) + org : __umul24(byte_x128(aq, s & 3), q) + org;
        }
    }

    // Row addresses a * q * 128 + origin of every slot's residue at site pos.
    __device__ __forceinline__ void row_bases(uint32_t pos, uint32_t lane, uint32_t q,
                                              uint32_t origin, uint32_t (&base)[S]) const {
        uint32_t org = origin;
        asm("" : "+v"(org));   // as in bases()
        uint32_t apk[NP];
        residues(pos, lane, apk);
#pragma unroll
        for (int s = 0; s < S; s++) {
            if constexpr (QB) {
                if (s % 4 == 0) apk[s / 4] *= q;
                base[s] = byte_x128(apk[s / 4], s & 3) + org;
            } else {
                base[s] = __umul24(byte_x128(apk[s / 4], s & 3), q) + org;
            }
        }
    }

    // LDS or memory addresses of a slot's gathers from chunk k
    __device__ __forceinline__ void gather_addr(int s, int k, uint32_t baseA, uint32_t baseB,
                                                uint32_t& aA, uint32_t& aB) const {
        const uint32_t off = byte_x128(st[s][k >> 2], k & 3);
        aA = baseA + off;
        aB = baseB + off;
    }

    // Accept or reject: this lane decides for its slot, and the owner lanes
    // of pos take every slot's residue, the proposal or the current one.
    // Residues and decisions reach them as packed bytes, so a slot costs one
    // byte permute there, with no lane mask of its own.
    __device__ __forceinline__ void accept(uint32_t pos, uint32_t lane, float (&acc)[S],
                                           uint32_t Pcur, float nbeta) {
        const uint32_t kp = pos >> 5, owner = pos & 31;
        const uint32_t wd = kp >> 2, e0 = kp & 3;
        const float dE = transposed_sum<S>(acc, lane);
        const float u = (float)(Pcur >> 8) * 0x1.0p-24f;
        // byte 0 the proposal, byte 1 all ones where it is accepted
        uint32_t v = (Pcur & 0xffu) | (__expf(nbeta * dE) > u ? 0xff00u : 0u);
        v = (uint32_t)__builtin_amdgcn_ds_bpermute(remap, (int)v);
        // row lane 4g: the four slots' proposals and masks
        const uint32_t y =
            (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xF5, 0xF, 0xF, false);  // quad 1,1,3,3
        const uint32_t z = __builtin_amdgcn_perm(y, v, 0x05010400u);
        const uint32_t y2 =
            (uint32_t)__builtin_amdgcn_mov_dpp((int)z, 0xAA, 0xF, 0xF, false);  // quad 2,2,2,2
        const uint32_t bp = __builtin_amdgcn_perm(y2, z, 0x05040100u);
        const uint32_t mp = __builtin_amdgcn_perm(y2, z, 0x07060302u);
        uint32_t npk[NP];
        if constexpr (KEEP) {
#pragma unroll
            for (int g = 0; g < NP; g++) npk[g] = kept[g];
        } else {
            residues(pos, lane, npk);
        }
#pragma unroll
        for (int g = 0; g < NP; g++) {
            const uint32_t m = row_bcast(mp, 4 * g);
            npk[g] = (row_bcast(bp, 4 * g) & m) | (npk[g] & ~m);
        }
        // owner lanes put byte e of the new residues at pos's byte; the
        // others keep their word
        const bool own = (lane & 31) == owner;
        const uint32_t keep = 0x07060504u & ~(0xffu << (8 * e0));
        uint32_t sel[S < 4 ? S : 4];
#pragma unroll
        for (int e = 0; e < (S < 4 ? S : 4); e++)
            sel[e] = own ? keep | ((uint32_t)e << (8 * e0)) : 0x07060504u;
#pragma unroll
        for (int i = 0; i < KW; i++) {
            if (KW == 1 || wd == (uint32_t)i) {
#pragma unroll
                for (int s = 0; s < S; s++)
                    st[s][i] = perm_apart(st[s][i], npk[s / 4], sel[s & 3]);
            }
        }
    }
};

// sweep_block runs the walkers of work-group tile `block` (W = 2*S*NWAVES
// walkers starting at walker block*W); k_sweep is one tile per work-group,
// k_sweep_batch a persistent loop over the tiles of many models.
template <int KW, int S, int NWAVES, int PF>
__device__ __forceinline__ void sweep_block(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t nchunk, uint32_t nsteps, uint32_t k0,
    uint32_t k1, uint64_t step0, uint32_t walker_base, float nbeta, uint32_t block) {
    constexpr int NT = 64 * NWAVES;
    constexpr int K = 4 * KW;
    using W = Walkers<KW, S, (PF <= 4)>;
    extern __shared__ f4v lds4[];
    char* ldsb = reinterpret_cast<char*>(lds4);

    // the padded chunk is PF float4 per thread of the first DMA_T threads
    // (the chunk layout's unit); waves beyond them take no part in staging
    constexpr int DMA_T = NT < 512 ? NT : 512;
    constexpr uint32_t chb = PF * DMA_T * 16;  // padded chunk (bytes)
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wfirst = block * (2 * S * NWAVES) + (wave * 2 + (lane >> 5)) * S;
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * nchunk * chb);
    const uint32_t voff = tid * 16;
    // staging waves: each copies one float4 per lane per pass; a single-pass
    // chunk (PF = 1, q <= 8) needs only the first ceil(q*q/8) waves, whose
    // 1 KB pieces hold its q*q*32 floats (the rest is padding nobody reads:
    // 3-4% faster at q = 3..4 than copying all 8 KB)
    const bool stage = (PF == 1) ? (uint32_t)wave < (q * q + 7) / 8 : wave < DMA_T / 64;

    W w;
    w.load(seq, ldseq, L, wfirst, lane);
    uint32_t baseA[S], baseB[S];  // LDS byte offsets of rows a and b (+ lane column)
    float acc[S];

    if (nsteps == 0) return;
    // site of the current step; the next one is read one step ahead (with
    // the prefetch of its first chunk), so no step waits on a scalar load
    // (readfirstlane: the site is wave-uniform whatever the compiler can prove
    // about the list's memory, so masks built from it stay in SGPRs)
    uint32_t pos = __builtin_amdgcn_readfirstlane(pos_list[0]);
    uint32_t pos_next = nsteps > 1 ? __builtin_amdgcn_readfirstlane(pos_list[1]) : 0u;
    if (stage) chunk_dma<PF, DMA_T>(rJ, voff, pos * nchunk * chb, ldsb, wave);
    wait_vmem();
    __syncthreads();
    const uint32_t j4 = j * 4;

    // one step whose chunk 0 is in buffer b0: chunk k is in buffer (b0 + k) % 2.
    // For up to two state words the step is compiled for either b0, so that
    // the buffer is a constant offset of each read and an address one plain
    // add (half the time of a three-operand one); two copies of the longer
    // steps spill registers.
    constexpr bool TWICE = KW <= 2;
    auto step = [&](auto b0c, uint32_t b0v, uint32_t t) __attribute__((always_inline)) {
        const uint32_t b0 = TWICE ? decltype(b0c)::value : b0v;
        const uint32_t pos_after =
            (t + 2 < nsteps) ? __builtin_amdgcn_readfirstlane(pos_list[t + 2]) : 0u;
        const uint32_t Pcur =
            w.draws(t, step0, walker_base + wfirst + (j >> W::SH), lane, q, k0, k1);
        w.bases(pos, lane, Pcur & 0xffu, q, j4, baseA, baseB);
        // stream the couplings of site pos, chunk by chunk
#pragma unroll
        for (int k = 0; k < K; k++) {
            // (chunk 0 always exists: nchunk >= 1)
            if (k == 0 || (uint32_t)k < nchunk) {
                const bool last_chunk = (uint32_t)k + 1 == nchunk;
                const bool has_next = !last_chunk || (t + 1 < nsteps);
                const uint32_t buf = (b0 + k) & 1;
                if (has_next) {
                    uint32_t npos = last_chunk ? pos_next : pos;
                    uint32_t nc = last_chunk ? 0u : (uint32_t)k + 1;
                    if (stage)
                        chunk_dma<PF, DMA_T>(rJ, voff, (npos * nchunk + nc) * chb,
                                             ldsb + (buf ^ 1) * chb, wave);
                }
                const char* cb = ldsb + buf * chb;
                // gathers in groups of G slots, P groups in flight: the reads
                // of group i are issued before the sums of group i - P + 1,
                // and scheduling barriers keep the compiler from interleaving
                // them slot by slot (which exposes the LDS latency per slot)
                constexpr int G = (S < SWEEP_G) ? S : SWEEP_G;
                constexpr int NG = S / G;
                constexpr int P = (NG < SWEEP_P) ? NG : SWEEP_P;
                float vA[S], vB[S];
#pragma unroll
                for (int i = 0; i < NG + P - 1; i++) {
                    if (i < NG) {
#pragma unroll
                        for (int g = 0; g < G; g++) {
                            const int s = i * G + g;
                            static_assert(CH * 4 == 128, "row stride of a chunk");
                            uint32_t aA, aB;
                            w.gather_addr(s, k, baseA[s], baseB[s], aA, aB);
                            vA[s] = *reinterpret_cast<const float*>(cb + aA);
                            vB[s] = *reinterpret_cast<const float*>(cb + aB);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (i >= P - 1) {
#pragma unroll
                        for (int g = 0; g < G; g++) {
                            const int s = (i - P + 1) * G + g;
                            // the first chunk starts the sums
                            if (k == 0) acc[s] = vB[s] - vA[s];
                            else acc[s] += vB[s] - vA[s];
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                wait_vmem();
                __syncthreads();
            }
        }
        w.accept(pos, lane, acc, Pcur, nbeta);
        pos = pos_next;
        pos_next = pos_after;
    };
    uint32_t b0 = 0;
    const uint32_t flip = nchunk & 1;
    for (uint32_t t = 0; t < nsteps; t++) {
        if (TWICE && b0) step(std::integral_constant<uint32_t, 1>{}, b0, t);
        else step(std::integral_constant<uint32_t, 0>{}, b0, t);
        b0 ^= flip;
    }
    w.store(seq, ldseq, L, wfirst, lane);
}

// The whole rows of several steps staged at once: a stage holds `nst` steps
// (nst * nchunk chunks of NPC KB, of which the first ceil(q*q/8) KB are
// copied), double-buffered, one barrier per stage.  Inside a stage no wave
// waits for another, so the latencies of one wave's reduction and acceptance
// overlap the gathers of the others.
template <int KW, int S, int NWAVES, int NPC>
__device__ __forceinline__ void sweep_steps(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t nchunk, uint32_t nsteps, uint32_t k0,
    uint32_t k1, uint64_t step0, uint32_t walker_base, float nbeta, uint32_t block, uint32_t nst) {
    constexpr int K = 4 * KW;
    constexpr uint32_t SLOT = NPC * 1024;     // a chunk in LDS
    constexpr uint32_t chb = 8192;            // a padded chunk in memory (q <= 8)
    using W = Walkers<KW, S, true>;
    extern __shared__ f4v lds4[];
    char* ldsb = reinterpret_cast<char*>(lds4);
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wfirst = block * (2 * S * NWAVES) + (wave * 2 + (lane >> 5)) * S;
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * nchunk * chb);
    const uint32_t voff = lane * 16;
    if (nsteps == 0) return;
    const uint32_t rowb = nchunk * SLOT, stageb = nst * rowb;
    // KB pieces of a row, dealt to the waves over all steps of a stage
    const uint32_t npc = (q * q + 7) / 8, rp = nchunk * npc;
    const uint32_t inv = 65536 / npc + 1;     // r / npc for r < 256
    auto copy_stage = [&](uint32_t t0, uint32_t buf) {
        const uint32_t n = nsteps - t0 < nst ? nsteps - t0 : nst;
        uint32_t g = 0, r = wave;
        while (r >= rp) {
            r -= rp;
            g++;
        }
        while (g < n) {
            const uint32_t pos = __builtin_amdgcn_readfirstlane(pos_list[t0 + g]);
            const uint32_t k = (r * inv) >> 16, piece = r - k * npc;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rJ, (lds_void*)(ldsb + buf * stageb + g * rowb + k * SLOT + piece * 1024), 16, voff,
                (pos * nchunk + k) * chb + piece * 1024, 0, 0);
            r += NWAVES;
            while (r >= rp) {
                r -= rp;
                g++;
            }
        }
    };
    W w;
    w.load(seq, ldseq, L, wfirst, lane);
    uint32_t baseA[S], baseB[S];
    float acc[S];
    copy_stage(0, 0);
    wait_vmem();
    __syncthreads();
    uint32_t buf = 0;
    uint32_t pos = __builtin_amdgcn_readfirstlane(pos_list[0]);
    for (uint32_t t0 = 0; t0 < nsteps; t0 += nst) {
        if (t0 + nst < nsteps) copy_stage(t0 + nst, buf ^ 1);
        const uint32_t t1 = t0 + nst < nsteps ? t0 + nst : nsteps;
        uint32_t origin = j * 4 + buf * stageb;
        for (uint32_t t = t0; t < t1; t++) {
            const uint32_t pos_next =
                (t + 1 < nsteps) ? __builtin_amdgcn_readfirstlane(pos_list[t + 1]) : 0u;
            const uint32_t Pcur =
                w.draws(t, step0, walker_base + wfirst + (j >> W::SH), lane, q, k0, k1);
            w.bases(pos, lane, Pcur & 0xffu, q, origin, baseA, baseB);
#pragma unroll
            for (int k = 0; k < K; k++) {
                if (k == 0 || (uint32_t)k < nchunk) {
                    const char* cb = ldsb + k * SLOT;
                    constexpr int G = (S < SWEEP_G) ? S : SWEEP_G;
#pragma unroll
                    for (int i = 0; i < S / G; i++) {
                        float vA[G], vB[G];
#pragma unroll
                        for (int g = 0; g < G; g++) {
                            const int s = i * G + g;
                            uint32_t aA, aB;
                            w.gather_addr(s, k, baseA[s], baseB[s], aA, aB);
                            vA[g] = *reinterpret_cast<const float*>(cb + aA);
                            vB[g] = *reinterpret_cast<const float*>(cb + aB);
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int g = 0; g < G; g++) {
                            const int s = i * G + g;
                            if (k == 0) acc[s] = vB[g] - vA[g];
                            else acc[s] += vB[g] - vA[g];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            w.accept(pos, lane, acc, Pcur, nbeta);
            pos = pos_next;
            origin += rowb;
        }
        wait_vmem();
        __syncthreads();
        buf ^= 1;
    }
    w.store(seq, ldseq, L, wfirst, lane);
}

// No staging: every lane reads the couplings it needs from memory (the rows
// of a step are shared by all walkers, so they come from L2).  One wave per
// work-group, no barrier, no LDS.  NC = nchunk, so that the loads of a step
// are straight-line code and all in flight together.
template <int NC, int S>
__device__ __forceinline__ void sweep_direct(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t chb, uint32_t nsteps, uint32_t k0, uint32_t k1,
    uint64_t step0, uint32_t walker_base, float nbeta, uint32_t block) {
    constexpr int KW = (NC + 3) / 4;
    using W = Walkers<KW, S, false>;
    const uint32_t lane = threadIdx.x;
    const uint32_t j = lane & 31;
    const uint32_t wfirst = block * (2 * S) + (lane >> 5) * S;
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * NC * chb);
    if (nsteps == 0) return;
    W w;
    w.load(seq, ldseq, L, wfirst, lane);
    uint32_t baseA[S], baseB[S];
    float acc[S];
    uint32_t pos = __builtin_amdgcn_readfirstlane(pos_list[0]);
    for (uint32_t t = 0; t < nsteps; t++) {
        const uint32_t pos_next =
            (t + 1 < nsteps) ? __builtin_amdgcn_readfirstlane(pos_list[t + 1]) : 0u;
        const uint32_t Pcur =
            w.draws(t, step0, walker_base + wfirst + (j >> W::SH), lane, q, k0, k1);
        w.bases(pos, lane, Pcur & 0xffu, q, j * 4, baseA, baseB);
        const uint32_t row = pos * NC * chb;
        float vA[NC][S], vB[NC][S];
#pragma unroll
        for (int k = 0; k < NC; k++) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                uint32_t aA, aB;
                w.gather_addr(s, k, baseA[s], baseB[s], aA, aB);
                vA[k][s] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(rJ, aA, row + k * chb, 0));
                vB[k][s] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(rJ, aB, row + k * chb, 0));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NC; k++) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                if (k == 0) acc[s] = vB[k][s] - vA[k][s];
                else acc[s] += vB[k][s] - vA[k][s];
            }
        }
        w.accept(pos, lane, acc, Pcur, nbeta);
        pos = pos_next;
    }
    w.store(seq, ldseq, L, wfirst, lane);
}

template <int KW, int S, int NWAVES, int NPC>
__global__ __launch_bounds__(64 * NWAVES) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_sweep_steps(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t nchunk, uint32_t nsteps, uint32_t k0,
    uint32_t k1, uint64_t step0, uint32_t walker_base, float nbeta, uint32_t nst) {
    sweep_steps<KW, S, NWAVES, NPC>(Ju, seq, pos_list, ldseq, L, q, nchunk, nsteps, k0, k1, step0,
                                    walker_base, nbeta, blockIdx.x, nst);
}

template <int NC, int S>
__global__ __launch_bounds__(64) void k_sweep_direct(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t chb, uint32_t nsteps, uint32_t k0, uint32_t k1,
    uint64_t step0, uint32_t walker_base, float nbeta) {
    sweep_direct<NC, S>(Ju, seq, pos_list, ldseq, L, q, chb, nsteps, k0, k1, step0, walker_base,
                        nbeta, blockIdx.x);
}

template <int KW, int S, int NWAVES, int PF>
__global__ __launch_bounds__(64 * NWAVES) __attribute__((amdgpu_waves_per_eu(NWAVES / 4, NWAVES / 4))) void k_sweep(
    const float* __restrict__ Ju, uint8_t* __restrict__ seq, const uint32_t* __restrict__ pos_list,
    uint32_t ldseq, uint32_t L, uint32_t q, uint32_t nchunk, uint32_t nsteps, uint32_t k0,
    uint32_t k1, uint64_t step0, uint32_t walker_base, float nbeta) {
    sweep_block<KW, S, NWAVES, PF>(Ju, seq, pos_list, ldseq, L, q, nchunk, nsteps, k0, k1, step0,
                                   walker_base, nbeta, blockIdx.x);
}

// A model's descriptor with every field wave-uniform (the kernel's own stores
// to walker memory keep the compiler from proving it).
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    // (readfirstlane returns int: widen through uint32_t, or a low word
    // with bit 31 set would sign-extend over the high word)
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return (uint64_t)lo | ((uint64_t)hi << 32);
}
__device__ __forceinline__ BatchModel uniform_model(const BatchModel& m) {
    auto u32 = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    BatchModel r;
    r.Ju = (const float*)uniform64((uint64_t)m.Ju);
    r.seq = (uint8_t*)uniform64((uint64_t)m.seq);
    r.pos = (const uint32_t*)uniform64((uint64_t)m.pos);
    r.step = (const uint64_t*)uniform64((uint64_t)m.step);
    r.ld = u32(m.ld);
    r.L = u32(m.L);
    r.q = u32(m.q);
    r.nchunk = u32(m.nchunk);
    r.nsteps = u32(m.nsteps);
    r.k0 = u32(m.k0);
    r.k1 = u32(m.k1);
    r.walker_base = u32(m.walker_base);
    r.nbeta = __uint_as_float(u32(__float_as_uint(m.nbeta)));
    r.pad_ = 0;
    return r;
}

// Persistent sweep over the tiles of one (KW, PF) class of a batch of
// models: every work-group takes tiles from a shared counter until none is
// left (the counter is cleared before each launch).
template <int KW, int S, int NWAVES, int PF>
__global__ __launch_bounds__(64 * NWAVES) __attribute__((amdgpu_waves_per_eu(NWAVES / 4, NWAVES / 4))) void
k_sweep_batch(const BatchModel* __restrict__ models, const BatchTile* __restrict__ tiles,
              uint32_t ntiles, uint32_t* __restrict__ counter) {
    // the tile's number; two chunks of q > 21 take all of the LDS, so there it goes
    // through their first word
    constexpr bool OWN_WORD = PF < 10;
    uint32_t* s_tile;
    if constexpr (OWN_WORD) {
        __shared__ uint32_t word;
        s_tile = &word;
    } else {
        extern __shared__ f4v lds4[];
        s_tile = reinterpret_cast<uint32_t*>(lds4);
    }
    for (;;) {
        __syncthreads();   // previous tile's LDS reads done; s_tile free
        if (threadIdx.x == 0) *s_tile = atomicAdd(counter, 1u);
        __syncthreads();
        const uint32_t t = __builtin_amdgcn_readfirstlane(*s_tile);  // uniform: scalar loads below
        if (t >= ntiles) break;
        if constexpr (!OWN_WORD) __syncthreads();   // read by all before a copy overwrites it
        const BatchTile tl = tiles[t];
        const BatchModel m = uniform_model(models[tl.model]);
        const uint64_t step0 = uniform64(*m.step);
        sweep_block<KW, S, NWAVES, PF>(
            m.Ju, m.seq, m.pos, m.ld, m.L, m.q, m.nchunk, m.nsteps, m.k0, m.k1, step0,
            m.walker_base, m.nbeta, (uint32_t)__builtin_amdgcn_readfirstlane((int)tl.block));
    }
}

// Unstaged sweep over the walkers of one class of a batch: `sub` waves of
// 2*S walkers per tile.  Work-groups go to the eight XCDs in turn, so each XCD
// takes a contiguous range of `per` waves: it sweeps few models, and its L2
// holds their rows.
template <int KW, int S>
__global__ __launch_bounds__(64) void k_sweep_batch_direct(const BatchModel* __restrict__ models,
                                                           const BatchTile* __restrict__ tiles,
                                                           uint32_t sub, uint32_t waves,
                                                           uint32_t per) {
    const uint32_t v = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (v >= waves) return;
    const uint32_t t = v / sub;
    const BatchTile tl = tiles[t];
    const BatchModel m = uniform_model(models[tl.model]);
    const uint64_t step0 = uniform64(*m.step);
    const uint32_t block = tl.block * sub + (v - t * sub);
    const uint32_t chb = chunk_floats(m.q) * 4;
#define MI3_NC(NC)                                                                              \
    if (m.nchunk == NC)                                                                         \
        sweep_direct<NC, S>(m.Ju, m.seq, m.pos, m.ld, m.L, m.q, chb, m.nsteps, m.k0, m.k1, step0, \
                            m.walker_base, m.nbeta, block);
    MI3_NC(4 * KW - 3) MI3_NC(4 * KW - 2) MI3_NC(4 * KW - 1) MI3_NC(4 * KW)
#undef MI3_NC
}

// ---------------------------------------------------------------------------
// Coupling-row staging alone: the sweep's per-step copies of J[pos] (the same
// chunks of the same sites, from the same chunked layout, by the same waves
// and instructions, one barrier per chunk) with no gathers, reduction or
// accept.  With INFLIGHT = 1 each chunk's copy is awaited before the barrier
// that follows its issue, as in the sweep; with INFLIGHT = 2 the copy of the
// chunk just issued stays in flight across the barrier (a barrier without
// the vmcnt(0) of __syncthreads; the LDS contents are not used).  The first
// is the staging time of the sweep's double-buffered launch shape, the
// second that of the copies alone, overlapped.
template <int PF, int NWAVES, int INFLIGHT>
__global__ __launch_bounds__(64 * NWAVES) void k_stage_probe(const float* __restrict__ Ju,
                                                             const uint32_t* __restrict__ pos_list,
                                                             uint32_t L, uint32_t nchunk,
                                                             uint32_t nsteps) {
    constexpr int NT = 64 * NWAVES;
    constexpr int DMA_T = NT < 512 ? NT : 512;
    constexpr uint32_t chb = PF * DMA_T * 16;
    extern __shared__ f4v lds4[];
    char* ldsb = reinterpret_cast<char*>(lds4);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * nchunk * chb);
    const uint32_t voff = tid * 16;
    uint32_t buf = 0;
    for (uint32_t t = 0; t < nsteps; t++) {
        const uint32_t pos = __builtin_amdgcn_readfirstlane(pos_list[t]);
        for (uint32_t k = 0; k < nchunk; k++) {
            if (wave < DMA_T / 64)
                chunk_dma<PF, DMA_T>(rJ, voff, (pos * nchunk + k) * chb, ldsb + buf * chb, wave);
            if constexpr (INFLIGHT == 1) {
                wait_vmem();
                __syncthreads();
            } else {
                wait_vmem_upto<PF>();
                barrier_copies_in_flight();
            }
            buf ^= 1;
        }
    }
    wait_vmem();
}

// ---------------------------------------------------------------------------
// Batch energies E(s) = sum_{i<m} J_{i,m}(s_i, s_m) of nseq sequences.
// Restates getEnergies (mcmc.cl:249-345); the sweep's layout, with, for each
// row i, only the chunks holding partners m > i.  As the sweep, in three forms:
// chunks staged one at a time, the rows of a stage staged at once (q <= 8), and
// unstaged (few sequences).

// Sum of the gathers of chunk k over the lane's slots.  MASK: the diagonal
// chunk, where only partners m > i count, as a 0/1 factor (fma(v, 1, acc) is
// acc + v exactly).  The other chunks add without it for up to two state words
// (an add takes half the time of an fma); beyond, two copies spill.
template <bool MASK, int KW, int S, bool QB>
__device__ __forceinline__ void energy_chunk(const Walkers<KW, S, QB>& w, int k, const char* cb,
                                             const uint32_t (&base)[S], float keep,
                                             float (&acc)[S]) {
    constexpr int G = (S < 16) ? S : 16;
#pragma unroll
    for (int s0 = 0; s0 < S; s0 += G) {
        float v[G];
#pragma unroll
        for (int g = 0; g < G; g++)
            v[g] = *reinterpret_cast<const float*>(
                cb + (base[s0 + g] + byte_x128(w.st[s0 + g][k >> 2], k & 3)));
#pragma unroll
        for (int g = 0; g < G; g++)
            acc[s0 + g] = MASK ? __fmaf_rn(v[g], keep, acc[s0 + g]) : acc[s0 + g] + v[g];
    }
}

template <int KW, int S, bool QB>
__device__ __forceinline__ void store_energies(const float (&acc)[S], float* E, uint32_t wfirst,
                                               uint32_t lane, uint32_t nseq) {
#pragma unroll
    for (int s = 0; s < S; s++) {
        const float e = half_wave_sum(acc[s]);
        if ((lane & 31) == 0 && wfirst + s < nseq) E[wfirst + s] = e;
    }
}

template <int KW, int S, int NWAVES, int PF, bool OVL>
__global__ __launch_bounds__(64 * NWAVES) void k_energies(
    const float* __restrict__ Ju, const uint8_t* __restrict__ seq, float* __restrict__ E,
    uint32_t ldseq, uint32_t nseq, uint32_t L, uint32_t q, uint32_t nchunk) {
    constexpr int NT = 64 * NWAVES;
    constexpr int K = 4 * KW;
    using W = Walkers<KW, S, (PF <= 4)>;
    extern __shared__ f4v lds4[];

    // the padded chunk is PF float4 per thread of the first DMA_T threads
    // (the chunk layout's unit); waves beyond them take no part in staging
    constexpr int DMA_T = 512;
    static_assert(NT >= DMA_T, "a chunk is copied in one pass");
    constexpr uint32_t chb = PF * DMA_T * 16;  // padded chunk (bytes)
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wfirst = blockIdx.x * (2 * S * NWAVES) + (wave * 2 + (lane >> 5)) * S;
    W w;
    w.load(seq, ldseq, L, wfirst, lane, nseq);
    float acc[S];
#pragma unroll
    for (int s = 0; s < S; s++) acc[s] = 0.f;
    uint32_t base[S];

    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * nchunk * chb);
    const uint32_t voff = tid * 16;
    // staging waves, as in the sweep
    const bool stage = (PF == 1) ? (uint32_t)wave < (q * q + 7) / 8 : wave < DMA_T / 64;
    char* ldsb = reinterpret_cast<char*>(lds4);
    // OVL: copy cursor (row ci, chunk ck) two units ahead of the gathers
    // and the byte offset of the unit one ahead; at the last unit the
    // cursor stays, so copies past the end repeat it into unread slots
    uint32_t ci = 0, ck = 0, off_next = 0;
    auto advance = [&]() {
        const bool wrap = ck + 1 >= nchunk;
        const bool stay = wrap && ci + 2 >= L;
        ck = stay ? ck : (wrap ? (ci + 2) >> 5 : ck + 1);
        ci = (wrap && !stay) ? ci + 1 : ci;
    };
    if constexpr (OVL) {
        static_assert(PF == 7 && DMA_T == 512, "overlapping ring: chunks of q = 17..21");
        // unit (0, 0) whole into slot 0, then the early part of the next
        if (wave < 8) {
            OverlapRing::copy<OverlapRing::EARLY_OPS>(rJ, voff, 0, ldsb, 0,
                                                      OverlapRing::early_first(0), wave);
            OverlapRing::copy<OverlapRing::LATE_OPS>(rJ, voff, 0, ldsb, 0,
                                                     OverlapRing::late_first(0), wave);
        }
        advance();
        off_next = (ci * nchunk + ck) * chb;
        if (wave < 8)
            OverlapRing::copy<OverlapRing::EARLY_OPS>(rJ, voff, off_next, ldsb, 1,
                                                      OverlapRing::early_first(1), wave);
        advance();
        wait_vmem_upto<OverlapRing::EARLY_OPS>();
        barrier_copies_in_flight();
    } else {
        // first unit: row 0, chunk 0
        if (stage) chunk_dma<PF, DMA_T>(rJ, voff, 0, ldsb, wave);
        wait_vmem();
        __syncthreads();
    }
    uint32_t ring = 0;
    // one row whose chunk k is in buffer (p + k) % 2; as the sweep's step,
    // compiled for either p where that does not spill
    constexpr bool TWICE = KW <= 2 && !OVL;
    auto row = [&](auto pc, uint32_t pv, uint32_t i) __attribute__((always_inline)) {
        const uint32_t p = TWICE ? decltype(pc)::value : pv;
        const uint32_t kp = i >> 5, c0 = (i + 1) >> 5;
        w.row_bases(i, lane, q, j * 4, base);
        const float keep = (c0 != kp || j > (i & 31)) ? 1.f : 0.f;
#pragma unroll
        for (int k = 0; k < K; k++) {
            if ((uint32_t)k >= c0 && (uint32_t)k < nchunk) {
                const char* cb;
                if constexpr (OVL) {
                    // late part of the next unit, early part of the one after
                    if (wave < 8) {
                        OverlapRing::copy<OverlapRing::LATE_OPS>(
                            rJ, voff, off_next, ldsb, (ring + 1) & 3,
                            OverlapRing::late_first((ring + 1) & 3), wave);
                        OverlapRing::copy<OverlapRing::EARLY_OPS>(
                            rJ, voff, (ci * nchunk + ck) * chb, ldsb, (ring + 2) & 3,
                            OverlapRing::early_first((ring + 2) & 3), wave);
                    }
                    off_next = (ci * nchunk + ck) * chb;
                    advance();
                    cb = ldsb + OverlapRing::base(ring);
                } else {
                    const uint32_t buf = (p + k) & 1;
                    const bool last_chunk = (uint32_t)k + 1 == nchunk;
                    const bool has_next = !last_chunk || (i + 2 < L);
                    if (has_next) {
                        const uint32_t ni = last_chunk ? i + 1 : i;
                        const uint32_t nc = last_chunk ? ((i + 2) >> 5) : (uint32_t)k + 1;
                        if (stage)
                            chunk_dma<PF, DMA_T>(rJ, voff, (ni * nchunk + nc) * chb,
                                                        ldsb + (buf ^ 1) * chb, wave);
                    }
                    cb = ldsb + buf * chb;
                }
                if constexpr (KW <= 2) {
                    if ((uint32_t)k == c0) energy_chunk<true>(w, k, cb, base, keep, acc);
                    else energy_chunk<false>(w, k, cb, base, keep, acc);
                } else {
                    energy_chunk<true>(w, k, cb, base, (uint32_t)k == c0 ? keep : 1.f, acc);
                }
                if constexpr (OVL) {
                    // the next unit has landed (only the early part of
                    // the one after may be in flight)
                    wait_vmem_upto<OverlapRing::EARLY_OPS>();
                    barrier_copies_in_flight();
                    ring = (ring + 1) & 3;
                } else {
                    wait_vmem();
                    __syncthreads();
                }
            }
        }
    };
    uint32_t p = 0;
    for (uint32_t i = 0; i + 1 < L; i++) {
        if (TWICE && p) row(std::integral_constant<uint32_t, 1>{}, p, i);
        else row(std::integral_constant<uint32_t, 0>{}, p, i);
        // the next row's first chunk follows this row's last
        p = (p + nchunk + ((i + 2) >> 5)) & 1;
    }
    // copies issued past the last unit
    if constexpr (OVL) wait_vmem();
    store_energies<KW, S, (PF <= 4)>(acc, E, wfirst, lane, nseq);
}

// Rows staged `nrow` at a time (all chunks of a row, NPC KB each; of the first
// row's chunks those before its diagonal are not read), one barrier per stage.
template <int KW, int S, int NWAVES, int NPC>
__global__ __launch_bounds__(64 * NWAVES) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_energies_rows(
    const float* __restrict__ Ju, const uint8_t* __restrict__ seq, float* __restrict__ E,
    uint32_t ldseq, uint32_t nseq, uint32_t L, uint32_t q, uint32_t nchunk, uint32_t nrow) {
    constexpr int K = 4 * KW;
    constexpr uint32_t SLOT = NPC * 1024, chb = 8192;
    extern __shared__ f4v lds4[];
    char* ldsb = reinterpret_cast<char*>(lds4);
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wfirst = blockIdx.x * (2 * S * NWAVES) + (wave * 2 + (lane >> 5)) * S;
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * nchunk * chb);
    const uint32_t voff = lane * 16;
    const uint32_t rowb = nchunk * SLOT, stageb = nrow * rowb;
    const uint32_t npc = (q * q + 7) / 8, rp = nchunk * npc;
    const uint32_t inv = 65536 / npc + 1;     // r / npc for r < 256
    auto copy_stage = [&](uint32_t i0, uint32_t buf) {
        const uint32_t n = L - 1 - i0 < nrow ? L - 1 - i0 : nrow;
        uint32_t g = 0, r = wave;
        while (r >= rp) {
            r -= rp;
            g++;
        }
        while (g < n) {
            const uint32_t k = (r * inv) >> 16, piece = r - k * npc;
            if (k >= (i0 + g + 1) >> 5)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rJ, (lds_void*)(ldsb + buf * stageb + g * rowb + k * SLOT + piece * 1024), 16,
                    voff, ((i0 + g) * nchunk + k) * chb + piece * 1024, 0, 0);
            r += NWAVES;
            while (r >= rp) {
                r -= rp;
                g++;
            }
        }
    };
    Walkers<KW, S, true> w;
    w.load(seq, ldseq, L, wfirst, lane, nseq);
    float acc[S];
#pragma unroll
    for (int s = 0; s < S; s++) acc[s] = 0.f;
    uint32_t base[S];
    copy_stage(0, 0);
    wait_vmem();
    __syncthreads();
    uint32_t buf = 0;
    for (uint32_t i0 = 0; i0 + 1 < L; i0 += nrow) {
        if (i0 + nrow + 1 < L) copy_stage(i0 + nrow, buf ^ 1);
        const uint32_t i1 = i0 + nrow < L - 1 ? i0 + nrow : L - 1;
        uint32_t origin = j * 4 + buf * stageb;
        for (uint32_t i = i0; i < i1; i++) {
            const uint32_t kp = i >> 5, c0 = (i + 1) >> 5;
            w.row_bases(i, lane, q, origin, base);
            const float keep = (c0 != kp || j > (i & 31)) ? 1.f : 0.f;
#pragma unroll
            for (int k = 0; k < K; k++) {
                if ((uint32_t)k < c0 || (uint32_t)k >= nchunk) continue;
                if constexpr (KW <= 2) {
                    if ((uint32_t)k == c0)
                        energy_chunk<true>(w, k, ldsb + k * SLOT, base, keep, acc);
                    else
                        energy_chunk<false>(w, k, ldsb + k * SLOT, base, keep, acc);
                } else {
                    energy_chunk<true>(w, k, ldsb + k * SLOT, base,
                                       (uint32_t)k == c0 ? keep : 1.f, acc);
                }
            }
            origin += rowb;
        }
        wait_vmem();
        __syncthreads();
        buf ^= 1;
    }
    store_energies<KW, S, true>(acc, E, wfirst, lane, nseq);
}

// No staging: one wave per work-group, ROWS neighbouring rows at a time (of one
// chunk, so that they share its partners), all their gathers of a chunk in
// flight.  Lanes whose partner does not count read the row all the same, and
// select its couplings away (as a 0 factor, an infinite one would make NaN of
// the energies of sequences that do not hold it, or hold it in a row that counts).
template <int NC>
__global__ __launch_bounds__(64) void k_energies_direct(
    const float* __restrict__ Ju, const uint8_t* __restrict__ seq, float* __restrict__ E,
    uint32_t ldseq, uint32_t nseq, uint32_t L, uint32_t q, uint32_t chb) {
    constexpr int KW = (NC + 3) / 4, S = 1, ROWS = 4;
    const uint32_t lane = threadIdx.x;
    const uint32_t j = lane & 31;
    const uint32_t wfirst = blockIdx.x * 2 + (lane >> 5);
    const __amdgpu_buffer_rsrc_t rJ = make_rsrc(Ju, L * NC * chb);
    Walkers<KW, S, false> w;
    w.load(seq, ldseq, L, wfirst, lane, nseq);
    float acc[1] = {0.f};
    for (uint32_t i0 = 0; i0 + 1 < L; i0 += ROWS) {
        const uint32_t kp = i0 >> 5;
        uint32_t base[ROWS][S];
        // whether a coupling counts: in the first chunk those of partners past the
        // row, then all; none in rows past the last, which repeat it
        bool all[ROWS], counts[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const uint32_t i = i0 + r + 1 < L ? i0 + r : L - 2;
            w.row_bases(i, lane, q, j * 4 + i * NC * chb, base[r]);
            all[r] = i == i0 + r;
            counts[r] = all[r] && j > (i & 31);
        }
#pragma unroll
        for (int k = 0; k < NC; k++) {
            if ((uint32_t)k < kp) continue;
            float v[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; r++)
                v[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    rJ, base[r][0] + byte_x128(w.st[0][k >> 2], k & 3), k * chb, 0));
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                acc[0] += counts[r] ? v[r] : 0.f;
                counts[r] = all[r];
            }
        }
    }
    store_energies<KW, S, false>(acc, E, wfirst, lane, nseq);
}

}  // namespace mi3
