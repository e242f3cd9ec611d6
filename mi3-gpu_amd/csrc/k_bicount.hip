// Bimarginal counts as a one-hot Gram product on the matrix cores, in 4-bit
// floats.
//
// With X[n][r] = [s_{n, r/q} == r % q] (N x L*q, one-hot, never stored),
// count_{ij}(a, b) = (X^T X)[i*q + a][j*q + b] for i < j.  Each wave owns a
// T x T block of the flattened L*q x L*q Gram matrix (tiles of
// v_mfma_scale_f32_32x32x64_f8f6f4 with e2m1 operands, twice the rate of the
// 8-bit ones), builds its operands on the fly from residues packed to bit
// planes (32 sequences per lane per k-step of 64), contracts over its range of
// sequences and scatters the i < j entries into the packed (L(L-1)/2, q*q)
// uint32 table.  Every product is 0 or 1 and a wave sums at most 2^23 sequences
// before it stores, so the float32 sums are exact integers and the result does
// not depend on the order of any addition.
// Replaces countBivariate (mcmc.cl:464-516); matches np.bincount per pair
// (getMarginals.py:80-86).
#include "common.h"

namespace mi3 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Residues packed for the operands: bit planes.  A unit is 128 sequences of a
// site in 16 * PL consecutive bytes, [plane][half] of 64 bits; a lane's 32
// sequences of the unit's first k-step are the low word of its half, those of
// the second the high word.
//   PL = 3 (q <= 7), PL = 5 (q <= 25).
// A residue equals a letter where every plane agrees with the letter's bit: PL
// instructions for 32 sequences.  Sequences past the end are all ones, which is
// no residue, and so is a byte that takes more than PL bits.  The bits of a word
// are in the same order at every site, which is all that a sum over sequences needs.
template <int PL>
__global__ __launch_bounds__(256) void k_pack_residues(const uint8_t* __restrict__ seq,
                                                       uint32_t ldseq, uint32_t nseq,
                                                       uint32_t nunits, uint8_t* __restrict__ out) {
    // thread: 64 sequences of a site
    const uint32_t c = blockIdx.x * 256 + threadIdx.x, site = blockIdx.y;
    if (c >= nunits * 2) return;
    const uint4* row = reinterpret_cast<const uint4*>(seq + (size_t)site * ldseq);
    uint32_t w[2][8];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
        const uint32_t n = c * 64 + k * 16;
        uint4 v = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (n < nseq) v = row[n / 16];   // rows are multiples of 16 bytes long
        uint32_t x[4] = {v.x, v.y, v.z, v.w};
        if (n < nseq && n + 16 > nseq) {
#pragma unroll
            for (uint32_t e = 0; e < 16; e++)
                if (n + e >= nseq) x[e >> 2] |= 0xffu << (8 * (e & 3));
        }
#pragma unroll
        for (uint32_t e = 0; e < 4; e++) w[k >> 1][(k & 1) * 4 + e] = x[e];
    }
    // bit 0 of a byte: it takes more than PL bits
    constexpr uint32_t LOW = 0x01010101u * ((1u << PL) - 1);
    uint32_t no[2][8];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 8; e++)
            no[h][e] = (((w[h][e] & 0x7f7f7f7fu) + (0x7f7f7f7fu - LOW)) | w[h][e]) >> 7;
    uint2* o = reinterpret_cast<uint2*>(out + ((size_t)site * nunits + (c >> 1)) * (16 * PL) +
                                        (c & 1) * 8);
#pragma unroll
    for (int p = 0; p < PL; p++) {
        uint32_t m[2] = {0u, 0u};
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) m[h] |= (((w[h][e] >> p) | no[h][e]) & 0x01010101u) << e;
        o[2 * p] = make_uint2(m[0], m[1]);
    }
}

// Staging: STAGE units of the sites that a block's rows and columns touch (at
// most T/q + 2 each), double-buffered; one LDS DMA instruction moves 16 bytes
// per lane.  An odd number of 16-byte pieces per site keeps the sites that one
// read touches (at most 17) in different banks.  The host takes the longer stage
// (5 units, else 3) whose buffers fit 40 KiB, so that four waves share a CU.
constexpr uint32_t BC_PLANES_Q = 7;   // largest q of three planes
constexpr uint32_t BC_UNIT = 128;     // sequences
// most units that a wave sums in float32 (2^23 sequences; whole numbers are exact to
// 2^24).  Parts reach it from 2^28 sequences on for few blocks (32 parts), and
// from 2^23 on where a wave takes whole blocks (L=255 q=25)
constexpr uint32_t BC_PART = 65536;
inline uint32_t bc_planes(uint32_t q) { return q <= BC_PLANES_Q ? 3 : 5; }
inline size_t bc_lds_bytes(uint32_t q, uint32_t tile, uint32_t stage) {
    const uint32_t sites = 2 * (tile / q + 2);
    return 2ull * ((sites * bc_planes(q) * stage + 63) / 64) * 1024;
}
inline uint32_t bc_stage_for(uint32_t q, uint32_t tile) {
    return bc_lds_bytes(q, tile, 5) <= 40960 ? 5 : 3;
}
typedef __attribute__((address_space(3))) void bc_lds_void;

// s_waitcnt vmcnt(0): every vector-memory operation of this wave, LDS DMA
// included, has completed.
__device__ __forceinline__ void wait_vmem_bc() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The work is `total` units: the blocks (rb, cb), rb <= cb, of T = 32 * NT rows and
// columns, nunits units each, in one sequence that the waves of the grid divide
// evenly, so that all SIMDs end together however many blocks there are.  A
// wave that holds the whole of a block stores its counts; the parts of a shared
// block are added with integer atomics (exact in any order; the table must be
// zeroed first).  NT = 4 keeps 256 sums per lane in AGPRs, one wave to a SIMD;
// NT = 2 is for problems too small for that (rule at the launch).
//
// Bound by the issue of the one wave that a SIMD holds: a matrix instruction takes 37
// cycles (at 2.4 GHz) alone and one is issued every 58 here.  So the operands of a
// k-step are built between the products of the one before, evenly and two at a
// time (their chains of dependent instructions otherwise stall; four at a time, or
// the reads later, took 3-5% longer); reads are eight bytes wide (2.6 cycles of a CU;
// 16 bytes 7.6).  Measured (us; 8-bit one-hot products built from bytes, 4-bit ones from
// nibbles, this form with a fixed number of parts per block, with even shares,
// and with this order of the building):
//   L    q   sequences   8-bit  nibbles  planes  even shares  order
//   232  21  1000003     10653     7020    5595         5533   4783
//   232  21  262144       3103     2063    1661         1525   1342
//   232  21  16384         459      400     378          207    197
//   150  12  100001        434      377     367          202    202
//   93   4   262144        163       84      70           70     70
//   99   4   16384          70       26      25           25     25
template <int NT, int PL, int STAGE>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(1, NT == 4 ? 1 : 2))) void k_bicounts_fp4(
    const uint8_t* __restrict__ pk, uint32_t nunits, uint32_t L, uint32_t q, uint32_t nblk,
    uint64_t total, uint32_t* __restrict__ counts) {
    extern __shared__ __attribute__((aligned(16))) uint8_t bc_lds[];
    constexpr uint32_t T = 32 * NT;
    constexpr uint32_t KB = 16 * PL;          // bytes of a site's unit
    constexpr uint32_t LPS = PL * STAGE;      // 16-byte pieces of a site's stage
    constexpr uint32_t SB = 16 * LPS;
    static_assert(LPS % 2 == 1, "sites in different banks");
    const uint32_t l = threadIdx.x;
    const uint32_t lr = l & 31, g = l >> 5;
    const uint32_t Lq = L * q;
    const uint32_t ldp = nunits * KB;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(pk), (short)0, (int)(ldp * L), 0x00020000);
    const uint64_t end = total * (blockIdx.x + 1) / gridDim.x;
    for (uint64_t cur = total * blockIdx.x / gridDim.x; cur < end;) {
        // units [u0, u1) of block t
        uint32_t t = (uint32_t)(cur / nunits);
        const uint32_t u0 = (uint32_t)(cur - (uint64_t)t * nunits);
        uint32_t u1 = u0 + BC_PART < nunits ? u0 + BC_PART : nunits;
        if (end - cur < u1 - u0) u1 = u0 + (uint32_t)(end - cur);
        cur += u1 - u0;
        uint32_t rb = 0;
        while (t >= nblk - rb) {
            t -= nblk - rb;
            rb++;
        }
        const uint32_t cb = rb + t;

        // the sites of this block's rows (A) and columns (B), staged as
        // [A sites..., B sites...] x SB bytes per buffer
        const uint32_t rA0 = rb * T, rA1 = (rA0 + T - 1 < Lq) ? rA0 + T - 1 : Lq - 1;
        const uint32_t cB0 = cb * T, cB1 = (cB0 + T - 1 < Lq) ? cB0 + T - 1 : Lq - 1;
        const uint32_t siA0 = rA0 / q, nsA = rA1 / q - siA0 + 1;
        const uint32_t siB0 = cB0 / q, nsB = cB1 / q - siB0 + 1;
        const uint32_t ninst = ((nsA + nsB) * LPS + 63) / 64;
        const uint32_t bufbytes = ninst * 1024;

        // per operand: LDS address of this lane's words, and the letter's bits as masks
        // (rows past L*q count the first row's site again and are not stored)
        uint32_t at[2 * NT], let[2 * NT][PL];
        auto operand = [&](int w, uint32_t r, uint32_t first, uint32_t slot0) {
            const uint32_t si = r < Lq ? r / q : first;
            const uint32_t a = r < Lq ? r - si * q : 0u;
            at[w] = (slot0 + si - first) * SB + g * 8;
#pragma unroll
            for (int p = 0; p < PL; p++) let[w][p] = 0u - ((a >> p) & 1u);
        };
#pragma unroll
        for (int x = 0; x < NT; x++) {
            operand(x, rA0 + x * 32 + lr, siA0, 0);
            operand(NT + x, cB0 + x * 32 + lr, siB0, nsA);
        }
        v16f acc[NT][NT];
#pragma unroll
        for (int x = 0; x < NT; x++)
#pragma unroll
            for (int y = 0; y < NT; y++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[x][y][e] = 0.f;

        // LDS DMA of one stage: piece P is piece P % LPS of site P / LPS; pieces past
        // the block's sites load a valid site that nothing reads.  The last stage of a
        // range can reach past the last unit (and, for the last site, past the
        // buffer): such pieces are never counted, and their source offsets are clamped
        // into the buffer.
        const uint32_t last16 = ldp * L - 16;
        auto stage = [&](uint32_t buf, uint32_t unit) {
            for (uint32_t k = 0; k < ninst; k++) {
                const uint32_t ts = (64 * k + l) / LPS, piece = (64 * k + l) - ts * LPS;
                const uint32_t site =
                    ts < nsA ? siA0 + ts : (ts < nsA + nsB ? siB0 + (ts - nsA) : siA0);
                const uint32_t off = site * ldp + unit * KB + 16 * piece;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs, (bc_lds_void*)(bc_lds + buf * bufbytes + k * 1024), 16,
                    off < last16 ? off : last16, 0, 0, 0);
            }
        };
        // operands: NT of rows, then NT of columns
        struct Raw {
            u2v f[2 * NT][PL];   // (as a uint2, each iteration waits for the LDS DMA in flight)
        };
        struct Ops {
            v4i f[2 * NT];
        };
        auto read = [&](const uint8_t* unit, int w, Raw& r) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < PL; p++)
                r.f[w][p] = *reinterpret_cast<const u2v*>(unit + at[w] + 16 * p);
        };
        // planes [p0, p1) of the matches of operand w at k-step h of the unit in r
        auto match = [&](const Raw& r, int w, int h, int p0, int p1,
                         uint32_t& m) __attribute__((always_inline)) {
            auto word = [&](int p) { return h ? r.f[w][p].y : r.f[w][p].x; };
#pragma unroll
            for (int p = p0; p < p1; p++)   // m & ~(word ^ letter)
                m = p == 0 ? ~(word(0) ^ let[w][0])
                           : (uint32_t)__builtin_amdgcn_bitop3_b32((int)m, (int)word(p),
                                                                   (int)let[w][p], 0x90);
        };
        // the matches as operand w: bits 4n + e go to nibble n of word e.  As e2m1, nibbles 1,
        // 2 and 4 are 0.5, 1 and 2: rows hold word e at (0.5, 1, 2, 2) and columns at (2, 1,
        // 0.5, 0.5), so that each product is 1 and most words need no shift.
        auto spread = [&](uint32_t m, int w, Ops& o) __attribute__((always_inline)) {
            if (w < NT)
                o.f[w] = v4i{(int)(m & 0x11111111u), (int)(m & 0x22222222u), (int)(m & 0x44444444u),
                             (int)((m >> 1) & 0x44444444u)};
            else
                o.f[w] = v4i{(int)((m << 2) & 0x44444444u), (int)(m & 0x22222222u),
                             (int)((m >> 2) & 0x11111111u), (int)((m >> 3) & 0x11111111u)};
            asm volatile("" : "+v"(o.f[w]));
        };
        // the products of o, and between them the building of the operands `on` of the
        // next k-step (step h of the unit in r); next: the registers of r take the next
        // unit's words as they come free.  Scheduling barriers and an empty asm at each
        // operand keep this order: left to itself, or to scheduling groups, the compiler
        // issues all products and then all the building.
        auto step = [&](const Ops& o, Ops& on, Raw& r, int h, bool next,
                        const uint8_t* unit) __attribute__((always_inline)) {
            uint32_t m[2] = {0, 0};
#pragma unroll
            for (int i = 0; i < NT * NT; i++) {
                const int x = i / NT, y = i % NT;
                const v4i f = o.f[x], c = o.f[NT + y];
                acc[x][y] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                    __builtin_shufflevector(f, f, 0, 1, 2, 3, -1, -1, -1, -1),
                    __builtin_shufflevector(c, c, 0, 1, 2, 3, -1, -1, -1, -1), acc[x][y], 4, 4, 0,
                    127, 0, 127);
                if (NT == 2) {
                    match(r, i, h, 0, PL, m[0]);
                    if (next) read(unit, i, r);
                    spread(m[0], i, on);
                } else {
                    const int w = i / 4 * 2;   // two operands to four products
                    if (i % 4 < 2) {
                        const int p0 = i % 4 ? (PL + 1) / 2 : 0, p1 = i % 4 ? PL : (PL + 1) / 2;
                        match(r, w, h, p0, p1, m[0]);
                        match(r, w + 1, h, p0, p1, m[1]);
                        asm volatile("" : "+v"(m[0]), "+v"(m[1]));   // formed here, not at their use
                        if (i % 4 && next) {
                            read(unit, w, r);
                            read(unit, w + 1, r);
                        }
                    } else {
                        spread(m[i % 2], w + i % 2, on);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        {
            // entering a stage: its bytes have landed, and the reads of the stage before
            // have completed, so its buffer takes the stage after
            uint32_t buf = 1;
            const uint8_t* sbase = bc_lds;
            auto enter = [&](uint32_t u) __attribute__((always_inline)) {
                wait_vmem_bc();
                __syncthreads();
                buf ^= 1;
                sbase = bc_lds + buf * bufbytes;
                if (u + STAGE < u1) stage(buf ^ 1, u + STAGE);
            };
            stage(0, u0);
            enter(u0);
            Raw r;
            Ops o0, o1;
#pragma unroll
            for (int w = 0; w < 2 * NT; w++) read(sbase, w, r);
#pragma unroll
            for (int w = 0; w < 2 * NT; w++) {
                uint32_t m = 0;
                match(r, w, 0, 0, PL, m);
                spread(m, w, o0);
            }
            // the operands built from the unit past the end (bytes of the last stage's
            // buffers) are not multiplied
            uint32_t k = 0;   // unit of the stage
            for (uint32_t u = u0; u < u1; u++) {
                if (++k == STAGE) {
                    k = 0;
                    if (u + 1 < u1) enter(u + 1);
                }
                step(o0, o1, r, 1, true, sbase + k * KB);
                step(o1, o0, r, 0, false, sbase);
            }
        }

        const uint32_t qq = q * q;
        // r / q as a product: r < 2^15 and r * q < 2^20, so 2^20 / q rounded up is exact
        const uint32_t inv = ((1u << 20) + q - 1) / q;
#pragma unroll
        for (int x = 0; x < NT; x++) {
#pragma unroll
            for (int y = 0; y < NT; y++) {
                const uint32_t c = cb * T + y * 32 + lr;
                if (c >= Lq) continue;
                const uint32_t jsite = (c * inv) >> 20, b = c - jsite * q;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const uint32_t r = rb * T + x * 32 + 8 * (e / 4) + 4 * g + (e % 4);
                    if (r >= Lq) continue;
                    const uint32_t isite = (r * inv) >> 20, a = r - isite * q;
                    if (isite < jsite) {
                        const uint32_t cnt = (uint32_t)acc[x][y][e];
                        uint32_t* dst = counts + (size_t)pair_index(isite, jsite, L) * qq + a * q + b;
                        if (u1 - u0 == nunits)
                            *dst = cnt;
                        else
                            atomicAdd(dst, cnt);
                    }
                }
            }
        }
        __syncthreads();   // the last stage has been read
    }
}

}  // namespace mi3
