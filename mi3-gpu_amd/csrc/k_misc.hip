// Layout, fill, random-site and independent-reseed kernels.
#include "common.h"

namespace mi3 {

// Packed (L(L-1)/2, q*q) couplings -> chunked symmetric layout
// Ju[i][c][a*q+b][jl] = J_{i,m}(a,b), m = 32c + jl (zero for m == i, m >= L).
// Same role as unpackfV (mcmc.cl:43-65): the (j,i) block is the transpose of
// the stored (i,j) block; the reference leaves the diagonal unfilled and
// skips it, here it is zero so no skip is needed.
// Every chunk is padded to `chf` floats (zeros after the q*q*32 used ones).
__global__ void k_unpack_chunked(const float* __restrict__ J, float* __restrict__ Ju, uint32_t L,
                                 uint32_t q, uint32_t nchunk, uint32_t chf, uint64_t total) {
    uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const uint32_t qq = q * q;
    uint64_t unit = idx / chf;
    uint32_t within = (uint32_t)(idx - unit * chf);
    uint32_t c = (uint32_t)(unit % nchunk);
    uint32_t i = (uint32_t)(unit / nchunk);
    uint32_t jl = within & 31;
    uint32_t ac = within >> 5;
    uint32_t m = c * CH + jl;
    float v = 0.f;
    if (ac < qq && m < L && m != i) {
        uint32_t a = ac / q, b = ac - a * q;
        if (i < m)
            v = J[(size_t)pair_index(i, m, L) * qq + a * q + b];
        else
            v = J[(size_t)pair_index(m, i, L) * qq + b * q + a];
    }
    Ju[idx] = v;
}

// Folded model for energies: k neighbouring sites as one of q^k letters, so that
// one gather adds k*k couplings (rule at fold_sites).  Couplings of the folded
// sites i < m in the chunked layout above, and zeros for the partners m <= i, which
// the energies do not count; what lies within a folded site is added to its
// couplings with the next one (the last site's to those with the one before).
// Sites past L have no couplings.
__global__ void k_fold_chunked(const float* __restrict__ J, float* __restrict__ Ju, uint32_t L,
                               uint32_t q, uint32_t k, uint32_t Q, uint32_t nfold, uint32_t nchunk,
                               uint32_t chf, uint32_t total) {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const uint32_t unit = idx / chf, within = idx - unit * chf;
    const uint32_t i = unit / nchunk, c = unit - i * nchunk;
    const uint32_t m = c * CH + (within & 31), ab = within >> 5;
    float v = 0.f;
    if (ab < Q * Q && m < nfold && m > i) {
        const uint32_t a = ab / Q, b = ab - a * Q;
        auto letter = [&](uint32_t x, uint32_t t) {   // of site t of a folded one
            for (uint32_t u = t + 1; u < k; u++) x /= q;
            return x % q;
        };
        auto coupling = [&](uint32_t x, uint32_t y, uint32_t sx, uint32_t sy) {
            return y < L ? J[(size_t)pair_index(x, y, L) * q * q + sx * q + sy] : 0.f;
        };
        for (uint32_t t = 0; t < k; t++)
            for (uint32_t u = 0; u < k; u++)
                v += coupling(i * k + t, m * k + u, letter(a, t), letter(b, u));
        if (m == i + 1)
            for (uint32_t t = 0; t < k; t++)
                for (uint32_t u = t + 1; u < k; u++) {
                    v += coupling(i * k + t, i * k + u, letter(a, t), letter(a, u));
                    if (m == nfold - 1)
                        v += coupling(m * k + t, m * k + u, letter(b, t), letter(b, u));
                }
    }
    Ju[idx] = v;
}

// Sequences of the folded model: 16 of a folded site per thread, site-major rows of
// ldp bytes (ld and ldp are multiples of 16).  Residues are cut to 3 bits, so that none reaches its neighbour's
// byte.
__global__ __launch_bounds__(256) void k_fold_residues(const uint8_t* __restrict__ seq, uint32_t ld,
                                                       uint32_t L, uint32_t q, uint32_t k,
                                                       uint8_t* __restrict__ out, uint32_t ldp) {
    const uint32_t n = (blockIdx.x * 256 + threadIdx.x) * 16, I = blockIdx.y;
    if (n >= ldp) return;
    uint32_t x = 0, y = 0, z = 0, w = 0;
    for (uint32_t t = 0; t < k; t++) {
        uint4 s = make_uint4(0, 0, 0, 0);
        if (I * k + t < L && n < ld) s = *reinterpret_cast<const uint4*>(seq + (size_t)(I * k + t) * ld + n);
        x = x * q + (s.x & 0x07070707u);
        y = y * q + (s.y & 0x07070707u);
        z = z * q + (s.z & 0x07070707u);
        w = w * q + (s.w & 0x07070707u);
    }
    *reinterpret_cast<uint4*>(out + (size_t)I * ldp + n) = make_uint4(x, y, z, w);
}

// Plain streaming kernels over n 16-byte words (grid-stride, eight
// nontemporal loads in flight per thread): the references for the HBM
// bandwidth a kernel reaches.  The read kernel stores the xor of the data
// only if it equals a key the caller passes, so that the loads stay.
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
constexpr int STREAM_U = 8;

__global__ __launch_bounds__(256) void k_stream_copy(const u4v* __restrict__ src,
                                                     u4v* __restrict__ dst, uint64_t n) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + (STREAM_U - 1) * stride < n; i += STREAM_U * stride) {
        u4v v[STREAM_U];
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) v[u] = __builtin_nontemporal_load(&src[i + u * stride]);
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) __builtin_nontemporal_store(v[u], &dst[i + u * stride]);
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void k_stream_read(const u4v* __restrict__ src, uint64_t n,
                                                     uint32_t key, uint32_t* __restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0;
    for (; i + (STREAM_U - 1) * stride < n; i += STREAM_U * stride) {
        u4v v[STREAM_U];
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) v[u] = __builtin_nontemporal_load(&src[i + u * stride]);
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    for (; i < n; i += stride) {
        const u4v a = src[i];
        acc ^= a.x ^ a.y ^ a.z ^ a.w;
    }
    if (acc == key) out[0] = acc;
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t val, uint64_t n) {
    uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < n) p[idx] = val;
}

// Shared site sequence for global steps step0 .. step0+n-1:
// pos = mulhi(Philox(key, (g, 0, TAG_POS)).x, L).  Replaces the host
// RandomState position list (mcmcGPU.py:447-458).
__global__ void k_positions(uint32_t* __restrict__ pos, uint32_t n, uint32_t L, uint32_t k0,
                            uint32_t k1, uint64_t step0) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    uint64_t g = step0 + t;
    uint4 r = philox4x32_10(make_uint4((uint32_t)g, (uint32_t)(g >> 32), 0u, TAG_POS), k0, k1);
    pos[t] = mulhi_range(r.x, L);
}

// Independent-site reseed (gen_indep, mcmc.cl:170-244): residue at site i is
// the number of cumulative probabilities cprob[i][0..q-2] that the uniform
// u = (r >> 8) * 2^-24 reaches, which is what the reference's binary search
// returns for a monotone row.  One thread per walker, site-major output.
__global__ void k_gen_indep(uint8_t* __restrict__ seq, uint32_t ldseq, uint32_t nwalk,
                            const float* __restrict__ cprob, uint32_t L, uint32_t q, uint32_t k0,
                            uint32_t k1, uint32_t call, uint32_t walker_base) {
    uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nwalk) return;
    for (uint32_t k = 0; 4 * k < L; k++) {
        uint4 r = philox4x32_10(make_uint4(k, call, walker_base + w, TAG_INDEP), k0, k1);
        uint32_t rr[4] = {r.x, r.y, r.z, r.w};
        for (uint32_t e = 0; e < 4 && 4 * k + e < L; e++) {
            uint32_t i = 4 * k + e;
            float u = (float)(rr[e] >> 8) * 0x1.0p-24f;
            uint32_t res = 0;
            const float* cp = cprob + (size_t)i * (q - 1);
            for (uint32_t a = 0; a + 1 < q; a++) res += (u >= cp[a]) ? 1u : 0u;
            seq[(size_t)i * ldseq + w] = (uint8_t)res;
        }
    }
}

// Fill every walker with the same sequence (fillSeqs, mcmcGPU.py:927-932).
__global__ void k_fill_seqs(uint8_t* __restrict__ seq, uint32_t ldseq, uint32_t nwalk,
                            const uint8_t* __restrict__ s, uint32_t L) {
    uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (uint64_t)L * nwalk) return;
    uint32_t i = (uint32_t)(idx / nwalk), w = (uint32_t)(idx - (uint64_t)i * nwalk);
    seq[(size_t)i * ldseq + w] = s[i];
}

// Subsequence substitution (copySubseq, mcmc.cl:98-122): every sequence of
// dst takes, at each marked site, the residue of sequence `seqind` of src.
__global__ void k_copy_subseq(uint8_t* __restrict__ dst, uint32_t lddst, uint32_t ndst,
                              const uint8_t* __restrict__ src, uint32_t ldsrc, uint32_t seqind,
                              const uint8_t* __restrict__ marks, uint32_t L) {
    uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (uint64_t)L * ndst) return;
    uint32_t i = (uint32_t)(idx / ndst), w = (uint32_t)(idx - (uint64_t)i * ndst);
    if (marks[i]) dst[(size_t)i * lddst + w] = src[(size_t)i * ldsrc + seqind];
}

}  // namespace mi3
