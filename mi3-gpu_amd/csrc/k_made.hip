// Learned proposal: a masked autoregressive MLP over sequence positions
// (MADE, Germain et al. 2015) used as an independence Metropolis-Hastings
// proposal beside the single-site sweep.
//
// Network (L sites, q letters, H hidden units per layer):
//   h1 = relu(b1 + sum_i W1[:, q*i + s_i])          (one-hot input: a gather-sum)
//   h2 = relu(W2 h1 + b2)
//   logits = W3 h2 + b3,  p(s_j | s_<j) = softmax over the q logits of site j
// with MADE masks baked into the weights (site j's logits see only s_<j).
// GEMMs run in bf16 on the matrix cores with float32 accumulation; the
// one-hot layer, softmax and sampling run in float32.  Sequences are
// site-major (L rows of `ld` bytes), the engine's walker layout.
#include "common.h"

#include <type_traits>

namespace mi3 {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// C = alpha * op(A) op(B) + beta * C + bias[col], optionally relu; fp32 C
// and/or bf16 Cb.  op(A) is M x K (A row-major M x K, or K x M if TA),
// op(B) is K x N (B row-major K x N, or N x K if TB).  Requires M, N, K, lda,
// ldb multiples of 8 and 16-byte aligned A, B (host-checked).
//
// Work-group tile BM x BN, 4 waves (2 x 2), each a (BM/2) x (BN/2) block of
// v_mfma_f32_32x32x16_bf16 tiles; K in steps of 64, both operands in LDS as
// [row or column][k], double-buffered, the next step's global loads in flight
// during this step's products, one barrier a step.  An operand whose memory is
// k-major is transposed on the way: a thread loads 4 (or, in the small tile, 2)
// k-rows of 8 columns and interleaves them in registers (byte permutes), so LDS
// takes 8- or 4-byte stores, not one 2-byte store per element (4872 x 512 x 4096, A k-major: 560 us
// before).  LDS rows are 128 bytes; the 16-byte pieces of row r are permuted
// by r ^ (r >> 3), which spreads both the stores and the reads over the banks.
// Products accumulate in ascending k, 16 at a time, whatever the tile.
constexpr int GK = 64;   // k step

template <int ROWS>
struct GemmStage {
    static constexpr int CHUNKS = ROWS * GK / 8 / 256;   // 16-byte loads per thread
    uint4 v[CHUNKS];
    // LDS byte address of piece kc (8 k) of row r
    __device__ static __forceinline__ uint32_t at(int r, int kc) {
        return (uint32_t)(r * (GK * 2) + ((kc ^ ((r ^ (r >> 3)) & 7)) << 4));
    }
    // T: the operand's memory is k-major (K rows of `rows`), else row-major
    template <bool T>
    __device__ __forceinline__ void load(const bf16* __restrict__ X, int ld, int r0, int rows,
                                         int k0, int K, int tid) {
#pragma unroll
        for (int c = 0; c < CHUNKS; c++) {
            uint4 x = make_uint4(0, 0, 0, 0);
            if (!T) {
                const int i = tid + 256 * c, r = r0 + (i >> 3), k = k0 + (i & 7) * 8;
                if (r < rows && k < K)
                    x = *reinterpret_cast<const uint4*>(X + (size_t)r * ld + k);
            } else {
                // rows 8*rb .. 8*rb + 7 of CHUNKS neighbouring k
                const int r = r0 + 8 * (tid % (ROWS / 8));
                const int k = k0 + CHUNKS * (tid / (ROWS / 8)) + c;
                if (r < rows && k < K)
                    x = *reinterpret_cast<const uint4*>(X + (size_t)k * ld + r);
            }
            v[c] = x;
        }
    }
    template <bool T>
    __device__ __forceinline__ void store(char* lds, int tid) const {
        if (!T) {
#pragma unroll
            for (int c = 0; c < CHUNKS; c++) {
                const int i = tid + 256 * c;
                *reinterpret_cast<uint4*>(lds + at(i >> 3, i & 7)) = v[c];
            }
        } else {
            static_assert(CHUNKS == 4 || CHUNKS == 2, "k-rows of a thread");
            const int rb = tid % (ROWS / 8), kq = tid / (ROWS / 8);
            const uint32_t* q0 = reinterpret_cast<const uint32_t*>(v);
#pragma unroll
            for (int p = 0; p < 4; p++) {   // rows 8*rb + 2p and 2p + 1
                const int r = 8 * rb + 2 * p;
                const uint32_t a0 = q0[p], a1 = q0[4 + p];
                const uint32_t lo = __builtin_amdgcn_perm(a1, a0, 0x05040100u);
                const uint32_t hi = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
                if constexpr (CHUNKS == 4) {
                    const uint32_t a2 = q0[8 + p], a3 = q0[12 + p];
                    *reinterpret_cast<uint2*>(lds + at(r, kq >> 1) + (kq & 1) * 8) =
                        make_uint2(lo, __builtin_amdgcn_perm(a3, a2, 0x05040100u));
                    *reinterpret_cast<uint2*>(lds + at(r + 1, kq >> 1) + (kq & 1) * 8) =
                        make_uint2(hi, __builtin_amdgcn_perm(a3, a2, 0x07060302u));
                } else {
                    *reinterpret_cast<uint32_t*>(lds + at(r, kq >> 2) + (kq & 3) * 4) = lo;
                    *reinterpret_cast<uint32_t*>(lds + at(r + 1, kq >> 2) + (kq & 3) * 4) = hi;
                }
            }
        }
    }
};

template <bool TA, bool TB, int BM, int BN>
__global__ __launch_bounds__(256) void k_gemm_bf16(int M, int N, int K, float alpha,
                                                   const bf16* __restrict__ A, int lda,
                                                   const bf16* __restrict__ B, int ldb,
                                                   float beta, float* __restrict__ C, int ldc,
                                                   bf16* __restrict__ Cb, int ldcb,
                                                   const float* __restrict__ bias, int relu) {
    constexpr int MT = BM / 64, NT = BN / 64;   // 32x32 tiles of a wave
    __shared__ __attribute__((aligned(16))) char As[2][BM * GK * 2];
    __shared__ __attribute__((aligned(16))) char Bs[2][BN * GK * 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    const int lr = lane & 31, lg = lane >> 5;
    f32x16 acc[MT][NT];
#pragma unroll
    for (int x = 0; x < MT; x++)
#pragma unroll
        for (int y = 0; y < NT; y++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[x][y][e] = 0.f;

    GemmStage<BM> a;
    GemmStage<BN> b;
    a.template load<TA>(A, lda, m0, M, 0, K, tid);
    b.template load<!TB>(B, ldb, n0, N, 0, K, tid);
    a.template store<TA>(As[0], tid);
    b.template store<!TB>(Bs[0], tid);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += GK) {
        const bool more = k0 + GK < K;
        if (more) {
            a.template load<TA>(A, lda, m0, M, k0 + GK, K, tid);
            b.template load<!TB>(B, ldb, n0, N, k0 + GK, K, tid);
        }
#pragma unroll
        for (int kk = 0; kk < GK; kk += 16) {
            bf16x8 fa[MT], fb[NT];
#pragma unroll
            for (int x = 0; x < MT; x++)
                fa[x] = *reinterpret_cast<const bf16x8*>(
                    As[buf] + GemmStage<BM>::at(wm + 32 * x + lr, (kk >> 3) + lg));
#pragma unroll
            for (int y = 0; y < NT; y++)
                fb[y] = *reinterpret_cast<const bf16x8*>(
                    Bs[buf] + GemmStage<BN>::at(wn + 32 * y + lr, (kk >> 3) + lg));
#pragma unroll
            for (int x = 0; x < MT; x++)
#pragma unroll
                for (int y = 0; y < NT; y++)
                    acc[x][y] =
                        __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[x], fb[y], acc[x][y], 0, 0, 0);
        }
        if (more) {
            a.template store<TA>(As[buf ^ 1], tid);
            b.template store<!TB>(Bs[buf ^ 1], tid);
        }
        __syncthreads();
        buf ^= 1;
    }
    // D layout of a 32x32 tile: value e of lane l is row 8*(e/4) + 4*(l/32) + e%4,
    // column l%32
#pragma unroll
    for (int x = 0; x < MT; x++)
#pragma unroll
        for (int y = 0; y < NT; y++) {
            const int col = n0 + wn + 32 * y + lr;
            if (col >= N) continue;
            const float bc = bias ? bias[col] : 0.f;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int row = m0 + wm + 32 * x + 8 * (e >> 2) + 4 * lg + (e & 3);
                if (row >= M) continue;
                float v = alpha * acc[x][y][e] + bc;
                if (beta != 0.f) v += beta * C[(size_t)row * ldc + col];
                if (relu) v = fmaxf(v, 0.f);
                if (C) C[(size_t)row * ldc + col] = v;
                if (Cb) Cb[(size_t)row * ldcb + col] = (bf16)v;
            }
        }
}

// h1[b][k] = b1[k] + sum_i W1t[(q*i + s_i)*H + k]  (W1t: (L*q, H), masked);
// h1b = bf16(relu(h1)).  A thread forms V neighbouring units of EMB
// neighbouring sequences, sites in order, four sites' loads in flight.  Bound by
// their latency while the chip has waves to spare, then by the gathered rows from
// L2, which wide loads and several sequences to a thread take in fewer
// instructions.
template <int V, int EMB>
__global__ __launch_bounds__(256) void k_made_embed(const uint8_t* __restrict__ seq, uint32_t ld,
                                                    uint32_t B, uint32_t L, uint32_t q, uint32_t H,
                                                    const float* __restrict__ W1t,
                                                    const float* __restrict__ b1,
                                                    float* __restrict__ h1,
                                                    bf16* __restrict__ h1b) {
    typedef float fv __attribute__((ext_vector_type(V)));
    typedef bf16 bv __attribute__((ext_vector_type(V)));
    const uint32_t nk = H / V, nb = (B + EMB - 1) / EMB;
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (uint64_t)nb * nk) return;
    const uint32_t bg = (uint32_t)(idx / nk), k = (uint32_t)(idx - (uint64_t)bg * nk) * V;
    // sequences past the batch repeat its last one and are not stored
    uint32_t col[EMB];
    fv v[EMB];
#pragma unroll
    for (int e = 0; e < EMB; e++) {
        const uint32_t b = bg * EMB + e;
        col[e] = b < B ? b : B - 1;
        v[e] = *reinterpret_cast<const fv*>(b1 + k);
    }
#pragma unroll 4
    for (uint32_t i = 0; i < L; i++) {
        fv w[EMB];
#pragma unroll
        for (int e = 0; e < EMB; e++)
            w[e] = *reinterpret_cast<const fv*>(
                W1t + (size_t)(q * i + seq[(size_t)i * ld + col[e]]) * H + k);
#pragma unroll
        for (int e = 0; e < EMB; e++) v[e] += w[e];
    }
#pragma unroll
    for (int e = 0; e < EMB; e++) {
        const uint32_t b = bg * EMB + e;
        if (b >= B) break;
        *reinterpret_cast<fv*>(h1 + (size_t)b * H + k) = v[e];
        bv r;
#pragma unroll
        for (int x = 0; x < V; x++) r[x] = (bf16)fmaxf(v[e][x], 0.f);
        *reinterpret_cast<bv*>(h1b + (size_t)b * H + k) = r;
    }
}

// dW1t[(q*i + a)*H + k] = sum over b with s_i(b) == a of dh1[b][k], in batch
// order.  One work-group per (site, 64*V units): it sorts EG_CHUNK sequences
// at a time by their letter at the site (a stable counting sort: the groups of
// 64 sequences are ranked by ballots, and their counts prefixed), and each
// wave sums the rows of every EG_WAVES-th letter in registers, several loads
// in flight.  Bound by the reads of dh1 (once per site) from L2; the sums of
// all letters in LDS instead are a chain of dependent read, add and write per
// sequence (4096 x 232 x 512 units: 273 us, 328 us in groups of four).  Writes
// every entry, so no zeroing is needed; deterministic.
constexpr int EG_WAVES = 4, EG_CHUNK = 2048, EG_GROUPS = EG_CHUNK / 64, EG_QMAX = 25;
constexpr int EG_LPW = (EG_QMAX + EG_WAVES - 1) / EG_WAVES;   // letters of a wave
template <int V>
__global__ __launch_bounds__(64 * EG_WAVES) void k_made_embed_grad(
    const uint8_t* __restrict__ seq, uint32_t ld, uint32_t B, uint32_t L, uint32_t q, uint32_t H,
    const float* __restrict__ dh1, float* __restrict__ dW1t) {
    typedef float fv __attribute__((ext_vector_type(V)));
    __shared__ uint16_t list[EG_CHUNK];             // sequences of the chunk by letter
    __shared__ uint32_t cnt[EG_GROUPS][32];         // per group and letter: count, then place
    __shared__ uint32_t off[33];                    // first place of each letter
    const uint32_t nkb = (H + 64 * V - 1) / (64 * V);
    const uint32_t i = blockIdx.x / nkb;
    const uint32_t lane = threadIdx.x & 63, k = ((blockIdx.x % nkb) * 64 + lane) * V;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool on = k < H;
    const float* gk = dh1 + (on ? k : 0);
    const uint8_t* si = seq + (size_t)i * ld;
    fv acc[EG_LPW];
#pragma unroll
    for (int x = 0; x < EG_LPW; x++) acc[x] = (fv)0.f;
    for (uint32_t c0 = 0; c0 < B; c0 += EG_CHUNK) {
        const uint32_t n = B - c0 < EG_CHUNK ? B - c0 : EG_CHUNK;
        // (a whole chunk with its number of groups known to the compiler: 4% of 4096 x 232
        // x 512)
        auto sort = [&](auto full) __attribute__((always_inline)) {
            // groups, dealt to the waves in turn
            const uint32_t ng = decltype(full)::value ? (uint32_t)EG_GROUPS : (n + 63) / 64;
            // ranks within groups of 64 (sequences past the batch: letter q)
            uint32_t s[EG_GROUPS / EG_WAVES], rank[EG_GROUPS / EG_WAVES];
#pragma unroll
            for (int x = 0; x < EG_GROUPS / EG_WAVES; x++) {
                const uint32_t g = EG_WAVES * x + wave, b = g * 64 + lane;
                s[x] = q;
                if (!decltype(full)::value && g >= ng) continue;
                if (b < n) {
                    s[x] = si[c0 + b];
                    if (s[x] >= q) s[x] = q - 1;
                }
                rank[x] = 0;
                uint32_t c = 0;
                for (uint32_t a = 0; a < q; a++) {
                    const uint64_t m = __ballot(s[x] == a);
                    const uint32_t r = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
                    rank[x] = s[x] == a ? r : rank[x];
                    c = lane == a ? (uint32_t)__popcll(m) : c;
                }
                if (lane < 32) cnt[g][lane] = c;
            }
            __syncthreads();
            // places: letters in order, within a letter the groups in order
            if (threadIdx.x < 32) {
                uint32_t t = 0;
                for (uint32_t g = 0; g < ng; g++) t += cnt[g][threadIdx.x];
                uint32_t before = 0;
                for (uint32_t a = 0; a < q; a++) {
                    const uint32_t ta = __shfl(t, a, 32);
                    before += a < threadIdx.x ? ta : 0u;
                }
                off[threadIdx.x] = before;
                for (uint32_t g = 0; g < ng; g++) {
                    const uint32_t c = cnt[g][threadIdx.x];
                    cnt[g][threadIdx.x] = before;
                    before += c;
                }
                if (threadIdx.x == 31) off[32] = before;
            }
            __syncthreads();
#pragma unroll
            for (int x = 0; x < EG_GROUPS / EG_WAVES; x++) {
                const uint32_t g = EG_WAVES * x + wave;
                if (s[x] < q) list[cnt[g][s[x]] + rank[x]] = (uint16_t)(g * 64 + lane);
            }
            __syncthreads();
        };
        if (n == EG_CHUNK) sort(std::true_type{});
        else sort(std::false_type{});
#pragma unroll
        for (int x = 0; x < EG_LPW; x++) {
            const uint32_t a = wave + EG_WAVES * x;
            if (a >= q) continue;
            const uint32_t e1 = __builtin_amdgcn_readfirstlane(off[a + 1]);
            for (uint32_t e0 = __builtin_amdgcn_readfirstlane(off[a]); e0 < e1; e0 += 64) {
                const uint32_t m = e1 - e0 < 64 ? e1 - e0 : 64;
                const uint32_t mine = lane < m ? list[e0 + lane] : 0u;
                constexpr int U = 8;
                uint32_t u0 = 0;
                for (; u0 + U <= m; u0 += U) {
                    fv g[U];
#pragma unroll
                    for (int u = 0; u < U; u++)
                        g[u] = *reinterpret_cast<const fv*>(
                            gk + (size_t)(c0 + __builtin_amdgcn_readlane(mine, u0 + u)) * H);
#pragma unroll
                    for (int u = 0; u < U; u++) acc[x] += g[u];
                }
                for (; u0 < m; u0++)
                    acc[x] += *reinterpret_cast<const fv*>(
                        gk + (size_t)(c0 + __builtin_amdgcn_readlane(mine, u0)) * H);
            }
        }
        __syncthreads();
    }
    if (!on) return;
#pragma unroll
    for (int x = 0; x < EG_LPW; x++) {
        const uint32_t a = wave + EG_WAVES * x;
        if (a < q) *reinterpret_cast<fv*>(dW1t + (size_t)(q * i + a) * H + k) = acc[x];
    }
}

// The same for few sequences: one work-group per (site, 256 units), a thread keeps
// its unit's sums of every letter in an LDS column of its own and walks the batch,
// eight sequences' letters and gradients loaded before their additions.  No
// sort, whose passes over the letters come to 4 us (rule at the launch).
constexpr int EGF_T = 256;
__global__ __launch_bounds__(EGF_T) void k_made_embed_grad_few(
    const uint8_t* __restrict__ seq, uint32_t ld, uint32_t B, uint32_t q, uint32_t H,
    const float* __restrict__ dh1, float* __restrict__ dW1t) {
    __shared__ float sum[EG_QMAX][EGF_T];
    const uint32_t nkb = (H + EGF_T - 1) / EGF_T, t = threadIdx.x;
    const uint32_t i = blockIdx.x / nkb, k = (blockIdx.x % nkb) * EGF_T + t;
    if (k >= H) return;
    const uint8_t* si = seq + (size_t)i * ld;
    for (uint32_t a = 0; a < q; a++) sum[a][t] = 0.f;
    constexpr uint32_t U = 8;
    auto add = [&](uint32_t letter, float g) {
        const uint32_t a = __builtin_amdgcn_readfirstlane(letter);
        sum[a < q ? a : q - 1][t] += g;
    };
    uint32_t b = 0;
    for (; b + U <= B; b += U) {
        uint32_t s[U];
        float g[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            s[u] = si[b + u];
            g[u] = dh1[(size_t)(b + u) * H + k];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) add(s[u], g[u]);
    }
    for (; b < B; b++) add(si[b], dh1[(size_t)b * H + k]);
    for (uint32_t a = 0; a < q; a++) dW1t[(size_t)(q * i + a) * H + k] = sum[a][t];
}

// Per sequence b (one work-group): nll[b] = -sum_j log softmax(logits_j)[s_j]
// and dlogits = gscale * (softmax - onehot), written bf16 (and fp32 if
// dlf != null).  The sequence's logits go through LDS, so that memory is read
// and written in whole lines (V values a thread) while each thread works on
// its sites' q letters (read and written by their own threads, 84 bytes apart,
// before: 727 us at 4096 x 232 x 21); threads stride over the sites, and the
// block sum is a fixed tree, so nll is deterministic.
template <int V>
__global__ __launch_bounds__(256) void k_made_xent(const float* __restrict__ logits,
                                                   const uint8_t* __restrict__ seq, uint32_t ld,
                                                   uint32_t B, uint32_t L, uint32_t q, float gscale,
                                                   float* __restrict__ nll, bf16* __restrict__ dlb,
                                                   float* __restrict__ dlf) {
    typedef float fv __attribute__((ext_vector_type(V)));
    typedef bf16 bv __attribute__((ext_vector_type(V)));
    extern __shared__ __attribute__((aligned(16))) float xrow[];   // 256 sites x q
    __shared__ float red[256];
    const uint32_t b = blockIdx.x, tid = threadIdx.x;
    const size_t row = (size_t)b * L * q;
    float part = 0.f;
    for (uint32_t j0 = 0; j0 < L; j0 += 256) {
        const uint32_t n = (L - j0 < 256 ? L - j0 : 256) * q;
        const size_t at = row + (size_t)j0 * q;
        for (uint32_t e = tid * V; e < n; e += 256 * V)
            *reinterpret_cast<fv*>(xrow + e) = *reinterpret_cast<const fv*>(logits + at + e);
        __syncthreads();
        const uint32_t j = j0 + tid;
        if (j < L) {
            float* z = xrow + tid * q;
            float mx = -INFINITY;
            for (uint32_t a = 0; a < q; a++) mx = fmaxf(mx, z[a]);
            float se = 0.f;
            for (uint32_t a = 0; a < q; a++) se += expf(z[a] - mx);
            const float lse = mx + logf(se);
            const uint32_t s = seq[(size_t)j * ld + b];
            part += lse - z[s];
            if (dlb || dlf)
                for (uint32_t a = 0; a < q; a++)
                    z[a] = gscale * (expf(z[a] - lse) - (a == s ? 1.f : 0.f));
        }
        __syncthreads();
        if (dlb || dlf) {
            for (uint32_t e = tid * V; e < n; e += 256 * V) {
                const fv g = *reinterpret_cast<const fv*>(xrow + e);
                if (dlf) *reinterpret_cast<fv*>(dlf + at + e) = g;
                if (dlb) {
                    bv r;
#pragma unroll
                    for (int x = 0; x < V; x++) r[x] = (bf16)g[x];
                    *reinterpret_cast<bv*>(dlb + at + e) = r;
                }
            }
            __syncthreads();
        }
    }
    red[tid] = part;
    __syncthreads();
    for (uint32_t off = 128; off > 0; off >>= 1) {
        if (tid < off) red[tid] += red[tid + off];
        __syncthreads();
    }
    if (tid == 0) nll[b] = red[0];
}

// out = dh * (hpre > 0) (fp32) and its bf16 copy.
__global__ void k_relu_grad(uint64_t n, const float* __restrict__ dh,
                            const float* __restrict__ hpre, float* __restrict__ out,
                            bf16* __restrict__ outb) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = hpre[i] > 0.f ? dh[i] : 0.f;
    if (out) out[i] = v;
    if (outb) outb[i] = (bf16)v;
}

// Fused autoregressive pass over all L sites for tiles of MF_T = 16 walkers,
// one work-group of 4 waves per tile (several tiles share a CU): with
// draw != 0 it samples s_j by inversion of u = Philox((j, walker_base + b,
// counter, TAG_MADE)) and writes it to row j of seq; with draw == 0 it reads
// s_j from seq (teacher forcing).  Either way nll[b] = -sum_j log p(s_j).
//
// The degree masks make each hidden unit final once: unit k (degree
// m_k = 1 + k mod (L-1)) of layer 1 sees sites i < m_k, unit k of layer 2
// sees layer-1 units of degree <= m_k, and site j's logits see layer-2 units
// of degree <= j.  So at site j the layer-1 units of degree j have all their
// inputs, the layer-2 units of degree j can be formed from them, and the
// logits need nothing newer: each unit is computed once per walker, at its
// degree, instead of the whole hidden layer at every site (L times less
// matrix-core work than a GEMM per site).
//
// Per site j: (A) layer-1 units of degree j, kept as float32 sums in
// registers (thread t owns units t and t + 256 for the tile's walkers), go
// to LDS as bf16(relu); (B) layer-2 units of degree j: [16 walkers x H] x W2b
// rows of those units on v_mfma_f32_16x16x32_bf16, the k-steps dealt to the
// 4 waves (wave 0 starts from the bias) and the partials summed in a fixed
// order, then bf16(relu(.)) into LDS; (C) site j's q logits the same way
// (one or two column tiles) from the layer-2 units, W3b rows q*j..q*j+q-1 and
// b3; (D) 16 lanes per walker: softmax, draw or read; (E) the float32 layer-1
// sums of units of degree > j add W1t's row of the site's letter (the sums
// are formed in site order, as the teacher-forced embedding forms them).  The
// uniforms of 16 sites are drawn together, one per thread.
//
// Bound by the chain of a site's phases (five barriers, two LDS exchanges of
// partial products, the gather of W1t rows once the letters are known) and,
// with many tiles, by instruction issue and the vector L1.  So a tile takes 40 KiB
// of LDS and 128 registers per lane, four tiles to a CU; the softmax exchanges
// values within its 16 lanes by data-parallel primitives and sums the partials
// itself; loads have no branches and one 32-bit offset per lane.  The
// operands of (B) for site j+1 are loaded after those of site j are used, those of
// (C) after the gathers of (E); when teacher forcing, so are the next site's
// letters.  Measured (us; three tiles to a CU, logits through LDS, shuffles, one
// wave drawing, branches around loads; and this form), draws, L=232 q=21 H=512:
// 65536 walkers 5532 and 4270, 4096 walkers (one tile per CU) 846 and 576; L=96
// q=4 H=256, 32768 walkers 924 and 434.
// Requires H % 32 == 0, H <= 512, q <= 25.
constexpr int MF_T = 16, MF_WAVES = 4, MF_THREADS = 64 * MF_WAVES, MF_HMAX = 512;
constexpr int MF_QMAX = 25;
constexpr int MF_NC = MF_QMAX;                  // columns of the partial products (odd)
static_assert(MF_THREADS == 16 * MF_T, "16 lanes per walker in the softmax");

// KS: k-steps of 32 units per wave; rows are padded by 8 units
template <int KS>
struct MadeFusedLds {
    bf16 h1[MF_T][32 * MF_WAVES * KS + 8]; // bf16(relu(layer 1)), final units only
    bf16 h2[MF_T][32 * MF_WAVES * KS + 8]; // bf16(relu(layer 2)), final units only
    float part[MF_WAVES][MF_T][MF_NC];     // per-wave partial products
    float u[MF_T][MF_T];                   // uniforms of 16 sites
    uint32_t s[MF_T];                      // offsets of the letters' rows of W1t
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

// B operand of one wave's k-steps for one 16-column tile: this lane's 8
// k-values of column lane%16, and the column's bias (the accumulator's start in
// wave 0).  Buffer loads: a uniform base per site, one 32-bit offset per lane for
// all sites, and no branches; what lies past the rows' end reads as zero.
// Columns that nobody reads and k-steps past H, which are not multiplied, hold
// whatever is there.
template <int KS>
struct MadeB {
    bf16x8 b[KS];
    float bias;
};
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t made_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// rows of W from `at` bytes, columns' biases from `bat` bytes
template <int KS>
__device__ __forceinline__ void made_load_b(MadeB<KS>& r, __amdgpu_buffer_rsrc_t W, uint32_t at,
                                            __amdgpu_buffer_rsrc_t bias, uint32_t bat) {
#pragma unroll
    for (int t = 0; t < KS; t++) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(W, (int)(at + 64 * MF_WAVES * t), 0, 0);
        r.b[t] = __builtin_bit_cast(bf16x8, v);
    }
    r.bias = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(bias, (int)bat, 0, 0));
}

// part[wave][.][16 c + .] = bias (wave 0) + X[16 x H] . (this wave's k-steps of b[c])
template <int KS, int NC>
__device__ __forceinline__ void made_product(const bf16 (*X)[32 * MF_WAVES * KS + 8],
                                             const MadeB<KS> (&b)[NC], uint32_t H,
                                             float (*part)[MF_NC], int lr, int lg, int wave) {
    f32x4 acc[NC];
    bf16x8 a[KS];
#pragma unroll
    for (int t = 0; t < KS; t++)
        a[t] = *reinterpret_cast<const bf16x8*>(&X[lr][32 * (wave + MF_WAVES * t) + 8 * lg]);
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[c][e] = wave == 0 ? b[c].bias : 0.f;
#pragma unroll
    for (int t = 0; t < KS; t++) {
        if (t < KS - 1 || 32u * (wave + MF_WAVES * t) < H) {
#pragma unroll
            for (int c = 0; c < NC; c++)
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[c].b[t], acc[c], 0, 0, 0);
        }
    }
    // D layout: value e of lane l is row 4*(l/16) + e, column l%16
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (16 * c + lr < MF_NC) part[4 * lg + e][16 * c + lr] = acc[c][e];
}

__device__ __forceinline__ float made_part_sum(const float (*part)[MF_T][MF_NC], uint32_t r,
                                               uint32_t c) {
    return ((part[0][r][c] + part[1][r][c]) + part[2][r][c]) + part[3][r][c];
}

// Value of another lane of the row of 16 by data-parallel primitives: rotated by
// n lanes, shifted up by n lanes (zero where none is), or lane n's.
constexpr int DPP_ROW_SHR = 0x110, DPP_ROW_ROR = 0x120, DPP_ROW_BCAST = 0x150;
template <int CTRL>
__device__ __forceinline__ float row_dpp(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// KS = ceil(H / 128), NC = ceil(q / 16): smaller networks take less LDS and fewer
// registers, so more tiles share a CU.
template <int KS, int NC>
__global__ __launch_bounds__(MF_THREADS, KS > 2 ? 4 : 5) void k_made_fused(
    uint32_t L, uint32_t q, uint32_t H, uint32_t B, const float* __restrict__ W1t,
    const float* __restrict__ b1, const bf16* __restrict__ W2b, const float* __restrict__ b2,
    const bf16* __restrict__ W3b, const float* __restrict__ b3, uint32_t k0, uint32_t k1,
    uint32_t counter, uint32_t walker_base, uint8_t* __restrict__ seq, uint32_t ld,
    float* __restrict__ nll, int draw) {
    constexpr int HU = (KS + 1) / 2;   // layer-1 units per thread
    __shared__ MadeFusedLds<KS> sm;
    int tid = threadIdx.x, lr = tid & 15, lg = (tid >> 4) & 3;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tile0 = blockIdx.x * MF_T;
    const uint32_t Lm1 = L - 1;
    // units of degree jj: k = (jj - 1) + c (L - 1), c = 0, 1, ...
    auto n_units = [&](uint32_t jj) -> uint32_t {
        return (jj >= 1 && jj < L && jj - 1 < H) ? (H - (jj - 1) + Lm1 - 1) / Lm1 : 0u;
    };
    uint32_t deg[HU];
    float h1r[HU][MF_T];
#pragma unroll
    for (int u = 0; u < HU; u++) {
        const uint32_t k = tid + MF_THREADS * u;
        deg[u] = k < H ? 1 + k % Lm1 : 0xffffffffu;
        const float v = k < H ? b1[k] : 0.f;
#pragma unroll
        for (int w = 0; w < MF_T; w++) h1r[u][w] = v;
    }
    for (uint32_t e = tid; e < sizeof(sm.h1) / sizeof(bf16); e += MF_THREADS) {
        (&sm.h1[0][0])[e] = (bf16)0.f;
        (&sm.h2[0][0])[e] = (bf16)0.f;
    }
    MadeB<KS> w2r[1], w3r[NC];
    const __amdgpu_buffer_rsrc_t w2 = made_rsrc(W2b, H * H * 2), bias2 = made_rsrc(b2, H * 4);
    // operands of the 16 layer-2 units jj - 1 + (c0 + lane % 16) (L - 1)
    auto load_w2 = [&](uint32_t jj, uint32_t c0) {
        const uint32_t row = (jj > 0 ? jj - 1 : 0) + (c0 + lr) * Lm1;
        made_load_b(w2r[0], w2, row * H * 2 + 2 * (32 * wave + 8 * lg), bias2, row * 4);
    };
    auto load_w3 = [&](uint32_t jj) {
        const size_t r0 = (size_t)q * (jj < L ? jj : 0u);
        const __amdgpu_buffer_rsrc_t w3 = made_rsrc(W3b + r0 * H, q * H * 2);
        const __amdgpu_buffer_rsrc_t bias3 = made_rsrc(b3 + r0, q * 4);
#pragma unroll
        for (int t = 0; t < NC; t++)
            made_load_b(w3r[t], w3, (16 * t + lr) * H * 2 + 2 * (32 * wave + 8 * lg), bias3, (16 * t + lr) * 4);
    };
    // teacher forcing: every lane of walker w's group holds its letter at the
    // next site
    uint32_t s_next = 0;
    auto load_s = [&](uint32_t jj) {
        const uint32_t b = tile0 + ((uint32_t)tid >> 4);
        s_next = (!draw && b < B && jj < L) ? seq[(size_t)jj * ld + b] : 0u;
    };
    load_w2(0, 0);
    load_w3(0);
    load_s(0);
    float nacc = 0.f;    // nll of walker tile0 + tid / 16 (every lane of its group)

    for (uint32_t j = 0; j < L; j++) {
        // what depends on the lane is formed anew at each site: kept over the sites, it
        // takes the registers of a fourth tile on the CU
        asm volatile("" : "+v"(tid));
        lr = tid & 15;
        lg = (tid >> 4) & 3;
        // uniforms of sites j .. j + MF_T - 1, one per thread (their last reads, in
        // (D) of site j - 1, lie before the barrier that follows it; the next ones, in
        // (D) of this site, after those of (A) and (C))
        if (draw && j % MF_T == 0) {
            const uint4 r = philox4x32_10(
                make_uint4(j + ((uint32_t)tid >> 4), walker_base + tile0 + (tid & 15), counter,
                           TAG_MADE), k0, k1);
            sm.u[tid >> 4][tid & 15] = (float)(r.x >> 8) * 0x1.0p-24f;
        }
        // (A) layer-1 units of degree j are final
#pragma unroll
        for (int u = 0; u < HU; u++) {
            if (deg[u] == j) {
                const uint32_t k = tid + MF_THREADS * u;
#pragma unroll
                for (int w = 0; w < MF_T; w++) sm.h1[w][k] = (bf16)fmaxf(h1r[u][w], 0.f);
            }
        }
        __syncthreads();
        // (B) layer-2 units of degree j, 16 at a time
        const uint32_t nU = n_units(j);
        for (uint32_t c0 = 0; c0 < nU; c0 += MF_T) {
            if (c0 > 0) load_w2(j, c0);   // the first 16 are there
            made_product(sm.h1, w2r, H, sm.part[wave], lr, lg, wave);
            __syncthreads();
            {
                const uint32_t r = tid / MF_T, c = tid % MF_T;   // 256 = 16 x 16 entries
                if (c0 + c < nU)
                    sm.h2[r][(j - 1) + (c0 + c) * Lm1] =
                        (bf16)fmaxf(made_part_sum(sm.part, r, c), 0.f);
            }
            __syncthreads();
        }
        // (C) logits of site j (columns a < q), b3 included
        made_product(sm.h2, w3r, H, sm.part[wave], lr, lg, wave);
        __syncthreads();
        load_w2(j + 1, 0);
        // (D) softmax and the letter: 16 lanes per walker (walker tid / 16; lane l
        // holds letters l and l + 16): max by row rotations, prefix sums by row
        // shifts, the inverse-CDF search by a ballot for each half of the letters
        float zs, mxs, ses;   // this lane's logit if the letter is s % 16, max, sum
        uint32_t ls;
        {
            const uint32_t w = (uint32_t)tid >> 4, l = (uint32_t)tid & 15;
            const float z1 = (l < q) ? made_part_sum(sm.part, w, l) : -INFINITY;
            const float z2 = (NC > 1 && l + 16 < q) ? made_part_sum(sm.part, w, l + 16) : -INFINITY;
            float mx = fmaxf(z1, z2);
            mx = fmaxf(mx, row_dpp<DPP_ROW_ROR + 8>(mx));
            mx = fmaxf(mx, row_dpp<DPP_ROW_ROR + 4>(mx));
            mx = fmaxf(mx, row_dpp<DPP_ROW_ROR + 2>(mx));
            mx = fmaxf(mx, row_dpp<DPP_ROW_ROR + 1>(mx));
            float c1 = (l < q) ? __expf(z1 - mx) : 0.f;
            float c2 = (l + 16 < q) ? __expf(z2 - mx) : 0.f;
            // inclusive prefix sums over the group (letters in order)
            c1 += row_dpp<DPP_ROW_SHR + 1>(c1), c2 += row_dpp<DPP_ROW_SHR + 1>(c2);
            c1 += row_dpp<DPP_ROW_SHR + 2>(c1), c2 += row_dpp<DPP_ROW_SHR + 2>(c2);
            c1 += row_dpp<DPP_ROW_SHR + 4>(c1), c2 += row_dpp<DPP_ROW_SHR + 4>(c2);
            c1 += row_dpp<DPP_ROW_SHR + 8>(c1), c2 += row_dpp<DPP_ROW_SHR + 8>(c2);
            const float tot1 = row_dpp<DPP_ROW_BCAST + 15>(c1);
            const float se = tot1 + row_dpp<DPP_ROW_BCAST + 15>(c2);
            uint32_t s;
            if (draw) {
                // first letter a (a + 1 < q) whose cumulative mass exceeds u
                const float uu = sm.u[j % MF_T][w] * se;
                const uint64_t m1 = __ballot((l + 1 < q) && uu < c1);
                const uint64_t m2 = __ballot((l + 17 < q) && uu < tot1 + c2);
                const uint32_t sh = (uint32_t)tid & 48u;
                const uint32_t g1 = (uint32_t)(m1 >> sh) & 0xffffu;
                const uint32_t g2 = (uint32_t)(m2 >> sh) & 0xffffu;
                s = g1 ? (uint32_t)__builtin_ctz(g1)
                       : (g2 ? 16u + (uint32_t)__builtin_ctz(g2) : q - 1);
                if (l == 0 && tile0 + w < B) seq[(size_t)j * ld + tile0 + w] = (uint8_t)s;
            } else {
                s = s_next < q ? s_next : q - 1;
            }
            if (l == 0) sm.s[w] = s * H * 4;   // bytes of its row of W1t
            zs = s < 16 ? z1 : z2;
            ls = s & 15;
            mxs = mx;
            ses = se;
        }
        load_s(j + 1);
        __syncthreads();
        // (E) sums of the layer-1 units that see site j.  Waves that hold none read
        // nothing (an empty buffer, zeros); sums that are final already may change.
        float v[HU][MF_T];
#pragma unroll
        for (int u = 0; u < HU; u++) {
            const bool sees = __any(deg[u] != 0xffffffffu && deg[u] > j);
            const __amdgpu_buffer_rsrc_t w1 =
                made_rsrc(W1t + (size_t)(q * j) * H, sees ? q * H * 4 : 0u);
#pragma unroll
            for (int w = 0; w < MF_T; w++)
                v[u][w] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    w1, (int)(sm.s[w] + 4 * (tid + MF_THREADS * u)), 0, 0));
        }
        nacc += mxs + __logf(ses) - __shfl(zs, (int)ls, 16);
#pragma unroll
        for (int u = 0; u < HU; u++)
#pragma unroll
            for (int w = 0; w < MF_T; w++) h1r[u][w] += v[u][w];
        load_w3(j + 1);
    }
    if ((tid & 15) == 0 && tile0 + (tid >> 4) < B) nll[tile0 + (tid >> 4)] = nacc;
}

// Independence Metropolis-Hastings: walker w moves to its proposal with
// probability min(1, exp(-(Ep - Ec) + log q(cur) - log q(prop))), with the
// proposal's negative log-likelihoods nc = -log q(cur), np = -log q(prop);
// u from Philox((counter lo, hi, walker, TAG_MHAC)).  Accepted columns are
// copied (site-major, L rows), with the energy and nll.
__global__ void k_mh_accept(uint32_t N, uint32_t L, uint8_t* __restrict__ cur, uint32_t ldc,
                            const uint8_t* __restrict__ prop, uint32_t ldp,
                            float* __restrict__ Ec, const float* __restrict__ Ep,
                            float* __restrict__ nc, const float* __restrict__ np, uint32_t k0,
                            uint32_t k1, uint64_t counter, uint32_t walker_base,
                            uint32_t* __restrict__ naccept) {
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= N) return;
    const uint4 r = philox4x32_10(
        make_uint4((uint32_t)counter, (uint32_t)(counter >> 32), walker_base + w, TAG_MHAC), k0,
        k1);
    const float u = ((float)(r.x >> 8) + 0.5f) * 0x1.0p-24f;
    const float logr = -(Ep[w] - Ec[w]) - nc[w] + np[w];
    if (logf(u) < logr) {
        for (uint32_t i = 0; i < L; i++) cur[(size_t)i * ldc + w] = prop[(size_t)i * ldp + w];
        Ec[w] = Ep[w];
        nc[w] = np[w];
        atomicAdd(naccept, 1u);
    }
}

// Adam step on float32 parameters p with gradient g (times the 0/1 mask if
// given): m, v moments; bias-corrected with step t >= 1.  Optionally writes
// the bf16 copy pb used by the matrix-core products.
__global__ void k_adam(uint64_t n, float* __restrict__ p, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v,
                       const float* __restrict__ mask, float lr, float b1, float b2, float eps,
                       float c1, float c2, bf16* __restrict__ pb) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    if (mask) gi *= mask[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    if (mask) pi *= mask[i];
    p[i] = pi;
    if (pb) pb[i] = (bf16)pi;
}

// out[c] = sum over rows r of x[r][c] (rows x cols row-major).  A work-group
// takes 32 columns with 8 row lanes each: row lane t sums rows t, t + 8, ...
// in order (each load instruction reads 8 rows x 128 contiguous bytes), then
// the 8 partial sums are added in a fixed order, so the result is
// deterministic.  Bound by the latency of its loads, CS_U of which are in
// flight (one at a time: 440 us at 4096 x 4872).
constexpr int CS_COLS = 32, CS_ROWL = 8, CS_U = 32;
__global__ __launch_bounds__(CS_COLS * CS_ROWL) void k_colsum(uint32_t rows, uint32_t cols,
                                                              const float* __restrict__ x,
                                                              float* __restrict__ out) {
    __shared__ float part[CS_ROWL][CS_COLS + 1];
    const uint32_t cl = threadIdx.x % CS_COLS, t = threadIdx.x / CS_COLS;
    const uint32_t c = blockIdx.x * CS_COLS + cl;
    float s = 0.f;
    if (c < cols) {
        uint32_t r = t;
        for (; r + (CS_U - 1) * CS_ROWL < rows; r += CS_U * CS_ROWL) {
            float v[CS_U];
#pragma unroll
            for (int u = 0; u < CS_U; u++) v[u] = x[(size_t)(r + u * CS_ROWL) * cols + c];
#pragma unroll
            for (int u = 0; u < CS_U; u++) s += v[u];
        }
        for (; r < rows; r += CS_ROWL) s += x[(size_t)r * cols + c];
    }
    part[t][cl] = s;
    __syncthreads();
    if (t == 0 && c < cols) {
        float v = part[0][cl];
#pragma unroll
        for (int k = 1; k < CS_ROWL; k++) v += part[k][cl];
        out[c] = v;
    }
}

// pb = bf16(p).
__global__ void k_to_bf16(uint64_t n, const float* __restrict__ p, bf16* __restrict__ pb) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) pb[i] = (bf16)p[i];
}

}  // namespace mi3
