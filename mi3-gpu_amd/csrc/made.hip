// libmi3hip.so: C ABI of the learned-proposal kernels (k_made.hip).  The
// launchers take raw device pointers and a HIP stream, so that the caller's
// own allocator and stream (the training step's framework) own the memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "k_made.hip"
#include "launch.h"
#include "mi3hip.h"

using namespace mi3;

namespace {
thread_local std::string g_made_error;

int mfail(int code, const std::string& m) {
    g_made_error = m;
    return code;
}

inline hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

inline uint32_t blocks(uint64_t n, uint32_t bs = 256) { return (uint32_t)((n + bs - 1) / bs); }

int launched() {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? MI3_OK : mfail(MI3_EHIP, hipGetErrorString(e));
}

bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Compute units of the current device.
int compute_units() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        return 256;
    return n;
}
}  // namespace

extern "C" {

const char* mi3_made_last_error(void) { return g_made_error.c_str(); }

int mi3_gemm_bf16(void* stream, int transA, int transB, int M, int N, int K, float alpha,
                  const void* A, int lda, const void* B, int ldb, float beta, float* C, int ldc,
                  void* Cb, int ldcb, const float* bias, int relu) {
    if (M <= 0 || N <= 0 || K <= 0 || !A || !B || (!C && !Cb))
        return mfail(MI3_EINVAL, "gemm: bad sizes or null operands");
    if (M % 8 || N % 8 || K % 8 || lda % 8 || ldb % 8 || !al16(A) || !al16(B))
        return mfail(MI3_EINVAL, "gemm: M, N, K, lda, ldb must be multiples of 8, A and B "
                                 "16-byte aligned");
    if ((!transA && lda < K) || (transA && lda < M) || (!transB && ldb < N) ||
        (transB && ldb < K) || (C && ldc < N) || (Cb && ldcb < N))
        return mfail(MI3_EINVAL, "gemm: leading dimension too small");
    if (beta != 0.f && !C) return mfail(MI3_EINVAL, "gemm: beta needs C");
    const bf16* a = static_cast<const bf16*>(A);
    const bf16* b = static_cast<const bf16*>(B);
    bf16* cb = static_cast<bf16*>(Cb);
    // 128 x 128 tiles where they give every CU two and have enough products to pay
    // for their fewer waves; else 64 x 64, which read LDS twice as often per product
    // but are four times as many, and six instead of two to a CU (us, 128 and 64: 4096
    // x 4872 over K = 512 64 and 74, 256 49 and 45, 64 38 and 26; 2904 x 3888 over 8 25
    // and 16; 4872 x 512 over 4096, 156 and 616 tiles, 72 and 62)
    auto tiles = [&](int t) { return (int64_t)((N + t - 1) / t) * ((M + t - 1) / t); };
    const int t = K >= 384 && tiles(128) >= 2 * compute_units() ? 128 : 64;
    const dim3 grid((N + t - 1) / t, (M + t - 1) / t);
#define MI3_G(TA_, TB_)                                                                        \
    if (t == 128)                                                                              \
        hipLaunchKernelGGL((k_gemm_bf16<TA_, TB_, 128, 128>), grid, dim3(256), 0, S(stream), M, N, \
                           K, alpha, a, lda, b, ldb, beta, C, ldc, cb, ldcb, bias, relu);      \
    else                                                                                       \
        hipLaunchKernelGGL((k_gemm_bf16<TA_, TB_, 64, 64>), grid, dim3(256), 0, S(stream), M, N, \
                           K, alpha, a, lda, b, ldb, beta, C, ldc, cb, ldcb, bias, relu)
    if (!transA && !transB) { MI3_G(false, false); }
    else if (!transA && transB) { MI3_G(false, true); }
    else if (transA && !transB) { MI3_G(true, false); }
    else { MI3_G(true, true); }
#undef MI3_G
    return launched();
}

int mi3_made_embed(void* stream, const uint8_t* seq, uint32_t ld, uint32_t B, uint32_t L,
                   uint32_t q, uint32_t H, const float* W1t, const float* b1, float* h1,
                   void* h1b) {
    if (!seq || !W1t || !b1 || !h1 || !h1b || ld < B || q < 2 || q > MAX_Q)
        return mfail(MI3_EINVAL, "made_embed: bad arguments");
    if (B == 0 || H == 0) return mfail(MI3_EHIP, "made_embed: no sequences or no units");
    bf16* hb = static_cast<bf16*>(h1b);
    // One unit of one sequence to a thread while those are few, else four units of one
    // sequence, then of four (us alone at L=232 q=21, 512 units, by units and sequences
    // of a thread: 64 sequences 1/1 16, 4/1 26, 4/4 66; 512 34, 34, 72; 2048 73, 47, 68;
    // 4096 145, 91, 83, and 76 of 4/2, which beside other contexts' steps cost 4 more
    // than 4/4; where units are no multiple of 4, 1024 38 and 1/4 47, 2048 73 and 61)
    const uint64_t n = (uint64_t)B * H;
#define MI3_EMBED(V, E)                                                                          \
    hipLaunchKernelGGL((k_made_embed<V, E>), dim3(blocks((uint64_t)((B + E - 1) / E) * (H / V))), \
                       dim3(256), 0, S(stream), seq, ld, B, L, q, H, W1t, b1, h1, hb)
    const bool wide = H % 4 == 0 && al16(W1t) && al16(b1) && al16(h1) && al16(h1b);
    if (wide && n > 3ull << 19) MI3_EMBED(4, 4);
    else if (wide && n > 3ull << 17) MI3_EMBED(4, 1);
    else if (n > 3ull << 18) MI3_EMBED(1, 4);
    else MI3_EMBED(1, 1);
#undef MI3_EMBED
    return launched();
}

static_assert(MAX_Q <= (uint32_t)EG_QMAX, "letter sums of the embedding gradient");

int mi3_made_embed_grad(void* stream, const uint8_t* seq, uint32_t ld, uint32_t B, uint32_t L,
                        uint32_t q, uint32_t H, const float* dh1, float* dW1t) {
    if (!seq || !dh1 || !dW1t || ld < B || q < 2 || q > MAX_Q)
        return mfail(MI3_EINVAL, "made_embed_grad: bad arguments");
    if (L == 0 || H == 0) return MI3_OK;
    // sorting takes longer by the letters, and by the work-groups that share a CU, summing
    // in LDS by the sequences (us, sorted and not: 64 sequences of L=232 q=21, 512 units
    // 10.6 and 7.4, 128 12.3 and 11.2, 256 14.1 and 18.1; q=25, 200 sequences of L=100 12.6
    // and 12.6; q=4, 64 sequences of L=93 4.9 and 5.1; L=318 in 6 work-groups a site,
    // 359 units, 128 sequences q=2 11.5 and 9.9, q=25 22.6 and 12.4, 256 17.1 and 17.4,
    // 25.2 and 20.2)
    const bool wide = H % 4 == 0 && al16(dh1) && al16(dW1t);
    const int64_t groups = (int64_t)L * (wide ? (H + 255) / 256 : (H + 63) / 64);
    const int64_t few = 7 * q + std::max<int64_t>(0, groups - 4 * compute_units()) / 4;
    if (B <= few)
        hipLaunchKernelGGL(k_made_embed_grad_few, dim3(L * ((H + EGF_T - 1) / EGF_T)), dim3(EGF_T), 0,
                           S(stream), seq, ld, B, q, H, dh1, dW1t);
    else if (wide)
        hipLaunchKernelGGL(k_made_embed_grad<4>, dim3(L * ((H + 255) / 256)), dim3(64 * EG_WAVES), 0,
                           S(stream), seq, ld, B, L, q, H, dh1, dW1t);
    else
        hipLaunchKernelGGL(k_made_embed_grad<1>, dim3(L * ((H + 63) / 64)), dim3(64 * EG_WAVES), 0,
                           S(stream), seq, ld, B, L, q, H, dh1, dW1t);
    return launched();
}

int mi3_made_xent(void* stream, const float* logits, const uint8_t* seq, uint32_t ld, uint32_t B,
                  uint32_t L, uint32_t q, float gscale, float* nll, void* dlogits_bf16,
                  float* dlogits) {
    if (!logits || !seq || !nll || ld < B || q < 2 || q > MAX_Q || B == 0)
        return mfail(MI3_EINVAL, "made_xent: bad arguments");
    const size_t lds = (size_t)(L < 256 ? L : 256) * q * sizeof(float);   // logits of 256 sites
    bf16* dlb = static_cast<bf16*>(dlogits_bf16);
    auto kern = ((uint64_t)L * q % 4 == 0 && al16(logits) && al16(dlogits) && al16(dlb))
                    ? k_made_xent<4> : k_made_xent<1>;
    hipLaunchKernelGGL(kern, dim3(B), dim3(256), lds, S(stream), logits, seq, ld, B, L, q, gscale,
                       nll, dlb, dlogits);
    return launched();
}

int mi3_relu_grad(void* stream, uint64_t n, const float* dh, const float* hpre, float* out,
                  void* outb) {
    if (!dh || !hpre || (!out && !outb)) return mfail(MI3_EINVAL, "relu_grad: bad arguments");
    hipLaunchKernelGGL(k_relu_grad, dim3(blocks(n)), dim3(256), 0, S(stream), n, dh, hpre, out,
                       static_cast<bf16*>(outb));
    return launched();
}

int mi3_made_fused(void* stream, uint32_t L, uint32_t q, uint32_t H, uint32_t B, const float* W1t,
                   const float* b1, const void* W2b, const float* b2, const void* W3b,
                   const float* b3, uint64_t seed, uint32_t counter, uint32_t walker_base,
                   uint8_t* seq, uint32_t ld, float* nll, int draw) {
    if (!W1t || !b1 || !W2b || !b2 || !W3b || !b3 || !seq || !nll || L < 2 || q < 2 ||
        ld < B || !al16(W2b) || !al16(W3b))
        return mfail(MI3_EINVAL, "made_fused: bad arguments");
    if (q > (uint32_t)MF_QMAX || H == 0 || H % 32 || H > (uint32_t)MF_HMAX)
        return mfail(MI3_EUNSUP, "made_fused: needs q <= 25 and H a multiple of 32 up to 512");
    if (B == 0) return MI3_OK;
    const uint32_t ks = (H + 127) / 128;
    auto kern = q > 16 ? (ks == 1 ? k_made_fused<1, 2> : ks == 2 ? k_made_fused<2, 2>
                          : ks == 3 ? k_made_fused<3, 2> : k_made_fused<4, 2>)
                       : (ks == 1 ? k_made_fused<1, 1> : ks == 2 ? k_made_fused<2, 1>
                          : ks == 3 ? k_made_fused<3, 1> : k_made_fused<4, 1>);
    hipLaunchKernelGGL(kern, dim3((B + MF_T - 1) / MF_T), dim3(MF_THREADS), 0, S(stream),
                       L, q, H, B, W1t, b1, static_cast<const bf16*>(W2b), b2,
                       static_cast<const bf16*>(W3b), b3, (uint32_t)seed, (uint32_t)(seed >> 32),
                       counter, walker_base, seq, ld, nll, draw);
    return launched();
}

int mi3_mh_accept(void* stream, uint32_t N, uint32_t L, uint8_t* cur, uint32_t ldc,
                  const uint8_t* prop, uint32_t ldp, float* Ecur, const float* Eprop,
                  float* nll_cur, const float* nll_prop, uint64_t seed, uint64_t counter,
                  uint32_t walker_base, uint32_t* naccept) {
    if (!cur || !prop || !Ecur || !Eprop || !nll_cur || !nll_prop || !naccept || ldc < N ||
        ldp < N)
        return mfail(MI3_EINVAL, "mh_accept: bad arguments");
    hipLaunchKernelGGL(k_mh_accept, dim3(blocks(N)), dim3(256), 0, S(stream), N, L, cur, ldc, prop,
                       ldp, Ecur, Eprop, nll_cur, nll_prop, (uint32_t)seed,
                       (uint32_t)(seed >> 32), counter, walker_base, naccept);
    return launched();
}

int mi3_adam_step(void* stream, uint64_t n, float* p, const float* g, float* m, float* v,
                  const float* mask, float lr, float beta1, float beta2, float eps, uint32_t t,
                  void* pb) {
    if (!p || !g || !m || !v || t == 0) return mfail(MI3_EINVAL, "adam: bad arguments");
    const float c1 = 1.f - powf(beta1, (float)t), c2 = 1.f - powf(beta2, (float)t);
    hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(256), 0, S(stream), n, p, g, m, v, mask, lr,
                       beta1, beta2, eps, c1, c2, static_cast<bf16*>(pb));
    return launched();
}

int mi3_colsum(void* stream, uint32_t rows, uint32_t cols, const float* x, float* out) {
    if (!x || !out) return mfail(MI3_EINVAL, "colsum: bad arguments");
    if (cols == 0) return MI3_OK;
    hipLaunchKernelGGL(k_colsum, dim3((cols + CS_COLS - 1) / CS_COLS), dim3(CS_COLS * CS_ROWL), 0,
                       S(stream), rows, cols, x, out);
    return launched();
}

int mi3_to_bf16(void* stream, uint64_t n, const float* p, void* pb) {
    if (!p || !pb) return mfail(MI3_EINVAL, "to_bf16: bad arguments");
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks(n)), dim3(256), 0, S(stream), n, p,
                       static_cast<bf16*>(pb));
    return launched();
}

}  // extern "C"
