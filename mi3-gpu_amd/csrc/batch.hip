// libmi3hip.so, batched models: many independent Potts models of uneven L
// and q, each with its own walkers, couplings and random streams, swept by
// (state words, chunk class) class: unstaged, one class after another, or by a
// persistent kernel per class on parallel branches.  One round (positions of
// every model, the class sweeps, the step-counter advance) is captured once into
// a HIP graph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "common.h"
#include "launch.h"
#include "mi3hip.h"

using namespace mi3;

namespace {

// Site lists of every model for this launch:
// pos_m[t] = mulhi(Philox((step_m + t, 0, TAG_POS)).x, L_m), the stream of
// a single-model context keyed by the model's seed.
__global__ void k_batch_positions(const BatchModel* __restrict__ models, uint32_t* const* pos) {
    const BatchModel m = models[blockIdx.y];
    const uint64_t step0 = *m.step;
    uint32_t* p = pos[blockIdx.y];
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < m.nsteps;
         t += gridDim.x * blockDim.x) {
        const uint64_t g = step0 + t;
        uint4 r = philox4x32_10(make_uint4((uint32_t)g, (uint32_t)(g >> 32), 0u, TAG_POS), m.k0,
                                m.k1);
        p[t] = mulhi_range(r.x, m.L);
    }
}

// Step counters move past this launch, kept even (as a single-model context).
__global__ void k_batch_advance(const BatchModel* __restrict__ models, uint64_t* steps,
                                uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) steps[i] += models[i].nsteps + (models[i].nsteps & 1u);
}

__global__ void k_batch_zero(uint32_t* __restrict__ p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

struct ClassKey {
    uint32_t kw, pf;
    bool operator<(const ClassKey& o) const { return kw != o.kw ? kw < o.kw : pf < o.pf; }
};

struct ClassRun {
    std::vector<uint32_t> models;
    bool fixed = false;      // form and tile asked for, or kept by the autotuner
    uint32_t wpb = 0;        // walkers per tile
    bool direct = false;     // swept without staging
    BatchTile* tiles = nullptr;
    uint32_t ntiles = 0;
    hipStream_t side = nullptr;
};

}  // namespace

struct mi3_batch {
    int dev = 0;
    hipStream_t stream = nullptr;
    std::string err;
    uint64_t seed = 0;
    uint32_t n = 0;
    std::vector<uint32_t> L, q, N, nchunk;
    std::vector<float*> Jp, Ju;      // packed / chunked couplings
    std::vector<uint8_t*> seq;
    std::vector<uint32_t*> pos;
    std::vector<uint32_t> pos_cap;
    std::vector<BatchModel> host_models;
    BatchModel* models = nullptr;    // device copy
    uint32_t** pos_ptrs = nullptr;   // device array of the pos pointers
    uint64_t* steps = nullptr;
    uint32_t* counters = nullptr;    // one per class
    std::map<ClassKey, ClassRun> classes;
    uint32_t nsweeps = 0;            // of the captured graph
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph = nullptr;
    uint32_t ncu = 0;
};

namespace {

int bfail(mi3_batch* b, int code, const std::string& m) {
    if (b) b->err = m;
    return code;
}

#define BCHK(b, call)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (call);                                                            \
        if (e_ != hipSuccess)                                                              \
            return bfail(b, MI3_EHIP, std::string(#call) + ": " + hipGetErrorString(e_));  \
    } while (0)

thread_local std::string g_batch_create_error;

void drop_graph(mi3_batch* b) {
    if (b->exec) hipGraphExecDestroy(b->exec);
    if (b->graph) hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->nsweeps = 0;
}

// Walkers per tile allowed for a class.
std::vector<uint32_t> tile_options(uint32_t kw) {
    if (kw >= 5) return {128, 256};
    return {128, 256, 512};
}

uint32_t units(const mi3_batch* b) { return b->ncu ? b->ncu : 256; }

// Walkers up to which a class may be swept unstaged.  Beyond, the rows that its
// waves read at a time leave the L2s (us a step, unstaged and in tiles of 128:
// 8192 walkers of L=232 q=21 5.6 and 6.9, L=93 2.5 and 2.8, but L=300 11.0 and
// 8.6, L=400 19 and 11; 4096 of L=300 4.1 and 8.6, L=600 8.8 and 20).
bool may_be_unstaged(const mi3_batch* b, const ClassKey& key, const ClassRun& cr) {
    uint64_t total = 0;
    for (uint32_t m : cr.models) total += b->N[m];
    return total <= (uint64_t)(key.pf == 1 ? 24 : key.kw <= 2 ? 32 : 16) * units(b);
}

// A class whose couplings an XCD's L2 holds (4 MiB).
bool l2_resident(const mi3_batch* b, const ClassRun& cr) {
    uint64_t bytes = 0;
    for (uint32_t m : cr.models) bytes += (uint64_t)b->L[m] * b->nchunk[m] * b->q[m] * b->q[m] * CH * 4;
    return bytes <= 4u << 20;
}

// Times of a sweep of a class alone on the card: unstaged; staged, and then its
// share of the card's CUs.
struct ClassTimes {
    double direct, staged, card;
    bool resident;
};

// What a batch takes whose classes d are swept unstaged: those run one after
// another, and the staged ones beside each other, after them or beside those
// whose couplings the L2s hold (enqueue_round).
double batch_time(const std::vector<ClassTimes>& t, const std::vector<bool>& d) {
    double first = 0, beside = 0, longest = 0, card = 0;
    for (size_t i = 0; i < t.size(); i++) {
        if (d[i]) {
            (t[i].resident ? beside : first) += t[i].direct;
        } else {
            longest = std::max(longest, t[i].staged);
            card += t[i].card;
        }
    }
    return first + std::max(std::max(longest, card), beside);
}

// The classes to sweep unstaged: of those that may be, the first of the longest
// staged ones, the first two, and so on are tried; times(d) gives the classes'
// times if the classes d are unstaged.
template <typename F>
std::vector<bool> choose_unstaged(const std::vector<bool>& may, F times) {
    std::vector<bool> d(may.size(), false), best = d;
    const std::vector<ClassTimes> t = times(d);
    std::vector<size_t> order;
    for (size_t i = 0; i < may.size(); i++)
        if (may[i]) order.push_back(i);
    std::sort(order.begin(), order.end(),
              [&](size_t x, size_t y) { return t[x].staged > t[y].staged; });
    double least = batch_time(t, d);
    for (size_t i : order) {
        d[i] = true;
        const double all = batch_time(times(d), d);
        if (all < least) {
            least = all;
            best = d;
        }
    }
    return best;
}

// Estimate of those times in tiles of w walkers, in us (within a third of what
// L=40 to 1000 with 512 to 8192 walkers took, to where may_be_unstaged ends).  An
// unstaged step waits for its gathers, and shares the L2s' lines (as many of a
// chunk as its 32 sites have letters) with the class's other walkers; a staged
// step takes the copies of its chunks, or the gathers of the tile's walkers.
ClassTimes estimate(const mi3_batch* b, const ClassKey& key, const ClassRun& cr, uint32_t w) {
    static const double per_chunk[4][3] = {
        {0.37, 0.55, 0.92}, {0.66, 0.70, 1.0}, {0.90, 0.94, 1.05}, {1.15, 1.2, 1.3}};
    const double chunk = per_chunk[key.pf == 1 ? 0 : key.pf == 4 ? 1 : key.pf == 7 ? 2 : 3]
                                  [w == 128 ? 0 : w == 256 ? 1 : 2] *
                         (key.kw >= 5 && key.pf > 1 ? 1.15 : key.kw == 4 && w == 512 ? 1.2 : 1.0);
    ClassTimes t{0, 0, 0, l2_resident(b, cr)};
    double gathers = 0, tiles = 0;
    for (uint32_t m : cr.models) {
        const double L = b->L[m], q = b->q[m], nc = b->nchunk[m];
        t.direct = std::max(t.direct, L * (0.55 + 0.05 * nc));
        gathers += L * nc * b->N[m] * q * (1 - std::pow(1 - 1 / q, 32)) * 4.9e-6;
        const double step = L * (0.3 + chunk * nc);
        t.staged = std::max(t.staged, step);
        tiles += step * (b->N[m] / w);
    }
    t.direct += gathers;
    t.card = tiles / units(b);
    t.staged = std::max(t.staged, t.card);
    return t;
}

// Tiles of a class of w walkers; larger models first so that the tail of the
// persistent loop is short.
int build_tiles(mi3_batch* b, ClassRun& cr, uint32_t w, bool direct) {
    std::vector<BatchTile> t;
    std::vector<uint32_t> order = cr.models;
    std::stable_sort(order.begin(), order.end(),
                     [&](uint32_t x, uint32_t y) { return b->L[x] > b->L[y]; });
    for (uint32_t m : order)
        for (uint32_t blk = 0; blk < b->N[m] / w; blk++) t.push_back({m, blk});
    if (cr.tiles) hipFree(cr.tiles);
    cr.tiles = nullptr;
    BCHK(b, hipMalloc(&cr.tiles, std::max<size_t>(1, t.size()) * sizeof(BatchTile)));
    BCHK(b, hipMemcpy(cr.tiles, t.data(), t.size() * sizeof(BatchTile), hipMemcpyHostToDevice));
    cr.ntiles = (uint32_t)t.size();
    cr.wpb = w;
    cr.direct = direct;
    return MI3_OK;
}

// Forms and tiles of the classes that nobody fixed: tiles of the most walkers, or
// smaller where all staged classes' together leave most of the card free.
int choose_tiles(mi3_batch* b) {
    std::vector<bool> may;
    for (auto& kv : b->classes) may.push_back(!kv.second.fixed && may_be_unstaged(b, kv.first, kv.second));
    auto tile = [&](const std::vector<bool>& d) {
        uint64_t walkers = 0;
        size_t i = 0;
        for (auto& kv : b->classes)
            if (!d[i++])
                for (uint32_t m : kv.second.models) walkers += b->N[m];
        // (a third of the card: three batches beside each other find room)
        return chunk_tile((uint32_t)std::min<uint64_t>(walkers, 1u << 30), 512, units(b) * 4 / 3);
    };
    auto class_tile = [](const ClassKey& key, uint32_t w) {
        return std::min(w, tile_options(key.kw).back());
    };
    const std::vector<bool> direct = choose_unstaged(may, [&](const std::vector<bool>& d) {
        std::vector<ClassTimes> t;
        const uint32_t w = tile(d);
        for (auto& kv : b->classes) {
            const ClassRun& cr = kv.second;
            t.push_back(estimate(b, kv.first, cr, cr.fixed ? cr.wpb : class_tile(kv.first, w)));
            if (cr.fixed && cr.direct) t.back().staged = t.back().card = t.back().direct;
        }
        return t;
    });
    const uint32_t w = tile(direct);
    size_t i = 0;
    for (auto& kv : b->classes) {
        if (!kv.second.fixed)
            if (const int rc = build_tiles(b, kv.second, class_tile(kv.first, w), direct[i])) return rc;
        i++;
    }
    return MI3_OK;
}

uint32_t class_grid(mi3_batch* b, const ClassRun& cr) {
    return std::min<uint32_t>(cr.ntiles, units(b));
}

// The sweep of one class on stream st.
hipError_t sweep_class(mi3_batch* b, const ClassKey& key, const ClassRun& cr, uint32_t* counter,
                       hipStream_t st) {
    if (cr.direct) {
        uint32_t qmin = MAX_Q;
        for (uint32_t m : cr.models) qmin = std::min(qmin, b->q[m]);
        return launch_sweep_batch_direct(key.kw, qmin, cr.wpb, cr.ntiles * cr.wpb, units(b), b->models,
                                         cr.tiles, cr.ntiles, st);
    }
    return launch_sweep_batch(key.kw, key.pf, cr.wpb, b->models, cr.tiles, cr.ntiles, counter,
                              class_grid(b, cr), st);
}

// Per-model descriptors for nsweeps sweeps (nsteps = nsweeps * L).
int upload_models(mi3_batch* b, uint32_t nsweeps) {
    for (uint32_t m = 0; m < b->n; m++) {
        const uint32_t ns = nsweeps * b->L[m];
        if (b->pos_cap[m] < ns) {
            if (b->pos[m]) hipFree(b->pos[m]);
            b->pos[m] = nullptr;
            BCHK(b, hipMalloc(&b->pos[m], (size_t)ns * 4));
            b->pos_cap[m] = ns;
        }
        BatchModel& d = b->host_models[m];
        d.Ju = b->Ju[m];
        d.seq = b->seq[m];
        d.pos = b->pos[m];
        d.step = b->steps + m;
        d.ld = b->N[m];
        d.L = b->L[m];
        d.q = b->q[m];
        d.nchunk = b->nchunk[m];
        d.nsteps = ns;
        d.k0 = (uint32_t)(b->seed + m);
        d.k1 = (uint32_t)((b->seed + m) >> 32);
        d.walker_base = 0;
        d.nbeta = -1.f;
        d.pad_ = 0;
    }
    BCHK(b, hipMemcpy(b->models, b->host_models.data(), b->n * sizeof(BatchModel),
                      hipMemcpyHostToDevice));
    BCHK(b, hipMemcpy(b->pos_ptrs, b->pos.data(), b->n * sizeof(uint32_t*),
                      hipMemcpyHostToDevice));
    return MI3_OK;
}

uint32_t max_steps(mi3_batch* b) {
    uint32_t mx = 0;
    for (auto& d : b->host_models) mx = std::max(mx, d.nsteps);
    return mx;
}

// Enqueue one round on b->stream (also used under stream capture):
// positions, class sweeps forked onto side streams, join, step advance.
int enqueue_round(mi3_batch* b, std::vector<hipEvent_t>& events) {
    const uint32_t nclass = (uint32_t)b->classes.size();
    hipLaunchKernelGGL(k_batch_zero, dim3(1), dim3(64), 0, b->stream, b->counters, nclass);
    const uint32_t mx = max_steps(b);
    hipLaunchKernelGGL(k_batch_positions, dim3(std::max(1u, std::min(64u, (mx + 255) / 256)), b->n),
                       dim3(256), 0, b->stream, (const BatchModel*)b->models,
                       (uint32_t* const*)b->pos_ptrs);
    BCHK(b, hipGetLastError());
    // unstaged classes first, one after another: side by side, or beside staged ones,
    // their waves start or drift apart, the rows they share leave the L2s, and
    // each takes several times as long (L=301 q=4 and L=400 q=21, 1024 walkers, 4
    // sweeps: 1.0 and 3.2 ms alone, 9.2 ms together; L=400 and 600 q=21, 2048 walkers, 2
    // sweeps: 8.7 ms one after another, 16.6 with the first staged beside the second).
    // Those that the L2s hold follow each other beside the staged ones
    for (auto& kv : b->classes)
        if (kv.second.direct && !l2_resident(b, kv.second)) {
            const hipError_t e = sweep_class(b, kv.first, kv.second, nullptr, b->stream);
            if (e != hipSuccess)
                return bfail(b, MI3_EHIP, std::string("batch sweep: ") + hipGetErrorString(e));
        }
    hipEvent_t fork;
    BCHK(b, hipEventCreateWithFlags(&fork, hipEventDisableTiming));
    events.push_back(fork);
    BCHK(b, hipEventRecord(fork, b->stream));
    uint32_t ci = 0;
    int rc = MI3_OK;
    hipStream_t beside = nullptr;
    for (auto& kv : b->classes) {
        ClassRun& cr = kv.second;
        if (cr.direct && !l2_resident(b, cr)) continue;
        if (cr.direct && !beside) beside = cr.side;
        hipStream_t s = cr.direct ? beside : cr.side;
        if (hipStreamWaitEvent(s, fork, 0) != hipSuccess) { rc = bfail(b, MI3_EHIP, "fork"); break; }
        hipError_t e = sweep_class(b, kv.first, cr, b->counters + ci, s);
        if (e != hipSuccess) {
            rc = bfail(b, MI3_EHIP, std::string("batch sweep: ") + hipGetErrorString(e));
            break;
        }
        hipEvent_t j;
        if (hipEventCreateWithFlags(&j, hipEventDisableTiming) != hipSuccess) {
            rc = bfail(b, MI3_EHIP, "event");
            break;
        }
        events.push_back(j);
        if (hipEventRecord(j, s) != hipSuccess || hipStreamWaitEvent(b->stream, j, 0) != hipSuccess) {
            rc = bfail(b, MI3_EHIP, "join");
            break;
        }
        ci++;
    }
    if (rc == MI3_OK) {
        hipLaunchKernelGGL(k_batch_advance, dim3((b->n + 255) / 256), dim3(256), 0, b->stream,
                           (const BatchModel*)b->models, b->steps, b->n);
        if (hipGetLastError() != hipSuccess) rc = bfail(b, MI3_EHIP, "advance");
    }
    return rc;
}

}  // namespace

extern "C" {

int mi3_batch_create(int device, uint32_t nmodels, const uint32_t* L, const uint32_t* q,
                     const uint32_t* nwalkers, uint64_t seed, mi3_batch** out) {
    if (!out) return MI3_EINVAL;
    *out = nullptr;
    if (nmodels == 0 || !L || !q || !nwalkers) {
        g_batch_create_error = "need at least one model";
        return MI3_EINVAL;
    }
    for (uint32_t m = 0; m < nmodels; m++) {
        if (L[m] < 2 || q[m] < 2 || q[m] > MAX_Q || L[m] > MAX_L || !chunked_fits(L[m], q[m])) {
            g_batch_create_error = "model " + std::to_string(m) + ": need 2 <= L <= " +
                                   std::to_string(MAX_L) + " and 2 <= q <= " +
                                   std::to_string(MAX_Q) +
                                   ", with chunked couplings under 4 GiB";
            return MI3_EUNSUP;
        }
        if (nwalkers[m] == 0 || nwalkers[m] % 512) {
            g_batch_create_error = "model " + std::to_string(m) +
                                   ": walkers must be a positive multiple of 512";
            return MI3_EINVAL;
        }
    }
    if (hipSetDevice(device) != hipSuccess) {
        g_batch_create_error = "bad device";
        return MI3_EHIP;
    }
    mi3_batch* b = new mi3_batch();
    b->dev = device;
    b->seed = seed;
    b->n = nmodels;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) b->ncu = prop.multiProcessorCount;
    int rc = MI3_OK;
    auto bad = [&](const char* what) {
        g_batch_create_error = what;
        rc = MI3_ENOMEM;
    };
    if (hipStreamCreate(&b->stream) != hipSuccess) bad("stream");
    b->L.assign(L, L + nmodels);
    b->q.assign(q, q + nmodels);
    b->N.assign(nwalkers, nwalkers + nmodels);
    b->nchunk.resize(nmodels);
    b->Jp.assign(nmodels, nullptr);
    b->Ju.assign(nmodels, nullptr);
    b->seq.assign(nmodels, nullptr);
    b->pos.assign(nmodels, nullptr);
    b->pos_cap.assign(nmodels, 0);
    b->host_models.resize(nmodels);
    for (uint32_t m = 0; m < nmodels && rc == MI3_OK; m++) {
        const uint32_t nc = (L[m] + CH - 1) / CH;
        b->nchunk[m] = nc;
        const size_t np = (size_t)L[m] * (L[m] - 1) / 2 * q[m] * q[m];
        if (hipMalloc(&b->Jp[m], np * 4) != hipSuccess ||
            hipMalloc(&b->Ju[m], (size_t)L[m] * nc * chunk_floats(q[m]) * 4) != hipSuccess ||
            hipMalloc(&b->seq[m], (size_t)L[m] * nwalkers[m]) != hipSuccess)
            bad("device memory for a model");
        else {
            hipMemset(b->Jp[m], 0, np * 4);
            hipMemset(b->seq[m], 0, (size_t)L[m] * nwalkers[m]);
        }
        ClassKey k{state_words(L[m]), pf_class(q[m])};
        b->classes[k].models.push_back(m);
    }
    if (rc == MI3_OK &&
        (hipMalloc(&b->models, nmodels * sizeof(BatchModel)) != hipSuccess ||
         hipMalloc(&b->pos_ptrs, nmodels * sizeof(uint32_t*)) != hipSuccess ||
         hipMalloc(&b->steps, nmodels * sizeof(uint64_t)) != hipSuccess ||
         hipMalloc(&b->counters, b->classes.size() * sizeof(uint32_t)) != hipSuccess))
        bad("device memory for descriptors");
    if (rc == MI3_OK) {
        hipMemset(b->steps, 0, nmodels * sizeof(uint64_t));
        for (uint32_t m = 0; m < nmodels && rc == MI3_OK; m++)
            if (launch_unpack_chunked(b->Jp[m], b->Ju[m], L[m], q[m], b->nchunk[m], b->stream) !=
                hipSuccess)
                bad("unpack");
        for (auto& kv : b->classes) {
            if (rc != MI3_OK) break;
            if (hipStreamCreate(&kv.second.side) != hipSuccess) bad("stream");
        }
        if (rc == MI3_OK && choose_tiles(b) != MI3_OK) bad("tiles");
        if (hipStreamSynchronize(b->stream) != hipSuccess) bad("sync");
    }
    if (rc != MI3_OK) {
        mi3_batch_destroy(b);
        return rc;
    }
    *out = b;
    return MI3_OK;
}

int mi3_batch_destroy(mi3_batch* b) {
    if (!b) return MI3_EINVAL;
    hipSetDevice(b->dev);
    if (b->stream) hipStreamSynchronize(b->stream);
    drop_graph(b);
    for (auto& kv : b->classes) {
        if (kv.second.side) {
            hipStreamSynchronize(kv.second.side);
            hipStreamDestroy(kv.second.side);
        }
        hipFree(kv.second.tiles);
    }
    for (uint32_t m = 0; m < b->n; m++) {
        hipFree(b->Jp[m]);
        hipFree(b->Ju[m]);
        hipFree(b->seq[m]);
        hipFree(b->pos[m]);
    }
    hipFree(b->models);
    hipFree(b->pos_ptrs);
    hipFree(b->steps);
    hipFree(b->counters);
    if (b->stream) hipStreamDestroy(b->stream);
    delete b;
    return MI3_OK;
}

const char* mi3_batch_last_error(mi3_batch* b) {
    return b ? b->err.c_str() : g_batch_create_error.c_str();
}

int mi3_batch_set_couplings(mi3_batch* b, uint32_t model, const float* J) {
    if (!b || !J) return MI3_EINVAL;
    if (model >= b->n) return bfail(b, MI3_EINVAL, "model index out of range");
    hipSetDevice(b->dev);
    const size_t np = (size_t)b->L[model] * (b->L[model] - 1) / 2 * b->q[model] * b->q[model];
    BCHK(b, hipStreamSynchronize(b->stream));
    BCHK(b, hipMemcpy(b->Jp[model], J, np * 4, hipMemcpyHostToDevice));
    BCHK(b, launch_unpack_chunked(b->Jp[model], b->Ju[model], b->L[model], b->q[model],
                                  b->nchunk[model], b->stream));
    BCHK(b, hipStreamSynchronize(b->stream));
    return MI3_OK;
}

int mi3_batch_set_seqs(mi3_batch* b, uint32_t model, const uint8_t* seqs) {
    if (!b || !seqs) return MI3_EINVAL;
    if (model >= b->n) return bfail(b, MI3_EINVAL, "model index out of range");
    hipSetDevice(b->dev);
    const size_t nb = (size_t)b->L[model] * b->N[model];
    for (size_t i = 0; i < nb; i++)
        if (seqs[i] >= b->q[model]) return bfail(b, MI3_EINVAL, "residues must be < q");
    BCHK(b, hipStreamSynchronize(b->stream));
    BCHK(b, hipMemcpy(b->seq[model], seqs, nb, hipMemcpyHostToDevice));
    return MI3_OK;
}

int mi3_batch_get_seqs(mi3_batch* b, uint32_t model, uint8_t* out) {
    if (!b || !out) return MI3_EINVAL;
    if (model >= b->n) return bfail(b, MI3_EINVAL, "model index out of range");
    hipSetDevice(b->dev);
    BCHK(b, hipStreamSynchronize(b->stream));
    BCHK(b, hipMemcpy(out, b->seq[model], (size_t)b->L[model] * b->N[model],
                      hipMemcpyDeviceToHost));
    return MI3_OK;
}

int mi3_batch_run(mi3_batch* b, uint32_t nsweeps) {
    if (!b || nsweeps == 0) return MI3_EINVAL;
    hipSetDevice(b->dev);
    if (!b->exec || b->nsweeps != nsweeps) {
        drop_graph(b);
        BCHK(b, hipStreamSynchronize(b->stream));
        int rc = upload_models(b, nsweeps);
        if (rc) return rc;
        BCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        std::vector<hipEvent_t> events;   // fork/join events, alive until capture ends
        rc = enqueue_round(b, events);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(b->stream, &g);
        for (auto ev : events) hipEventDestroy(ev);
        if (rc) {
            if (g) hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return bfail(b, MI3_EHIP, std::string("capture: ") + hipGetErrorString(e));
        b->graph = g;
        BCHK(b, hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
        b->nsweeps = nsweeps;
    }
    BCHK(b, hipGraphLaunch(b->exec, b->stream));
    return MI3_OK;
}

int mi3_batch_synchronize(mi3_batch* b) {
    if (!b) return MI3_EINVAL;
    hipSetDevice(b->dev);
    BCHK(b, hipStreamSynchronize(b->stream));
    return MI3_OK;
}

int mi3_batch_tune(mi3_batch* b, uint32_t nsweeps) {
    if (!b || nsweeps == 0) return MI3_EINVAL;
    hipSetDevice(b->dev);
    drop_graph(b);
    BCHK(b, hipStreamSynchronize(b->stream));
    int rc = upload_models(b, nsweeps);
    if (rc) return rc;
    hipEvent_t e0, e1;
    BCHK(b, hipEventCreate(&e0));
    BCHK(b, hipEventCreate(&e1));
    uint32_t ci = 0;
    std::vector<ClassTimes> times;
    std::vector<bool> may;
    for (auto& kv : b->classes) {
        ClassRun& cr = kv.second;
        // the class sweep alone, in the present tiles; the step counters advance as
        // after any launch
        auto sweep_ms = [&](float& ms) {
            hipLaunchKernelGGL(k_batch_zero, dim3(1), dim3(64), 0, b->stream, b->counters + ci, 1u);
            const uint32_t mx = max_steps(b);
            hipLaunchKernelGGL(k_batch_positions,
                               dim3(std::max(1u, std::min(64u, (mx + 255) / 256)), b->n), dim3(256),
                               0, b->stream, (const BatchModel*)b->models,
                               (uint32_t* const*)b->pos_ptrs);
            hipEventRecord(e0, b->stream);
            hipError_t e = sweep_class(b, kv.first, cr, b->counters + ci, b->stream);
            hipEventRecord(e1, b->stream);
            hipLaunchKernelGGL(k_batch_advance, dim3((b->n + 255) / 256), dim3(256), 0, b->stream,
                               (const BatchModel*)b->models, b->steps, b->n);
            if (e != hipSuccess || hipEventSynchronize(e1) != hipSuccess)
                return bfail(b, MI3_EHIP, "tuning launch failed");
            hipEventElapsedTime(&ms, e0, e1);
            return MI3_OK;
        };
        float best = 1e30f, ms = 0.f;
        uint32_t best_w = 0;
        for (uint32_t w : tile_options(kv.first.kw)) {
            rc = build_tiles(b, cr, w, false);
            if (!rc) rc = sweep_ms(ms);
            if (rc) break;
            if (ms < best) {
                best = ms;
                best_w = w;
            }
        }
        if (rc) break;
        may.push_back(may_be_unstaged(b, kv.first, cr));
        float unstaged = 0.f;
        if (may.back()) {
            rc = build_tiles(b, cr, best_w, true);
            if (!rc) rc = sweep_ms(unstaged);
            if (rc) break;
        }
        rc = build_tiles(b, cr, best_w, false);
        if (rc) break;
        cr.fixed = true;
        times.push_back({unstaged, best, best * class_grid(b, cr) / units(b), l2_resident(b, cr)});
        ci++;
    }
    if (!rc) {
        const std::vector<bool> direct =
            choose_unstaged(may, [&](const std::vector<bool>&) { return times; });
        size_t i = 0;
        for (auto& kv : b->classes) kv.second.direct = direct[i++];
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    return rc;
}

int mi3_batch_tile(mi3_batch* b, uint32_t model, uint32_t* wpb) {
    if (!b || !wpb || model >= b->n) return MI3_EINVAL;
    ClassKey k{state_words(b->L[model]), pf_class(b->q[model])};
    const ClassRun& cr = b->classes[k];
    *wpb = cr.fixed && !cr.direct ? cr.wpb : tile_options(k.kw).back();
    return MI3_OK;
}

int mi3_batch_set_tile(mi3_batch* b, uint32_t model, uint32_t wpb) {
    if (!b || model >= b->n) return MI3_EINVAL;
    ClassKey k{state_words(b->L[model]), pf_class(b->q[model])};
    auto opts = tile_options(k.kw);
    if (std::find(opts.begin(), opts.end(), wpb) == opts.end())
        return bfail(b, MI3_EINVAL, "walkers per tile must be 128, 256 or 512 (128 or 256 for L > 512)");
    hipSetDevice(b->dev);
    BCHK(b, hipStreamSynchronize(b->stream));
    drop_graph(b);
    ClassRun& cr = b->classes[k];
    if (const int rc = build_tiles(b, cr, wpb, false)) return rc;
    cr.fixed = true;
    return choose_tiles(b);
}

int mi3_batch_step_count(mi3_batch* b, uint32_t model, uint64_t* steps) {
    if (!b || !steps || model >= b->n) return MI3_EINVAL;
    hipSetDevice(b->dev);
    BCHK(b, hipStreamSynchronize(b->stream));
    BCHK(b, hipMemcpy(steps, b->steps + model, sizeof(uint64_t), hipMemcpyDeviceToHost));
    return MI3_OK;
}

}  // extern "C"
