// Model apply on the device: raw predictions of an oblivious float ensemble.
//
// Mirrors the reference's device apply (crates/cb-backend/src/kernels.rs:629
// apply_oblivious_float_kernel, launched by launch_apply_oblivious_f64,
// crates/cb-backend/src/gpu_runtime/mod.rs:337) and its CPU twin predict_raw
// (crates/cb-model/src/apply.rs): one object per thread over a feature-major matrix, each
// tree's leaf from its float splits (value > border, forward bit order), contributions
// summed in tree order from 0, the bias added once after the trees.  A split on a feature
// the matrix does not have is absent (bit 0); a NaN value fails every split unless its
// feature is flagged nan_as_true (borders of nan_mode=Max, apply.rs:160-166); a leaf index
// beyond the tree's leaves contributes 0.  Multi-output models (approx_dim K) store the K
// values of a leaf contiguously; the output is dim-major [K][n].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/cbhip.h"
#include "common.hpp"
#include "copy_threads.hpp"

int cbh_internal_fail(int code, const std::string& msg);  // session.hip

namespace {

#define APPLY_TRY(expr)                                                                          \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return cbh_internal_fail(CBH_ERR_DEVICE, std::string(#expr ": ") + hipGetErrorString(e_)); \
    } while (0)

// The model on the device.  Split arrays hold kSplitPad entries past the last split, so that a
// tree's splits are read eight at a time whatever its depth.
constexpr uint32_t kSplitPad = 8;
struct Model {
    const uint32_t* sf;    // [splits + pad] feature
    const double* sb;      // [splits + pad] border
    const uint32_t* so;    // [trees + 1]
    const double* lv;
    const uint32_t* lo;    // [trees + 1]
    const double* bias;          // nullable
    const uint8_t* nan_true;     // nullable [F]
    uint32_t trees, F;
};

// 64 objects (lanes) a workgroup, its eight waves sharing the trees: what bounds a tree is the chain
// of its scalar loads (offsets, then features and borders) and its objects' values, about 1 us,
// so eight chains run side by side, two trees to a wave and step, their splits read eight at a
// time.  The objects' values are staged in LDS [F][64] (kLds; more features than fit are read
// through the caches).  The leaf indices of kApplyTrees trees go to LDS, and wave d adds dimension
// d's leaf values in tree order while the other waves go on to the next trees (two index buffers).
// One object a thread over all trees, value by value from memory, took 240 us for 1024 x 50 and
// 30 trees with its allocations, and read 6 GB through the caches for 500k x 100 and 500 trees.
constexpr uint32_t kApplyObj = 64, kApplyWaves = 8, kApplyTrees = 32;
constexpr uint32_t kNoLeaf = 0xFFFFFFFFu;
template <int K, bool kLds>
__global__ __launch_bounds__(kApplyObj * kApplyWaves) void apply_oblivious_kernel(
    const float* __restrict__ x /* value of feature f, object i at x[f * ld + i] */, uint64_t ld, uint64_t n,
    uint32_t chunk /* 0, or a multiple of kApplyObj: the table comes in chunks of so many objects, */,
    uint64_t cstride /* chunk c at x + c cstride, its values [F][objects of it] */, Model M,
    double* __restrict__ out /* [K][ldo] */, uint64_t ldo) {
    __shared__ uint32_t leaves[2][kApplyTrees][kApplyObj];
    extern __shared__ float xs[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kApplyObj), lane = threadIdx.x % kApplyObj;
    const uint64_t obj = (uint64_t)blockIdx.x * kApplyObj + lane;
    uint64_t oc = obj, end = n;
    if (chunk) {   // (a workgroup's objects lie in one chunk)
        const uint32_t c = blockIdx.x / (chunk / kApplyObj);
        const uint64_t o0 = (uint64_t)c * chunk;
        x += c * cstride;
        oc = obj - o0;
        end = n - o0 < chunk ? n - o0 : chunk;
        ld = end;
    }
    if (oc >= end) oc = end - 1;
    if (kLds) {
#pragma unroll 4
        for (uint32_t f = wave; f < M.F; f += kApplyWaves) xs[f * kApplyObj + lane] = x[(size_t)f * ld + oc];
        __syncthreads();
    }
    auto bits8 = [&](uint32_t s) -> uint32_t {   // the tests of splits s .. s + 7
        uint32_t f[8];
        double b[8];
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            f[k] = M.sf[s + k];
            b[k] = M.sb[s + k];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t fc = f[k] < M.F ? f[k] : 0u;
            v[k] = M.F == 0 ? 0.0f : kLds ? xs[fc * kApplyObj + lane] : x[(size_t)fc * ld + oc];
        }
        uint32_t bits = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool have = f[k] < M.F;   // (a split on an absent feature fails)
            bool pass = (double)v[k] > b[k];   // false for NaN
            if (M.nan_true) pass |= v[k] != v[k] && M.nan_true[have ? f[k] : 0u] != 0;
            bits |= (uint32_t)(pass && have) << k;
        }
        return bits;
    };
    constexpr int KD = (K + (int)kApplyWaves - 1) / (int)kApplyWaves;   // dimensions of a wave
    double acc[KD];
#pragma unroll
    for (int j = 0; j < KD; ++j) acc[j] = 0.0;
    uint32_t buf = 0;
    for (uint32_t t0 = 0; t0 < M.trees; t0 += kApplyTrees, buf ^= 1u) {
        const uint32_t nt = min(kApplyTrees, M.trees - t0);
        for (uint32_t i = wave; i < nt; i += 2 * kApplyWaves) {   // wave-uniform
            const uint32_t i1 = min(i + kApplyWaves, nt - 1);     // (the second tree, or a repeat)
            const uint32_t t[2] = {t0 + i, t0 + i1};
            uint32_t s0[2], s1[2], l0[2], l1[2], leaf[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                s0[u] = M.so[t[u]];
                s1[u] = M.so[t[u] + 1];
                l0[u] = M.lo[t[u]];
                l1[u] = M.lo[t[u] + 1];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {   // bits past the tree's last split: another tree's, or padding
                const uint32_t m = s1[u] - s0[u];
                leaf[u] = bits8(s0[u]);
                if (m < 8) leaf[u] &= (1u << m) - 1u;
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                for (uint32_t s = s0[u] + 8; s < s1[u]; s += 8) {
                    const uint32_t m = s1[u] - s;
                    const uint32_t bits = bits8(s);
                    leaf[u] |= (m < 8 ? bits & ((1u << m) - 1u) : bits) << (s - s0[u]);
                }
                const uint32_t li = l0[u] + leaf[u];
                leaves[buf][t[u] - t0][lane] = li < l1[u] ? li : kNoLeaf;
            }
        }
        // one barrier a chunk: the other buffer's readers pass it only after reading it
        __syncthreads();
#pragma unroll
        for (int j = 0; j < KD; ++j) {
            const uint32_t d = wave + (uint32_t)j * kApplyWaves;
            if (d >= (uint32_t)K) break;
#pragma unroll 1
            for (uint32_t i = 0; i < nt; i += 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t li = leaves[buf][min(i + (uint32_t)u, nt - 1)][lane];
                    v[u] = li != kNoLeaf ? M.lv[(size_t)li * K + d] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (i + (uint32_t)u < nt) acc[j] += v[u];
            }
        }
    }
    if (obj >= n) return;
#pragma unroll
    for (int j = 0; j < KD; ++j) {
        const uint32_t d = wave + (uint32_t)j * kApplyWaves;
        if (d < (uint32_t)K) out[(size_t)d * ldo + obj] = acc[j] + (M.bias ? M.bias[d] : 0.0);
    }
}

constexpr size_t kApplyLdsMax = 128 * 1024;
constexpr uint64_t kMaxBlocks = (uint64_t)1 << 22;

struct Table {   // on the device: one block of leading dimension ld, or chunks (the kernel's arguments)
    const float* x;
    uint64_t ld;
    uint32_t chunk;
    uint64_t cstride;
};

template <int K>
int launch(const Table& t, uint64_t n, const Model& M, double* out, uint64_t ldo, hipStream_t st) {
    const size_t lds = (size_t)M.F * kApplyObj * sizeof(float);
    const uint64_t blocks = (n + kApplyObj - 1) / kApplyObj;
    if (blocks > kMaxBlocks) {   // (a launch holds fewer than 2^32 threads; chunks are far smaller)
        const uint64_t n0 = kMaxBlocks * kApplyObj;
        const int rc = launch<K>(t, n0, M, out, ldo, st);
        return rc != CBH_OK ? rc : launch<K>(Table{t.x + n0, t.ld, 0, 0}, n - n0, M, out + n0, ldo, st);
    }
    const unsigned grid = (unsigned)blocks;
    if (lds <= kApplyLdsMax) {
        if (lds > 32 * 1024)
            APPLY_TRY(hipFuncSetAttribute((const void*)apply_oblivious_kernel<K, true>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)kApplyLdsMax));
        apply_oblivious_kernel<K, true><<<grid, kApplyObj * kApplyWaves, lds, st>>>(t.x, t.ld, n, t.chunk, t.cstride, M,
                                                                                    out, ldo);
    } else {
        apply_oblivious_kernel<K, false><<<grid, kApplyObj * kApplyWaves, 0, st>>>(t.x, t.ld, n, t.chunk, t.cstride, M,
                                                                                   out, ldo);
    }
    APPLY_TRY(hipGetLastError());
    return CBH_OK;
}

int launch_k(uint32_t K, const Table& t, uint64_t n, const Model& M, double* out, uint64_t ldo, hipStream_t st) {
    switch (K) {
#define CASE(k) case k: return launch<k>(t, n, M, out, ldo, st);
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(10) CASE(12) CASE(16)
#undef CASE
        default: return cbh_internal_fail(CBH_ERR_UNSUPPORTED, "approx_dim " + std::to_string(K) + " has no apply variant");
    }
}
bool has_variant(uint32_t K) { return (K >= 1 && K <= 8) || K == 10 || K == 12 || K == 16; }

// A call's buffers: a device block, a pinned block and its streams.  Allocating and freeing them per
// call (eight of each, each free a device synchronization) was most of a small call's time, so
// up to kKeep idle workspaces are kept, each a call's own while it runs (any number of threads); one
// more is freed with its call.  A block that has grown past kKeepBytes goes with its call, the streams
// and the rest stay: freed whole and made anew by each call, 10M x 1 (an 80 MB result) took 17.7 ms, 10.3
// this way.  The kept blocks go when an allocation fails.  Two are kept because streams that stay
// share the few hardware queues as they were dealt: with 16 kept, calls of four threads on 50k x 50
// took 230 to 320 us each from run to run, 235 with two.
struct Workspace {
    int device = -1;
    hipStream_t stream = nullptr, copy = nullptr;   // copy: a large table's uploads, beside the kernels
    unsigned char* dev = nullptr;
    unsigned char* pin = nullptr;
    size_t dev_cap = 0, pin_cap = 0;
    hipEvent_t ev[6] = {};   // of the three chunk buffers: uploaded, then read by the kernel

    void release() {
        drop_dev();
        drop_pin();
        for (auto& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (stream) (void)hipStreamDestroy(stream);
        if (copy) (void)hipStreamDestroy(copy);
        copy = stream = nullptr;
    }
    void drop_dev() {
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        dev_cap = 0;
    }
    void drop_pin() {
        if (pin) (void)hipHostFree(pin);
        pin = nullptr;
        pin_cap = 0;
    }
    int grow(size_t need_dev, size_t need_pin);
};
constexpr size_t kKeep = 2, kKeepBytes = (size_t)64 << 20;
std::mutex g_ws_mu;
std::vector<Workspace>& idle_workspaces() {
    static std::vector<Workspace>* v = [] {   // (never destroyed: no frees after the runtime has gone)
        auto* p = new std::vector<Workspace>();
        p->reserve(kKeep);
        return p;
    }();
    return *v;
}
// The idle workspaces' blocks are given back (to a call that found no memory).
void drop_idle_blocks() {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    for (Workspace& w : idle_workspaces()) {
        w.drop_dev();
        w.drop_pin();
    }
}
int Workspace::grow(size_t need_dev, size_t need_pin) {
    if (!stream) APPLY_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    if (need_dev > dev_cap) {
        drop_dev();
        need_dev = std::max<size_t>(need_dev, 1 << 20);
        if (hipMalloc((void**)&dev, need_dev) != hipSuccess) {
            (void)hipGetLastError();
            drop_idle_blocks();
            APPLY_TRY(hipMalloc((void**)&dev, need_dev));
        }
        dev_cap = need_dev;
    }
    if (need_pin > pin_cap) {
        drop_pin();
        need_pin = std::max<size_t>(need_pin, 1 << 20);
        if (hipHostMalloc((void**)&pin, need_pin, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            drop_idle_blocks();
            APPLY_TRY(hipHostMalloc((void**)&pin, need_pin, hipHostMallocDefault));
        }
        pin_cap = need_pin;
    }
    return CBH_OK;
}
struct Lease {
    Workspace ws;
    bool ok = false;   // the call went through: nothing is running on the stream
    explicit Lease(int device) {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        auto& idle = idle_workspaces();
        for (size_t k = idle.size(); k-- > 0;)   // the one given back last
            if (idle[k].device == device) {
                ws = idle[k];
                idle.erase(idle.begin() + (long)k);
                return;
            }
        ws.device = device;
    }
    ~Lease() {
        if (!ok && ws.copy) (void)hipStreamSynchronize(ws.copy);
        if (!ok && ws.stream) (void)hipStreamSynchronize(ws.stream);
        if (ok) {
            if (ws.dev_cap > kKeepBytes) ws.drop_dev();
            if (ws.pin_cap > kKeepBytes) ws.drop_pin();
            std::lock_guard<std::mutex> lock(g_ws_mu);
            auto& idle = idle_workspaces();
            if (idle.size() < kKeep) {
                idle.push_back(ws);
                return;
            }
        }
        ws.release();
    }
};

// Leaf values that go up through the pinned block: what fits its smallest size beside the other
// arrays.  More go up from the caller's memory: pinning 3 MB for them took the first call on 100 trees
// of depth 12 from 1.2 to 2.2 ms, which a call's 0.1 ms of copying does not pay back.
constexpr size_t kPinModel = (size_t)512 << 10;

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Host threads that copy a large table into pinned memory (the CPU share of a shared host).
unsigned copy_threads() {
    unsigned t = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
    if (const char* e = std::getenv("OMP_NUM_THREADS")) {
        const long v = std::strtol(e, nullptr, 10);
        if (v >= 1 && (unsigned long)v < t) t = (unsigned)v;
    }
    return t;
}

constexpr size_t kChunkBytes = (size_t)6 << 20;   // of a table in pinned chunks, three in flight

// A large table in chunks of objects: the threads copy a chunk's runs of every feature into one of
// three pinned buffers, which goes to its device buffer and through the kernel while the next one
// fills (the runtime's own path for pageable memory copies with one thread: 200 MB in 7 ms).
//
// A kernel takes a group of chunks: one where the model takes less time than a chunk's upload (135 us),
// three groups in flight, else as many as fill the CUs, two groups in flight.  A chunk of 100 features is
// 245 workgroups, one a CU and bound by the latency of its trees (0.2 us each up to 8 splits): a
// launch a chunk fell behind the uploads at large models, and behind one launch over the whole
// table.  500k x 100, a launch a chunk / a group / one launch after the upload: 500 trees 4.6 / 4.6 / 9.5 ms,
// 1000 6.9 / 4.9 / 11.0, 5000 30.3 / 16.6 / 23.8; 300k x 300, 3000 trees of depth 8 38.5 / 13.9 / 27.0.
// (The three buffers' kernels on streams of their own gave the same where the streams had hardware
// queues of their own, and nothing where they had not.)
struct ChunkPlan {
    uint64_t chunk, n_chunks;   // objects, a multiple of kApplyObj
    uint32_t group, ring;       // chunks a launch, groups in flight
    size_t cbytes;              // of a chunk's buffer
};
constexpr uint64_t kGroupWork = 800;    // trees and groups of 8 splits past which a launch takes several chunks
constexpr uint32_t kGroupMax = 10;      // (60 MB)
ChunkPlan plan_chunks(uint64_t n, uint32_t F, uint32_t n_trees, uint32_t n_splits, uint32_t cus) {
    ChunkPlan p{};
    p.chunk = kChunkBytes / (sizeof(float) * F) / kApplyObj * kApplyObj;
    p.n_chunks = (n + p.chunk - 1) / p.chunk;
    p.cbytes = align256(sizeof(float) * p.chunk * F);
    p.group = 1;
    p.ring = 3;
    if ((uint64_t)n_trees + n_splits / 8 > kGroupWork) {
        // workgroups a CU holds: 32 waves, and the objects' values in its LDS
        const size_t lds = (size_t)F * kApplyObj * sizeof(float) + sizeof(uint32_t) * 2 * kApplyTrees * kApplyObj;
        const uint32_t per_cu = lds <= kApplyLdsMax + 16 * 1024 ? std::max<uint32_t>(1, std::min<uint32_t>(4, 160 * 1024 / lds)) : 4u;
        const uint64_t wgs = p.chunk / kApplyObj;
        p.group = (uint32_t)std::min<uint64_t>({std::max<uint64_t>(1, (uint64_t)cus * per_cu / wgs), kGroupMax, p.n_chunks});
        if (p.group > 1) p.ring = (uint32_t)std::min<uint64_t>(2, (p.n_chunks + p.group - 1) / p.group);
    }
    return p;
}
int apply_chunks(Workspace& w, const float* features, uint64_t n, uint32_t F, uint32_t K, const Model& M, size_t dev_x,
                 size_t pin_x, const ChunkPlan& p, double* d_out) {
    const uint64_t chunk = p.chunk, n_chunks = p.n_chunks;
    const size_t cbytes = p.cbytes;
    for (auto& e : w.ev)
        if (!e) APPLY_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (!w.copy) APPLY_TRY(hipStreamCreateWithFlags(&w.copy, hipStreamNonBlocking));
    auto copy_chunk = [&](uint64_t c, uint32_t first, uint32_t step) {
        const uint64_t o0 = c * chunk, m = std::min(chunk, n - o0);
        float* dst = (float*)(w.pin + pin_x + (c % 3) * cbytes);
        for (uint32_t f = first; f < F; f += step)
            std::memcpy(dst + (size_t)f * m, features + (size_t)f * n + o0, sizeof(float) * m);
    };
    cbh::CopyThreads<decltype(copy_chunk)> threads(copy_threads(), n_chunks, std::min<uint64_t>(2, n_chunks), copy_chunk);
    int rc = CBH_OK;
    for (uint64_t c = 0; c < n_chunks && rc == CBH_OK; ++c) {
        threads.wait(c);
        const uint64_t o0 = c * chunk, m = std::min(chunk, n - o0);
        const uint64_t grp = c / p.group, slot = grp % p.ring, in = c - grp * p.group;   // its place on the device
        float* dx = (float*)(w.dev + dev_x + slot * p.group * cbytes);
        hipEvent_t up = w.ev[c % 3], read = w.ev[3 + slot];
        if ((in == 0 && grp >= p.ring && hipStreamWaitEvent(w.copy, read, 0) != hipSuccess) ||   // the slot's last kernel
            hipMemcpyAsync((unsigned char*)dx + in * cbytes, w.pin + pin_x + (c % 3) * cbytes, sizeof(float) * m * F,
                           hipMemcpyHostToDevice, w.copy) != hipSuccess ||
            hipEventRecord(up, w.copy) != hipSuccess)
            rc = cbh_internal_fail(CBH_ERR_DEVICE, "table upload failed");
        if (rc == CBH_OK && (in + 1 == p.group || c + 1 == n_chunks)) {   // the group is on its way
            const uint64_t g0 = grp * p.group * chunk;
            if (hipStreamWaitEvent(w.stream, up, 0) != hipSuccess)
                rc = cbh_internal_fail(CBH_ERR_DEVICE, "table upload failed");
            if (rc == CBH_OK)
                rc = launch_k(K, Table{dx, m, in ? (uint32_t)chunk : 0u, cbytes / sizeof(float)}, o0 + m - g0, M,
                              d_out + g0, n, w.stream);
            if (rc == CBH_OK && hipEventRecord(read, w.stream) != hipSuccess)
                rc = cbh_internal_fail(CBH_ERR_DEVICE, "table upload failed");
        }
        if (rc == CBH_OK && c + 2 < n_chunks) {   // chunk c + 2 takes the buffer of chunk c - 1
            if (c >= 1 && hipEventSynchronize(w.ev[(c - 1) % 3]) != hipSuccess)
                rc = cbh_internal_fail(CBH_ERR_DEVICE, "table upload failed");
            else
                threads.open(c + 3);
        }
    }
    return rc;
}

}  // namespace

extern "C" int cbh_apply_oblivious(const float* features_fm, uint64_t n_objects, uint32_t n_features,
                                   const uint32_t* split_features, const double* split_borders,
                                   const uint32_t* tree_split_offsets, const double* leaf_values,
                                   const uint32_t* tree_leaf_offsets, uint32_t n_trees, uint32_t approx_dim,
                                   const double* bias, const uint8_t* nan_as_true, double* out) {
    if (!tree_split_offsets || !tree_leaf_offsets || !out)
        return cbh_internal_fail(CBH_ERR_INVALID_ARG, "offset arrays and out are required");
    if (n_objects > 0 && n_features > 0 && !features_fm)
        return cbh_internal_fail(CBH_ERR_INVALID_ARG, "features are null");
    // CSR offsets: start at 0, non-decreasing (gpu_runtime/mod.rs:306-330); a leaf index has
    // one bit per split, so a tree has at most 31 splits
    if (tree_split_offsets[0] != 0 || tree_leaf_offsets[0] != 0)
        return cbh_internal_fail(CBH_ERR_OUT_OF_RANGE, "CSR offsets must start at 0");
    for (uint32_t t = 0; t < n_trees; ++t) {
        if (tree_split_offsets[t + 1] < tree_split_offsets[t] || tree_leaf_offsets[t + 1] < tree_leaf_offsets[t])
            return cbh_internal_fail(CBH_ERR_OUT_OF_RANGE, "CSR offsets must be non-decreasing");
        if (tree_split_offsets[t + 1] - tree_split_offsets[t] > 31)
            return cbh_internal_fail(CBH_ERR_OUT_OF_RANGE, "a tree has more than 31 splits");
    }
    const uint32_t n_splits = tree_split_offsets[n_trees];
    const uint32_t n_leaves = tree_leaf_offsets[n_trees];
    if ((n_splits && (!split_features || !split_borders)) || (n_leaves && !leaf_values))
        return cbh_internal_fail(CBH_ERR_INVALID_ARG, "model arrays are null");
    const uint32_t K = approx_dim;
    if (n_objects == 0) return CBH_OK;
    if (!has_variant(K))
        return cbh_internal_fail(CBH_ERR_UNSUPPORTED, "approx_dim " + std::to_string(K) + " has no apply variant");
    const uint64_t n = n_objects;
    const uint32_t F = n_features;
    // one block: the model (and a small table) as uploaded in one copy, the table's chunks, the output
    const size_t o_sb = 0, o_bias = o_sb + align256(sizeof(double) * ((size_t)n_splits + kSplitPad));
    const size_t o_sf = o_bias + align256(sizeof(double) * K);
    const size_t o_so = o_sf + align256(sizeof(uint32_t) * ((size_t)n_splits + kSplitPad));
    const size_t o_lo = o_so + align256(sizeof(uint32_t) * ((size_t)n_trees + 1));
    const size_t o_na = o_lo + align256(sizeof(uint32_t) * ((size_t)n_trees + 1)), o_lv = o_na + align256(F);
    const size_t o_x = o_lv + align256(sizeof(double) * n_leaves * K);
    const size_t x_bytes = sizeof(float) * n * F, out_bytes = sizeof(double) * n * K;
    // a table in chunks of at least 64 objects; one with more features than that leaves room for,
    // and a model's leaf values past kPinModel, are uploaded from the caller's memory (pinning
    // them would take longer than the runtime's copy)
    const bool big = x_bytes > 2 * kChunkBytes, chunked = big && kChunkBytes / (sizeof(float) * F) >= 64;
    const bool pin_table = !big, pin_lv = sizeof(double) * n_leaves * K <= kPinModel;
    int dev = 0, cus = 0;
    APPLY_TRY(hipGetDevice(&dev));
    if (chunked) APPLY_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const ChunkPlan plan = chunked ? plan_chunks(n, F, n_trees, n_splits, (uint32_t)cus) : ChunkPlan{};
    const size_t x_dev = chunked ? plan.ring * plan.group * plan.cbytes : align256(x_bytes);
    const size_t o_out = o_x + x_dev;
    Lease L(dev);
    Workspace& w = L.ws;
    const bool pin_out = out_bytes <= ((size_t)4 << 20);   // the kernel's results through pinned memory
    // the pinned block: the model's arrays and a small table laid out as on the device, so that they
    // go up in one copy, or the chunk buffers, then the results
    const size_t h_x = pin_lv ? o_x : o_lv, h_out = h_x + (chunked ? 3 * plan.cbytes : pin_table ? x_dev : 0);
    int rc = w.grow(o_out + out_bytes, h_out + (pin_out ? out_bytes : 0));
    if (rc != CBH_OK) return rc;
    unsigned char* h = w.pin;
    if (n_splits) std::memcpy(h + o_sb, split_borders, sizeof(double) * n_splits);
    std::memset(h + o_sb + sizeof(double) * n_splits, 0, sizeof(double) * kSplitPad);
    if (n_leaves && pin_lv) std::memcpy(h + o_lv, leaf_values, sizeof(double) * n_leaves * K);
    if (bias) std::memcpy(h + o_bias, bias, sizeof(double) * K);
    if (n_splits) std::memcpy(h + o_sf, split_features, sizeof(uint32_t) * n_splits);
    std::memset(h + o_sf + sizeof(uint32_t) * n_splits, 0, sizeof(uint32_t) * kSplitPad);
    std::memcpy(h + o_so, tree_split_offsets, sizeof(uint32_t) * ((size_t)n_trees + 1));
    std::memcpy(h + o_lo, tree_leaf_offsets, sizeof(uint32_t) * ((size_t)n_trees + 1));
    if (nan_as_true && F) std::memcpy(h + o_na, nan_as_true, F);
    if (pin_table && x_bytes) std::memcpy(h + h_x, features_fm, x_bytes);
    const Model M{(const uint32_t*)(w.dev + o_sf), (const double*)(w.dev + o_sb), (const uint32_t*)(w.dev + o_so),
                  (const double*)(w.dev + o_lv), (const uint32_t*)(w.dev + o_lo),
                  bias ? (const double*)(w.dev + o_bias) : nullptr,
                  nan_as_true && F ? (const uint8_t*)(w.dev + o_na) : nullptr, n_trees, F};
    double* d_out = (double*)(w.dev + o_out);
    const bool one_copy = pin_lv && pin_table;
    APPLY_TRY(hipMemcpyAsync(w.dev, h, one_copy ? o_x + x_bytes : h_x, hipMemcpyHostToDevice, w.stream));
    if (!pin_lv)
        APPLY_TRY(hipMemcpyAsync(w.dev + o_lv, leaf_values, sizeof(double) * n_leaves * K, hipMemcpyHostToDevice, w.stream));
    if (!one_copy && !chunked && x_bytes)
        APPLY_TRY(hipMemcpyAsync(w.dev + o_x, pin_table ? (const void*)(h + h_x) : features_fm, x_bytes,
                                 hipMemcpyHostToDevice, w.stream));
    if (chunked) {
        try {
            rc = apply_chunks(w, features_fm, n, F, K, M, o_x, h_x, plan, d_out);
        } catch (const std::exception& e) {   // (its threads are joined)
            rc = cbh_internal_fail(CBH_ERR_DEVICE, std::string("table upload: ") + e.what());
        }
    } else {
        rc = launch_k(K, Table{(const float*)(w.dev + o_x), n, 0, 0}, n, M, d_out, n, w.stream);
    }
    if (rc != CBH_OK) return rc;
    if (pin_out) {
        unsigned char* ho = h + h_out;
        APPLY_TRY(hipMemcpyAsync(ho, d_out, out_bytes, hipMemcpyDeviceToHost, w.stream));
        APPLY_TRY(hipStreamSynchronize(w.stream));
        std::memcpy(out, ho, out_bytes);
    } else {
        APPLY_TRY(hipMemcpyAsync(out, d_out, out_bytes, hipMemcpyDeviceToHost, w.stream));
        APPLY_TRY(hipStreamSynchronize(w.stream));
    }
    L.ok = true;
    return CBH_OK;
}
