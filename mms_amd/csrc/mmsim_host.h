// Host-side objects of libmmsim shared by its translation units: error reporting, device memory, and what the
// opaque handles of the C ABI point at.
#pragma once

#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

#include "mmsim_internal.h"

namespace mmsim {

inline thread_local std::string g_last_error;

inline int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}

// What an entry point returns for an exception that reached it (host memory or threads that were not to be had): none
// leaves the C ABI.
inline int caught() noexcept {
    try {
        return fail(MMSIM_E_NOMEM, "host allocation failed");
    } catch (...) {
        return MMSIM_E_NOMEM;  // (not even the message: the one before stays)
    }
}

inline int hip_fail(hipError_t e, const char *what) {
    return fail(e == hipErrorOutOfMemory ? MMSIM_E_NOMEM : MMSIM_E_HIP,
                std::string(what) + ": " + hipGetErrorString(e));
}

#define HIP_TRY(expr)                                      \
    do {                                                   \
        hipError_t e__ = (expr);                           \
        if (e__ != hipSuccess) return hip_fail(e__, #expr); \
    } while (0)

// Copies on a stream read and write host memory until the stream has been waited for.  Declared behind that memory, this
// waits for them on every way out of a function.
struct StreamWait {
    hipStream_t stream;
    bool pending = true;
    explicit StreamWait(hipStream_t st) : stream(st) {}
    StreamWait(const StreamWait &) = delete;
    StreamWait &operator=(const StreamWait &) = delete;
    hipError_t now() {
        pending = false;
        return hipStreamSynchronize(stream);
    }
    ~StreamWait() {
        if (pending) (void)hipStreamSynchronize(stream);
    }
};

// Device memory for a batch comes either from hipMalloc or, while g_arena is set (mmsim_eval_batch_static), from
// a bump allocator over the library's static device scratch: such buffers are never freed one by one.
struct Arena {
    unsigned char *base = nullptr;
    size_t cap = 0, used = 0;
    bool overflow = false;
};
inline thread_local Arena *g_arena = nullptr;
struct ArenaScope {
    explicit ArenaScope(Arena *a) { g_arena = a; }
    ~ArenaScope() { g_arena = nullptr; }
};

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    bool owned = true;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p && owned) (void)hipFree(p);
        p = nullptr;
        n = 0;
        owned = true;
    }
    hipError_t alloc(size_t count) {
        release();
        n = count;
        const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
        if (Arena *ar = g_arena) {
            const size_t rounded = (bytes + 255) & ~(size_t)255;
            if (rounded > ar->cap - ar->used) {
                ar->overflow = true;
                n = 0;
                return hipErrorOutOfMemory;
            }
            p = reinterpret_cast<T *>(ar->base + ar->used);
            ar->used += rounded;
            owned = false;
            return hipSuccess;
        }
        return hipMalloc(reinterpret_cast<void **>(&p), bytes);
    }
    size_t bytes() const { return n * sizeof(T); }
};

}  // namespace mmsim


using namespace mmsim;

namespace mmsim {

// Host memory the GPU copies from and to directly, kept by a context between calls: packed inputs and results pass
// through it.  Grows on demand; a call that needs more than kMost gives its memory back at the end.
struct Staging {
    static constexpr size_t kMost = (size_t)64 << 20;
    unsigned char *p = nullptr;
    size_t n = 0;
    Staging() = default;
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;
    ~Staging() { release(); }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        n = 0;
    }
    hipError_t ensure(size_t bytes) {
        if (bytes <= n) return hipSuccess;
        release();
        const size_t want = std::max<size_t>(bytes, std::min(kMost, std::max<size_t>((size_t)1 << 20, 2 * bytes)));
        const hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&p), want, hipHostMallocDefault);
        if (e != hipSuccess) {
            p = nullptr;
            return e;
        }
        n = want;
        return hipSuccess;
    }
    void trim() {
        if (n > kMost) release();
    }
};

// What a launch of simulations that are cut into runs has of device memory beside its batch's: no launch needs what another left
// there, and those of a context follow one another on its stream, so all of its batches share one buffer.
struct RunMemory {
    // Most bytes of a launch, and most that are kept while no batch is there that may be run again (a gigabyte costs 0.3 ms to
    // allocate and free).  A launch takes no more than a quarter of what is free either: it can do without.
    static constexpr size_t kMost = (size_t)16 << 30, kMostKept = (size_t)2 << 30;
    DevBuf<uint8_t> buf;
    int batches = 0;  // that may be run again
    bool fits(size_t bytes) const {
        if (bytes <= buf.n) return true;
        size_t free = 0, total = 0;
        if (bytes > kMost || hipMemGetInfo(&free, &total) != hipSuccess) return false;
        return bytes <= (free + buf.n) / 4;
    }
    // nullptr: there is no room, simulations are not cut
    uint8_t *ensure(size_t bytes, hipStream_t stream) {
        if (bytes <= buf.n) return buf.p;
        if (!fits(bytes) || hipStreamSynchronize(stream) != hipSuccess) return nullptr;  // (a launch before this one may still use it)
        if (buf.alloc(bytes) != hipSuccess) {
            (void)hipGetLastError();
            buf.release();
            return nullptr;
        }
        return buf.p;
    }
    void trim() {
        if (batches == 0 && buf.n > kMostKept) buf.release();
    }
};

// Runs fn(lo, hi) on slices of [0, n) on up to 16 host threads (one slice per thread; the caller's
// slices write disjoint memory).  Small ranges run on the calling thread.  What a slice throws is thrown to the caller
// when all have ended; a slice for which there is no thread runs on the calling one.
template <class F>
void parallel_slices(int64_t n, int64_t min_per_thread, F &&fn) {
    int64_t threads = std::min<int64_t>(16, std::max(1u, std::thread::hardware_concurrency()));
    threads = std::min<int64_t>(threads, n / std::max<int64_t>(1, min_per_thread));
    if (threads <= 1) {
        fn((int64_t)0, n);
        return;
    }
    const int64_t per = (n + threads - 1) / threads;
    std::mutex thrown_mutex;
    std::exception_ptr thrown;
    auto slice = [&](int64_t lo) noexcept {
        try {
            fn(lo, std::min(n, lo + per));
        } catch (...) {
            std::lock_guard<std::mutex> lock(thrown_mutex);
            if (!thrown) thrown = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve((size_t)threads);
    for (int64_t lo = per; lo < n; lo += per) {
        try {
            pool.emplace_back(slice, lo);
        } catch (const std::system_error &) {
            slice(lo);
        }
    }
    slice(0);
    for (std::thread &th : pool) th.join();
    if (thrown) std::rethrow_exception(thrown);
}

}  // namespace mmsim

struct mmsim_ctx {
    Staging staging;
    RunMemory runs;
    int device = 0;
    hipStream_t stream = nullptr;
    hipDeviceProp_t prop{};
    int max_lds = 0;
    unsigned char *scratch = nullptr;     // this device's copy of the static scratch (mmsim_eval_batch_static)
    hipEvent_t ev_static[2] = {};         // timing events of batches that live in the static scratch
    mmsim_options opt{};                  // what batches made without options of their own use (mmsim_ctx_set_options)
    std::atomic<int> users{1};            // its owner, and the workloads and batches that were made of it
    void drop() {
        if (users.fetch_sub(1) != 1) return;
        (void)hipSetDevice(device);
        if (stream) (void)hipStreamDestroy(stream);
        for (hipEvent_t e : ev_static)
            if (e) (void)hipEventDestroy(e);
        delete this;
    }
};

// The context of a workload or batch, which lives until they are gone as well (a garbage collector may end it first).
struct CtxRef {
    mmsim_ctx *p = nullptr;
    CtxRef() = default;
    CtxRef(const CtxRef &) = delete;
    ~CtxRef() {
        if (p) p->drop();
    }
    CtxRef &operator=(const CtxRef &) = delete;
    CtxRef &operator=(mmsim_ctx *ctx) {
        if (ctx) ctx->users.fetch_add(1);
        if (p) p->drop();
        p = ctx;
        return *this;
    }
    operator mmsim_ctx *() const { return p; }
    mmsim_ctx *operator->() const { return p; }
};

inline std::atomic<uint64_t> g_next_workload_id{1};

struct mmsim_workload {
    CtxRef ctx;
    uint64_t id = 0;  // unique per mmsim_workload_create: a batch remembers which streams it was made from
    int64_t R = 0;
    int32_t M = 0;
    std::shared_ptr<DevBuf<Req>> reqs = std::make_shared<DevBuf<Req>>();  // shared with batches that read it in place
    std::vector<int32_t> model_num_requests;  // requests per model id (placement independent)
    double span = 0.0;                        // from the first arrival to the last
    bool sorted = true;                       // arrivals ascend
    double burst = 1.0;                       // of streams that may be cut into runs: standard deviation of the time between a model's
                                              // arrivals, over its mean (of the models, as often as they are asked for)
    int64_t repeats = 0;                      // requests with the model of the request before
    int64_t run_repeats = 0;                  // ... and with its SLO (bit for bit)
    // arrivals regrouped by model (batching simulator): offsets per model, then per arrival
    // its time, its deadline time + (double)slo and its index in the stream
    std::vector<int64_t> mq_off;
    DevBuf<MqEntry> mq;
};

// How busy the streams keep the groups, about: requests of a second, times the time a group needs for one (the longest of
// its stages, alone in its batch, over the models as often as they are asked for), over the groups of a placement (of some
// sixty that are looked at).
inline double offered_load(const mmsim_workload *const *wls, int32_t n_streams, const mmsim_tables *t, int32_t B, int32_t Gmax,
                           const int32_t *num_groups, const int32_t *group_cfg) {
    double requests = 0.0, seconds = 0.0;
    std::vector<double> weight(t->M, 0.0), busy(t->C, 0.0);
    for (int s = 0; s < n_streams; ++s) {
        seconds += wls[s]->span;
        for (int32_t m = 0; m < t->M; ++m) {
            weight[m] += (double)wls[s]->model_num_requests[m];
            requests += (double)wls[s]->model_num_requests[m];
        }
    }
    for (int32_t c = 0; c < t->C; ++c)
        for (int32_t m = 0; m < t->M; ++m) {
            float longest = 0.0f;
            for (int k = 0; k < t->cfg_pp[c]; ++k) longest = std::max(longest, t->cfg_lat[(((size_t)m * t->C + c) * t->Smax + k) * t->NB]);
            if (std::isfinite(longest)) busy[c] += weight[m] / requests * (double)longest;
        }
    double a_second = 0.0;  // requests that the groups of `looked` placements take in a second
    const int32_t every = std::max(1, B / 64), looked = (B + every - 1) / every;
    for (int32_t p = 0; p < B; p += every)
        for (int32_t g = 0; g < num_groups[p]; ++g) a_second += 1.0 / std::max(1e-9, busy[group_cfg[(size_t)p * Gmax + g]]);
    return a_second > 0.0 && seconds > 0.0 ? requests / seconds * looked / a_second : 0.0;
}

// Replicas that a request may choose from, on average (over the placements that offered_load looks at).
inline double replicas_of_a_request(const mmsim_workload *const *wls, int32_t n_streams, const mmsim_placements *p, int32_t M) {
    std::vector<double> weight(M, 0.0);
    double requests = 0.0, replicas = 0.0;
    for (int s = 0; s < n_streams; ++s)
        for (int32_t m = 0; m < M; ++m) {
            weight[m] += (double)wls[s]->model_num_requests[m];
            requests += (double)wls[s]->model_num_requests[m];
        }
    const int32_t every = std::max(1, p->B / 64), looked = (p->B + every - 1) / every;
    for (int32_t b = 0; b < p->B; b += every) {
        const int64_t *off = p->gm_off + (size_t)b * (p->Gmax + 1);
        for (int64_t x = off[0]; x < off[p->num_groups[b]]; ++x) replicas += weight[p->gm_idx[x]];
    }
    return requests > 0.0 ? replicas / requests / looked : 0.0;
}

// Whether it pays to cut simulations into runs: groups that are busy all along, and requests that may go to several of them, keep runs
// that once chose differently apart; pauses between a model's bursts bring them together.  Cut against not cut, random batches of 1 to 1100
// placements, 7700 to 121000 requests, loads of 0.3 to 8, times between arrivals that vary by 1 to 8 times their mean, lines at
// load x replicas = most x burst.  Plain, 806 batches, most = 1: 70 of the 462 that are cut are more than 5 % slower for it (worst 2.8 -> 4.3 ms), and 13
// of the 326 that cutting makes a quarter or more faster are not cut; most = 2: 143 of 572, and 2; all cut 298; a line at load >= 2.5 and load x
// replicas >= 2.2 128 of 574, and 20.  Batching, 413 batches, where runs that never agree cost less (13 % at most): most = 1 16 of 259, and 11 of the 196 not
// cut, some of which take 8 times as long for it; 2: 34 of 324, and 2; all cut 76.
inline bool runs_agree_early(const mmsim_workload *const *wls, int32_t n_streams, double load, double replicas, double most) {
    double requests = 0.0, burst = 0.0;
    for (int s = 0; s < n_streams; ++s) {
        requests += (double)wls[s]->R;
        burst += (double)wls[s]->R * wls[s]->burst;
    }
    return load * replicas * requests < most * burst;
}

// Ordered replica lists per (placement, model): the rows of m_id2g_id.
struct RepLists {
    int32_t B = 0, M = 0, Gmax = 0;
    std::vector<int32_t> num_groups;  // [B]
    std::vector<int32_t> group_cfg;   // [B][Gmax]
    std::vector<int64_t> off;         // [B*M+1]
    std::vector<int32_t> grp;         // group index per replica
    // models of each group in the order the batching simulator scans them (g_id2m_id);
    // left empty, they are derived from the replica lists as the reference does (:424-430)
    std::vector<int64_t> g2m_off;     // [B*Gmax+1]
    std::vector<int32_t> g2m_m;
    bool models_ascend() const {  // every group lists its models in ascending order
        for (size_t g = 0; g + 1 < g2m_off.size(); ++g)
            for (int64_t x = g2m_off[g] + 1; x < g2m_off[g + 1]; ++x)
                if (g2m_m[(size_t)x] <= g2m_m[(size_t)x - 1]) return false;
        return true;
    }
};

// Replicas that a request may choose from, on average (over the placements that offered_load looks at).
inline double replicas_of_a_request(const mmsim_workload *const *wls, int32_t n_streams, const RepLists &rl) {
    double requests = 0.0, replicas = 0.0;
    const int32_t every = std::max(1, rl.B / 64), looked = (rl.B + every - 1) / every;
    for (int s = 0; s < n_streams; ++s)
        for (int32_t m = 0; m < rl.M; ++m) {
            const double n = (double)wls[s]->model_num_requests[m];
            requests += n;
            for (int32_t p = 0; p < rl.B; p += every) replicas += n * (double)(rl.off[(size_t)p * rl.M + m + 1] - rl.off[(size_t)p * rl.M + m]);
        }
    return requests > 0.0 ? replicas / requests / looked : 0.0;
}

struct mmsim_batch {
    CtxRef ctx;
    uint32_t flags = 0;
    int32_t n_seeds = 0, B = 0, M = 0, Gmax = 0, tiles = 0, waves = 0;
    int32_t smax_bucket = 0, rmax_all = 0, nslots = 0, waves_per_block = 1;
    size_t lds_bytes = 0;
    int64_t Rmax = 0, Rtotal = 0;
    std::vector<int64_t> wl_R;                           // [n_seeds] stream lengths
    std::vector<uint64_t> wl_id;                         // [n_seeds] ids of the workloads the batch was made from
    std::vector<std::vector<int32_t>> wl_model_requests;  // [n_seeds][M] requests per model of each stream
    int32_t row = kWave;       // width of the rows of the device tables and results: 64, or 1 if every simulation has a wavefront
    std::vector<int32_t> pos;  // pos[placement] = tile * row + lane it is simulated on
    // Paired batch (mmsim_eval_pairs): placement p is simulated on stream stream_of[p] only; a tile holds
    // placements of one stream, and results are laid out as for a single seed.
    bool paired = false;
    std::vector<int32_t> stream_of;   // [B]
    DevBuf<int32_t> tile_seed;        // [tiles]
    int32_t out_seeds = 1;            // seeds of the result layout: n_seeds, or 1 for a paired batch
    size_t wave_bytes = 0;     // LDS bytes of one wavefront's region (chunked loop, batching simulator)
    // Plain simulator, loop over runs: one launch of `sched_groups` workgroups, each owning a set of (tile, stream)
    // items that its wavefronts simulate segment by segment (clocks parked in `state` between segments).
    int32_t sched_groups = 0, sched_waves = 0, seg_requests = 0, max_nseg = 1;
    DevBuf<int32_t> plan;      // wg_off | item_tile | item_seed | item_nslots | item_bytes | item_nseg | part_off | part_bytes
    DevBuf<double> state;
    // ... with lanes at their own pace
    DevBuf<int64_t> run_base;
    DevBuf<uint32_t> run_off;
    DevBuf<Run> run_list;
    DevBuf<double> run_times;
    DevBuf<uint2> rep16, stage;

    DevBuf<Req> streams;
    DevBuf<int64_t> stream_off;
    DevBuf<uint32_t> rep32, repx32;
    DevBuf<uint64_t> rep8;
    DevBuf<uint8_t> repx;
    DevBuf<uint8_t> rmax;
    DevBuf<int32_t> kerr;
    DevBuf<uint32_t> ginfo;
    DevBuf<float> lat;
    DevBuf<int32_t> n_good;
    DevBuf<double> lat_sum;
    DevBuf<int32_t> model_good, group_req, group_good;
    DevBuf<unsigned long long> slot_cnt;      // plain simulator: per-group counts by last clock slot [waves][nslots][64]
    std::vector<int16_t> group_last_slot;     // [B][Gmax] last clock slot of each group, -1: no such group
    int32_t group_by_slot = 0, slot_rows = 0; // group_by_slot: the group counts are in slot_cnt (else in group_req / group_good)
    int32_t group_lds = 0;                    // the kernel keeps the slot counters in LDS while it runs
    DevBuf<double> finish;
    DevBuf<uint8_t> good;
    DevBuf<int64_t> fp_ops;
    // batching simulator
    DevBuf<int64_t> mq_off;
    DevBuf<MqEntry> mq;
    DevBuf<int32_t> status, batch_sizes;
    DevBuf<uint16_t> g2m_off, g2m_idx;
    DevBuf<float> lat_nb;
    std::vector<uint8_t> hosted;  // [B][M] model has a replica (batching: decides model_num_requests)
    BatchingArgs bargs{};
    // device buffers of mmsim_batch_model_stats, made by its first call and kept for the next ones
    DevBuf<const MqEntry *> st_mq;
    DevBuf<int64_t> st_i64;   // mq_off | lo | hi | sim_base
    DevBuf<int32_t> st_i32;   // sim_stream | model_req | model_good
    DevBuf<double> st_f64;    // the seven double results
    DevBuf<uint64_t> st_scratch;

    // Requests side by side (window_batch.hip): all inputs in one buffer, all outputs in another
    bool window = false;
    WindowArgs wargs{};
    DevBuf<uint8_t> win_in, win_out;
    size_t run_bytes = 0, run_ends = 0, run_pieces = 0, run_vals = 0;  // simulations cut into runs: of RunMemory, and offsets there
    RunMemory *runs_again = nullptr;                                   // ... of a batch that may be run again
    DevBuf<uint32_t> run_sync;                                         // ... batching simulator
    std::vector<std::shared_ptr<DevBuf<Req>>> win_streams;
    size_t win_lat_sum = 0, win_model = 0, win_group = 0, win_finish = 0, win_good = 0;  // offsets in win_out (n_good: 0)

    MixedArgs args{};
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    bool own_events = true;  // false: the context's events (batch in the static scratch)
    bool in_scratch = false; // the batch lives in the static scratch: nothing is allocated for it, pinned memory included
    bool ran = false;
    mmsim_options opt{};     // the options the batch was built with

    void run_again(RunMemory *runs) {
        runs_again = runs;
        runs->batches += 1;
    }
    ~mmsim_batch() {
        if (own_events && ev_start) (void)hipEventDestroy(ev_start);
        if (own_events && ev_stop) (void)hipEventDestroy(ev_stop);
        if (runs_again) --runs_again->batches;
    }
};

namespace mmsim {

// The latency table as the plain simulator's kernels read it: [M][lat_row], per model the latencies of configuration
// 0, then 1, ... (its cfg_pp[c] stages, or one value per configuration when every (model, configuration) has one
// latency for all its stages), then one +inf entry, the latency of "no such replica".
struct CompactLatency {
    bool uniform = true;
    int32_t row = 0;
    std::vector<int32_t> off;  // [C+1]
    std::vector<float> lat;
};
int compact_latency(const mmsim_tables *t, bool all_batch_sizes, CompactLatency *out);

// Builds the batch for the kernel of sim_window.hip if that is the one for it.  Returns MMSIM_OK, an error code, or 1
// when the batch is for the other kernels (or is not valid: they say what is wrong with it).
int build_window(mmsim_ctx *ctx, const mmsim_workload *const *wls, int32_t n_seeds, const mmsim_tables *t,
                 const mmsim_placements *p, const int32_t *stream_of, uint32_t flags, const mmsim_options &o, bool events,
                 mmsim_batch **out);
int run_window(mmsim_batch *b);
int fetch_window(mmsim_batch *b, mmsim_result *out);

}  // namespace mmsim
