// Host paths of libmmsim against a HIP runtime that lives in this program: copies to and from host memory are carried
// out when their stream is waited for, and not before, and the n-th call that can fail does.  For every n, the calls below
// must leave no copy behind whose host memory is gone, and no device memory.  Nothing here needs or touches a GPU.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <malloc.h>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../include/mmsim.h"

namespace {
struct Copy {
    void *dst;
    const void *src;
    size_t n;
};
template <class T>
struct Plain {  // (memory that operator delete below does not see)
    using value_type = T;
    Plain() = default;
    template <class U> Plain(const Plain<U> &) {}
    T *allocate(size_t n) { return static_cast<T *>(std::malloc(n * sizeof(T))); }
    void deallocate(T *p, size_t) { std::free(p); }
    template <class U> bool operator==(const Plain<U> &) const { return true; }
    template <class U> bool operator!=(const Plain<U> &) const { return false; }
};
std::recursive_mutex lock;
std::vector<Copy, Plain<Copy>> pending;
std::map<char *, size_t, std::less<char *>, Plain<std::pair<char *const, size_t>>> device;
long calls = 0, fail_at = 0;
int dangling = 0;
hipError_t last = hipSuccess;

void carry_out() {
    for (const Copy &c : pending) std::memcpy(c.dst, c.src, c.n);
    pending.clear();
}
bool fails() { return ++calls == fail_at; }
hipError_t result(hipError_t failure) {
    if (!fails()) return hipSuccess;
    return last = failure;
}
void gone(void *p, size_t n) {  // host memory that a copy still needs
    std::lock_guard<std::recursive_mutex> hold(lock);
    for (const Copy &c : pending)
        for (const void *q : {c.src, static_cast<const void *>(c.dst)})
            if (q >= p && q < static_cast<char *>(p) + n) {
                ++dangling;
                carry_out();
                return;
            }
}
}  // namespace

void *operator new(size_t n) {
    void *p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept {
    if (p) gone(p, malloc_usable_size(p));
    std::free(p);
}
void operator delete(void *p, size_t) noexcept { operator delete(p); }

extern "C" {
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) { *g = *b = dim3(1); *s = 0; *st = nullptr; return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return result(hipErrorLaunchFailure); }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 163840; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return result(hipErrorOutOfMemory); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 0.0f; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return result(hipErrorUnknown); }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { std::memset(a, 0, sizeof(*a)); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetSymbolAddress(void **p, const void *) { static char scratch[256]; *p = scratch; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (result(hipErrorOutOfMemory) != hipSuccess) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    if (p) gone(p, malloc_usable_size(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    if (result(hipErrorOutOfMemory) != hipSuccess) return hipErrorOutOfMemory;
    *p = std::calloc(n, 1);
    device[static_cast<char *>(*p)] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    if (!p) return hipSuccess;
    carry_out();
    device.erase(static_cast<char *>(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    if (result(hipErrorUnknown) != hipSuccess) return hipErrorUnknown;
    pending.push_back({dst, src, n});
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    carry_out();
    if (result(hipErrorUnknown) != hipSuccess) return hipErrorUnknown;
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int v, size_t n, hipStream_t) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    carry_out();
    if (result(hipErrorUnknown) != hipSuccess) return hipErrorUnknown;
    std::memset(dst, v, n);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::recursive_mutex> hold(lock);
    carry_out();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
}

namespace {
const int M = 3, C = 2, G = 2, B = 70;
const int64_t R = 9000;  // two blocks of runs
struct Problem {
    std::vector<double> t;
    std::vector<int32_t> m, pp{2, 4}, sizes{1, 2}, groups, cfg, idx;
    std::vector<float> slo, lat;
    std::vector<int64_t> off;
    mmsim_tables tables{};
    mmsim_placements places{};
    Problem() : t(R), m(R), groups(B, G), cfg(B * G), slo(R, 1.0f), lat(M * C * 4 * 2, 0.05f), off(B * (G + 1)) {
        for (int64_t i = 0; i < R; ++i) {
            t[i] = 0.001 * (double)i;
            m[i] = (int32_t)(i / 8 % M);
        }
        for (int b = 0; b < B; ++b)
            for (int g = 0; g < G; ++g) {
                cfg[b * G + g] = (b + g) % C;
                off[b * (G + 1) + g] = (int64_t)idx.size();
                idx.push_back((b + g) % M);
                off[b * (G + 1) + g + 1] = (int64_t)idx.size();
            }
        tables = {M, C, 4, 2, lat.data(), pp.data(), sizes.data(), 0.011};
        places = {B, G, groups.data(), cfg.data(), off.data(), idx.data()};
    }
};

std::string kernel;  // of the batch that was made last
int batch(mmsim_ctx *ctx, Problem &p, uint32_t flags, int32_t skip_ahead, int32_t window) {
    mmsim_workload *w = nullptr;
    mmsim_batch *b = nullptr;
    int rc = mmsim_workload_create(ctx, R, M, p.t.data(), p.m.data(), p.slo.data(), &w);
    if (rc == MMSIM_OK) {
        mmsim_options o;
        mmsim_options_default(&o);
        o.skip_ahead = skip_ahead;
        o.window_lanes = window;
        rc = mmsim_batch_create_ex(ctx, &w, 1, &p.tables, &p.places, flags, &o, &b);
    }
    if (rc == MMSIM_OK) {
        char name[200];
        mmsim_batch_kernel_name(b, name, sizeof(name));
        kernel = name;
        rc = mmsim_batch_run(b);
    }
    if (rc == MMSIM_OK && (flags & MMSIM_WANT_PER_REQUEST)) {
        std::vector<int32_t> a(B * M), c(B * M);
        std::vector<double> d[7];
        for (auto &v : d) v.resize(B * M);
        mmsim_model_stats out{a.data(), c.data(), d[0].data(), d[1].data(), d[2].data(), d[3].data(), d[4].data(), d[5].data(), d[6].data()};
        const int64_t skip = 0;
        rc = mmsim_batch_model_stats(b, &w, 1, &skip, &out);
    }
    if (rc == MMSIM_OK && window > 0) {  // (the other kernels say that they completed every item, which a launch here does not)
        std::vector<int64_t> good(B);
        std::vector<double> sum(B), finish(B * R);
        std::vector<uint8_t> flags_of(B * R);
        mmsim_result out{};
        out.n_good = good.data();
        out.latency_sum = sum.data();
        out.finish = finish.data();
        out.good = flags_of.data();
        rc = mmsim_batch_fetch(b, &out);
    }
    mmsim_batch_destroy(b);
    mmsim_workload_destroy(w);
    return rc;
}

int scalar(mmsim_ctx *ctx, Problem &p) {
    std::vector<double> finish(R);
    std::vector<uint8_t> good(R);
    std::vector<int32_t> rows{0, -1, 1, -1, 0, 1}, counts(2 * M + 2 * G);
    std::vector<float> most(M * G, 0.1f), sum(M * G, 0.2f);
    return mmsim_simulate_requests(ctx, finish.data(), good.data(), p.t.data(), p.m.data(), p.slo.data(), rows.data(), most.data(), sum.data(), R, M, G,
                                   0.011, counts.data(), counts.data() + M, counts.data() + 2 * M, counts.data() + 2 * M + G);
}
}  // namespace

int main() {
    Problem p;
    mmsim_ctx *ctx = nullptr;
    if (mmsim_ctx_create(0, &ctx) != MMSIM_OK) return std::printf("no context: %s\n", mmsim_last_error()), 1;
    struct Path {
        const char *name, *kernel;
        uint32_t flags;
        int32_t skip_ahead, window;
    } paths[] = {{"lanes at their own pace", "sim_lanes_kernel", 0, 2, -1},
                 {"loop over runs", "sim_mixed_kernel", MMSIM_WANT_MODEL_COUNTS | MMSIM_WANT_GROUP_COUNTS, 1, -1},
                 {"outputs of every request", "sim_mixed_kernel", MMSIM_WANT_PER_REQUEST, 1, -1},
                 {"requests side by side", "sim_window_kernel", MMSIM_WANT_PER_REQUEST, -1, 64},
                 {"batching", "sim_batching", MMSIM_BATCHING | MMSIM_WANT_MODEL_COUNTS, -1, 0},
                 {"one clock a group", "", 0, 0, 0}};
    int bad = 0;
    for (const Path &path : paths) {
        long n = 0, other = 0;
        for (fail_at = 0;; ++fail_at) {
            calls = 0;
            kernel.clear();
            const int before = dangling;
            const int rc = *path.kernel ? batch(ctx, p, path.flags, path.skip_ahead, path.window) : scalar(ctx, p);
            const bool failed = fail_at > 0 && calls >= fail_at;
            if (dangling != before) bad += std::printf("%s: call %ld of %ld failed: a copy outlived its host memory\n", path.name, fail_at, n) > 0;
            if (!device.empty()) {
                bad += std::printf("%s: call %ld of %ld failed: device memory was not given back\n", path.name, fail_at, n) > 0;
                device.clear();
            }
            if (fail_at == 0) {
                n = calls;
                if (rc != MMSIM_OK || kernel.compare(0, std::strlen(path.kernel), path.kernel) != 0)
                    bad += std::printf("%s: %d %s %s\n", path.name, rc, kernel.c_str(), mmsim_last_error()) > 0;
            } else if (!failed) {
                break;
            } else if (rc == MMSIM_OK) {
                other += kernel.compare(0, std::strlen(path.kernel), path.kernel) != 0;
            }
        }
        std::printf("%s: %ld calls that can fail, %ld of them answered by another kernel\n", path.name, n, other);
        // lanes at their own pace need memory that the other loops do without
        if (path.skip_ahead == 2 && other == 0) bad += std::printf("%s: a batch without memory for its tables was refused\n", path.name) > 0;
    }
    fail_at = 0;
    mmsim_ctx_destroy(ctx);
    std::printf(bad ? "%d problems\n" : "ok\n", bad);
    return bad != 0;
}
