// Library context: device, stream and the per-context error message that
// the C-ABI reports through fyzz_hip_last_error().
#pragma once
#include <cstring>
#include <exception>
#include <initializer_list>
#include <map>
#include <mutex>
#include <vector>
#include <new>
#include <string>

#include "common.hpp"

namespace fyzz_hip {
// Optional per-stage timing with HIP events recorded on the context's
// stream around named launches; read back (and reset) on demand.
struct Profiler {
    struct Span {
        hipEvent_t a, b;
    };
    bool enabled = false;
    std::map<std::string, std::vector<Span>> spans;
    std::vector<hipEvent_t> pool;
    hipEvent_t take() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        FYZZ_HIP_CHECK(hipEventCreate(&e));
        return e;
    }
    // Returns the span index to close with end(), or -1 when disabled.
    long begin(const std::string& name, hipStream_t st) {
        if (!enabled) return -1;
        Span s{take(), take()};
        FYZZ_HIP_CHECK(hipEventRecord(s.a, st));
        auto& v = spans[name];
        v.push_back(s);
        return static_cast<long>(v.size() - 1);
    }
    void end(const std::string& name, long idx, hipStream_t st) {
        if (idx < 0) return;
        FYZZ_HIP_CHECK(hipEventRecord(spans[name][static_cast<std::size_t>(idx)].b, st));
    }
    // Sum of elapsed ms and span count for `name`; releases its events.
    void read(const std::string& name, double* total_ms, std::uint64_t* count) {
        double t = 0.0;
        std::uint64_t c = 0;
        auto it = spans.find(name);
        if (it != spans.end()) {
            for (auto& s : it->second) {
                FYZZ_HIP_CHECK(hipEventSynchronize(s.b));
                float ms = 0.f;
                FYZZ_HIP_CHECK(hipEventElapsedTime(&ms, s.a, s.b));
                t += ms;
                ++c;
                pool.push_back(s.a);
                pool.push_back(s.b);
            }
            spans.erase(it);
        }
        *total_ms = t;
        *count = c;
    }
    ~Profiler() {
        for (auto& kv : spans)
            for (auto& s : kv.second) {
                (void)hipEventDestroy(s.a);
                (void)hipEventDestroy(s.b);
            }
        for (auto e : pool) (void)hipEventDestroy(e);
    }
};
struct ProfScope {
    Profiler* p;
    std::string name;
    long idx;
    hipStream_t st;
    ProfScope(Profiler* prof, const char* n, hipStream_t s) : p(prof), name(n), idx(-1), st(s) {
        if (p && p->enabled) idx = p->begin(name, st);
    }
    ~ProfScope() {
        try {
            if (p && idx >= 0) p->end(name, idx, st);
        } catch (...) {
        }
    }
};
// Pinned host memory for small readbacks: a copy into pageable memory is
// staged by the runtime and synchronizes by itself, about 20 us each against
// half of that into pinned memory. At most kMax bytes per context, given
// back with it; larger readbacks go straight to the caller's memory.
struct HostStage {
    static constexpr std::size_t kMax = 1u << 20;
    std::mutex mu;
    unsigned char* p = nullptr;
    std::size_t cap = 0;
    ~HostStage() {
        if (p) (void)hipHostFree(p);
    }
    void reserve(std::size_t n) {
        if (n <= cap) return;
        std::size_t want = 4096;
        while (want < n) want <<= 1;
        if (p) FYZZ_HIP_CHECK(hipHostFree(p));
        p = nullptr;
        cap = 0;
        void* q = nullptr;
        FYZZ_HIP_CHECK(hipHostMalloc(&q, want, hipHostMallocDefault));
        p = static_cast<unsigned char*>(q);
        cap = want;
    }
};
struct Readback {
    void* dst;        // host
    const void* src;  // device
    std::size_t bytes;
};
}  // namespace fyzz_hip

struct fyzz_hip_context {
    int device = 0;
    hipStream_t stream = nullptr;  // null = the device's default stream
    bool cooperative = true;       // the Dy sweeps: cooperative or plain launches
    std::string last_error;
    fyzz_hip::Profiler prof;
    fyzz_hip::HostStage stage;
};

namespace fyzz_hip {

// Device words read back in stream order with one synchronization.
inline void read_back(fyzz_hip_context* ctx, std::initializer_list<Readback> parts) {
    hipStream_t st = ctx->stream;
    std::size_t total = 0;
    for (const Readback& r : parts) total += (r.bytes + 15) & ~std::size_t{15};
    if (total > HostStage::kMax) {
        for (const Readback& r : parts)
            if (r.bytes) FYZZ_HIP_CHECK(hipMemcpyAsync(r.dst, r.src, r.bytes, hipMemcpyDeviceToHost, st));
        FYZZ_HIP_CHECK(hipStreamSynchronize(st));
        return;
    }
    if (!total) {
        FYZZ_HIP_CHECK(hipStreamSynchronize(st));
        return;
    }
    std::lock_guard<std::mutex> lock(ctx->stage.mu);
    ctx->stage.reserve(total);
    std::size_t at = 0;
    for (const Readback& r : parts) {
        if (r.bytes)
            FYZZ_HIP_CHECK(hipMemcpyAsync(ctx->stage.p + at, r.src, r.bytes, hipMemcpyDeviceToHost, st));
        at += (r.bytes + 15) & ~std::size_t{15};
    }
    FYZZ_HIP_CHECK(hipStreamSynchronize(st));
    at = 0;
    for (const Readback& r : parts) {
        if (r.bytes) std::memcpy(r.dst, ctx->stage.p + at, r.bytes);
        at += (r.bytes + 15) & ~std::size_t{15};
    }
}

// Runs f, converting exceptions into a status code and the context's
// last-error string; no exception crosses the C-ABI.
template <class F>
int guarded(fyzz_hip_context* ctx, F&& f) {
    if (!ctx) return kInvalidArgument;
    try {
        FYZZ_HIP_CHECK(hipSetDevice(ctx->device));
        f();
        ctx->last_error.clear();
        return kOk;
    } catch (const Error& e) {
        ctx->last_error = e.what();
        return e.code;
    } catch (const std::bad_alloc&) {
        ctx->last_error = "host allocation failed";
        return kOutOfMemory;
    } catch (const std::exception& e) {
        ctx->last_error = e.what();
        return kLogicError;
    } catch (...) {
        ctx->last_error = "unknown failure";
        return kLogicError;
    }
}

}  // namespace fyzz_hip
