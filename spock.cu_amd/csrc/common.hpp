// Host-side pieces shared by the C ABI translation units: the context, device buffers and
// HIP error checks.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "handles.hpp"

struct spk_ctx : spk::Counted {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    double tickRateHz = 1e8;
    // two pinned pieces of spk::STAGE_BYTES for reading large results back; made at the first one
    std::mutex stageLock;
    void *stage = nullptr;
};

namespace spk {

// Frees a context whose last reference was dropped: its stream, then the object.
inline void freeCtx(spk_ctx *c) {
    if (c->stream) {
        (void) hipStreamSynchronize(c->stream);
        (void) hipStreamDestroy(c->stream);
    }
    if (c->stage) (void) hipHostFree(c->stage);
    delete c;
}

inline void releaseCtx(spk_ctx *c) { release(c, freeCtx); }

struct HipError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

inline void check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw HipError(std::string(what) + ": " + hipGetErrorString(e));
}

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void) hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    void alloc(size_t b) {
        release();
        if (b == 0) b = 16;
        check(hipMalloc(&p, b), "hipMalloc");
        bytes = b;
    }
    template <typename T>
    T *as() const {
        return static_cast<T *>(p);
    }
};

// Reads n words of type S back into dst (type D).  put(first, count, to) queues the words first .. first + count
// on the context's stream to pinned memory.  The device fills one piece while up to 8 threads convert the
// other: what bounds a large read is the host, above all the page faults of a destination nobody has touched
// yet (26.9 M FP32 parameters: 10.6 ms by one copy to pageable memory, now 4.0).
constexpr size_t STAGE_BYTES = 4 << 20;

template <typename S, typename D, typename F>
void readBack(spk_ctx *c, D *dst, size_t n, F put) {
    std::lock_guard<std::mutex> guard(c->stageLock);
    if (!c->stage) check(hipHostMalloc(&c->stage, 2 * STAGE_BYTES, hipHostMallocDefault), "hipHostMalloc");
    const size_t per = STAGE_BYTES / sizeof(S);
    const long pieces = (long) ((n + per - 1) / per);
    auto piece = [&](long i) { return static_cast<S *>(c->stage) + (i & 1) * per; };
    auto size = [&](long i) { return std::min(per, n - (size_t) i * per); };
    auto convert = [&](long i, size_t part, size_t parts) {
        const size_t len = size(i), a = len * part / parts, b = len * (part + 1) / parts;
        std::copy(piece(i) + a, piece(i) + b, dst + (size_t) i * per + a);
    };
    if (pieces <= 1) {
        if (n == 0) return;
        put(0, n, piece(0));
        check(hipStreamSynchronize(c->stream), "read back");
        convert(0, 0, 1);
        return;
    }
    std::atomic<long> ready{0}, done{0};  // pieces in pinned memory (< 0: give up), parts converted
    std::atomic<int> threads{0};
    auto work = [&](int t) {
        for (long i = 0; i < pieces; i++) {
            long r;
            while ((r = ready.load()) >= 0 && r <= i) ready.wait(r);
            if (r < 0) return;
            convert(i, t, threads.load());
            done.fetch_add(1);
            done.notify_one();
        }
    };
    std::vector<std::thread> pool;
    auto end = [&](long r) {
        ready.store(r);
        ready.notify_all();
        for (auto &t : pool) t.join();
    };
    try {
        put(0, size(0), piece(0));
        const int want = (int) std::clamp(std::thread::hardware_concurrency(), 1u, 8u);
        try {
            for (int t = 0; t < want; t++) pool.emplace_back(work, t);
        } catch (const std::system_error &) {  // fewer threads, or this one alone
        }
        const int got = (int) pool.size();
        threads.store(std::max(1, got));
        for (long i = 0; i < pieces; i++) {
            check(hipStreamSynchronize(c->stream), "read back");
            if (got) {
                // everyone is done with the pieces before i, so the other one is free; only then may i be started,
                // or its parts would be counted for a part of i - 1
                for (long d; (d = done.load()) < i * got;) done.wait(d);
                ready.store(i + 1);
                ready.notify_all();
            }
            if (i + 1 < pieces) put((size_t) (i + 1) * per, size(i + 1), piece(i + 1));
            if (!got) convert(i, 0, 1);
        }
    } catch (...) {
        end(-1);
        throw;
    }
    end(pieces);
}

// The same from one device array; a small one needs no pinned memory.
template <typename S, typename D>
void readBack(spk_ctx *c, D *dst, const S *src, size_t n) {
    if (n * sizeof(S) <= STAGE_BYTES / 4) {
        std::vector<S> tmp(n);
        check(hipMemcpy(tmp.data(), src, n * sizeof(S), hipMemcpyDeviceToHost), "read back");
        std::copy(tmp.begin(), tmp.end(), dst);
        return;
    }
    readBack<S>(c, dst, n, [&](size_t first, size_t count, S *to) {
        check(hipMemcpyAsync(to, src + first, count * sizeof(S), hipMemcpyDeviceToHost, c->stream), "read back");
    });
}

// A cooperative launch the device refused; it queued nothing and can be retried with one
// workgroup (the C ABI returns SPK_ERR_COOPERATIVE_LAUNCH for it).
struct CoopRefused : HipError {
    using HipError::HipError;
};

inline int fail(spk_ctx *ctx, const std::exception &e) {
    if (ctx) ctx->err = e.what();
    return dynamic_cast<const CoopRefused *>(&e) ? -2 : -1;
}

// For a writer of all of a batch's iterates on context c's stream: where a shared FP32 batch of c holds them
// (16 instances to a block, instance fastest) if an iterate has n words, its residuals cleared; else null.
float *laneIterates(spk_batch *b, const spk_ctx *c, long n);

}  // namespace spk
