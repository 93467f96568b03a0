"""Reading results back (spk::readBack of spock.cu_amd/csrc/common.hpp), on the CPU: the piece and thread protocol
against a stand-in for the HIP runtime whose stream does nothing before it is waited for, under
ThreadSanitizer.  A second build refuses new threads after a given number (0: the caller converts alone).

Sizes lie around multiples of a piece.  Every word arrives once and converted, and an error of the copy or of the
wait ends the call with that error, its threads joined and the next call working."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r'''
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>
enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum { hipHostMallocDefault = 0 };
enum hipMemcpyKind { hipMemcpyDeviceToHost };
typedef void *hipStream_t;
inline std::vector<std::function<void()>> queued;
inline int syncs = 0, failSync = -1, copies = 0, failCopy = -1;
inline const char *hipGetErrorString(hipError_t) { return "stub error"; }
inline hipError_t hipStreamSynchronize(hipStream_t) {
    if (syncs++ == failSync) { queued.clear(); return hipErrorUnknown; }
    for (auto &f : queued) f();
    queued.clear();
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, int) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    if (copies++ == failCopy) return hipErrorUnknown;
    queued.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
'''

HARNESS = r'''
#include <cstdio>
struct spk_batch;
#include "common.hpp"

#ifdef REFUSE
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
static int allowed = 0;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    if (allowed-- <= 0) return EAGAIN;
    static auto next = (int (*)(pthread_t *, const pthread_attr_t *, void *(*) (void *), void *)) dlsym(RTLD_NEXT, "pthread_create");
    return next(t, a, f, arg);
}
#endif

template <typename S, typename D>
void once(spk_ctx *c, size_t n) {
    std::vector<S> src(n);
    for (size_t k = 0; k < n; k++) src[k] = (S) (k % 1000003) + (S) 0.5;
    std::vector<D> dst(n + 2, (D) -1);
    spk::readBack(c, dst.data() + 1, (const S *) src.data(), n);
    if (dst[0] != (D) -1 || dst[n + 1] != (D) -1) { std::printf("%zu: out of range\n", n); std::exit(2); }
    for (size_t k = 0; k < n; k++)
        if (dst[k + 1] != (D) src[k]) { std::printf("%zu: word %zu\n", n, k); std::exit(3); }
}

template <typename S, typename D>
void sizes(spk_ctx *c) {
    const size_t per = spk::STAGE_BYTES / sizeof(S);
    for (size_t n : {(size_t) 0, (size_t) 1, per / 4, per / 4 + 1, per - 1, per, per + 1, 2 * per, 3 * per - 1, 5 * per + 3}) once<S, D>(c, n);
}

int main() {
    spk_ctx *c = new spk_ctx;
#ifdef REFUSE
    for (int k : {0, 1, 3}) { allowed = k; once<float, double>(c, 5 * spk::STAGE_BYTES / 4 + 3); allowed = k; once<double, double>(c, 2 * spk::STAGE_BYTES / 8); }
#else
    sizes<float, double>(c);
    sizes<float, float>(c);
    sizes<double, double>(c);
    int errors = 0;
    for (int at = 0; at < 4; at++)
        for (int what = 0; what < 2; what++) {
            syncs = copies = 0;
            failSync = what ? at : -1;
            failCopy = what ? -1 : at;
            try { once<float, double>(c, 4 * spk::STAGE_BYTES / 4); } catch (const spk::HipError &) { errors++; }
            failSync = failCopy = -1;
            queued.clear();
            once<float, double>(c, 3 * spk::STAGE_BYTES / 4);
        }
    if (errors != 8) { std::printf("%d errors\n", errors); return 4; }
#endif
    spk::releaseCtx(c);
    std::puts("done");
    return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("flags", [["-fsanitize=thread"], ["-DREFUSE", "-ldl"]], ids=["threads", "refused"])
def test_read_back(tmp_path, flags):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    src, exe = tmp_path / "r.cpp", tmp_path / "r"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-pthread", f"-I{tmp_path}",
                    f"-I{os.path.join(ROOT, 'spock.cu_amd', 'csrc')}", str(src), "-o", str(exe)] + flags, check=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, (run.stdout + run.stderr)[-3000:]
    assert run.stdout.strip() == "done"
