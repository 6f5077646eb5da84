"""Staged copies (golaypair_amd/csrc/copies.hip) over a stand-in of the runtime calls that
they make: every byte arrives at sizes around the chunks, a call that fails for want of
pinned memory hands back what it had taken, and a buffer is not freed under its last copy."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r'''
#pragma once
#include <cstdlib>
#include <cstring>
struct uint4 { unsigned x, y, z, w; };
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
typedef void* hipGraphExec_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipHostMallocDefault, hipEventDisableTiming };
inline int host_mallocs_left = 1 << 30;
inline const char* hipGetErrorString(hipError_t) { return "failed"; }
inline hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
    if (host_mallocs_left-- <= 0) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
inline int recorded = 0, freed_in_flight = 0;  // events recorded and not waited for; buffers freed meanwhile
inline hipError_t hipHostFree(void* p) { freed_in_flight += recorded; std::free(p); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = std::malloc(1); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { ++recorded; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { recorded = 0; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
'''

PROG = r'''
#include "copies.hip"
int main() {
    gp_ctx ctx;
    const size_t chunk = 4 << 20;
    for (size_t n : {size_t(0), size_t(5), gp::kStagedCopy - 1, gp::kStagedCopy, gp::kStagedCopy + 1, 3 * chunk, 5 * chunk + 77}) {
        std::vector<unsigned char> a(n + 1), b(n + 1, 1), c(n + 1, 2);
        for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 2654435761u >> 13);
        gp::copy_to_device(&ctx, b.data(), a.data(), n);
        gp::copy_to_host(&ctx, c.data(), b.data(), n);
        if (std::memcmp(a.data(), c.data(), n) || b[n] != 1 || c[n] != 2) { std::puts("bytes"); return 1; }
    }
    const size_t held = ctx.copy_pinned.bufs.size();
    if (held != 3) { std::puts("buffers"); return 1; }
    for (int left = 0; left < 3; ++left) {
        gp_ctx poor;
        std::vector<unsigned char> a(gp::kStagedCopy), b(gp::kStagedCopy);
        host_mallocs_left = left;
        bool failed = false;
        try { gp::copy_to_device(&poor, b.data(), a.data(), a.size()); } catch (const gp::HipError&) { failed = true; }
        if (!failed) { std::puts("no failure"); return 1; }
        for (auto& x : poor.copy_pinned.bufs) if (x->busy) { std::puts("kept a buffer"); return 1; }
        host_mallocs_left = 1 << 30;
        gp::copy_to_device(&poor, b.data(), a.data(), a.size());
        if (poor.copy_pinned.bufs.size() > 3) { std::puts("more buffers"); return 1; }
    }
    {   // a buffer that grows while its last upload may still run
        gp::PinnedPool pool;
        gp::PinnedBuf* b = pool.acquire(100);
        recorded = freed_in_flight = 0;
        b->record_upload(nullptr);
        pool.release(b);
        if (pool.acquire(1 << 20) != b || freed_in_flight) { std::puts("freed in flight"); return 1; }
    }
    std::puts("ok");
    return 0;
}
'''


def test_staged_copies(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    src = tmp_path / "copies_test.cpp"
    src.write_text(PROG)
    exe = tmp_path / "copies_test"
    subprocess.run(["g++", "-O2", "-std=c++20", "-pthread", "-I", str(tmp_path),
                    "-I", os.path.join(ROOT, "golaypair_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
