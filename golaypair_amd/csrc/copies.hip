// Copies between the caller's ordinary memory and the device.  The runtime's copy
// of unpinned memory runs at 30 GB/s to the device and 18 GB/s back, one thread
// filling or emptying its staging memory.  A large copy goes through pinned
// buffers of the context instead, filled or emptied by the host threads
// while the DMA of the chunks before runs (57 GB/s).  Sorting 4e6 records of 22
// bytes, 88 MB each way, takes 5.0 ms instead of 8.5 ms; chunks of 1 MB give 7.5 ms
// (the threads' start and end shows), of 8 MB 4.9 ms.  Copies below kStagedCopy gain
// nothing (6 MB: 1.04 ms a call against 1.19 ms staged in smaller chunks).
#include <array>
#include <cstring>

#include "gp_internal.hpp"
#include "threadpool.hpp"

namespace gp {

namespace {

constexpr size_t kChunk = 4 << 20;
constexpr int kBufs = 3;

struct Ring {
    PinnedPool& pool;
    std::array<PinnedBuf*, kBufs> b{};
    explicit Ring(PinnedPool& p) : pool(p) {
        try {
            for (auto& x : b) x = pool.acquire(kChunk);
        } catch (...) {  // (no destructor runs)
            give_back();
            throw;
        }
    }
    ~Ring() { give_back(); }
    void give_back() {
        for (PinnedBuf* x : b) pool.release(x);  // (a copy from it that still runs is waited for by the next user)
    }
};

void copy_on_threads(char* dst, const char* src, size_t n) {
    constexpr size_t piece = 256 << 10;
    pool().parallel_for((n + piece - 1) / piece, [&](size_t i) {
        const size_t at = i * piece;
        std::memcpy(dst + at, src + at, std::min(piece, n - at));
    });
}

}  // namespace

void copy_to_device(gp_ctx* ctx, void* dst, const void* src, size_t bytes) {
    hipStream_t st = ctx->stream;
    if (bytes < kStagedCopy) {
        if (bytes) GP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
        return;
    }
    Ring ring(ctx->copy_pinned);
    int i = 0;
    for (size_t at = 0; at < bytes; at += kChunk, i = (i + 1) % kBufs) {
        PinnedBuf& b = *ring.b[i];
        if (b.upload_pending) GP_HIP(hipEventSynchronize(b.upload));
        const size_t n = std::min(kChunk, bytes - at);
        copy_on_threads(static_cast<char*>(b.p), static_cast<const char*>(src) + at, n);
        GP_HIP(hipMemcpyAsync(static_cast<char*>(dst) + at, b.p, n, hipMemcpyHostToDevice, st));
        b.record_upload(st);
    }
}

void copy_to_host(gp_ctx* ctx, void* dst, const void* src, size_t bytes) {
    hipStream_t st = ctx->stream;
    if (bytes < kStagedCopy) {
        if (bytes) GP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
        return;
    }
    Ring ring(ctx->copy_pinned);
    size_t sent = 0, at = 0;  // bytes whose DMA is queued; bytes delivered
    int is = 0, ia = 0;
    while (at < bytes) {
        for (; sent < bytes && sent < at + kBufs * kChunk; is = (is + 1) % kBufs) {
            const size_t n = std::min(kChunk, bytes - sent);
            GP_HIP(hipMemcpyAsync(ring.b[is]->p, static_cast<const char*>(src) + sent, n, hipMemcpyDeviceToHost, st));
            ring.b[is]->record_upload(st);
            sent += n;
        }
        PinnedBuf& b = *ring.b[ia];
        GP_HIP(hipEventSynchronize(b.upload));
        const size_t n = std::min(kChunk, bytes - at);
        copy_on_threads(static_cast<char*>(dst) + at, static_cast<const char*>(b.p), n);
        at += n;
        ia = (ia + 1) % kBufs;
    }
}

}  // namespace gp
