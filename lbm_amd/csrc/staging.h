// Large copies between device memory and a caller's ordinary host memory.
//
// The runtime's own path for pageable memory copies through one pinned buffer
// with one thread: 17.7 GB/s out, 29 GB/s in, and the first touch of the
// caller's pages (a fresh 134 MB array: 5 ms) in the same thread, where the
// link takes 57 GB/s.  Here four threads each own two pinned 1 MB chunks: a
// thread keeps one chunk in flight on the object's stream while it copies the
// other, and touches its pages before it first waits, while the stream's earlier
// work is still running.  134 MB after 50 ms of steps: 13.0 -> 4.5 ms.
//
// The chunks are moved by a kernel and not by the copy engines: those also clear
// the memory of allocations given back, and a chunk waits its turn behind such a
// job.  For seconds after grids of 240 MB were destroyed a chunk took 150 us
// instead of 20 and a read of 27 MB 3.9 ms, the runtime's own path 1.7, with the
// kernel 0.67 (0.9 with free engines; 134 MB: 20 ms, 4.2 with free engines, 3.0).
//
// An object (grid, batch, network, solver) owns one Staging, made on its first
// large copy and freed with it; it is used by the object's own calls only, which
// are not concurrent.
//
// Memory the runtime knows (a caller's own pinned buffer) takes the runtime's copy,
// which is one transfer at the link's rate: three planes of 8192 x 4096 into
// pinned memory 7.1 ms that way, 12.7 through the chunks.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace {

struct Piece {
    void *host, *device;
    size_t bytes;
};

// n bytes (of 4-byte aligned addresses) between device and pinned host memory, 16 a thread
__global__ void k_move(const char *src, char *dst, uint32_t n) {
    typedef uint32_t Quad __attribute__((vector_size(16), aligned(4), may_alias));
    const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 16;
    if (i + 16 <= n) *(Quad *)(dst + i) = *(const Quad *)(src + i);
    else
        for (uint32_t b = i; b < n; ++b) dst[b] = src[b];
}

struct Staging {
    static constexpr size_t kChunk = (size_t)1 << 20;
    static constexpr int kThreads = 4, kSlots = 2 * kThreads;
    // below these the threads' start costs what they save (4 MB: 240 us out, 140 in)
    static constexpr size_t kLeastOut = (size_t)4 << 20, kLeastIn = (size_t)8 << 20;
    char *buf = nullptr;
    hipEvent_t done[kSlots] = {};  // the last copy through each chunk
    bool unavailable = false;

    bool ready() {
        if (buf || unavailable) return buf != nullptr;
        if (hipHostMalloc((void **)&buf, kSlots * kChunk, hipHostMallocDefault) != hipSuccess) buf = nullptr;
        for (int i = 0; buf && i < kSlots; ++i)
            if (hipEventCreateWithFlags(&done[i], hipEventDisableTiming | hipEventBlockingSync) != hipSuccess) {
                done[i] = nullptr;
                release();
            }
        if (!buf) {
            (void)hipGetLastError();
            unavailable = true;  // this object copies the plain way from now on
        }
        return buf != nullptr;
    }
    void release() {
        for (hipEvent_t &e : done) {
            if (e) {
                (void)hipEventSynchronize(e);
                (void)hipEventDestroy(e);
            }
            e = nullptr;
        }
        if (buf) (void)hipHostFree(buf);
        buf = nullptr;
    }

    // is every piece's host memory the process's own, unknown to the runtime?
    static bool ordinary(const Piece *pieces, int n) {
        for (int i = 0; i < n; ++i) {
            hipPointerAttribute_t a;
            if (hipPointerGetAttributes(&a, pieces[i].host) != hipSuccess)
                (void)hipGetLastError();  // (how older runtimes answer for such memory)
            else if (a.type != hipMemoryTypeUnregistered)
                return false;
        }
        return true;
    }

    // Copies the pieces in stream order after the stream's earlier work.  Out of
    // the device it returns when they are there; into it, the caller waits for
    // the stream before it gives the host memory back.
    hipError_t copy(int dev, hipStream_t s, const Piece *pieces, int n, bool out) {
        size_t total = 0;
        for (int i = 0; i < n; ++i) total += pieces[i].bytes;
        if (total < (out ? kLeastOut : kLeastIn) || !ordinary(pieces, n) || !ready()) {
            for (int i = 0; i < n; ++i) {
                const Piece &p = pieces[i];
                const hipError_t e = out ? hipMemcpyAsync(p.host, p.device, p.bytes, hipMemcpyDeviceToHost, s)
                                         : hipMemcpyAsync(p.device, p.host, p.bytes, hipMemcpyHostToDevice, s);
                if (e != hipSuccess) return e;
            }
            return out ? hipStreamSynchronize(s) : hipSuccess;
        }
        std::vector<Piece> chunks;
        chunks.reserve(total / kChunk + (size_t)n);
        for (int i = 0; i < n; ++i)
            for (size_t at = 0; at < pieces[i].bytes; at += kChunk)
                chunks.push_back({(char *)pieces[i].host + at, (char *)pieces[i].device + at,
                                  pieces[i].bytes - at < kChunk ? pieces[i].bytes - at : kChunk});
        hipError_t err[kThreads] = {};
        std::thread threads[kThreads];
        auto work = [&](int t) { err[t] = out ? share_out(dev, s, chunks, t) : share_in(dev, s, chunks, t); };
        int started = 1;
        try {
            for (; started < kThreads; ++started) threads[started] = std::thread(work, started);
        } catch (const std::exception &) {  // no thread, or no memory for one: the shares left are done here
        }
        work(0);
        for (int t = started; t < kThreads; ++t) work(t);
        for (int t = 1; t < started; ++t) threads[t].join();
        for (hipError_t e : err)
            if (e != hipSuccess) {
                (void)hipStreamSynchronize(s);
                return e;
            }
        return hipSuccess;
    }

private:
    // a chunk in stream order
    static hipError_t move(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t s) {
        if (((uintptr_t)dst | (uintptr_t)src) & 3) return hipMemcpyAsync(dst, src, n, kind, s);
        hipLaunchKernelGGL(k_move, dim3((unsigned)((n + 4095) / 4096)), dim3(256), 0, s, (const char *)src, (char *)dst,
                           (uint32_t)n);
        return hipGetLastError();
    }

    // thread t's chunks: t, t + kThreads, ...; the i-th of them through slot
    // t + kThreads (i % 2)
    hipError_t share_out(int dev, hipStream_t s, const std::vector<Piece> &chunks, int t) {
        hipError_t e = hipSetDevice(dev);
        auto issue = [&](size_t c) {
            const int slot = (int)(c % kSlots);
            if (e == hipSuccess) e = hipEventSynchronize(done[slot]);  // an earlier call's copy through it
            if (e == hipSuccess)
                e = move(buf + slot * kChunk, chunks[c].device, chunks[c].bytes, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(done[slot], s);
        };
        for (size_t c = t; c < chunks.size() && c < kSlots; c += kThreads) issue(c);
        // first touch of the pages, without changing what they hold
        for (size_t c = t; c < chunks.size(); c += kThreads)
            for (size_t b = 0; b < chunks[c].bytes; b += 4096)
                (void)__atomic_fetch_or((char *)chunks[c].host + b, 0, __ATOMIC_RELAXED);
        for (size_t c = t; c < chunks.size() && e == hipSuccess; c += kThreads) {
            e = hipEventSynchronize(done[c % kSlots]);
            if (e != hipSuccess) break;
            std::memcpy(chunks[c].host, buf + (c % kSlots) * kChunk, chunks[c].bytes);
            if (c + kSlots < chunks.size()) issue(c + kSlots);
        }
        return e;
    }
    hipError_t share_in(int dev, hipStream_t s, const std::vector<Piece> &chunks, int t) {
        hipError_t e = hipSetDevice(dev);
        for (size_t c = t; c < chunks.size() && e == hipSuccess; c += kThreads) {
            const int slot = (int)(c % kSlots);
            e = hipEventSynchronize(done[slot]);
            if (e != hipSuccess) break;
            std::memcpy(buf + slot * kChunk, chunks[c].host, chunks[c].bytes);
            e = move(chunks[c].device, buf + slot * kChunk, chunks[c].bytes, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(done[slot], s);
        }
        return e;
    }
};

}  // namespace
