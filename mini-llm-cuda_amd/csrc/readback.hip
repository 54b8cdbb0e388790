#include "readback.h"

#include <sched.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23 // Linux 5.14; older kernels answer EINVAL and the copy faults the pages in
#endif

// Threads from this many bytes on (starting them costs 0.1 ms).  Four of them: 84 MB of fresh pages are mapped in 1.2 ms, in
// 2.2 ms by eight, which get in each other's way and, holding the address space's lock, in the way of the thread that launches.
#define RB_WORKERS 4
#define RB_THREADED ((size_t)4 << 20)

Readback::Readback(const Part* parts, int n) {
    size_t total = 0;
    for (int i = 0; i < n; i++) total += parts[i].bytes;
    for (int i = 0; i < n; i++)
        for (size_t o = 0; o < parts[i].bytes; o += RB_CHUNK)
            chunks.push_back({parts[i].src + o, parts[i].dst + o, std::min((size_t)RB_CHUNK, parts[i].bytes - o)});
    if (total < RB_THREADED) return;
    const int nw = std::max(1, std::min(RB_WORKERS, (int)std::thread::hardware_concurrency() - 1));
    done.reset(new std::atomic<int>[chunks.size()]);
    for (size_t k = 0; k < chunks.size(); k++) done[k] = 0;
    workers.reserve(nw);
    try {
        for (int w = 0; w < nw; w++) workers.emplace_back(&Readback::work, this, w, nw);
    } catch (...) { // fewer threads than wanted: none at all, every piece is copied by the caller
        stop();
        workers.clear();
    }
}

Readback::~Readback() { stop(); }

void Readback::stop() {
    {
        std::lock_guard<std::mutex> g(m);
        abandoned = true;
    }
    cv.notify_all();
    for (std::thread& t : workers)
        if (t.joinable()) t.join();
}

void Readback::work(int w, int nw) {
    const size_t page = (size_t)sysconf(_SC_PAGESIZE);
    auto piece = [&](const Part& c, size_t& a, size_t& b) {
        const size_t each = ((c.bytes + nw - 1) / nw + 63) & ~(size_t)63;
        a = std::min(c.bytes, each * w);
        b = std::min(c.bytes, a + each);
    };
    for (size_t k = w; k < chunks.size(); k += nw) { // whole chunks here: neighbouring pieces share pages
        const uintptr_t a = ((uintptr_t)chunks[k].dst + page - 1) & ~(page - 1), b = ((uintptr_t)chunks[k].dst + chunks[k].bytes) & ~(page - 1);
        if (b > a) (void)madvise((void*)a, b - a, MADV_POPULATE_WRITE);
    }
    {
        std::unique_lock<std::mutex> g(m);
        cv.wait(g, [&] { return started || abandoned; });
    }
    for (size_t k = 0; k < chunks.size(); k++) {
        while (ready.load(std::memory_order_acquire) <= k) {
            if (abandoned) return;
            sched_yield();
        }
        size_t a, b;
        piece(chunks[k], a, b);
        memcpy(chunks[k].dst + a, stage + (k % RB_RING) * RB_CHUNK + a, b - a);
        done[k].fetch_add(1, std::memory_order_release);
    }
}

hipError_t Readback::run(hipStream_t st, unsigned char* stageBuf) {
    const size_t n = chunks.size();
    stage = stageBuf;
    hipEvent_t ev[RB_RING] = {};
    hipError_t e = hipSuccess;
    auto issue = [&](size_t k) {
        if (e == hipSuccess) e = hipMemcpyAsync(stage + (k % RB_RING) * RB_CHUNK, chunks[k].src, chunks[k].bytes, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev[k % RB_RING], st);
    };
    auto drained = [&](size_t k) { // chunk k is in the caller's memory
        while (done[k].load(std::memory_order_acquire) < (int)workers.size()) sched_yield();
    };
    for (int i = 0; i < RB_RING && e == hipSuccess; i++) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    {
        std::lock_guard<std::mutex> g(m);
        started = true;
    }
    cv.notify_all();
    for (size_t k = 0; k < std::min(n, (size_t)RB_RING); k++) issue(k);
    for (size_t k = 0; k < n && e == hipSuccess; k++) {
        e = hipEventSynchronize(ev[k % RB_RING]);
        if (e != hipSuccess) break;
        if (workers.empty()) {
            memcpy(chunks[k].dst, stage + (k % RB_RING) * RB_CHUNK, chunks[k].bytes);
            if (k + RB_RING < n) issue(k + RB_RING);
            continue;
        }
        ready.store(k + 1, std::memory_order_release);
        if (k > 0 && k - 1 + RB_RING < n) {
            drained(k - 1);
            issue(k - 1 + RB_RING);
        }
    }
    if (e == hipSuccess && !workers.empty())
        for (size_t k = n > RB_RING ? n - RB_RING : 0; k < n; k++) drained(k);
    else if (e != hipSuccess)
        (void)hipStreamSynchronize(st); // nothing may still be writing the staging memory
    for (int i = 0; i < RB_RING; i++)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    return e;
}
