// Device results into a caller's pageable memory: through a ring of pinned chunks, each shared out to a few host threads.
//
// What bounds it: a copy into pages that the caller has not touched yet costs their faults first (one thread, with or without
// the driver's own staging, gets 3 to 10 GB/s; the link does 53).  So the threads start when the call does and, while the
// GPU still computes, have the kernel map the pages (MADV_POPULATE_WRITE: the contents stay); then each copies its share of
// every chunk that lands.  Logits and probabilities of 517 tokens of a 20 160-word vocabulary (83 MB): 2.2 ms behind the last
// kernel, 8 before.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#define RB_CHUNK ((size_t)4 << 20)
#define RB_RING 4

class Readback {
  public:
    struct Part {
        const char* src; // device
        char* dst;
        size_t bytes;
    };
    Readback(const Part* parts, int n);
    ~Readback();
    // after the stream's work so far; stageBuf: RB_RING * RB_CHUNK bytes of pinned memory.  Returns when all is copied.
    hipError_t run(hipStream_t st, unsigned char* stageBuf);

  private:
    void work(int w, int nw);
    void stop();
    std::vector<Part> chunks;
    std::vector<std::thread> workers;
    std::unique_ptr<std::atomic<int>[]> done; // threads through with a chunk
    std::atomic<size_t> ready{0};             // chunks that have landed
    std::atomic<bool> abandoned{false};
    bool started = false;
    unsigned char* stage = nullptr;
    std::mutex m;
    std::condition_variable cv;
};
