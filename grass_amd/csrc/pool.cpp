// Working memory kept between calls: device blocks (per GPU) and pinned host blocks that calls
// return when they are done, for later calls to take instead of hipMalloc / hipHostMalloc.
//
// A call that builds or loads a graph or samples an MDRW batch takes a dozen blocks of working
// memory, up to gigabytes, and hands all of them back before it returns.  hipMalloc and hipFree of
// such blocks cost 0.1 to 0.8 ms each (every hipFree waits for the whole device), 6 ms of the 25 ms
// in which an edge list of 67 M edges becomes a resident graph, and an allocation after much
// memory was used and freed on the card waits for it to be cleared: the same call then took 85 to
// 129 ms.  A pinned staging chunk of 64 MB costs milliseconds to pin.
//
// What a block holds is never read by its next owner.  A block enters the cache idle: its owner has
// waited for the stream it was used on (WorkMem does).  Bounded: at most kDeviceMax bytes idle per
// GPU (and a sixteenth of its memory) and kPinnedMax of host memory, the longest idle freed first;
// blocks idle for kKeepSeconds go at the next call that takes or returns one or waits for the device anyway
// (a program that builds its graph and then samples makes only the latter), and all of them when an
// allocation fails or the caller asks (grass_trim).  Closing a graph does not free them: the next one
// is built with them (R-MAT s22 from an edge list: 9 ms, 25 without).  Memory that callers own (graphs,
// results) does not come from here.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <mutex>
#include <new>

#include "runtime.h"

namespace grass {
namespace {

using Clock = std::chrono::steady_clock;

// A failed allocation reaches its caller by the return value alone: HIP keeps it as the thread's last
// error through later successful calls, where the launch checks of a caller that goes on without the
// memory (or got it at the second attempt) would find it.
hipError_t quiet(hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

constexpr size_t kDeviceMax = 16ull << 30;
constexpr size_t kPinnedMax = 256ull << 20;
constexpr int kKeepSeconds = 10;
constexpr int kMaxDevices = 64;

struct Block {
    void* p;
    size_t bytes;
    Clock::time_point since;
};

// Idle blocks in the order they came back (fixed arrays: nothing here throws).
class BlockCache {
   public:
    BlockCache(bool pinned, size_t limit) : pinned_(pinned), limit_(limit) {}

    hipError_t take(size_t need, void** p, size_t* got) {
        *p = nullptr;
        Dropped drop;
        {
            std::lock_guard<std::mutex> lock(mu_);
            int best = -1;
            // the smallest block that fits and is at most a quarter (and 1 MB) too large
            for (int i = 0; i < count_; ++i)
                if (idle_[i].bytes >= need && idle_[i].bytes <= need + need / 4 + (1u << 20) &&
                    (best < 0 || idle_[i].bytes < idle_[best].bytes))
                    best = i;
            if (best >= 0) {
                const Block b = remove(best);
                *p = b.p;
                *got = b.bytes;
            }
            expire(drop);
        }
        release(drop);
        if (*p) return hipSuccess;
        const size_t unit = need >= (8u << 20) ? (2u << 20) : 4096;
        *got = (need + unit - 1) / unit * unit;
        hipError_t e = quiet(allocate(p, *got));
        if (e != hipSuccess) {
            clear();
            e = quiet(allocate(p, *got));
        }
        return e;
    }

    void give(void* p, size_t bytes) {
        Dropped drop;
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (count_ == kMaxBlocks) drop.add(remove(0));
            idle_[count_++] = Block{p, bytes, Clock::now()};
            held_ += bytes;
            expire(drop);
            while (held_ > limit_ && count_) drop.add(remove(0));
        }
        release(drop);
    }

    void clear() {
        Dropped drop;
        {
            std::lock_guard<std::mutex> lock(mu_);
            while (count_) drop.add(remove(0));
        }
        release(drop);
    }

    // Frees what is idle for too long (a look at the clock where nothing is).
    void age() {
        if (!count_.load(std::memory_order_relaxed)) return;
        Dropped drop;
        {
            std::lock_guard<std::mutex> lock(mu_);
            expire(drop);
        }
        release(drop);
    }

   private:
    static constexpr int kMaxBlocks = 64;
    struct Dropped {
        Block b[kMaxBlocks + 1];
        int n = 0;
        void add(const Block& x) { b[n++] = x; }
    };
    Block remove(int i) {  // under mu_
        const Block b = idle_[i];
        held_ -= b.bytes;
        for (--count_; i < count_; ++i) idle_[i] = idle_[i + 1];
        return b;
    }
    void expire(Dropped& drop) {  // under mu_
        const Clock::time_point old = Clock::now() - std::chrono::seconds(kKeepSeconds);
        while (count_ && idle_[0].since < old) drop.add(remove(0));
    }
    hipError_t allocate(void** p, size_t bytes) {
        return pinned_ ? hipHostMalloc(p, bytes, hipHostMallocDefault) : hipMalloc(p, bytes);
    }
    void release(const Dropped& drop) {
        if (!drop.n) return;
        // (another thread may be capturing a graph, which these calls are no part of)
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        for (int i = 0; i < drop.n; ++i) {
            if (pinned_) (void)hipHostFree(drop.b[i].p);
            else (void)hipFree(drop.b[i].p);
        }
        (void)hipThreadExchangeStreamCaptureMode(&mode);
    }

    const bool pinned_;
    const size_t limit_;
    std::mutex mu_;
    Block idle_[kMaxBlocks];
    std::atomic<int> count_{0};
    size_t held_ = 0;
};

// Never destroyed: the HIP runtime may be gone when static objects are.
BlockCache* device_cache(int dev) {
    static std::mutex mu;
    static BlockCache* caches[kMaxDevices] = {};
    if (dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (!caches[dev]) {
        size_t fr = 0, total = 0;
        if (hipMemGetInfo(&fr, &total) != hipSuccess) total = 0;
        caches[dev] = new (std::nothrow) BlockCache(false, std::min<size_t>(kDeviceMax, total / 16));
    }
    return caches[dev];
}

BlockCache* pinned_cache() {
    static BlockCache* c = new (std::nothrow) BlockCache(true, kPinnedMax);
    return c;
}

}  // namespace

hipError_t WorkMem::alloc(size_t need, hipStream_t stream) {
    reset();
    s = stream;
    need = std::max<size_t>(need, 256);
    if (hipGetDevice(&dev) != hipSuccess) return hipErrorNoDevice;
    BlockCache* c = device_cache(dev);
    return c ? c->take(need, &p, &bytes) : hipErrorOutOfMemory;
}

void WorkMem::reset() {
    if (!p) return;
    // idle from here on, or (a stream that failed) not to be used again
    const hipError_t e = whole_device ? hipDeviceSynchronize() : hipStreamSynchronize(s);
    if (e == hipSuccess) device_cache(dev)->give(p, bytes);
    else (void)hipFree(p);
    p = nullptr;
}

hipError_t PinnedWork::alloc(size_t need) {
    reset();
    BlockCache* c = pinned_cache();
    return c ? c->take(std::max<size_t>(need, 256), &p, &bytes) : hipErrorOutOfMemory;
}

void PinnedWork::reset() {
    if (p) pinned_cache()->give(p, bytes);
    p = nullptr;
}

void release_aged(int dev) {
    if (BlockCache* c = device_cache(dev)) c->age();
    if (BlockCache* c = pinned_cache()) c->age();
}

void release_idle(int dev) {
    if (BlockCache* c = device_cache(dev)) c->clear();
    if (BlockCache* c = pinned_cache()) c->clear();
}

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = quiet(hipMalloc(p, bytes));
    if (e == hipSuccess) return e;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return e;
    if (BlockCache* c = device_cache(dev)) c->clear();
    return quiet(hipMalloc(p, bytes));
}

hipError_t pinned_malloc(void** p, size_t bytes) {
    hipError_t e = quiet(hipHostMalloc(p, bytes, hipHostMallocDefault));
    if (e == hipSuccess) return e;
    if (BlockCache* c = pinned_cache()) c->clear();
    return quiet(hipHostMalloc(p, bytes, hipHostMallocDefault));
}

}  // namespace grass
