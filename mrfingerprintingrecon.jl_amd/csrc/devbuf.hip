// Idle device blocks, kept for the next buffer of about their size.  hipMalloc
// and hipFree map and unmap pages: a kernel construction (about 20 temporaries,
// 0.6 GB at 256 x 256, K = 5) spent as long in them as in its kernels, and
// with other allocations on the device up to 10 times that (measured 7 to
// 24 ms per construction for 5 ms of kernels in 2D, 28 to 520 ms for 22 ms in
// 3D).  A block is kept only after the device has finished everything queued
// before its release, as hipFree would have waited, so any stream or thread
// may take it; at most IDLE_LIMIT bytes stay idle per device, oldest freed
// first, and all of them when an allocation fails or a context is destroyed.
#include <cstdlib>
#include <mutex>
#include <vector>

#include "internal.hpp"

namespace msr {

constexpr size_t IDLE_LIMIT = (size_t)8 << 30;
constexpr size_t IDLE_BLOCKS = 512;

namespace {
struct Block {
    void* p;
    size_t cap;
    int device;
};
struct Idle {
    std::mutex mu;
    std::vector<Block> blocks;  // oldest first
};
// never destroyed: buffers may be released while the process ends
Idle& idle() {
    static Idle* c = new Idle;
    return *c;
}

// makes `device` current for its lifetime
struct OnDevice {
    int before = -1;
    bool ok;
    explicit OnDevice(int device) {
        ok = hipGetDevice(&before) == hipSuccess;
        if (ok && before != device) ok = hipSetDevice(device) == hipSuccess;
        else before = -1;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
};

// MSR_DEVICE_ALLOC_LIMIT=<bytes> in the environment: larger requests fail, as on
// a device without that much free memory (a check of the paths taken then)
bool over_limit(size_t n) {
    const char* e = getenv("MSR_DEVICE_ALLOC_LIMIT");
    return e && n > (size_t)strtoull(e, nullptr, 10);
}
}  // namespace

void* dev_acquire(size_t n, size_t& cap, int& device) {
    MSR_HIP(hipGetDevice(&device));
    cap = (n + 511) / 512 * 512;
    if (over_limit(cap)) {
        cap = SIZE_MAX / 4;  // more than any device has: fails below
    } else {
        Idle& c = idle();
        std::lock_guard<std::mutex> guard(c.mu);
        size_t best = c.blocks.size();
        for (size_t i = 0; i < c.blocks.size(); ++i) {
            const Block& b = c.blocks[i];
            if (b.device == device && b.cap >= cap && b.cap <= cap + cap / 4 + 65536 &&
                (best == c.blocks.size() || b.cap < c.blocks[best].cap))
                best = i;
        }
        if (best < c.blocks.size()) {
            void* p = c.blocks[best].p;
            cap = c.blocks[best].cap;
            c.blocks.erase(c.blocks.begin() + best);
            return p;
        }
    }
    void* p = nullptr;
    if (hipMalloc(&p, cap) != hipSuccess) {
        (void)hipGetLastError();
        dev_trim(device);
        MSR_HIP(hipMalloc(&p, cap));
    }
    return p;
}

void dev_release(void* p, size_t cap, int device) noexcept {
    OnDevice on(device);
    // not idle (or not known to be): hipFree waits by itself
    if (!on.ok || cap > IDLE_LIMIT || hipDeviceSynchronize() != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return;
    }
    std::vector<Block> out;
    try {
        Idle& c = idle();
        std::lock_guard<std::mutex> guard(c.mu);
        c.blocks.push_back({p, cap, device});
        p = nullptr;
        size_t bytes = 0, count = 0;
        for (const Block& b : c.blocks)
            if (b.device == device) {
                bytes += b.cap;
                ++count;
            }
        for (size_t i = 0; i < c.blocks.size() && (bytes > IDLE_LIMIT || count > IDLE_BLOCKS);) {
            if (c.blocks[i].device != device) {
                ++i;
                continue;
            }
            bytes -= c.blocks[i].cap;
            --count;
            out.push_back(c.blocks[i]);
            c.blocks.erase(c.blocks.begin() + i);
        }
    } catch (...) {
        if (p) (void)hipFree(p);
    }
    for (const Block& b : out) (void)hipFree(b.p);
}

void dev_trim(int device) noexcept {
    OnDevice on(device);
    Idle& c = idle();
    std::lock_guard<std::mutex> guard(c.mu);
    for (size_t i = 0; i < c.blocks.size();) {
        if (c.blocks[i].device != device) {
            ++i;
            continue;
        }
        (void)hipFree(c.blocks[i].p);
        c.blocks.erase(c.blocks.begin() + i);
    }
}

}  // namespace msr
