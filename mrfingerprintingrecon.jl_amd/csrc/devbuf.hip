// Idle device blocks, kept for the next buffer of about their size.  hipMalloc
// and hipFree map and unmap pages: a kernel construction (about 20 temporaries,
// 0.6 GB at 256 x 256, K = 5) spent as long in them as in its kernels, and
// with other allocations on the device up to 10 times that (measured 7 to
// 24 ms per construction for 5 ms of kernels in 2D, 28 to 520 ms for 22 ms in
// 3D).  A block is kept only after the device has finished everything queued
// before its release, as hipFree would have waited, so any stream or thread
// may take it; at most IDLE_LIMIT bytes stay idle per device, oldest freed
// first, and no large block while the device is nearly full.  All are given back when an allocation of this library fails, when a context is
// destroyed, and by msr_trim (another allocator in the process cannot ask).
#include <cstdlib>
#include <mutex>
#include <vector>

#include "internal.hpp"

namespace msr {

constexpr size_t IDLE_LIMIT = (size_t)8 << 30;
constexpr size_t IDLE_BLOCKS = 512;
// A buffer of `need` bytes takes a block of up to this many: the byte counts of
// operator footprints, the server's admission and the kernel cache's budget are
// those requested.  (Constructions of one protocol ask for the same sizes again;
// blocks up to a quarter larger gained nothing measurable.)
constexpr size_t block_for(size_t need) { return need + need / 64 + 65536; }
constexpr size_t LARGE_BLOCK = (size_t)512 << 20;

// Whether a block may stay idle: a large one (the grids of a 3D construction)
// only while an eighth of the device's memory is free besides.  Asking takes
// about 7 us, too long for the blocks of shorter calls (from 64 MiB on, a 256 x 256
// construction took 1.25 ms for 1.23; for every block, a calibration 5.5 for 4.3).
static bool may_stay(size_t cap) {
    if (cap > IDLE_LIMIT) return false;
    if (cap < LARGE_BLOCK) return true;
    size_t avail = 0, total = 0;
    return hipMemGetInfo(&avail, &total) == hipSuccess && avail >= total / 8;
}

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
            if (b.device == device && b.cap >= cap && b.cap <= block_for(cap) &&
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
    if (!on.ok || !may_stay(cap) || hipDeviceSynchronize() != hipSuccess) {
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

size_t dev_trim(int device) noexcept {
    OnDevice on(device);
    size_t bytes = 0;
    Idle& c = idle();
    std::lock_guard<std::mutex> guard(c.mu);
    for (size_t i = 0; i < c.blocks.size();) {
        if (c.blocks[i].device != device) {
            ++i;
            continue;
        }
        (void)hipFree(c.blocks[i].p);
        bytes += c.blocks[i].cap;
        c.blocks.erase(c.blocks.begin() + i);
    }
    return bytes;
}

}  // namespace msr
