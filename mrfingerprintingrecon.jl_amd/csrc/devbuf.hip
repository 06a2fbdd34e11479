// Idle device blocks, kept for the next buffer of about their size.  hipMalloc
// and hipFree map and unmap pages: a kernel construction (about 20 temporaries,
// 0.6 GB at 256 x 256, K = 5) spent as long in them as in its kernels, and
// with other allocations on the device up to 10 times that (measured 7 to
// 24 ms per construction for 5 ms of kernels in 2D, 28 to 520 ms for 22 ms in
// 3D).  A released block is handed out again once nothing queued before its
// release can use it: a temporary's at once (its function has waited for its
// stream), a destroyed handle's too (destroying waits for the device), any other
// after such a wait.  At most IDLE_LIMIT bytes are kept per device, oldest freed
// first, and no large block while the device is nearly full.  All are given back
// when an allocation of this library fails, when a context is destroyed, and by
// msr_trim (another allocator in the process cannot ask).
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
    bool done;  // nothing queued uses it
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

// Index of the smallest kept block for a buffer of `need` bytes, or -1.
static int best_block(const std::vector<Block>& blocks, int device, size_t need, bool done) {
    int best = -1;
    for (size_t i = 0; i < blocks.size(); ++i) {
        const Block& b = blocks[i];
        if (b.device == device && b.done == done && b.cap >= need && b.cap <= block_for(need) &&
            (best < 0 || b.cap < blocks[best].cap))
            best = (int)i;
    }
    return best;
}

static Block take(std::vector<Block>& blocks, int i) {
    const Block b = blocks[i];
    blocks.erase(blocks.begin() + i);
    return b;
}

bool dev_wait() noexcept {
    void* p = nullptr;
    if (hipMalloc(&p, 512) == hipSuccess && hipFree(p) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

static thread_local bool all_done = false;
DoneScope::DoneScope(bool done) noexcept : before(all_done) { all_done = all_done || done; }
DoneScope::~DoneScope() { all_done = before; }

// Waits until the blocks of the current device that may still be in use are
// idle.  They are out of other threads' reach meanwhile.
static void settle(Idle& c, int device) {
    std::vector<Block> busy;
    {
        std::lock_guard<std::mutex> guard(c.mu);
        for (size_t i = 0; i < c.blocks.size();)
            if (c.blocks[i].device == device && !c.blocks[i].done) busy.push_back(take(c.blocks, (int)i));
            else ++i;
    }
    const bool waited = dev_wait();
    std::lock_guard<std::mutex> guard(c.mu);
    for (Block& b : busy) {
        b.done = waited;
        c.blocks.push_back(b);
    }
}

void* dev_acquire(size_t n, size_t& cap, int& device) {
    MSR_HIP(hipGetDevice(&device));
    cap = (n + 511) / 512 * 512;
    if (over_limit(cap)) {
        cap = SIZE_MAX / 4;  // more than any device has: fails below
    } else {
        Idle& c = idle();
        std::unique_lock<std::mutex> guard(c.mu);
        int i = best_block(c.blocks, device, cap, true);
        if (i < 0 && best_block(c.blocks, device, cap, false) >= 0) {
            guard.unlock();
            settle(c, device);
            guard.lock();
            i = best_block(c.blocks, device, cap, true);
        }
        if (i >= 0) {
            const Block b = take(c.blocks, i);
            cap = b.cap;
            return b.p;
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

void dev_release(void* p, size_t cap, int device, bool done) noexcept {
    OnDevice on(device);
    if (!on.ok || !may_stay(cap)) {  // hipFree waits by itself
        (void)hipGetLastError();
        (void)hipFree(p);
        return;
    }
    std::vector<Block> out;
    try {
        Idle& c = idle();
        std::lock_guard<std::mutex> guard(c.mu);
        c.blocks.push_back({p, cap, device, done || all_done});
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
