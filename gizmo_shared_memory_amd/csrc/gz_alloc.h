// Errors, and the device memory that the library keeps between calls: host code only.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <mutex>

#include "gz_grav.h"

namespace gz {

// ---- errors ---------------------------------------------------------------------------------
void set_error(const char* fmt, ...);
gz_status fail(gz_status s, const char* fmt, ...);
gz_status hip_fail(hipError_t e, const char* what, const char* file, int line);
const char* last_error_cstr();
void clear_error();

#define GZ_HIP(call)                                                          \
    do {                                                                      \
        hipError_t gz_e_ = (call);                                            \
        if (gz_e_ != hipSuccess) return ::gz::hip_fail(gz_e_, #call, __FILE__, __LINE__); \
    } while (0)

#define GZ_TRY(expr)                       \
    do {                                   \
        gz_status gz_s_ = (expr);          \
        if (gz_s_ != GZ_OK) return gz_s_;  \
    } while (0)

// ---- device memory --------------------------------------------------------------------------
class BlockCache;

// Device memory for a context whose freed trees left their blocks in cache: on out of memory those,
// and scratch lent to it, are given back and the allocation is tried again.
gz_status device_alloc(BlockCache* cache, void** p, size_t bytes);

// Grow-only device allocation.
struct DevMem {
    void* p = nullptr;
    size_t bytes = 0;
    BlockCache* cache = nullptr; // the context's
    bool in_use = false;         // a call has its contents there (ScratchUse)
    gz_status reserve(size_t want);
    // The same for memory that a call can do without: false when there is not enough (what was
    // here is gone then).
    bool offer(size_t want);
    void release();
    template <class T> T* as() const { return static_cast<T*>(p); }
};

struct ScratchUse {
    DevMem& m;
    explicit ScratchUse(DevMem& mem) : m(mem) { m.in_use = true; }
    ~ScratchUse() { m.in_use = false; }
    ScratchUse(const ScratchUse&) = delete;
};

struct DevBlock {
    void* p;
    size_t bytes;
};

// Device blocks that freed trees leave for the next build on their context: a tree is some 25
// arrays, and at 4M particles freeing and allocating them took 4.6 of a rebuild's 5.3 ms. Blocks
// come in sizes an eighth of a power of two apart, so that a tree that grows a little from one
// rebuild to the next finds its blocks again (exact sizes left each tree's blocks useless to the
// next: a rebuild of a 4M tree that grows by 0.1% a time took 6.6 to 27 ms once the cache was full
// of them, now 2.6). It holds at most kBytes and kBlocks, since nothing outside the library can ask
// for them back (a rebuild of 16.8M particles, whose blocks are more, loses .1 of 5.1 ms to the
// bound, of 33.6M 1.7 of 11.4); beyond that the blocks put longest ago go back to the device, and
// everything does when its context is destroyed or an allocation of the context finds no memory.
// Trees may be freed by another thread than the one that builds (the list is locked), and after
// their context (they share the cache's ownership; it then keeps nothing).
class BlockCache {
public:
    static constexpr size_t kBytes = size_t(2) << 30;
    static constexpr int kBlocks = 64;
    // A block of at least `bytes`: a kept one if it is not much larger.
    gz_status get(size_t bytes, DevBlock* out);
    // A block that nothing on the device uses any more.
    void put(DevBlock b);
    // Blocks that work on any stream may still use: kept once the device is done. When it cannot
    // be waited for (some stream of the process is being captured) they go back to the device
    // instead, whose own free waits, or refuses.
    void retire(const DevBlock* b, int n);
    // Scratch of the context that drain gives back too when no call has its contents there: what is
    // large, kept for speed alone, and no captured graph reads.
    void lend(DevMem* m);
    void drain();
    void close(); // drain, and keep nothing from now on

private:
    void evict(int n); // the n put longest ago (the list is locked)
    std::mutex mu_;
    DevBlock kept_[kBlocks]; // in the order they were put
    int n_ = 0;
    size_t held_ = 0;
    bool open_ = true;
    DevMem* lent_[4];
    int n_lent_ = 0;
};

} // namespace gz
