// The library's error text and the device memory that it keeps between calls (gz_alloc.h).
#include "gz_alloc.h"

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <string>

namespace gz {

// ---- errors ----------------------------------------------------------------------------------
static thread_local std::string g_last_error;

void set_error(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

gz_status fail(gz_status s, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return s;
}

gz_status hip_fail(hipError_t e, const char* what, const char* file, int line) {
    set_error("%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
    return (e == hipErrorOutOfMemory) ? GZ_ERR_NOMEM : GZ_ERR_HIP;
}

const char* last_error_cstr() { return g_last_error.c_str(); }
void clear_error() { g_last_error.clear(); }

// ---- device memory ---------------------------------------------------------------------------
gz_status device_alloc(BlockCache* cache, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && cache) {
        (void)hipGetLastError();
        cache->drain();
        e = hipMalloc(p, bytes);
    }
    if (e == hipSuccess) return GZ_OK;
    (void)hipGetLastError(); // (reported here; the next launch's check is not to find it)
    *p = nullptr;
    return hip_fail(e, "hipMalloc", __FILE__, __LINE__);
}

gz_status DevMem::reserve(size_t want) {
    if (want <= bytes && p) return GZ_OK;
    if (p) {
        // work already queued may still read the old buffer
        GZ_HIP(hipDeviceSynchronize());
        GZ_HIP(hipFree(p));
        p = nullptr;
        bytes = 0;
    }
    const size_t b = std::max<size_t>(want, 256);
    GZ_TRY(device_alloc(cache, &p, b));
    bytes = b;
    return GZ_OK;
}

bool DevMem::offer(size_t want) {
    if (reserve(want) == GZ_OK) return true;
    clear_error();
    return false;
}

void DevMem::release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
}

// The block size that serves `bytes`: up to an eighth more, in whole pages.
static size_t block_size(size_t bytes) {
    size_t step = 4096;
    while (bytes > 16 * step) step *= 2;
    return (std::max<size_t>(bytes, 1) + step - 1) / step * step;
}

gz_status BlockCache::get(size_t bytes, DevBlock* out) {
    const size_t want = block_size(bytes);
    {
        std::lock_guard<std::mutex> lock(mu_);
        int best = -1;
        for (int i = 0; i < n_; ++i)
            if (kept_[i].bytes >= want && kept_[i].bytes - want <= want / 4 &&
                (best < 0 || kept_[i].bytes < kept_[best].bytes))
                best = i;
        if (best >= 0) {
            *out = kept_[best];
            held_ -= out->bytes;
            std::copy(kept_ + best + 1, kept_ + n_, kept_ + best);
            --n_;
            return GZ_OK;
        }
    }
    GZ_TRY(device_alloc(this, &out->p, want));
    out->bytes = want;
    return GZ_OK;
}

void BlockCache::put(DevBlock b) {
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (open_ && b.bytes <= kBytes) {
            int old = (n_ == kBlocks) ? 1 : 0;
            size_t held = held_;
            for (int i = 0; i < old; ++i) held -= kept_[i].bytes;
            while (held + b.bytes > kBytes) held -= kept_[old++].bytes;
            evict(old);
            kept_[n_++] = b;
            held_ += b.bytes;
            return;
        }
    }
    (void)hipFree(b.p);
}

void BlockCache::retire(const DevBlock* b, int n) {
    if (n <= 0) return;
    const bool idle = hipDeviceSynchronize() == hipSuccess;
    for (int i = 0; i < n; ++i) {
        if (idle) put(b[i]);
        else (void)hipFree(b[i].p);
    }
    if (!idle) (void)hipGetLastError(); // (the next launch's check is not to find it)
}

void BlockCache::evict(int n) {
    for (int i = 0; i < n; ++i) {
        (void)hipFree(kept_[i].p);
        held_ -= kept_[i].bytes;
    }
    std::copy(kept_ + n, kept_ + n_, kept_);
    n_ -= n;
}

void BlockCache::lend(DevMem* m) {
    if (n_lent_ < (int)(sizeof lent_ / sizeof *lent_)) lent_[n_lent_++] = m;
}

void BlockCache::drain() {
    std::lock_guard<std::mutex> lock(mu_);
    evict(n_);
    for (int i = 0; i < n_lent_; ++i) {
        DevMem& m = *lent_[i];
        // (queued work may still read it)
        if (m.p && !m.in_use && hipDeviceSynchronize() == hipSuccess) m.release();
    }
}

void BlockCache::close() {
    {
        std::lock_guard<std::mutex> lock(mu_);
        open_ = false;
        n_lent_ = 0; // (the context frees its scratch)
    }
    drain();
}

} // namespace gz
