// The device memory that the library keeps between calls (csrc/gz_alloc.cpp), on the CPU: the few
// HIP calls it makes are defined here, over a device of a given size whose waits can be refused.
// Run by tests/test_alloc.py with the name of one check.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "gz_alloc.h"

namespace {
struct Device {
    size_t room = size_t(64) << 30;
    bool refuse = false; // waits and frees, as while a stream is being captured
    hipError_t last = hipSuccess;
    std::map<void*, size_t> live;
    long mallocs = 0, frees = 0, waits = 0;
    uintptr_t next = uintptr_t(1) << 40;
    size_t used() const {
        size_t s = 0;
        for (auto& b : live) s += b.second;
        return s;
    }
} dev;

hipError_t note(hipError_t e) {
    if (e != hipSuccess) dev.last = e;
    return e;
}

#define CHECK(x)                                                              \
    do {                                                                      \
        if (!(x)) {                                                           \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);               \
            std::exit(1);                                                     \
        }                                                                     \
    } while (0)
} // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    ++dev.mallocs;
    if (dev.used() + bytes > dev.room) return note(hipErrorOutOfMemory);
    *p = reinterpret_cast<void*>(dev.next);
    dev.next += (bytes + 4095) & ~size_t(4095);
    dev.live[*p] = bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (dev.refuse) return note(hipErrorStreamCaptureUnsupported);
    CHECK(!p || dev.live.erase(p) == 1);
    ++dev.frees;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    ++dev.waits;
    return note(dev.refuse ? hipErrorStreamCaptureUnsupported : hipSuccess);
}
hipError_t hipGetLastError() {
    const hipError_t e = dev.last;
    dev.last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
}

using gz::BlockCache;
using gz::DevBlock;

// Blocks whose device could not be waited for never serve another allocation.
static void refused_wait() {
    BlockCache c;
    DevBlock b[3];
    for (auto& x : b) CHECK(c.get(100000, &x) == GZ_OK);
    dev.refuse = true;
    c.retire(b, 3);
    CHECK(hipGetLastError() == hipSuccess);
    dev.refuse = false;
    for (int i = 0; i < 3; ++i) {
        DevBlock n;
        CHECK(c.get(100000, &n) == GZ_OK);
        for (auto& x : b) CHECK(n.p != x.p);
        b[i] = n;
    }
    const long before = dev.waits;
    c.retire(b, 3);
    CHECK(dev.waits == before + 1);
    DevBlock n;
    CHECK(c.get(100000, &n) == GZ_OK);
    CHECK(n.p == b[0].p || n.p == b[1].p || n.p == b[2].p);
    c.retire(&n, 1);
    c.close();
    CHECK(dev.live.size() == 3); // those refused, which the device kept
}

// The blocks of a tree of n particles, as a build takes them.
static std::vector<DevBlock> tree(BlockCache& c, size_t n, double cells = 0.375) {
    const size_t nodes = (size_t)(cells * n) + 1024;
    const size_t sizes[] = {4 * n, 4 * n, 4 * n, 8 * n, 4 * n, 32 * n, 8 * n, 64 * nodes, 4 * nodes,
                            4 * nodes, 4 * nodes, 4 * nodes, 8 * nodes, 8 * nodes, 8 * nodes,
                            8 * nodes, 8 * nodes, 8 * nodes, 96, 6 * nodes, 8};
    std::vector<DevBlock> t;
    for (size_t s : sizes) {
        DevBlock b;
        CHECK(c.get(s, &b) == GZ_OK && b.bytes >= s);
        CHECK(4 * b.bytes <= 5 * (s + s / 8 + 4096)); // a kept one may be a quarter larger
        for (auto& o : t) CHECK(o.p != b.p);
        t.push_back(b);
    }
    return t;
}

static size_t held(const std::vector<DevBlock>& t) {
    size_t s = 0;
    for (auto& b : t) s += b.bytes;
    return s;
}

// A tree that grows a little from rebuild to rebuild keeps finding its blocks, and so does one that
// follows trees of quite other sizes.
static void growing_trees() {
    for (double n0 : {5e4, 1e6, 4e6}) {
        BlockCache c;
        long first = 0;
        for (int i = 0; i < 400; ++i) {
            const std::vector<DevBlock> t = tree(c, (size_t)(n0 * (1.0 + 1e-3 * i)));
            c.retire(t.data(), (int)t.size());
            CHECK(dev.used() <= BlockCache::kBytes && dev.live.size() <= BlockCache::kBlocks);
            if (i == 0) first = dev.mallocs;
        }
        // 1.4 times as large: some four steps of the sizes for each array
        CHECK(dev.mallocs - first <= 6 * first);
        for (double f : {2.0, 3.1, 0.4, 0.3, 5.0}) {
            const std::vector<DevBlock> t = tree(c, (size_t)(f * n0));
            c.retire(t.data(), (int)t.size());
        }
        std::vector<DevBlock> t = tree(c, (size_t)n0);
        c.retire(t.data(), (int)t.size());
        const long before = dev.mallocs;
        t = tree(c, (size_t)(1.0001 * n0));
        CHECK(dev.mallocs - before <= 2);
        c.retire(t.data(), (int)t.size());
        c.close();
        CHECK(dev.live.empty());
        dev.mallocs = 0;
    }
}

// A tree larger than what is kept: most of its blocks are.
static void large_tree() {
    BlockCache c;
    std::vector<DevBlock> t = tree(c, 20000000);
    CHECK(held(t) > BlockCache::kBytes);
    for (int i = 0; i < 5; ++i) {
        const long before = dev.mallocs;
        if (i) t = tree(c, 20000000);
        CHECK(i == 0 || dev.mallocs - before <= (long)t.size() / 2);
        c.retire(t.data(), (int)t.size());
        CHECK(dev.used() <= BlockCache::kBytes);
    }
    DevBlock b;
    CHECK(c.get(BlockCache::kBytes + 1, &b) == GZ_OK);
    const size_t kept = dev.live.size() - 1;
    c.retire(&b, 1); // larger than all that may be kept: straight back, the others stay
    CHECK(dev.live.size() == kept);
    c.close();
    CHECK(dev.live.empty());
}

// Kept blocks make way for every other allocation of their context, which fails only when the device
// is full without them, and leaves no error behind for the next call's check.
static void room_for_others() {
    BlockCache c;
    std::vector<DevBlock> t = tree(c, 4000000);
    c.retire(t.data(), (int)t.size());
    const size_t kept = dev.used();
    CHECK(kept > size_t(300) << 20);
    dev.room = kept + (size_t(64) << 20);
    gz::DevMem m;
    m.cache = &c;
    CHECK(m.reserve(size_t(32) << 20) == GZ_OK && dev.used() == kept + m.bytes);
    CHECK(m.reserve(kept) == GZ_OK && m.bytes == kept && dev.used() == kept);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(m.reserve(dev.room + 1) == GZ_ERR_NOMEM && m.p == nullptr && m.bytes == 0);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(m.reserve(kept) == GZ_OK);
    m.release();
    t = tree(c, 4000000);
    c.retire(t.data(), (int)t.size());
    void* p = nullptr;
    CHECK(gz::device_alloc(&c, &p, kept) == GZ_OK && dev.used() == kept);
    CHECK(gz::device_alloc(nullptr, &p, dev.room) == GZ_ERR_NOMEM && p == nullptr);
    c.close();
}

// So does scratch that no call is using; a call can do without what it only offers to take.
static void lent_scratch() {
    BlockCache c;
    gz::DevMem a, b;
    a.cache = b.cache = &c;
    c.lend(&a);
    c.lend(&b);
    dev.room = size_t(300) << 20;
    CHECK(a.reserve(size_t(200) << 20) == GZ_OK);
    {
        gz::ScratchUse use(a);
        CHECK(!b.offer(size_t(150) << 20) && b.p == nullptr && a.p != nullptr);
        CHECK(*gz::last_error_cstr() == 0);
        CHECK(b.offer(size_t(50) << 20));
        CHECK(b.offer(size_t(50) << 20) && b.bytes == size_t(50) << 20);
    }
    DevBlock t;
    CHECK(c.get(size_t(250) << 20, &t) == GZ_OK && !a.p && !b.p && dev.waits > 0);
    dev.refuse = true; // nothing is given back that may still be read
    c.put(t);
    CHECK(a.reserve(size_t(1) << 20) == GZ_OK);
    CHECK(b.reserve(size_t(300) << 20) == GZ_ERR_NOMEM && a.p);
    dev.refuse = false;
    c.close();
    DevBlock u;
    CHECK(c.get(size_t(290) << 20, &u) == GZ_ERR_NOMEM && a.p); // the context frees its scratch
    a.release();
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> checks = {{"refused_wait", refused_wait},
                                                         {"growing_trees", growing_trees},
                                                         {"large_tree", large_tree},
                                                         {"room_for_others", room_for_others},
                                                         {"lent_scratch", lent_scratch}};
    CHECK(argc == 2 && checks.count(argv[1]));
    checks.at(argv[1])();
    std::printf("ok\n");
    return 0;
}
