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

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> checks = {{"refused_wait", refused_wait}};
    CHECK(argc == 2 && checks.count(argv[1]));
    checks.at(argv[1])();
    std::printf("ok\n");
    return 0;
}
