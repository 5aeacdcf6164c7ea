// KeptScratch over a model of the HIP allocator: a freed address is given out
// again, every allocation has an identifier of its own, and a reset takes all of
// them away.  Ends with 0 when every check holds.
#include "../tatara_amd/csrc/kept_scratch.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <thread>
#include <vector>

namespace {
struct Block {
    uint64_t id;
    size_t bytes;
};
std::map<void*, Block> live;
uint64_t next_id = 1, mallocs = 0, bad_frees = 0;
int device = 0;
bool fail_malloc = false;
char space[64];

void reset() { live.clear(); }
}  // namespace

hipError_t hipMalloc(void** p, size_t bytes) {
    if (fail_malloc) return hipErrorOutOfMemory;
    for (char& c : space)  // the lowest address that is not in use
        if (!live.count(&c)) {
            live[&c] = {next_id++, bytes};
            ++mallocs;
            *p = &c;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    if (!live.erase(p)) ++bad_frees;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttribute(void* data, hipPointer_attribute what, hipDeviceptr_t p) {
    if (what != HIP_POINTER_ATTRIBUTE_BUFFER_ID || !live.count(p)) return hipErrorInvalidValue;
    *static_cast<uint64_t*>(data) = live[p].id;
    return hipSuccess;
}

#define CHECK(x)                                             \
    do {                                                     \
        if (!(x)) {                                          \
            std::printf("line %d: %s\n", __LINE__, #x);      \
            return 1;                                        \
        }                                                    \
    } while (0)

int main() {
    using tatara::KeptScratch;
    {
        KeptScratch k;
        void *p = nullptr, *q = nullptr;
        // kept between calls, grown when a call needs more, not lent twice
        CHECK(k.lend(1000, &p) == hipSuccess && p);
        CHECK(k.lend(10, &q) == hipSuccess && !q);
        k.give_back();
        CHECK(k.lend(500, &q) == hipSuccess && q == p && mallocs == 1);
        k.give_back();
        CHECK(k.lend(2000, &q) == hipSuccess && live[q].bytes == 2000 && live.size() == 1);
        k.release();  // lent: stays
        CHECK(live.size() == 1);
        k.give_back();
        CHECK(k.lend(KeptScratch::kMaxBytes + 1, &q) == hipSuccess && !q);
        CHECK(k.lend(KeptScratch::kMaxBytes, &q) == hipSuccess && q);
        k.give_back();
        // a reset: the next call allocates, and frees nothing that is gone
        reset();
        CHECK(k.lend(100, &q) == hipSuccess && live.count(q) && bad_frees == 0);
        k.give_back();
        // a reset, and the program owns the address now
        reset();
        void* theirs = nullptr;
        CHECK(hipMalloc(&theirs, 100) == hipSuccess && theirs == q);
        const uint64_t id = live[theirs].id;
        CHECK(k.lend(100, &p) == hipSuccess && p != theirs);
        k.give_back();
        k.release();
        CHECK(live.size() == 1 && live.count(theirs) && live[theirs].id == id && bad_frees == 0);
        // another device
        CHECK(k.lend(100, &p) == hipSuccess);
        k.give_back();
        const uint64_t before = mallocs;
        device = 1;
        CHECK(k.lend(100, &p) == hipSuccess && mallocs == before + 1 && live.size() == 2);
        k.give_back();
        // out of memory: reported, nothing kept, and the next call tries again
        fail_malloc = true;
        CHECK(k.lend(5000, &p) == hipErrorOutOfMemory && !p && live.size() == 1);
        fail_malloc = false;
        CHECK(k.lend(5000, &p) == hipSuccess && p);
        k.give_back();
    }
    CHECK(live.size() == 1 && bad_frees == 0);  // what is left is the program's
    // a thread's memory ends with the thread, also after a reset
    std::thread([] {
        thread_local KeptScratch k;
        void* p = nullptr;
        (void)k.lend(64, &p);
        k.give_back();
    }).join();
    CHECK(live.size() == 1 && bad_frees == 0);
    std::thread([] {
        thread_local KeptScratch k;
        void* p = nullptr;
        (void)k.lend(64, &p);
        k.give_back();
        reset();
        (void)hipMalloc(&p, 8);  // the addresses are the program's
        (void)hipMalloc(&p, 8);
    }).join();
    CHECK(live.size() == 2 && bad_frees == 0);
    return 0;
}
