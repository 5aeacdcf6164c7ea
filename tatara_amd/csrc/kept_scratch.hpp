// The scratch memory a thread keeps between the standalone ops.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace tatara {

// At most kMaxBytes on one device, freed when the thread ends, asks for it on
// another device or releases it.  An op has synchronised before it returns, so the
// memory is idle between calls.  Allocating and freeing an op's buffers on each
// call cost the f32 gradient op at ft_out 768, batch 16381 110 us of 358 (now
// 239), the f16 one at 1536, 16384 118 us of 440 (now 321).
//
// What 64 MB hold (an op that needs more allocates for the call): the occurrence
// lists (16 bytes an index slot and perspective) of 52,000 positions at 40 slots and
// 32,000 at 64; the block scan's schedule and tables (434 bytes a position at
// 1629 pieces) of 150,000, with the copy of a dft that is not read in place (f32,
// 260 columns) of 14,000; the forward's schedule of more than a million; the tile
// offsets of every table below 2^34 cells.
//
// A hipDeviceReset between two calls takes the memory away, and the program may
// then own the same address: the pointer is used and freed only while the
// runtime's identifier of its allocation, which is never given twice, is the one
// it had.
class KeptScratch {
   public:
    static constexpr size_t kMaxBytes = 64ull << 20;

    KeptScratch() = default;
    KeptScratch(const KeptScratch&) = delete;
    KeptScratch& operator=(const KeptScratch&) = delete;
    ~KeptScratch() { release(); }

    // Memory of `bytes` on the current device until give_back(); null when it is
    // lent already or `bytes` is too much to keep.
    hipError_t lend(size_t bytes, void** out) {
        *out = nullptr;
        if (lent_ || bytes > kMaxBytes) return hipSuccess;
        int device = 0;
        hipError_t e = hipGetDevice(&device);
        if (e != hipSuccess) return e;
        if (device != device_ || bytes > bytes_ || !alive()) {
            release();
            void* p = nullptr;
            if ((e = hipMalloc(&p, bytes ? bytes : 4)) != hipSuccess) return e;
            if ((e = identify(p, &id_)) != hipSuccess) {
                (void)hipFree(p);
                return e;
            }
            p_ = p;
            bytes_ = bytes;
            device_ = device;
        }
        lent_ = true;
        *out = p_;
        return hipSuccess;
    }
    void give_back() { lent_ = false; }
    // Frees the memory, unless it is lent.
    void release() {
        if (lent_) return;
        if (alive()) (void)hipFree(p_);
        p_ = nullptr;
        bytes_ = 0;
        device_ = -1;
    }

   private:
    static hipError_t identify(void* p, uint64_t* id) {
        return hipPointerGetAttribute(id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, p);
    }
    bool alive() const {
        if (!p_) return false;
        uint64_t id = 0;
        if (identify(p_, &id) == hipSuccess) return id == id_;
        (void)hipGetLastError();  // not an allocation any more
        return false;
    }

    void* p_ = nullptr;
    size_t bytes_ = 0;
    int device_ = -1;
    uint64_t id_ = 0;
    bool lent_ = false;
};

}  // namespace tatara
