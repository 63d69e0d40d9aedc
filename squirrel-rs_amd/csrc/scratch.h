// Device scratch of the operator-level entry points, kept between calls.
//
// A call's temporaries came from hipMalloc and went back with hipFree, which
// waits for the device: 30 to 130 us of a call whose kernels take 5 to 100.
// Idle blocks are kept per device instead.  Every user launches on the null
// stream, so a block that goes to another call, of this thread or another, is
// written there only behind the launches that still read it.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace sq {

constexpr size_t kScratchKeep = (size_t)256 << 20;  // idle bytes kept per device at most
constexpr unsigned kScratchAge = 256;               // an idle block is freed after so many returns without a use

// A block of at least n bytes on the current device; 0 or a status code.
int scratch_get(size_t n, void** p, size_t* size, int* device);
// Back to the pool (the block's launches may still be queued on the null stream).
void scratch_put(void* p, size_t size, int device);
// Frees the current device's idle blocks.
void scratch_trim();
// hipMalloc, tried again without the idle blocks where it fails.  A failure
// leaves no error behind for the next launch's check to find.
hipError_t device_alloc(void** p, size_t n);

// A temporary of one entry point's call.
struct Tmp {
    void* p = nullptr;
    size_t size = 0;
    int device = 0;
    Tmp() = default;
    Tmp(const Tmp&) = delete;
    Tmp& operator=(const Tmp&) = delete;
    ~Tmp() {
        if (p) scratch_put(p, size, device);
    }
    int alloc(size_t n) { return scratch_get(n, &p, &size, &device); }
};

}  // namespace sq
