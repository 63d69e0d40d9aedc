#include "scratch.h"

#include <mutex>
#include <vector>

#include "model.h"

namespace sq {
namespace {

struct Block {
    void* p;
    size_t size;
    unsigned returned;  // the pool's count when it came back
};
struct Pool {
    std::mutex mu;
    std::vector<Block> idle;
    size_t bytes = 0;
    unsigned returns = 0;
};
constexpr int kMaxDevices = 64;
// never destroyed: at process end the runtime may be gone before it
Pool& pool_of(int device) {
    static Pool* pools = new Pool[kMaxDevices];
    return pools[device];
}

// Sizes in steps of an eighth of their power of two (4 KB at least), so that
// calls of nearby sizes share blocks.
size_t rounded(size_t n) {
    size_t step = 4096;
    while (step * 16 <= n) step *= 2;
    return (n + step - 1) / step * step;
}

}  // namespace

hipError_t device_alloc(void** p, size_t n) {
    hipError_t e = hipMalloc(p, n);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        scratch_trim();
        if ((e = hipMalloc(p, n)) != hipSuccess) (void)hipGetLastError();
    }
    return e;
}

int scratch_get(size_t n, void** p, size_t* size, int* device) {
    SQ_HIP_CHECK(hipGetDevice(device));
    const size_t want = n ? n : 1;
    n = want > kScratchKeep ? want : rounded(want);  // (larger blocks are never kept)
    if (*device >= 0 && *device < kMaxDevices) {
        Pool& P = pool_of(*device);
        std::lock_guard<std::mutex> lk(P.mu);
        // the smallest block that holds n, unless it would waste as much again
        size_t best = P.idle.size();
        for (size_t i = 0; i < P.idle.size(); i++)
            if (P.idle[i].size >= n && P.idle[i].size <= 2 * n && (best == P.idle.size() || P.idle[i].size < P.idle[best].size))
                best = i;
        if (best < P.idle.size()) {
            *p = P.idle[best].p;
            *size = P.idle[best].size;
            P.bytes -= *size;
            P.idle[best] = P.idle.back();
            P.idle.pop_back();
            return 0;
        }
    }
    hipError_t e = device_alloc(p, n);
    if (e != hipSuccess && n > want) {  // rounding must not refuse what fits
        n = want;
        e = device_alloc(p, n);
    }
    if (e != hipSuccess) {
        *p = nullptr;
        return set_error(SQ_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    *size = n;
    return 0;
}

void scratch_put(void* p, size_t size, int device) {
    if (device < 0 || device >= kMaxDevices || size > kScratchKeep) {
        (void)hipFree(p);
        return;
    }
    std::vector<void*> drop;
    {
        Pool& P = pool_of(device);
        std::lock_guard<std::mutex> lk(P.mu);
        P.returns++;
        P.idle.push_back(Block{p, size, P.returns});
        P.bytes += size;
        for (;;) {
            size_t old = 0;
            for (size_t i = 1; i < P.idle.size(); i++)
                if (P.returns - P.idle[i].returned > P.returns - P.idle[old].returned) old = i;
            if (P.bytes <= kScratchKeep && P.returns - P.idle[old].returned < kScratchAge) break;
            drop.push_back(P.idle[old].p);
            P.bytes -= P.idle[old].size;
            P.idle[old] = P.idle.back();
            P.idle.pop_back();
        }
    }
    for (void* d : drop) (void)hipFree(d);
}

void scratch_trim() {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return;
    std::vector<Block> drop;
    {
        Pool& P = pool_of(device);
        std::lock_guard<std::mutex> lk(P.mu);
        drop.swap(P.idle);
        P.bytes = 0;
    }
    for (const Block& b : drop) (void)hipFree(b.p);
}

}  // namespace sq
