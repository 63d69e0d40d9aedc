// Host entry points of the persistent decode step for the CPU emulation
// build.  That kernel (its LDS ring fed by direct-to-LDS loads and its
// inter-workgroup polling) is not emulated: the stub reports that no
// persistent grid fits, so contexts take the one-kernel-per-op decode path.
// With SQEMU_STEP=1 it reports one that does, for what surrounds the step: the
// stream builder is then a kernel that reads the layer table as the real one
// does and stops the run where the table is not there yet, and a step writes
// the first word of its timeline and nothing else.
// TEST INFRASTRUCTURE ONLY.
#include <cstdlib>
#include <cstring>

#include "launch.h"

namespace sq {

namespace {
bool set_up() {
    const char* e = getenv("SQEMU_STEP");
    return e && !strcmp(e, "1");
}
__global__ void read_layers_kernel(const StepLayer* layers, int n) {
    for (int l = 0; l < n; l++)
        if (layers[l].qkv.rows <= 0 || layers[l].down.rows <= 0)
            ::sqemu::fatal("the stream builder ran before the layer table was written");
}
__global__ void trace_kernel(unsigned long long* trace) { *trace = 7; }
}  // namespace

bool decode_step_fits(int, int, int, int, int) { return set_up(); }
size_t decode_stream_stride(int, int, int, int, int, int, int, int) { return 0; }
size_t exchange_words(int dim, int ffn, int heads, int kv_heads, int tiles, int) {
    return set_up() ? (size_t)2 * dim + ffn + 64 * heads * (size_t)(tiles + 2) + 256 * kv_heads : 0;
}
int launch_build_stream(hipStream_t s, int, const StepArgs& a, int, void*) {
    if (!set_up()) return set_error(SQ_ERR_UNSUPPORTED, "persistent decode step is not emulated");
    hipLaunchKernelGGL(read_layers_kernel, dim3(1), dim3(1), 0, s, a.layers, a.n_layers);
    return 0;
}
int launch_decode_step(hipStream_t s, int, const StepArgs& a, int, int) {
    if (set_up() && a.trace) {
        hipLaunchKernelGGL(trace_kernel, dim3(1), dim3(1), 0, s, a.trace);
        return 0;
    }
    return set_error(SQ_ERR_UNSUPPORTED, "persistent decode step is not emulated");
}
int decode_step_max_grid(int, int* grid) {
    *grid = set_up() ? 1 : 0;
    return 0;
}

}  // namespace sq
