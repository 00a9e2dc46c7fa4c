// The HIP calls that libqgemm.so makes around a launch, without a GPU: a
// 256-CU gfx950 whose launches are recorded (thread, grid, block, kernel)
// instead of run.  Loaded before the library, so that its calls resolve here.
#include <hip/hip_runtime_api.h>
#include <sys/syscall.h>
#include <unistd.h>

#include <cstring>
#include <mutex>
#include <vector>

namespace {
struct Launch {
    long long thread, grid[3], block, kernel;
};
std::mutex mu;
std::vector<Launch> launches;
int pause_us = 0;
thread_local dim3 cfg_grid, cfg_block;
thread_local size_t cfg_lds;
thread_local hipStream_t cfg_stream;
}  // namespace

extern "C" {

hipError_t hipGetDevice(int* dev) {
    *dev = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) {
    *value = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = reinterpret_cast<void*>(1ull << 46);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
    {
        std::lock_guard<std::mutex> lock(mu);
        launches.push_back({(long long)syscall(SYS_gettid), {grid.x, grid.y, grid.z}, (long long)block.x * block.y * block.z,
                            (long long)(size_t)kernel});
    }
    if (pause_us) usleep(pause_us);
    // the runtime's own limit: threads per grid dimension fit 32 bits
    const bool fits = (unsigned long long)grid.x * block.x <= 0xffffffffull && (unsigned long long)grid.y * block.y <= 0xffffffffull;
    return fits ? hipSuccess : hipErrorInvalidConfiguration;
}

// microseconds a launch takes its caller from now on; forgets the launches so far
void stub_reset(int launch_us) {
    std::lock_guard<std::mutex> lock(mu);
    launches.clear();
    pause_us = launch_us;
}
int stub_count(void) {
    std::lock_guard<std::mutex> lock(mu);
    return (int)launches.size();
}
// thread, grid x / y / z, threads per block, kernel
void stub_launch(int i, long long* out) {
    std::lock_guard<std::mutex> lock(mu);
    const Launch& l = launches[i];
    const long long v[6] = {l.thread, l.grid[0], l.grid[1], l.grid[2], l.block, l.kernel};
    std::memcpy(out, v, sizeof(v));
}

}  // extern "C"
