// fake_hip.cpp -- the HIP runtime calls that libcoral_search.so makes, without a device: memory comes from the host,
// kernels are not run, and what was asked for is recorded.  Loaded in front of the real runtime by
// tests/test_host_launches.py, which looks at how the library plans, allocates and launches.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <vector>

namespace {
struct Launch {
    const void* fn;
    size_t lds;
    unsigned blocks, threads;
};
std::map<void*, size_t> live;          // device allocations
std::map<const void*, size_t> limits;  // dynamic LDS a kernel may ask for
std::vector<Launch> launches;
size_t live_bytes = 0, refuse_at_least = 0, refuse_below = 0;
dim3 c_grid, c_block;
size_t c_lds;
hipStream_t c_stream;
}  // namespace

extern "C" {
// ---- what a test asks and sets
size_t fake_live_bytes() { return live_bytes; }
size_t fake_live_of_size(size_t bytes) {
    size_t c = 0;
    for (auto& a : live) c += a.second == bytes;
    return c;
}
void fake_refuse(size_t at_least, size_t below) { refuse_at_least = at_least, refuse_below = below; }
void fake_forget() { launches.clear(); }
size_t fake_launches() { return launches.size(); }
size_t fake_launch_lds(size_t i) { return launches[i].lds; }
unsigned fake_launch_blocks(size_t i) { return launches[i].blocks; }
unsigned fake_launch_threads(size_t i) { return launches[i].threads; }
const void* fake_launch_fn(size_t i) { return launches[i].fn; }
// launches that asked for more LDS than their kernel's limit was raised to (64 KB before it is)
size_t fake_launches_beyond_limit() {
    size_t c = 0;
    for (auto& l : launches) c += l.lds > (limits.count(l.fn) ? limits[l.fn] : (size_t)65536);
    return c;
}

// ---- the runtime
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    c_grid = g, c_block = b, c_lds = lds, c_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = c_grid, *b = c_block, *lds = c_lds, *s = c_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void**, size_t lds, hipStream_t) {
    launches.push_back({fn, lds, g.x, b.x});
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* fn, hipFuncAttribute, int value) {
    limits[fn] = (size_t)value;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int threads, size_t lds) {
    const int by_threads = 2048 / threads, by_lds = (int)((160u << 10) / (lds + 128));
    *n = by_threads < by_lds ? by_threads : by_lds;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    *p = nullptr;
    if (bytes >= refuse_at_least && bytes < refuse_below) return hipErrorOutOfMemory;
    *p = calloc(bytes ? bytes : 1, 1);
    if (!*p) return hipErrorOutOfMemory;
    live[*p] = bytes, live_bytes += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = live.find(p);
    if (it == live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    live_bytes -= it->second;
    live.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = calloc(bytes, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind) {
    memcpy(d, s, bytes);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, bytes);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* a, size_t* b) {
    *a = *b = (size_t)200 << 30;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (a macro of the header names the symbol of this version)
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* block = calloc((size_t)40 << 20, 1);
    *p = block;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
}
