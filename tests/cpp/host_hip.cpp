#include "host_hip.h"

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#include "kernels.h"

namespace host_hip {
int units = 256;
bool no_pinned = false;
int64_t mallocs_left = INT64_MAX;
int64_t device_bytes = 0, mallocs = 0;
}  // namespace host_hip

namespace {
std::map<void*, size_t> sizes;
hipError_t last = hipSuccess;

hipError_t done(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}
}  // namespace

extern "C" {

hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = host_hip::units, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host error"; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

hipError_t hipMalloc(void** p, size_t n)
{
    if (host_hip::mallocs_left-- <= 0 || !(*p = std::malloc(n ? n : 1))) return done(hipErrorOutOfMemory);
    std::memset(*p, 0xa5, n);   // what was never written is no zero
    sizes[*p] = n;
    host_hip::device_bytes += (int64_t)n;
    host_hip::mallocs++;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    const auto it = sizes.find(p);
    if (it == sizes.end()) return done(hipErrorInvalidValue);
    host_hip::device_bytes -= (int64_t)it->second;
    sizes.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (host_hip::no_pinned || !(*p = std::malloc(n ? n : 1))) return done(hipErrorOutOfMemory);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }

hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    return std::memcpy(d, s, n), hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return *e = nullptr, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }

}  // extern "C"

// What the kernels' files say of their launches, and the fills, which the host code counts on.
namespace xpbd {

int compact_block() { return 256; }
int compact_blocks(int nf) { return ((nf > 0 ? nf : 1) + 255) / 256; }
int jacobi_patch_size() { return 256; }
size_t jacobi_patch_smem(int maxl, bool det)
{
    return (size_t)maxl * 28 + (det ? (size_t)12 * 256 * 4 + (size_t)4 * 256 * 2 : (size_t)maxl * 12);
}
size_t jacobi_fused_smem(int maxl, bool con)
{
    return jacobi_patch_smem(maxl, true) + (con ? (size_t)maxl * 12 + (size_t)256 * 40 : 0);
}
bool quad_split(int block) { return (block < 0 ? -block : block) > kQuadSplit; }
bool quad_block_supported(int block)
{
    const int b = (block < 0 ? -block : block) - (quad_split(block) ? kQuadSplit : 0);
    return b == 64 || b == 128 || b == 256;
}
hipError_t launch_fill_zero(hipStream_t, void* p, size_t bytes) { return std::memset(p, 0, bytes), hipSuccess; }

}  // namespace xpbd
