// A stand-in for the HIP runtime and the kernels, to run the host engine
// (nb_engine.cpp) without a GPU: device and pinned memory are host memory with
// limits that a test sets, streams and events do nothing because every launch is
// done when it returns, and the launches that move bodies move them. The others
// do nothing. Linked with nb_engine.cpp into a library of its own.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#include "nb_internal.h"

namespace {

struct Pool {
    std::mutex mu;
    std::map<void *, size_t> blocks;
    size_t used = 0, limit = ~(size_t)0;

    hipError_t get(void **p, size_t bytes)
    {
        std::lock_guard<std::mutex> lock(mu);
        *p = nullptr;
        if (bytes > limit - used) return hipErrorOutOfMemory;
        if (posix_memalign(p, 256, bytes ? bytes : 1)) return hipErrorOutOfMemory;
        blocks[*p] = bytes;
        used += bytes;
        return hipSuccess;
    }
    hipError_t give_back(void *p)
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto it = blocks.find(p);
        if (it == blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
        used -= it->second;
        blocks.erase(it);
        free(p);
        return hipSuccess;
    }
    void set_limit(long long more)
    {
        std::lock_guard<std::mutex> lock(mu);
        limit = more < 0 ? ~(size_t)0 : used + (size_t)more;
    }
};

Pool device, pinned;
std::atomic<int> fail_state{0}; // which set-state launch from now on fails (0: none)
// as the runtime keeps it: the last failure, until it is asked for; a launch asks
thread_local hipError_t last_error = hipSuccess;

hipError_t kept(hipError_t e)
{
    if (e != hipSuccess) last_error = e;
    return e;
}

} // namespace

extern "C" {

// bytes that may still be allocated (negative: no limit), and what is
void host_device_room(long long more) { device.set_limit(more); }
void host_pinned_room(long long more) { pinned.set_limit(more); }
long long host_device_used() { return (long long)device.used; }
long long host_pinned_used() { return (long long)pinned.used; }
void host_fail_state_launch(int nth) { fail_state = nth; }

hipError_t hipGetLastError()
{
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipMalloc(void **p, size_t bytes) { return kept(device.get(p, bytes)); }
hipError_t hipFree(void *p) { return device.give_back(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return kept(pinned.get(p, bytes)); }
hipError_t hipHostFree(void *p) { return pinned.give_back(p); }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int value, size_t bytes, hipStream_t)
{
    memset(dst, value, bytes);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol)
{
    *p = const_cast<void *>(symbol);
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = reinterpret_cast<hipEvent_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.0f;
    return hipSuccess;
}

} // extern "C"

namespace nb {

hipError_t launch_set_state(const Dev &d, int first, int count, const float *c, hipStream_t)
{
    if (fail_state > 0 && --fail_state == 0) return hipErrorLaunchFailure;
    for (int j = 0; j < count; ++j) {
        const int i = first + j;
        const float x = c[j], y = c[count + j], z = c[2 * count + j];
        d.pm4[i] = make_float4(x, y, z, c[6 * count + j]);
        d.vel4[i] = make_float4(c[3 * count + j], c[4 * count + j], c[5 * count + j], 0.0f);
        d.acc4[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (d.fp64) d.pos64[i] = make_double4(x, y, z, 0.0);
        d.sorted[i] = i;
    }
    if (first == 0) d.ctl->step = -1;
    return hipGetLastError();
}
hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t)
{
    if (((uintptr_t)dst | (uintptr_t)src) % 16) return hipErrorInvalidValue;
    memcpy(dst, src, bytes);
    return hipGetLastError();
}
hipError_t launch_columns(const float4 *src, int count, float *col, hipStream_t)
{
    for (int j = 0; j < count; ++j) {
        col[j] = src[j].x;
        col[count + j] = src[j].y;
        col[2 * count + j] = src[j].z;
    }
    return hipGetLastError();
}
hipError_t launch_copy_vertices(const Dev &d, int first, int count, float4 *pos, float4 *vel, hipStream_t)
{
    for (int j = 0; j < count; ++j) {
        const float4 p = d.pm4[first + j], v = d.vel4[first + j];
        if (pos) pos[j] = make_float4(p.x, p.y, p.z, 1.0f);
        if (vel) vel[j] = make_float4(v.x, v.y, v.z, 1.0f);
    }
    return hipGetLastError();
}

hipError_t launch_bbox(const Dev &, int, bool, hipStream_t) { return hipGetLastError(); }
hipError_t launch_build_keys(const Dev &d, bool, bool, bool, hipStream_t)
{
    for (int i = 0; i < d.n; ++i) d.kb_val[0][i] = i; // the order is an order
    return hipGetLastError();
}
hipError_t launch_levels(const Dev &, hipStream_t) { return hipGetLastError(); }
hipError_t launch_summarize_level(const Dev &, int, int, hipStream_t) { return hipGetLastError(); }
hipError_t launch_summarize_block(const Dev &, int, int, hipStream_t) { return hipGetLastError(); }
hipError_t launch_force(const Dev &, int, int, hipStream_t) { return hipGetLastError(); }
hipError_t launch_integrate(const Dev &, hipStream_t) { return hipGetLastError(); }
hipError_t launch_step_mark(const Dev &, bool, hipStream_t) { return hipGetLastError(); }
hipError_t launch_paths(const Dev &, unsigned long long *, int *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_moments(const Dev &, double *part, hipStream_t)
{
    memset(part, 0, sizeof(double) * 11 * kMomentBlocks);
    return hipGetLastError();
}
hipError_t launch_direct64(const Dev &, const int *, int ns, double4 *, double4 *out, DirectSum, hipStream_t)
{
    memset(out, 0, sizeof(double4) * (size_t)ns);
    return hipGetLastError();
}
hipError_t launch_gather_acc(const Dev &, const int *, int, float4 *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_group_order(const Dev &, hipStream_t) { return hipGetLastError(); }
hipError_t launch_coarse(const Dev &, const Learn &, int, const int *, int, float *, float4 *, int, hipStream_t)
{
    return hipGetLastError();
}
hipError_t launch_pair_records(const Dev &, const int *, int, float4 *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_pairs(const Dev &, const Learn &, const int *, int, const float4 *, float *, float4 *, float4 *,
                        hipStream_t)
{
    return hipGetLastError();
}
hipError_t launch_make_target(const float4 *, const float4 *, int, float *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_standardize(float *, int, int, float *, float *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_mlp_rows(const Learn &, const float *, int, float *, hipStream_t) { return hipGetLastError(); }
hipError_t launch_train_iter(const Train &, int, int, uint64_t, bool, float, float, float, float, float, float,
                             hipStream_t)
{
    return hipGetLastError();
}

} // namespace nb
