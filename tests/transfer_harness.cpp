// transfer.hip over a runtime of a few lines, for test_transfer.py: "device" memory is the process's own, a stream is a list of work that nothing is done of before somebody
// waits for the stream, and pinned memory can run out.
#include "../ferric_amd/csrc/transfer.hip"

#include <stdarg.h>
#include <stdlib.h>

#include <functional>
#include <map>

namespace {
struct Runtime {
    std::map<hipStream_t, std::vector<std::function<void()>>> work;
    size_t pinned = 0, pinned_limit = (size_t)1 << 40;
    int own_copies = 0;                // copies that the runtime was asked for
    hipError_t last = hipSuccess;      // what hipGetLastError would report
    hipError_t result(hipError_t e) { return e == hipSuccess ? e : last = e; }
} rt;
thread_local struct { dim3 grid, block; hipStream_t stream; } config;
char text[256];

template <class U, int N>
bool copy_launch(const void* kernel, void** args) {
    if (kernel != (const void*)&copy_kernel<U, N>) return false;
    auto src = *(const uint8_t**)args[0];
    auto dst = *(uint8_t**)args[1];
    auto parts = *(Parts<N>*)args[2];
    auto seq = *(uint32_t*)args[3];
    const unsigned wgs = config.grid.x;
    rt.work[config.stream].push_back([=] {
        const int count = N == 1 ? 1 : parts.count;
        memcpy(dst, src, parts.end[count - 1]);
        for (int p = 0; p < count; p++)
            for (unsigned w = 0; w < wgs; w++) parts.done[p][w] = seq;
    });
    return true;
}
}  // namespace

extern "C" {
char __hip_fatbin[4096];
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = nullptr;
    if (rt.pinned + n > rt.pinned_limit) return rt.result(hipErrorOutOfMemory);
    rt.pinned += n;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* h, size_t n, hipMemcpyKind, hipStream_t s) {
    rt.own_copies++;
    const std::vector<uint8_t> read((const uint8_t*)h, (const uint8_t*)h + n);
    rt.work[s].push_back([=] { memcpy(d, read.data(), n); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    for (auto& w : rt.work[s]) w();
    rt.work[s].clear();
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return rt.result(hipErrorOutOfMemory); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return rt.result(hipErrorInvalidValue); }   // plain host memory
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = rt.last; rt.last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t s) { config = {grid, block, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) { *grid = config.grid; *block = config.block; *lds = 0; *s = config.stream; return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    return copy_launch<u32x4, 1>(f, args) || copy_launch<uint32_t, 1>(f, args) || copy_launch<uint8_t, 1>(f, args) || copy_launch<u32x4, PARTS>(f, args) ||
                   copy_launch<uint32_t, PARTS>(f, args) || copy_launch<uint8_t, PARTS>(f, args) ? hipSuccess : hipErrorInvalidValue;
}

int h_upload(void* d, const void* h, size_t n, void* s) { return fhip::upload(d, h, n, (hipStream_t)s); }
int h_h2d(void* d, const void* h, size_t n, void* s) { return fhip::copy_h2d(d, h, n, (hipStream_t)s); }
int h_d2h(void* h, const void* d, size_t n, void* s) { return fhip::copy_d2h(h, d, n, (hipStream_t)s); }
size_t h_waiting(void* s) { return rt.work[(hipStream_t)s].size(); }
int h_runtime_copies() { return rt.own_copies; }
int h_stale_error() { return (int)hipGetLastError(); }
size_t h_pinned() { return rt.pinned; }
void h_no_more_pinned(size_t n) { rt.pinned_limit = rt.pinned + n; }
void h_hold_upload_slots(int n) {        // as uploads of other threads do
    int rc;
    Ring* r = ring(&rc);
    for (int i = 0; i < n; i++) (void)r->take(&rc, SLOTS, SMALL_SLOTS);
}
}

namespace fhip {
int set_error(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(text, sizeof(text), fmt, ap);
    va_end(ap);
    return code;
}
int check_hip(hipError_t e, const char* what) { return e == hipSuccess ? FHIP_OK : set_error(FHIP_ERR_HIP, "%s: %d", what, (int)e); }
Place pool_place(const void*, size_t, int) { return Place::inside; }
bool thread_captures() { return false; }
bool runtime_allocates() { return true; }
int device_malloc(void**, size_t, const char*) { return FHIP_ERR_HIP; }
int launch_dequant(uint32_t, const uint8_t*, size_t, float*, hipStream_t) { return FHIP_ERR_HIP; }
int launch_dequant_through(uint32_t, const uint8_t*, size_t, float*, uint32_t*, uint32_t, hipStream_t, int*) { return FHIP_ERR_HIP; }
}  // namespace fhip
