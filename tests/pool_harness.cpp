// memory.hip over a runtime of a few lines, for test_pool.py: addresses that nothing is ever read from, an allocation limit, and the rules about
// stream captures as the HIP runtime has them (a thread that captures may neither allocate, free nor wait, and is invalidated if it tries;
// hipDeviceSynchronize does that to the captures of all threads).
#include "../ferric_amd/csrc/memory.hip"

#include <stdarg.h>

#include <thread>

namespace {
struct Runtime {
    std::mutex mu;
    uintptr_t next = (uintptr_t)1 << 40;
    std::map<uintptr_t, size_t> blocks;
    size_t bytes = 0, limit = (size_t)8 << 30;
    bool busy = false;
    int waits = 0;
    std::map<hipStream_t, std::pair<std::thread::id, bool>> capture;   // of a stream: its thread, and whether it is still valid
    bool refuse() {
        bool r = false;
        for (auto& c : capture)
            if (c.second.first == std::this_thread::get_id()) { c.second.second = false; r = true; }
        return r;
    }
    void idle() { busy = false; waits++; }
} rt;
char text[256];
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lock(rt.mu);
    *p = nullptr;
    if (rt.refuse()) return hipErrorStreamCaptureUnsupported;
    if (n == 0) return hipSuccess;
    if (n > rt.limit || rt.bytes + n > rt.limit) return hipErrorOutOfMemory;
    rt.blocks[rt.next] = n;
    rt.bytes += n;
    *p = (void*)rt.next;
    rt.next += (n + 4095) / 4096 * 4096;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lock(rt.mu);
    if (rt.refuse()) return hipErrorStreamCaptureUnsupported;
    auto it = rt.blocks.find((uintptr_t)p);
    if (it == rt.blocks.end()) return hipErrorInvalidValue;
    rt.idle();
    rt.bytes -= it->second;
    rt.blocks.erase(it);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    std::lock_guard<std::mutex> lock(rt.mu);
    for (auto& c : rt.capture) c.second.second = false;
    if (!rt.capture.empty()) return hipErrorStreamCaptureUnsupported;
    rt.idle();
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    std::lock_guard<std::mutex> lock(rt.mu);
    auto it = rt.capture.find(s);
    *st = it == rt.capture.end() ? hipStreamCaptureStatusNone : it->second.second ? hipStreamCaptureStatusActive : hipStreamCaptureStatusInvalidated;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { static thread_local hipStreamCaptureMode now = hipStreamCaptureModeGlobal; std::swap(*m, now); return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

int h_malloc(size_t n, void** p) { return fhip::pool_malloc(p, n); }
int h_free(void* p) { return fhip::pool_free(p); }
void h_trim() { fhip::pool_trim(); }
size_t h_range(void* p) {            // bytes from p to the end of the block in use it lies in, 0: none
    uintptr_t base = 0, end = 0;
    return fhip::pool_range(p, &base, &end) ? end - (uintptr_t)p : 0;
}
int h_place(void* p, size_t n, int dev) { return (int)fhip::pool_place(p, n, dev); }
void* h_stream() { static uintptr_t n = 4096; return (void*)(n += 16); }
int h_stream_destroy(void* s) {
    fhip::capture_ended((hipStream_t)s, true);
    std::lock_guard<std::mutex> lock(rt.mu);
    rt.capture.erase((hipStream_t)s);
    return 0;
}
void h_begin(void* s, int through_library) {
    if (through_library) fhip::capture_begun((hipStream_t)s);
    std::lock_guard<std::mutex> lock(rt.mu);
    rt.capture[(hipStream_t)s] = {std::this_thread::get_id(), true};
}
int h_end(void* s) {                 // 0: a valid graph, 1: an invalidated one, 2: another thread's capture, or none
    std::unique_lock<std::mutex> lock(rt.mu);
    auto it = rt.capture.find((hipStream_t)s);
    const bool mine = it != rt.capture.end() && it->second.first == std::this_thread::get_id(), valid = mine && it->second.second;
    if (mine) rt.capture.erase(it);
    lock.unlock();
    fhip::capture_ended((hipStream_t)s, false);
    return mine ? !valid : 2;
}
void h_work() { rt.busy = true; }
int h_busy() { return rt.busy; }
int h_waits() { return rt.waits; }
size_t h_bytes() { return rt.bytes; }
const char* h_text() { return text; }
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
}  // namespace fhip
