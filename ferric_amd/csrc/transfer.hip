// Host <-> device copies of the library through its own pinned memory, and dequantization of host bytes to host floats.
//
// A pageable hipMemcpyAsync costs a staging copy inside the runtime and a switch between the compute queue and a DMA engine: behind
// a kernel, 20 KB to the device took 16 us with the synchronisation that lets the source go, 608 KB to the host 38 us, and 84 MB
// to fresh host memory 12.5 ms (a single thread taking page faults one by one). Here a copy goes through a slot of pinned memory
// that a small kernel on the caller's own stream reads or writes directly:
//   to the device   the source is in the slot when the call returns, so nobody waits (3 us of host time)
//   to the host     one kernel and one wait; more than a slot is cut into chunks, each copied out of its slot by a worker thread
//                   while the next ones cross the bus (page faults of the destination included, which is why there are several)
// The kernel's rate is the bus's: 84 MB in 1.6 ms (53 GB/s) from 64 workgroups on, where the DMA engines took 1.6 - 3.0 ms.
#include "hostmem.hpp"

#include <string.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <system_error>
#include <thread>

namespace {

constexpr size_t OUT_BYTES = (size_t)2 << 20;    // a slot's part for data on its way to the host ...
constexpr size_t IN_BYTES = fhip::H2D_STAGED;    // ... and to the device (OUT_BYTES of floats are at most 557 056 block bytes, Q8_0)
constexpr size_t SLOT_BYTES = OUT_BYTES + IN_BYTES;
constexpr int SLOTS = 12, JOB_SLOTS = 8;         // a chunked copy takes up to JOB_SLOTS and leaves the others to small copies
constexpr int MAX_WG = 32, THREADS = 512;        // workgroups of a small copy (each confirms its part in a word of its own)
constexpr int WORKERS = 6;
constexpr int MAX_DEVICES = 64;

// n bytes, each workgroup a strided share; U = 16, 4 or 1 bytes, what the addresses allow. done (may be null): workgroup w stores seq
// in done[w] once everything it reads has been read.
template <class U>
__global__ __launch_bounds__(THREADS) void copy_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, size_t n, uint32_t* done,
                                                       uint32_t seq) {
    const size_t units = n / sizeof(U), step = (size_t)gridDim.x * THREADS;
    const U* s = (const U*)src;
    U* d = (U*)dst;
    size_t i = (size_t)blockIdx.x * THREADS + threadIdx.x;
    for (; i + 3 * step < units; i += 4 * step) {       // four loads in flight: a load from host memory takes over a microsecond
        const U a = s[i], b = s[i + step], c = s[i + 2 * step], e = s[i + 3 * step];
        d[i] = a; d[i + step] = b; d[i + 2 * step] = c; d[i + 3 * step] = e;
    }
    for (; i < units; i += step) d[i] = s[i];
    if (sizeof(U) > 1 && blockIdx.x == 0)
        for (size_t k = units * sizeof(U) + threadIdx.x; k < n; k += THREADS) dst[k] = src[k];
    if (done) {
        __syncthreads();                                // every wave's stores, and so the loads in front of them, are issued
        if (threadIdx.x == 0) __hip_atomic_store(&done[blockIdx.x], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

int launch_copy(const void* src, void* dst, size_t n, int max_wg, uint32_t* done, uint32_t seq, hipStream_t s, int* wgs) {
    const uintptr_t a = (uintptr_t)src | (uintptr_t)dst;
    const size_t unit = a & 3 ? 1 : (a & 15 ? 4 : 16);
    size_t g = (n / unit + 4 * THREADS - 1) / (4 * THREADS);
    g = g < 1 ? 1 : (g > (size_t)max_wg ? (size_t)max_wg : g);
    *wgs = (int)g;
    const uint8_t* from = (const uint8_t*)src;
    uint8_t* to = (uint8_t*)dst;
    if (unit == 16) copy_kernel<uint4><<<(unsigned)g, THREADS, 0, s>>>(from, to, n, done, seq);
    else if (unit == 4) copy_kernel<uint32_t><<<(unsigned)g, THREADS, 0, s>>>(from, to, n, done, seq);
    else copy_kernel<uint8_t><<<(unsigned)g, THREADS, 0, s>>>(from, to, n, done, seq);
    return fhip::check_hip(hipGetLastError(), "copy kernel");
}

struct Slot {
    uint8_t* host = nullptr;     // SLOT_BYTES pinned: [OUT_BYTES][IN_BYTES]
    uint8_t* dev = nullptr;      // IN_BYTES of device memory (dequantization only)
    uint32_t* done = nullptr;    // MAX_WG pinned words
    uint32_t seq = 0;
    int wgs = 0;                 // words of `done` that have to reach seq before the GPU has read the slot
    bool held = false;
    hipEvent_t ev = nullptr;

    bool read_by_gpu() const {
        for (int i = 0; i < wgs; i++)
            if (__atomic_load_n(&done[i], __ATOMIC_ACQUIRE) != seq) return false;
        return true;
    }
};

struct Ring {                    // one per device
    std::mutex mu;
    Slot slot[SLOTS];
    uint32_t* words = nullptr;
    hipStream_t stream[2] = {nullptr, nullptr};   // of dequantizations

    // The lowest slot that neither the host holds nor the GPU still reads: low slots stay warm in the CPU's caches. A slot's
    // pinned memory is made when it is first taken. null: all are taken.
    Slot* take(int* rc) {
        std::lock_guard<std::mutex> lock(mu);
        *rc = FHIP_OK;
        for (int i = 0; i < SLOTS; i++) {
            Slot& q = slot[i];
            if (q.held || !q.read_by_gpu()) continue;
            if (!words) {
                if ((*rc = fhip::check_hip(hipHostMalloc((void**)&words, SLOTS * MAX_WG * sizeof(uint32_t), hipHostMallocPortable), "hipHostMalloc"))) return nullptr;
                memset(words, 0, SLOTS * MAX_WG * sizeof(uint32_t));
            }
            if (!q.host && (*rc = fhip::check_hip(hipHostMalloc((void**)&q.host, SLOT_BYTES, hipHostMallocPortable), "hipHostMalloc"))) { q.host = nullptr; return nullptr; }
            q.done = words + i * MAX_WG;
            q.held = true;
            q.wgs = 0;
            return &q;
        }
        return nullptr;
    }
    // take() until there is one; the device is waited for when none comes free by itself
    Slot* need(int* rc) {
        for (int tries = 0; tries < 1 << 20; tries++) {
            if (Slot* q = take(rc)) return q;
            if (*rc) return nullptr;
            if (tries == 1 << 14 && (*rc = fhip::check_hip(hipDeviceSynchronize(), "hipDeviceSynchronize"))) return nullptr;
            std::this_thread::yield();
        }
        *rc = fhip::set_error(FHIP_ERR_HIP, "transfer: no pinned slot came free");
        return nullptr;
    }
    void release(Slot* q) {
        std::lock_guard<std::mutex> lock(mu);
        q->held = false;
    }
};
Ring* ring(int* rc) {
    static Ring* all = new Ring[MAX_DEVICES];    // never destroyed, as the streams and the pinned memory are not
    int dev = 0;
    if ((*rc = fhip::check_hip(hipGetDevice(&dev), "hipGetDevice"))) return nullptr;
    if (dev >= MAX_DEVICES) { *rc = fhip::set_error(FHIP_ERR_ARG, "device %d out of range", dev); return nullptr; }
    return &all[dev];
}

// ---- chunks on their way to the host, copied out of their slots by worker threads ----------------------------------------------
struct Job {
    uint8_t* dst;
    size_t bytes, chunk, count;               // the destination, cut into `count` chunks of `chunk` bytes (the last: what is left)
    Slot** slots;
    size_t n_slots;
    int dev;
    std::atomic<size_t> launched{0}, next{0}, copied{0};
    std::atomic<uint8_t>* out;                // [count] chunk has left its slot
    std::atomic<int> abort{0};
    std::atomic<int> err{0};                  // hipError_t of an event
};

void work_on(Job* j) {
    (void)hipSetDevice(j->dev);
    for (;;) {
        const size_t c = j->next.fetch_add(1);
        if (c >= j->count) return;
        while (j->launched.load(std::memory_order_acquire) <= c) {
            if (j->abort.load()) return;
            std::this_thread::yield();
        }
        Slot* q = j->slots[c % j->n_slots];
        hipError_t e;
        while ((e = hipEventQuery(q->ev)) == hipErrorNotReady) {
            (void)hipGetLastError();
            if (j->abort.load()) return;
            std::this_thread::yield();
        }
        if (e != hipSuccess) { j->err.store((int)e); j->abort.store(1); return; }
        const size_t at = c * j->chunk, n = j->bytes - at < j->chunk ? j->bytes - at : j->chunk;
        memcpy(j->dst + at, q->host, n);
        j->out[c].store(1, std::memory_order_release);
        j->copied.fetch_add(1);
    }
}

struct Workers {
    std::mutex one;                           // one job at a time
    std::mutex mu;
    std::condition_variable wake, left;
    Job* job = nullptr;
    uint64_t id = 0;
    int inside = 0;
    int threads = 0;

    void start() {
        if (threads) return;
        for (int i = 0; i < WORKERS; i++) {
            try {
                std::thread(&Workers::loop, this).detach();
            } catch (const std::system_error&) {
                return;                       // the threads there are do the work
            }
            threads++;
        }
    }
    void loop() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lock(mu);
        for (;;) {
            wake.wait(lock, [&] { return job && id != seen; });
            seen = id;
            Job* j = job;
            inside++;
            lock.unlock();
            work_on(j);
            lock.lock();
            if (--inside == 0) left.notify_all();
        }
    }
    bool post(Job* j) {                       // false: there are no threads
        std::lock_guard<std::mutex> lock(mu);
        start();
        if (!threads) return false;
        job = j; id++;
        wake.notify_all();
        return true;
    }
    void finish() {                           // nobody looks at the job any more when this returns
        std::unique_lock<std::mutex> lock(mu);
        job = nullptr;
        left.wait(lock, [&] { return inside == 0; });
    }
};
Workers& workers() { static Workers* w = new Workers(); return *w; }

// fill(c, slot, stream, n): enqueue what puts chunk c (n bytes) into slot->host; streams are taken in turn
template <class Fill>
int run_chunks(Ring* r, uint8_t* dst, size_t bytes, size_t chunk, hipStream_t* streams, size_t n_streams, Fill fill) {
    Workers& w = workers();
    std::lock_guard<std::mutex> one(w.one);
    int rc = FHIP_OK;
    Job j;
    j.dst = dst; j.bytes = bytes; j.chunk = chunk; j.count = (bytes + chunk - 1) / chunk;
    Slot* slots[JOB_SLOTS];
    j.slots = slots;
    j.n_slots = 0;
    if ((rc = fhip::check_hip(hipGetDevice(&j.dev), "hipGetDevice"))) return rc;
    while (j.n_slots < JOB_SLOTS && j.n_slots < j.count) {
        Slot* q = j.n_slots ? r->take(&rc) : r->need(&rc);
        if (!q) break;
        slots[j.n_slots++] = q;
        if (!q->ev && (rc = fhip::check_hip(hipEventCreateWithFlags(&q->ev, hipEventDisableTiming), "hipEventCreate"))) { q->ev = nullptr; break; }
    }
    std::atomic<uint8_t>* out = nullptr;
    if (!rc) {
        out = new std::atomic<uint8_t>[j.count]();
        j.out = out;
        const bool helped = w.post(&j);
        for (size_t c = 0; c < j.count && !rc; c++) {
            if (c >= j.n_slots && helped)
                while (!out[c - j.n_slots].load(std::memory_order_acquire) && !j.abort.load()) std::this_thread::yield();
            if (j.abort.load()) break;
            Slot* q = slots[c % j.n_slots];
            hipStream_t s = streams[c % n_streams];
            const size_t at = c * chunk, n = bytes - at < chunk ? bytes - at : chunk;
            if (!(rc = fill(c, q, s, n))) rc = fhip::check_hip(hipEventRecord(q->ev, s), "hipEventRecord");
            if (!rc && !helped && !(rc = fhip::check_hip(hipEventSynchronize(q->ev), "hipEventSynchronize"))) {
                memcpy(dst + at, q->host, n);
                j.copied.fetch_add(1);
            }
            if (!rc) j.launched.store(c + 1, std::memory_order_release);
        }
        if (rc) j.abort.store(1);
        while (!j.abort.load() && j.copied.load() < j.count) std::this_thread::yield();
        w.finish();
        if (!rc && j.err.load()) rc = fhip::check_hip((hipError_t)j.err.load(), "hipEventQuery");
        if (rc)                                // an enqueued chunk may still write into a slot
            for (size_t i = 0; i < n_streams; i++) (void)hipStreamSynchronize(streams[i]);
        delete[] out;
    }
    for (size_t i = 0; i < j.n_slots; i++) r->release(slots[i]);
    return rc;
}

bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) { (void)hipGetLastError(); return false; }
    return st != hipStreamCaptureStatusNone;
}

}  // namespace

namespace fhip {

// Up to a slot's IN_BYTES: the source has been copied when the call returns. Longer sources go through the runtime (35 GB/s, and
// it returns when the source has been read or is known to be pinned). A copy in a stream capture stays a copy node.
int copy_h2d(void* d, const void* h, size_t n, hipStream_t s) {
    if (n > IN_BYTES || capturing(s)) return check_hip(hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
    int rc;
    Ring* r = ring(&rc);
    Slot* q = r ? r->need(&rc) : nullptr;
    if (!q) return rc;
    memcpy(q->host, h, n);
    int wgs = 0;
    if (!(rc = launch_copy(q->host, d, n, MAX_WG, q->done, q->seq + 1, s, &wgs))) { q->seq++; q->wgs = wgs; }
    r->release(q);
    return rc;
}

int copy_d2h(void* h, const void* d, size_t n, hipStream_t s) {
    if (capturing(s)) return check_hip(hipMemcpyAsync(h, d, n, hipMemcpyDeviceToHost, s), "hipMemcpyAsync D2H");
    int rc, wgs = 0;
    Ring* r = ring(&rc);
    if (!r) return rc;
    if (n > OUT_BYTES) {
        const uint8_t* from = (const uint8_t*)d;
        return run_chunks(r, (uint8_t*)h, n, OUT_BYTES, &s, 1, [&](size_t c, Slot* q, hipStream_t st, size_t bytes) {
            return launch_copy(from + c * OUT_BYTES, q->host, bytes, 64, nullptr, 0, st, &wgs);
        });
    }
    Slot* q = r->need(&rc);
    if (!q) return rc;
    if (!(rc = launch_copy(d, q->host, n, MAX_WG, nullptr, 0, s, &wgs)) && !(rc = check_hip(hipStreamSynchronize(s), "hipStreamSynchronize")))
        memcpy(h, q->host, n);
    r->release(q);
    return rc;
}

// nb blocks (bytes each, vals values) of host memory to nb * vals floats of host memory: chunk by chunk the bytes go up, the
// unpacker writes its floats straight into the slot and a worker copies them out. Two streams, so that the way up of one chunk
// runs beside the way down of the one before it.
int dequant_host(uint32_t type, const uint8_t* h_raw, size_t nb, size_t vals, size_t bytes, float* h_out) {
    int rc;
    Ring* r = ring(&rc);
    if (!r) return rc;
    {
        std::lock_guard<std::mutex> lock(r->mu);
        for (auto& st : r->stream)
            if (!st && (rc = check_hip(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate"))) { st = nullptr; return rc; }
    }
    const size_t per = OUT_BYTES / sizeof(float) / vals;   // blocks of a chunk
    auto fill = [&](size_t c, Slot* q, hipStream_t s, size_t out_bytes) {
        const size_t blocks = out_bytes / sizeof(float) / vals, in = blocks * bytes;
        int err, wgs;
        if (!q->dev && (err = device_malloc((void**)&q->dev, IN_BYTES, "hipMalloc"))) { q->dev = nullptr; return err; }
        uint8_t* up = q->host + OUT_BYTES;
        memcpy(up, h_raw + c * per * bytes, in);
        if ((err = launch_copy(up, q->dev, in, MAX_WG, nullptr, 0, s, &wgs))) return err;
        return launch_dequant(type, q->dev, blocks, (float*)q->host, s);
    };
    if (nb > per) return run_chunks(r, (uint8_t*)h_out, nb * vals * sizeof(float), OUT_BYTES, r->stream, 2, fill);
    Slot* q = r->need(&rc);
    if (!q) return rc;
    const size_t n = nb * vals * sizeof(float);
    if (!(rc = fill(0, q, r->stream[0], n)) && !(rc = check_hip(hipStreamSynchronize(r->stream[0]), "hipStreamSynchronize"))) memcpy(h_out, q->host, n);
    r->release(q);
    return rc;
}

}  // namespace fhip
