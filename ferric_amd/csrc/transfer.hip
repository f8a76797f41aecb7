// Host <-> device copies of the library through its own pinned memory, and dequantization of host bytes to host floats.
//
// A pageable hipMemcpyAsync costs a staging copy inside the runtime and a switch between the compute queue and a DMA engine: behind
// a kernel, 20 KB to the device took 16 us with the synchronisation that lets the source go, 608 KB to the host 38 us, and 84 MB
// to fresh host memory 12.5 ms (a single thread taking page faults one by one). Here a copy goes through slots of pinned memory
// that a small kernel on the caller's own stream reads or writes directly; the kernel's workgroups confirm in pinned words of
// their own, which a host thread polls without a call into the runtime.
//   to the device   up to H2D_STAGED the source is in a slot when the call returns, so nobody waits (3 us of host time); an upload of up to 12 MiB goes
//                   through several, one filled while the one before crosses the bus, and has arrived when the call returns, as longer ones have
//   to the host     up to a slot in one kernel that confirms part after part, the host copying one out while the next ones cross the bus
//                   (608 KB, idle device: 26 us; 37 with one part and a stream synchronisation), up to three slots likewise (one and a half into fresh memory); more is cut into chunks, each
//                   copied out of its slot by a worker thread while the next ones cross (page faults of the destination
//                   included, which is why there are several workers). While the stream has other work in front of the copy, the waiting thread makes the
//                   destination's pages: into fresh memory behind 350 us of work, us, 608 KB 477 -> 379, 2 MB 810 -> 417, 10.4 MB 2420 -> 1800
// The kernel's rate is the bus's: 84 MB in 1.6 ms (53 GB/s) from 64 workgroups on, where the DMA engines took 1.6 - 3.0 ms. A whole copy to the host reaches
// 40 - 42 GB/s (16 MB in 396 us), the host's side included.
// Nobody waits for another stream's work: a long copy takes the workers, which serve one at a time, once its own stream has got there, and who finds no slot
// goes through the runtime.
#include "hostmem.hpp"
#include "through.hpp"

#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace {

using fhip::store_through;
using fhip::u32x4;

constexpr size_t OUT_BYTES = (size_t)1 << 20;    // a slot's part for data on its way to the host ...
constexpr size_t IN_BYTES = fhip::H2D_STAGED;    // ... and to the device (a chunk of floats is at most 278 528 block bytes, Q8_0)
constexpr size_t CHUNK = OUT_BYTES;              // of a long copy
constexpr size_t SLOT_BYTES = OUT_BYTES + IN_BYTES;
constexpr int SLOTS = 28, JOB_SLOTS = 12;        // a chunked copy takes up to JOB_SLOTS of the first SMALL_SLOTS and leaves the others to small copies; ...
constexpr int SMALL_SLOTS = 16;                  // ... those behind are the chunked uploads', which hold them until their stream has got there
constexpr int MAX_WG = 64, THREADS = 512;        // workgroups of a copy (each confirms its part in a word of its own)
constexpr size_t IN_PARTS = (size_t)96 << 10;    // copies to the host from here on go in parts, the host copying one out while the next ones cross
constexpr int PARTS = 8;                         // at most
constexpr size_t D2H_ALONE = 3 * OUT_BYTES;      // longer copies to the host are the workers' ...
constexpr size_t D2H_ALONE_NEW = D2H_ALONE / 2;  // ... and those from here on whose destination has pages that nobody has touched
constexpr size_t IN_CHUNKS_TO = (SLOTS - SMALL_SLOTS) * OUT_BYTES;   // uploads up to there, from IN_BYTES on, the calling thread takes in chunks
constexpr int WORKERS = 10;
constexpr int MAX_DEVICES = 64;

// n bytes, each workgroup a strided share; U = 16, 4 or 1 bytes, what the addresses allow. Workgroup w stores seq
// in done[w] once everything it reads has been read and everything it writes has arrived.
// A confirmation is one store behind a wait, not a release: a release at system scope writes back the whole L2 (5 us of a 4 KB copy).
// The stores it stands for go through to memory themselves (sc0 sc1), and s_waitcnt holds the wave until they have arrived.

// The copy in up to N parts one after the other, each confirmed by itself: part p ends at byte end[p] (a multiple of 16 but for the last one's).
// A copy in one part is a kernel of its own: with eight parts' arguments and their loop it takes half a microsecond more (4096 bytes to the host
// 10.2 us, 9.6; 65536 12.5, 12.0).
template <int N>
struct Parts {
    int count;
    size_t end[N];
    uint32_t* done[N];           // MAX_WG words each
};
template <class U, int N>
__global__ __launch_bounds__(THREADS) void copy_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, Parts<N> parts, uint32_t seq) {
    const int count = N == 1 ? 1 : parts.count;
    const size_t step = (size_t)gridDim.x * THREADS, n = parts.end[count - 1];
    const U* s = (const U*)src;
    U* d = (U*)dst;
    size_t begin = 0;
#pragma unroll 1
    for (int p = 0; p < count; p++) {
        const size_t units = parts.end[p] / sizeof(U);
        size_t i = begin + (size_t)blockIdx.x * THREADS + threadIdx.x;
        for (; i + 3 * step < units; i += 4 * step) {   // four loads in flight: a load from host memory takes over a microsecond
            const U a = s[i], b = s[i + step], c = s[i + 2 * step], e = s[i + 3 * step];
            store_through(d + i, a); store_through(d + i + step, b); store_through(d + i + 2 * step, c); store_through(d + i + 3 * step, e);
        }
        for (; i < units; i += step) store_through(d + i, s[i]);
        if (sizeof(U) > 1 && blockIdx.x == 0 && p == count - 1)
            for (size_t k = units * sizeof(U) + threadIdx.x; k < n; k += THREADS) store_through(dst + k, src[k]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(&parts.done[p][blockIdx.x], seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        begin = units;
    }
}

template <int N>
int launch_copy(const void* src, void* dst, const Parts<N>& parts, int max_wg, int units_per_thread, uint32_t seq, hipStream_t s, int* wgs) {
    const uintptr_t a = (uintptr_t)src | (uintptr_t)dst;
    const size_t unit = a & 3 ? 1 : (a & 15 ? 4 : 16), per_wg = (size_t)units_per_thread * THREADS;
    size_t g = (parts.end[0] / unit + per_wg - 1) / per_wg;
    g = g < 1 ? 1 : (g > (size_t)max_wg ? (size_t)max_wg : g);
    *wgs = (int)g;
    const uint8_t* from = (const uint8_t*)src;
    uint8_t* to = (uint8_t*)dst;
    if (unit == 16) copy_kernel<u32x4, N><<<(unsigned)g, THREADS, 0, s>>>(from, to, parts, seq);
    else if (unit == 4) copy_kernel<uint32_t, N><<<(unsigned)g, THREADS, 0, s>>>(from, to, parts, seq);
    else copy_kernel<uint8_t, N><<<(unsigned)g, THREADS, 0, s>>>(from, to, parts, seq);
    return fhip::check_hip(hipGetLastError(), "copy kernel");
}
int launch_copy(const void* src, void* dst, size_t n, int units_per_thread, uint32_t* done, uint32_t seq, hipStream_t s, int* wgs) {
    return launch_copy(src, dst, Parts<1>{1, {n}, {done}}, MAX_WG, units_per_thread, seq, s, wgs);
}

struct Slot {
    uint8_t* host = nullptr;     // SLOT_BYTES pinned: [OUT_BYTES][IN_BYTES]; of a chunked upload's slots OUT_BYTES
    uint32_t* done = nullptr;    // MAX_WG pinned words, of a copy in parts the last part's ...
    uint32_t* early = nullptr;   // ... and (PARTS - 1) * MAX_WG for the parts before it
    uint32_t seq = 0;
    int wgs = 0;                 // words of `done` that have to reach seq before the GPU has read the slot
    bool held = false;

    bool read_by_gpu() const { return confirmed(seq, wgs); }
    bool confirmed(uint32_t want, int n) const { return confirmed(done, want, n); }
    static bool confirmed(const uint32_t* words, uint32_t want, int n) {
        for (int i = 0; i < n; i++)
            if (__atomic_load_n(&words[i], __ATOMIC_ACQUIRE) != want) return false;
        return true;
    }
};

// The pages of a destination, which a fresh allocation does not have until somebody writes to it, made a few at a time: by a thread that waits for the device
// anyway, in place of the copy behind the wait (0.16 us a KB). step() is false when all are there, or the kernel has no such call (Linux before 5.14).
class Pages {
    uintptr_t at, end;
    bool refused = false;

public:
    Pages(const void* h, size_t n) {
        static const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
        at = (uintptr_t)h / page * page;
        end = ((uintptr_t)h + n + page - 1) / page * page;
    }
    bool step() {
        constexpr int POPULATE_WRITE = 23;           // MADV_POPULATE_WRITE
        constexpr uintptr_t STEP = (uintptr_t)64 << 10;
        if (at >= end) return false;
        const uintptr_t n = end - at < STEP ? end - at : STEP;
        refused = madvise((void*)at, n, POPULATE_WRITE) != 0;
        at = refused ? end : at + n;
        return !refused;
    }
    bool made() const { return at >= end && !refused; }
};

// Until the first n of the words hold `want`: polled for two milliseconds (a decode step), then left to the runtime. `pages` are made meanwhile.
int await_words(const uint32_t* words, uint32_t want, int n, hipStream_t s, Pages* pages = nullptr) {
    const auto start = std::chrono::steady_clock::now();
    for (unsigned i = 0; !Slot::confirmed(words, want, n); i++) {
        if (pages && pages->step()) continue;
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
        if ((i & 255) == 255 && std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2))
            return fhip::check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
    }
    return FHIP_OK;
}

struct Ring {                    // one per device
    std::mutex mu;
    Slot slot[SLOTS];
    uint32_t* words = nullptr;
    hipStream_t stream[2] = {nullptr, nullptr};   // of dequantizations
    std::mutex spare_mu;
    uint8_t* spare = nullptr;    // SLOT_BYTES of device memory for a dequantization without a slot

    // The lowest slot that neither the host holds nor the GPU still reads: low slots stay warm in the CPU's caches. A slot's
    // pinned memory is made when it is first taken. null: all are taken.
    Slot* take(int* rc, int to = SMALL_SLOTS, int from = 0) {
        std::lock_guard<std::mutex> lock(mu);
        *rc = FHIP_OK;
        for (int i = from; i < to; i++) {
            Slot& q = slot[i];
            if (q.held || !q.read_by_gpu()) continue;
            if (!words) {
                if ((*rc = fhip::check_hip(hipHostMalloc((void**)&words, SLOTS * PARTS * MAX_WG * sizeof(uint32_t), hipHostMallocPortable), "hipHostMalloc"))) return nullptr;
                memset(words, 0, SLOTS * PARTS * MAX_WG * sizeof(uint32_t));
            }
            if (!q.host && (*rc = fhip::check_hip(hipHostMalloc((void**)&q.host, i < SMALL_SLOTS ? SLOT_BYTES : OUT_BYTES, hipHostMallocPortable), "hipHostMalloc"))) { q.host = nullptr; return nullptr; }
            q.done = words + i * PARTS * MAX_WG;
            q.early = q.done + MAX_WG;
            q.held = true;
            q.wgs = 0;
            return &q;
        }
        return nullptr;
    }
    // take(), for some milliseconds where all are taken. null without an error: copies that wait for other streams' work hold them, and
    // this one is better left to the runtime than made to wait for that work too
    Slot* get(int* rc) {
        const auto start = std::chrono::steady_clock::now();
        for (;;) {
            if (Slot* q = take(rc)) return q;
            if (*rc || std::chrono::steady_clock::now() - start > std::chrono::milliseconds(4)) return nullptr;
            std::this_thread::yield();
        }
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

// ---- chunks whose host side worker threads copy -------------------------------------------------------------------------------
// Task k of a job: the first n_slots are the ways up of chunks 0 .. n_slots - 1, then the way down of chunk c and the way up of chunk
// c + n_slots take turns. A job that goes one way only has the other kind as empty tasks.
struct Job {
    size_t count;                             // chunks; chunk c is [c * chunk, ..) of each side it has
    const uint8_t* up;                        // the caller's memory on the way up (may be null) ...
    size_t up_bytes, up_chunk, up_at;         // ... and where its chunks lie in a slot
    uint8_t* down;                            // and on the way down (may be null)
    size_t down_bytes, down_chunk;
    Slot** slots;
    size_t n_slots;
    std::atomic<size_t> launched{0}, next{0}, left{0};
    std::atomic<uint8_t>*filled, *emptied;    // [count] the chunk is in its slot / out of it
    uint32_t* want;                           // [count] what the slot's words hold once the device is done with the chunk ...
    int* words;                               // ... and how many do
    std::atomic<int> abort{0};

    bool device_done(size_t c) const { return launched.load(std::memory_order_acquire) > c && slots[c % n_slots]->confirmed(want[c], words[c]); }
};
// A wait's pause: the core is given away, and after a millisecond slept away
struct Pause {
    const std::chrono::steady_clock::time_point start = std::chrono::steady_clock::now();
    void operator()() const {
        if (std::chrono::steady_clock::now() - start < std::chrono::milliseconds(1)) std::this_thread::yield();
        else std::this_thread::sleep_for(std::chrono::microseconds(50));
    }
};
size_t part(size_t bytes, size_t chunk, size_t c) { return bytes - c * chunk < chunk ? bytes - c * chunk : chunk; }

// false: the job was aborted
bool go_up(Job* j, size_t c) {
    if (c >= j->count || !j->up) return true;
    auto free = [&] { return c < j->n_slots || (j->down ? j->emptied[c - j->n_slots].load(std::memory_order_acquire) != 0 : j->device_done(c - j->n_slots)); };
    for (Pause pause; !free(); pause())
        if (j->abort.load()) return false;
    memcpy(j->slots[c % j->n_slots]->host + j->up_at, j->up + c * j->up_chunk, part(j->up_bytes, j->up_chunk, c));
    j->filled[c].store(1, std::memory_order_release);
    return true;
}
bool go_down(Job* j, size_t c) {
    if (c >= j->count || !j->down) return true;
    for (Pause pause; !j->device_done(c); pause())
        if (j->abort.load()) return false;
    memcpy(j->down + c * j->down_chunk, j->slots[c % j->n_slots]->host, part(j->down_bytes, j->down_chunk, c));
    j->emptied[c].store(1, std::memory_order_release);
    j->left.fetch_add(1);
    return true;
}
void work_on(Job* j) {
    for (;;) {
        const size_t k = j->next.fetch_add(1);
        if (k >= 2 * j->count + j->n_slots) return;
        const size_t m = k - j->n_slots;
        if (!(k < j->n_slots ? go_up(j, k) : m % 2 ? go_up(j, m / 2 + j->n_slots) : go_down(j, m / 2))) return;
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

// launch(c, slot, stream, &words): enqueue what the device does with chunk c in slot->host, the last kernel confirming slot->seq + 1 in
// the slot's words; streams are taken in turn, and have no other work to finish first: a job is every other chunked copy's turn too. The
// caller sets the sides of `j` and its count. begun: the slots of the first n_begun chunks, which have been launched (they are released with the
// others). NO_SLOT: nothing was done.
constexpr int NO_SLOT = 1, BEGUN = 3;
template <class Launch>
int run_chunks(Ring* r, Job& j, hipStream_t* streams, size_t n_streams, Slot* const* begun, size_t n_begun, Launch launch) {
    Workers& w = workers();
    std::lock_guard<std::mutex> one(w.one);
    int rc = FHIP_OK;
    Slot* slots[JOB_SLOTS];
    j.slots = slots;
    j.n_slots = 0;
    while (j.n_slots < n_begun) { slots[j.n_slots] = begun[j.n_slots]; j.n_slots++; }
    while (j.n_slots < JOB_SLOTS && j.n_slots < j.count) {
        Slot* q = j.n_slots ? r->take(&rc) : r->get(&rc);
        if (!q) break;
        slots[j.n_slots++] = q;
    }
    if (!rc && !j.n_slots) return NO_SLOT;
    if (!rc) {
        std::vector<std::atomic<uint8_t>> flags(2 * j.count);
        std::vector<uint32_t> want(j.count);
        std::vector<int> words(j.count);
        j.filled = flags.data(); j.emptied = flags.data() + j.count; j.want = want.data(); j.words = words.data();
        for (size_t c = 0; c < n_begun; c++) { want[c] = begun[c]->seq; words[c] = begun[c]->wgs; }
        j.launched.store(n_begun);
        const bool helped = w.post(&j);
        for (size_t c = 0; c < n_begun && !helped && !rc; c++)
            if (!(rc = await_words(begun[c]->done, want[c], words[c], streams[0]))) (void)go_down(&j, c);
        auto wait_for = [&](auto ready) {       // also looks for a device error every few milliseconds: what waits here would wait for ever
            auto look = std::chrono::steady_clock::now();
            for (Pause pause; !ready() && !rc;) {
                pause();
                if (std::chrono::steady_clock::now() - look < std::chrono::milliseconds(5)) continue;
                look = std::chrono::steady_clock::now();
                for (size_t k = 0; k < n_streams && !rc; k++) {
                    const hipError_t e = hipStreamQuery(streams[k]);
                    if (e == hipErrorNotReady) (void)hipGetLastError();
                    else rc = fhip::check_hip(e, "hipStreamQuery");
                }
            }
        };
        for (size_t c = n_begun; c < j.count && !rc; c++) {
            Slot* q = slots[c % j.n_slots];
            hipStream_t s = streams[c % n_streams];
            if (!helped) {                       // without threads the chunks go one by one
                if (c >= j.n_slots) wait_for([&] { return j.device_done(c - j.n_slots); });
                if (!rc) (void)go_up(&j, c);
            } else if (j.up) {
                wait_for([&] { return j.filled[c].load(std::memory_order_acquire) != 0; });
            } else if (c >= j.n_slots) {
                wait_for([&] { return j.emptied[c - j.n_slots].load(std::memory_order_acquire) != 0; });
            }
            int wgs = 0;
            if (rc || (rc = launch(c, q, s, &wgs))) break;
            want[c] = ++q->seq; words[c] = q->wgs = wgs;
            j.launched.store(c + 1, std::memory_order_release);
            if (!helped && !(rc = await_words(q->done, want[c], wgs, s))) (void)go_down(&j, c);
        }
        if (j.down && !rc) wait_for([&] { return j.left.load() >= j.count; });
        if (rc) j.abort.store(1);
        w.finish();
        if (rc)                                 // an enqueued chunk may still use a slot
            for (size_t i = 0; i < n_streams; i++) (void)hipStreamSynchronize(streams[i]);
    }
    for (size_t i = 0; i < j.n_slots; i++) r->release(slots[i]);
    return rc;
}

bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) { (void)hipGetLastError(); return false; }
    return st != hipStreamCaptureStatusNone;
}

// no device memory: the host may touch it (0.1 us)
bool plain_host(const void* h) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, h) == hipSuccess) return a.type != hipMemoryTypeDevice && a.type != hipMemoryTypeArray;
    (void)hipGetLastError();                             // to some versions of the runtime, plain host memory is no pointer of its own
    return true;
}

// whether every page of the range is in memory: a fresh allocation's are made by whoever writes to them first
bool in_memory(const void* h, size_t n) {
    static const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
    const uintptr_t begin = (uintptr_t)h / page * page, pages = ((uintptr_t)h + n - begin + page - 1) / page;
    unsigned char there[D2H_ALONE / 4096 + 2];
    if (page < 4096 || mincore((void*)begin, pages * page, there) != 0) return false;
    unsigned char all = 1;
    for (uintptr_t i = 0; i < pages; i++) all &= there[i];
    return all & 1;
}

// Whether the copy kernels, which look nothing up, may take this copy (*yes): the device side inside one block of the library's on the current device,
// the host side no device memory. Other memory is the runtime's, to copy or to refuse; what leaves one of the library's blocks is refused
// here, since the runtime knows the block of the pool and not what was asked for. (0.15 us)
int for_kernels(const void* d, size_t n, const void* h, const char* who, bool* yes) {
    int dev = 0;
    *yes = false;
    if (const int rc = fhip::check_hip(hipGetDevice(&dev), "hipGetDevice")) return rc;
    const fhip::Place at = fhip::pool_place(d, n, dev);
    if (at == fhip::Place::outside) return fhip::set_error(FHIP_ERR_HIP, "%s: %zu bytes at %p are not within one allocation", who, n, d);
    *yes = at == fhip::Place::inside && plain_host(h);
    return FHIP_OK;
}

// A call that returns what the device has made of it has no place in a capture, where nothing runs: the host would go on with memory that
// nobody has written, and each replay would write to it, or read it, after it is gone. The runtime refuses such a thread its waits.
int may_wait(hipStream_t s, const char* who) {
    if (!fhip::thread_captures() && fhip::runtime_allocates() && !(s && capturing(s))) return FHIP_OK;
    return fhip::set_error(FHIP_ERR_HIP, "%s: waits for the device, which is not permitted while the stream is, or the thread has a stream, in a capture", who);
}

}  // namespace

namespace fhip {

// A source longer than a slot's IN_BYTES in chunks, by the calling thread, one crossing the bus while the next goes into its slot; the last one's words say that all
// have arrived. *took false: there were not enough slots at once, or no pinned memory for them, and nothing was done.
// us on an idle device, the runtime's copy and hipStreamSynchronize | this, of a source that was sent before: 0.66 MB 30 | 30, 1.04 43 | 43, 1.1 64 | 46, 1.5 59 | 54, 1.9 66 | 63, 2.2 91 | 71,
// 3.3 119 | 96, 5.0 154 | 131, 10.4 289 | 253, 12.5 343 | 312; of one that was not: 0.66 34 | 34, 1.04 52 | 46, 1.5 76 | 62, 1.9 87 | 73, 3.3 156 | 118. The first of a process 0.7 MB 6500 | 600,
// 10.4 9700 | 5000, and the runtime's staging memory is slow until 16 MB have gone through it, from whatever call (0.7 MB 290, 1.1 400, 10.4 2300), so that sizes left to it
// are slower the fewer others are: 56 prompt rows of 3072, 600 us a pass, took 842 where only uploads of up to 1 MiB still went that way.
// Two chunks at least: 0.66 MB in one 3 us more. A unit a thread: with four 1.9 MB 8 us more, 5.0 14. hipStreamSynchronize in place of the words 6.
static int upload_chunks(Ring* r, uint8_t* d, const uint8_t* h, size_t n, hipStream_t s, bool* took) {
    const size_t slots = (n + OUT_BYTES - 1) / OUT_BYTES, count = slots < 2 ? 2 : slots, each = ((n + count - 1) / count + 255) & ~(size_t)255;
    Slot* q[SLOTS - SMALL_SLOTS];
    size_t have = 0;
    int rc = FHIP_OK;
    while (have < count) {
        Slot* next = r->take(&rc, SLOTS, SMALL_SLOTS);
        if (!next) break;
        q[have++] = next;
    }
    *took = have == count;
    if (rc) {                               // the runtime's copy needs no slot, nor may the next launch be blamed for it
        (void)hipGetLastError();
        rc = FHIP_OK;
    }
    for (size_t c = 0; c < count && *took && !rc; c++) {
        int wgs = 0;
        const size_t bytes = part(n, each, c);
        memcpy(q[c]->host, h + c * each, bytes);
        if (!(rc = launch_copy(q[c]->host, d + c * each, bytes, 1, q[c]->done, q[c]->seq + 1, s, &wgs))) { q[c]->seq++; q[c]->wgs = wgs; }
    }
    if (*took && !rc) rc = await_words(q[count - 1]->done, q[count - 1]->seq, q[count - 1]->wgs, s);
    for (size_t i = 0; i < have; i++) r->release(q[i]);
    return rc;
}

// Up to a slot's IN_BYTES: the source has been copied when the call returns. Longer sources go through the runtime, which returns when the source has
// been read or is known to be pinned (upload(), which may wait, sends those of up to IN_CHUNKS_TO through slots). A copy in a stream capture stays a copy node; on another stream than the captured one it goes
// through the runtime too, since a slot may have to be made.
int copy_h2d(void* d, const void* h, size_t n, hipStream_t s) {
    int rc;
    bool kernels;
    if ((rc = for_kernels(d, n, h, "fhip_memcpy_h2d", &kernels))) return rc;
    const bool in_capture = capturing(s) || thread_captures();
    Ring* r = n > IN_BYTES || in_capture || !kernels ? nullptr : ring(&rc);
    Slot* q = r ? r->get(&rc) : nullptr;
    if (rc) return rc;
    if (!q) {
        rc = check_hip(hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
        return rc || n > IN_BYTES || in_capture ? rc : check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
    }
    memcpy(q->host, h, n);
    int wgs = 0;
    // One unit a thread while there are workgroups for it: a thread that has three makes three trips over the bus, one after the other. With the wait behind it, us, four units
    // a thread | one: 20 KB 17.8 | 15.8, 64 KB 18.1 | 17.1, 192 KB 21.6 | 20.7, 426 KB 31.2 | 29.3, 608 KB 34.3 | 35.4.
    if (!(rc = launch_copy(q->host, d, n, 1, q->done, q->seq + 1, s, &wgs))) { q->seq++; q->wgs = wgs; }
    r->release(q);
    return rc;
}

// A source of more than IN_BYTES has arrived when this returns, whichever way it went: other streams may use it.
int upload(void* d, const void* h, size_t n, hipStream_t s) {
    int rc = may_wait(s, "fhip_upload");
    if (rc) return rc;
    if (n > IN_BYTES && n <= IN_CHUNKS_TO) {
        bool kernels, took = false;
        if ((rc = for_kernels(d, n, h, "fhip_upload", &kernels))) return rc;
        Ring* r = kernels ? ring(&rc) : nullptr;
        if (r) rc = upload_chunks(r, (uint8_t*)d, (const uint8_t*)h, n, s, &took);
        if (rc || took) return rc;
    }
    rc = copy_h2d(d, h, n, s);
    return rc || n <= IN_BYTES ? rc : check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
}

// by the runtime: pointers that are not for kernels, or no slot
static int copy_d2h_plain(void* h, const void* d, size_t n, hipStream_t s) {
    const int rc = check_hip(hipMemcpyAsync(h, d, n, hipMemcpyDeviceToHost, s), "hipMemcpyAsync D2H");
    return rc ? rc : check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
}

// n bytes into the slot in parts, and out of it as they arrive.
// The host copies out at 30 GB/s what crosses at 53, so the total is the first part's way over and the host's whole copy: parts of 60 KB, at least four. A
// kernel of two thirds and one of the rest | four parts | eight, us on an idle device: 125 KB 15.4 | 13.3 | 16.6, 250 KB 19.3 | 16.5 | 17.7, 432 KB 25.0 |
// 22.8 | 21.7, 593 KB 31.5 | 28.4 | 26.1, 976 KB 45.4 | 41.5 | 39.0.
static int send_parts(Slot* q, const uint8_t* from, size_t n, hipStream_t s, Parts<PARTS>* out) {
    const size_t by_size = n / ((size_t)60 << 10);
    Parts<PARTS> parts{n < IN_PARTS ? 1 : by_size < 4 ? 4 : by_size < PARTS ? (int)by_size : PARTS, {}, {}};
    for (int p = 0; p < parts.count; p++) {
        const bool last = p == parts.count - 1;
        parts.end[p] = last ? n : (n / parts.count * (p + 1) + 255) & ~(size_t)255;
        parts.done[p] = last ? q->done : q->early + p * MAX_WG;
    }
    int wgs = 0;
    const uint32_t seq = q->seq + 1;
    const int rc = parts.count == 1 ? launch_copy(from, q->host, Parts<1>{1, {n}, {q->done}}, MAX_WG, 1, seq, s, &wgs) : launch_copy(from, q->host, parts, MAX_WG, 1, seq, s, &wgs);
    if (!rc) { q->seq = seq; q->wgs = wgs; }
    *out = parts;
    return rc;
}
static int take_parts(Slot* q, uint8_t* h, const Parts<PARTS>& parts, hipStream_t s, Pages* pages = nullptr) {
    int rc = FHIP_OK;
    for (int p = 0; p < parts.count && !rc; p++) {
        const size_t begin = p ? parts.end[p - 1] : 0;
        if (!(rc = await_words(parts.done[p], q->seq, q->wgs, s, p ? nullptr : pages))) memcpy(h + begin, q->host + begin, parts.end[p] - begin);
    }
    return rc;
}
// The same for two and three slots, all sent before the first is taken: up to D2H_ALONE the host by itself is done before the workers are awake. us, idle device, the workers | the
// host, a destination in memory: 1.04 MB 98 | 46, 1.5 99 | 60, 2.0 106 | 72, 2.36 105 | 80, 3.0 113 | 97 (4.0 125 | 131), 2 of them the question. Into fresh memory, whose pages are made on the way, one thread
// takes 0.16 us a KB more and ten share it: 1.04 MB 312 | 205, 1.5 326 | 290, 2.0 350 | 382, 2.36 365 | 450, 3.0 372 | 575. *took false: there were not enough slots at once, and
// nothing was done.
// A destination that is not in memory: its pages are made while the stream gets there; if they are not all there when the first part is, the workers take the slots.
static int copy_d2h_alone(Ring* r, uint8_t* h, const uint8_t* from, size_t n, bool there, hipStream_t s, bool* took) {
    constexpr size_t MOST = D2H_ALONE / OUT_BYTES;
    const size_t count = (n + OUT_BYTES - 1) / OUT_BYTES, each = ((n + count - 1) / count + 255) & ~(size_t)255;
    static_assert(D2H_ALONE % OUT_BYTES == 0 && MOST <= BEGUN, "as many slots as a chunked copy holds while its stream is behind other work");
    Slot* q[MOST];
    Parts<PARTS> parts[MOST];
    size_t have = 0, sent = 0;
    int rc = FHIP_OK;
    while (have < count && !rc) {
        Slot* next = r->take(&rc, JOB_SLOTS);
        if (!next) break;
        q[have++] = next;
    }
    *took = !rc && have == count;
    while (*took && !rc && sent < count) {
        const size_t at = sent * each;
        rc = send_parts(q[sent], from + at, n - at < each ? n - at : each, s, &parts[sent]);
        if (!rc) sent++;
    }
    Pages pages(h, n);
    if (*took && !rc && !there) {
        if (!(rc = await_words(parts[0].done[0], q[0]->seq, q[0]->wgs, s, &pages)) && !pages.made()) {
            Job j{};
            j.count = count;
            j.down = h; j.down_bytes = n; j.down_chunk = each;
            return run_chunks(r, j, &s, 1, q, count, [](size_t, Slot*, hipStream_t, int*) { return (int)FHIP_OK; });   // (everything has been launched)
        }
    }
    for (size_t i = 0; i < sent && !rc; i++) rc = take_parts(q[i], h + i * each, parts[i], s, i ? nullptr : &pages);
    if (rc && sent) (void)hipStreamSynchronize(s);      // an enqueued part may still use a slot
    for (size_t i = 0; i < have; i++) r->release(q[i]);
    return rc;
}

int copy_d2h(void* h, const void* d, size_t n, hipStream_t s) {
    int rc, wgs = 0;
    if ((rc = may_wait(s, "fhip_memcpy_d2h"))) return rc;
    bool kernels;
    if ((rc = for_kernels(d, n, h, "fhip_memcpy_d2h", &kernels))) return rc;
    if (!kernels) return copy_d2h_plain(h, d, n, s);
    Ring* r = ring(&rc);
    if (!r) return rc;
    const uint8_t* from = (const uint8_t*)d;
    if (n > OUT_BYTES && n <= D2H_ALONE) {
        bool took;
        if ((rc = copy_d2h_alone(r, (uint8_t*)h, from, n, n <= D2H_ALONE_NEW || in_memory(h, n), s, &took)) || took) return rc;
    }
    if (n > OUT_BYTES) {
        Job j{};
        j.count = (n + CHUNK - 1) / CHUNK;
        j.down = (uint8_t*)h; j.down_bytes = n; j.down_chunk = CHUNK;
        auto launch = [&](size_t c, Slot* to, hipStream_t st, int* w) {
            return launch_copy(from + c * CHUNK, to->host, part(n, CHUNK, c), 4, to->done, to->seq + 1, st, w);
        };
        // what the stream still has to do is waited for here, with the first chunk, and not by the workers and in front of other copies (hipStreamSynchronize in
        // its place: 8 us more of a 1.6 MB copy from an idle stream's 86); two more are on their way meanwhile, or the bus would wait too
        Slot* begun[BEGUN];
        size_t n_begun = 0;
        while (n_begun < BEGUN && n_begun < j.count && !rc) {
            Slot* q = n_begun ? r->take(&rc) : r->get(&rc);
            if (!q) break;
            begun[n_begun] = q;
            if (!(rc = launch(n_begun++, q, s, &wgs))) { q->seq++; q->wgs = wgs; }
        }
        if (!rc && !n_begun) return copy_d2h_plain(h, d, n, s);
        Pages pages(h, n);
        if (!rc) rc = await_words(begun[0]->done, begun[0]->seq, begun[0]->wgs, s, &pages);
        if (!rc) return run_chunks(r, j, &s, 1, begun, n_begun, launch);
        (void)hipStreamSynchronize(s);              // an enqueued chunk may still use a slot
        for (size_t i = 0; i < n_begun; i++) r->release(begun[i]);
        return rc;
    }
    Slot* q = r->get(&rc);
    if (!q) return rc ? rc : copy_d2h_plain(h, d, n, s);
    Parts<PARTS> parts;
    Pages pages(h, n);
    if (!(rc = send_parts(q, from, n, s, &parts))) rc = take_parts(q, (uint8_t*)h, parts, s, &pages);
    r->release(q);
    return rc;
}

// dequant_host with no slot to be had, or with device memory for a host side: a slot's worth of device memory kept for it, `per` blocks at a time, and the runtime's copies
static int dequant_plain(Ring* r, uint32_t type, const uint8_t* h_raw, size_t nb, size_t per, size_t vals, size_t bytes, float* h_out) {
    std::lock_guard<std::mutex> one(r->spare_mu);
    hipStream_t s = r->stream[0];
    int rc = FHIP_OK;
    if (!r->spare && (rc = device_malloc((void**)&r->spare, SLOT_BYTES, "hipMalloc"))) { r->spare = nullptr; return rc; }
    for (size_t b = 0; b < nb && !rc; b += per) {
        const size_t n = nb - b < per ? nb - b : per;
        if ((rc = check_hip(hipMemcpyAsync(r->spare + OUT_BYTES, h_raw + b * bytes, n * bytes, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D"))) break;
        if ((rc = launch_dequant(type, r->spare + OUT_BYTES, n, (float*)r->spare, s))) break;
        rc = copy_d2h_plain(h_out + b * vals, r->spare, n * vals * sizeof(float), s);
    }
    return rc;
}

// nb blocks (bytes each, vals values) of host memory to nb * vals floats of host memory: chunk by chunk a worker copies the bytes into a slot, one kernel takes
// them out of it and leaves the floats there, and a worker copies those out. Two streams, so that one chunk's bytes come up while the floats of the one
// before go down.
int dequant_host(uint32_t type, const uint8_t* h_raw, size_t nb, size_t vals, size_t bytes, float* h_out) {
    int rc;
    if ((rc = may_wait(nullptr, "fhip_deq_raw"))) return rc;
    Ring* r = ring(&rc);
    if (!r) return rc;
    {
        std::lock_guard<std::mutex> lock(r->mu);
        for (auto& st : r->stream)
            if (!st && (rc = check_hip(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate"))) { st = nullptr; return rc; }
    }
    const size_t per = CHUNK / sizeof(float) / vals, out_chunk = per * vals * sizeof(float);   // blocks of a chunk, and their floats
    const size_t n = nb * vals * sizeof(float);
    if (!plain_host(h_raw) || !plain_host(h_out)) return dequant_plain(r, type, h_raw, nb, per, vals, bytes, h_out);
    static_assert(CHUNK / sizeof(float) <= (size_t)4096 * MAX_WG, "a chunk's workgroups have a word each");
    auto launch = [&](size_t c, Slot* q, hipStream_t s, int* wgs) {
        return launch_dequant_through(type, q->host + OUT_BYTES, nb - c * per < per ? nb - c * per : per, (float*)q->host, q->done, q->seq + 1, s, wgs);
    };
    if (nb > per) {
        Job j{};
        j.count = (nb + per - 1) / per;
        j.up = h_raw; j.up_bytes = nb * bytes; j.up_chunk = per * bytes; j.up_at = OUT_BYTES;
        j.down = (uint8_t*)h_out; j.down_bytes = n; j.down_chunk = out_chunk;
        rc = run_chunks(r, j, r->stream, 2, nullptr, 0, launch);
        return rc == NO_SLOT ? dequant_plain(r, type, h_raw, nb, per, vals, bytes, h_out) : rc;
    }
    Slot* q = r->get(&rc);
    if (!q) return rc ? rc : dequant_plain(r, type, h_raw, nb, per, vals, bytes, h_out);
    int wgs = 0;
    memcpy(q->host + OUT_BYTES, h_raw, nb * bytes);
    if (!(rc = launch(0, q, r->stream[0], &wgs))) {
        q->seq++; q->wgs = wgs;
        if (!(rc = await_words(q->done, q->seq, wgs, r->stream[0]))) memcpy(h_out, q->host, n);
    }
    r->release(q);
    return rc;
}

}  // namespace fhip
