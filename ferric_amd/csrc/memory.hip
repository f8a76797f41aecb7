// Device memory of the library (fhip_malloc / fhip_free): freed blocks are kept for the next allocation of their size class.
//
// hipFree waits for the device, and a block of more than a few megabytes is mapped and unmapped on every call. An operator that
// allocates its output (and perhaps scratch) per call therefore paid a full drain of the queue per call, and the large ones the
// page tables of hundreds of megabytes: a 2048-row feed-forward block of 1.1 ms of kernels took 4.8 to 10.6 ms, a 5 us mat-vec 20 us.
//
// What hipFree's wait gave callers is kept: a freed block may still be in use by work enqueued on any stream, this library's or
// another's, so it is not handed out again before the device has been idle once since the free. Freed blocks collect on a `dirty`
// list; when an allocation finds no clean block and its class already holds keep_blocks() dirty ones, one wait for the device
// turns every dirty block of the device clean. Until then the class grows, so the wait comes once in up to 64 calls for small
// blocks and once in two for the largest, instead of at every free. A class of large blocks whose last free lies a millisecond back
// is drained at once instead of grown: the queue has most likely run empty since, and a new block would have to be mapped.
#include "hostmem.hpp"

#include <atomic>
#include <chrono>
#include <map>
#include <mutex>
#include <vector>

namespace {

constexpr size_t WEIGHT_SLACK = fhip::WEIGHT_SLACK;
constexpr size_t POOL_BLOCK_MAX = (size_t)768 << 20;   // larger blocks (weights, mostly) are freed at once
constexpr size_t POOL_CACHED_MAX = (size_t)2 << 30;    // cached bytes per device; beyond it the classes unused longest are freed
constexpr size_t LARGE = (size_t)1 << 20;              // blocks whose mapping costs more than a wait for an idle device
constexpr int MAX_DEVICES = 64;

// Every block fhip_malloc has from the runtime, in use or cached: a free has to know the ones that are free already.
struct Block {
    size_t asked, cls;                                 // cls: bytes there are
    int dev;
    bool pooled, live;
};
typedef std::map<uintptr_t, Block> Blocks;             // by address: fhip_weight_wrap_device looks up ranges
typedef std::vector<Blocks::iterator> Cached;
struct SizeClass {
    Cached clean, dirty;
    uint64_t last_use = 0;
    std::chrono::steady_clock::time_point last_free;
};
struct Pool {
    std::mutex mu;
    Blocks blocks;
    std::map<size_t, SizeClass> classes[MAX_DEVICES];
    size_t cached[MAX_DEVICES] = {};
    uint64_t clock = 0;
};
// never destroyed: objects of a host program may be freed after static destructors have begun to run
Pool& pool() { static Pool* p = new Pool(); return *p; }

// the calling thread's device; a process that sees one only is not asked every time (50 ns)
hipError_t current_device(int* dev) {
    static const bool one = [] { int n = 0; return hipGetDeviceCount(&n) == hipSuccess && n == 1; }();
    *dev = 0;
    return one ? hipSuccess : hipGetDevice(dev);
}

// The captures that fhip_graph_capture_begin opened and that have not ended, each with the thread it belongs to (the runtime lets no
// other thread end it). A thread that captures may not wait for the device nor map or unmap memory: the runtime refuses and
// invalidates the capture, and the stream then takes no work until it has been through another capture.
struct Captures {
    std::mutex mu;
    std::map<hipStream_t, uint64_t> owner;
    std::atomic<size_t> open{0};                       // = owner.size(), for threads that only want to know that there is none
};
Captures& captures() { static Captures* c = new Captures(); return *c; }
uint64_t this_thread() {
    static std::atomic<uint64_t> last{0};
    thread_local const uint64_t id = ++last;
    return id;
}

// Eight classes per power of two: at most an eighth of a block is not asked for. n: up to POOL_BLOCK_MAX, which is a class of its own.
size_t size_class(size_t n) {
    if (n <= 1024) return 1024;
    const int top = 63 - __builtin_clzll((unsigned long long)n - 1);   // 2^top < n <= 2^(top + 1)
    const size_t step = (size_t)1 << (top - 3);
    return (n + step - 1) / step * step;
}

// Dirty blocks a class may hold before an allocation waits for the device: 128 MiB of them, 2 to 64. A wait costs about 10 us and
// the gap behind it about as much, so a caller of microsecond kernels wants tens of calls between waits, while a class of
// hundreds of megabytes belongs to calls of a millisecond.
size_t keep_blocks(size_t cls) {
    const size_t k = ((size_t)128 << 20) / cls;
    return k < 2 ? 2 : (k > 64 ? 64 : k);
}

// Under p.mu: blocks out of the classes of `dev` that were unused longest, until at most `target` bytes stay cached. They are no blocks
// of the pool any more.
void take_oldest(Pool& p, int dev, size_t target, std::vector<void*>& out) {
    auto& cs = p.classes[dev];
    while (p.cached[dev] > target) {
        SizeClass* oldest = nullptr;
        size_t bytes = 0;
        for (auto& c : cs)
            if ((!c.second.clean.empty() || !c.second.dirty.empty()) && (!oldest || c.second.last_use < oldest->last_use)) {
                oldest = &c.second;
                bytes = c.first;
            }
        if (!oldest) return;
        for (auto* list : {&oldest->clean, &oldest->dirty})
            while (!list->empty() && p.cached[dev] > target) {
                out.push_back((void*)list->back()->first);
                p.blocks.erase(list->back());
                list->pop_back();
                p.cached[dev] -= bytes;
            }
    }
}

}  // namespace

namespace fhip {

void capture_begun(hipStream_t s) {
    Captures& c = captures();
    std::lock_guard<std::mutex> lock(c.mu);
    c.owner[s] = this_thread();
    c.open = c.owner.size();
}

void capture_ended(hipStream_t s, bool destroyed) {
    Captures& c = captures();
    if (c.open.load() == 0) return;
    std::lock_guard<std::mutex> lock(c.mu);
    auto it = c.owner.find(s);
    if (it == c.owner.end() || (!destroyed && it->second != this_thread())) return;
    c.owner.erase(it);
    c.open = c.owner.size();
}

bool thread_captures() {
    Captures& c = captures();
    if (c.open.load(std::memory_order_relaxed) == 0) return false;
    std::lock_guard<std::mutex> lock(c.mu);
    bool any = false;
    for (auto it = c.owner.begin(); it != c.owner.end();) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (it->second != this_thread()) { ++it; continue; }
        if (hipStreamIsCapturing(it->first, &st) != hipSuccess) (void)hipGetLastError();
        if (st == hipStreamCaptureStatusNone) { it = c.owner.erase(it); continue; }   // ended or destroyed through the runtime itself
        any = true;
        ++it;
    }
    c.open = c.owner.size();
    return any;
}

void pool_trim() {
    if (thread_captures() || !runtime_allocates()) return;   // hipFree would refuse, and the blocks would be nobody's
    Pool& p = pool();
    std::vector<void*> out;
    {
        std::lock_guard<std::mutex> lock(p.mu);
        for (int d = 0; d < MAX_DEVICES; d++) take_oldest(p, d, 0, out);
    }
    for (void* q : out) (void)hipFree(q);   // hipFree waits for whatever still uses the block
}

// Until all work enqueued on the device has ended. hipDeviceSynchronize fails while any thread of the process captures, and invalidates the
// capture: it is called where the library knows of none, and none can begin under the lock. Beside a capture it is hipFree's own wait, which
// the runtime permits, but which comes back only when the runtime has retired every launch (61 mat-vecs of 4.4 us: 52 us with the one, 104 - 110
// with the other; taken everywhere it cost 5 - 10 % of calls of 6 - 22 us that allocate their output).
static hipError_t device_wait() {
    {
        Captures& c = captures();
        std::lock_guard<std::mutex> lock(c.mu);
        if (c.owner.empty()) {
            const hipError_t e = hipDeviceSynchronize();
            if (e != hipErrorStreamCaptureUnsupported) return e;
            (void)hipGetLastError();                   // another thread captures through the runtime
        }
    }
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, 256);
    return e == hipSuccess ? hipFree(p) : e;
}

// A cached block must not go where a new one could not: a thread that captures a stream through the runtime itself would have a graph go
// on using scratch that its operator has freed. Only this thread's captures count: in the mode a thread has unless told otherwise the question would
// be refused for another thread's global capture too, and invalidate it. (0.2 us)
bool runtime_allocates() {
    hipStreamCaptureMode mode = hipStreamCaptureModeThreadLocal;
    void* none = nullptr;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t e = hipMalloc(&none, 0);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

int device_malloc(void** out, size_t n, const char* what) {
    hipError_t e = hipMalloc(out, n);
    if (e == hipErrorOutOfMemory) {         // what the pool holds back may be what is missing
        (void)hipGetLastError();
        pool_trim();
        e = hipMalloc(out, n);
    }
    return check_hip(e, what);
}

// A refused hipMalloc would invalidate the captures that refuse it; in this mode none does (the memory is no part of a graph).
void* device_malloc_beside_captures(size_t n) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    void* p = nullptr;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t e = hipMalloc(&p, n);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}

int pool_malloc(void** out, size_t nbytes) {
    *out = nullptr;
    if (thread_captures())
        return set_error(FHIP_ERR_HIP, "fhip_malloc: not while the thread captures a stream (the graph would go on using the memory after it is freed): allocate "
                         "before the capture begins");
    if (nbytes > SIZE_MAX - WEIGHT_SLACK) return check_hip(hipErrorOutOfMemory, "fhip_malloc");
    const size_t need = nbytes + WEIGHT_SLACK;
    int dev = 0;
    int rc = check_hip(current_device(&dev), "hipGetDevice");
    if (rc) return rc;
    Pool& p = pool();
    if (need > POOL_BLOCK_MAX || dev >= MAX_DEVICES) {
        if ((rc = device_malloc(out, need, "hipMalloc"))) return rc;
        std::lock_guard<std::mutex> lock(p.mu);
        p.blocks[(uintptr_t)*out] = Block{nbytes, need, dev, false, true};
        return FHIP_OK;
    }
    const size_t cls = size_class(need);
    const bool cached = runtime_allocates();           // otherwise the runtime is asked for a new block, and says why not
    for (bool waited = false; cached;) {
        std::vector<std::pair<size_t, Cached>> dirty;
        {
            std::lock_guard<std::mutex> lock(p.mu);
            SizeClass& c = p.classes[dev][cls];
            c.last_use = ++p.clock;
            if (!c.clean.empty()) {
                Blocks::iterator b = c.clean.back();
                c.clean.pop_back();
                p.cached[dev] -= cls;
                b->second.asked = nbytes;
                b->second.live = true;
                *out = (void*)b->first;
                return FHIP_OK;
            }
            if (waited || c.dirty.empty()) break;
            if (c.dirty.size() < keep_blocks(cls) &&
                (cls < LARGE || std::chrono::steady_clock::now() - c.last_free < std::chrono::milliseconds(1))) break;
            // every dirty block of the device leaves its list while the lock is given up for the wait: another thread that
            // comes for one of them meanwhile makes a new block
            for (auto& k : p.classes[dev])
                if (!k.second.dirty.empty()) {
                    dirty.emplace_back(k.first, Cached());
                    dirty.back().second.swap(k.second.dirty);
                }
        }
        const hipError_t e = device_wait();
        std::lock_guard<std::mutex> lock(p.mu);
        for (auto& d : dirty) {
            SizeClass& c = p.classes[dev][d.first];
            auto& to = e != hipSuccess ? c.dirty : c.clean;
            to.insert(to.end(), d.second.begin(), d.second.end());
        }
        if (e == hipErrorOutOfMemory) { (void)hipGetLastError(); break; }   // device_malloc gives back what is cached
        if (e != hipSuccess) return check_hip(e, "waiting for the device");
        waited = true;
    }
    if ((rc = device_malloc(out, cls, "hipMalloc"))) return rc;
    std::lock_guard<std::mutex> lock(p.mu);
    p.blocks[(uintptr_t)*out] = Block{nbytes, cls, dev, true, true};
    return FHIP_OK;
}

int pool_free(void* ptr) {
    Pool& p = pool();
    std::vector<void*> over;
    {
        std::lock_guard<std::mutex> lock(p.mu);
        auto it = p.blocks.find((uintptr_t)ptr);
        if (it == p.blocks.end()) {
            over.push_back(ptr);            // not of fhip_malloc: the runtime knows it, or says that it does not
        } else if (!it->second.live) {
            return set_error(FHIP_ERR_ARG, "fhip_free: the block has been freed already");
        } else if (!it->second.pooled) {
            p.blocks.erase(it);
            over.push_back(ptr);
        } else {
            Block& b = it->second;
            b.live = false;
            SizeClass& c = p.classes[b.dev][b.cls];
            c.dirty.push_back(it);
            c.last_use = ++p.clock;
            if (b.cls >= LARGE) c.last_free = std::chrono::steady_clock::now();
            p.cached[b.dev] += b.cls;
            if (p.cached[b.dev] > POOL_CACHED_MAX && !thread_captures() && runtime_allocates()) take_oldest(p, b.dev, POOL_CACHED_MAX, over);
        }
    }
    int rc = FHIP_OK;
    for (void* q : over) {
        const int r = check_hip(hipFree(q), "hipFree");
        if (r) rc = r;
    }
    return rc;
}

bool pool_range(const void* ptr, uintptr_t* base, uintptr_t* end) {
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.mu);
    auto it = p.blocks.upper_bound((uintptr_t)ptr);
    if (it == p.blocks.begin()) return false;
    --it;
    if (!it->second.live || (uintptr_t)ptr >= it->first + it->second.cls) return false;
    *base = it->first;
    *end = it->first + it->second.asked + WEIGHT_SLACK;
    return true;
}

Place pool_place(const void* ptr, size_t n, int dev) {
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.mu);
    auto it = p.blocks.upper_bound((uintptr_t)ptr);
    if (it == p.blocks.begin()) return Place::elsewhere;
    const Block& b = (--it)->second;
    const size_t at = (uintptr_t)ptr - it->first, size = b.asked + WEIGHT_SLACK;
    if (at >= b.cls) return Place::elsewhere;
    if (!b.live || at > size || n > size - at) return Place::outside;
    return b.dev == dev ? Place::inside : Place::elsewhere;
}

}  // namespace fhip
