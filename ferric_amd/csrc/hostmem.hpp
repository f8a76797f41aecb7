// Device memory and host <-> device copies of the library, as its other translation units see them.
#pragma once
#include "common.hpp"

namespace fhip {

// memory.hip: the library's device memory
constexpr size_t WEIGHT_SLACK = 256;   // readable bytes every weight and every block of fhip_malloc has behind its last byte
int pool_malloc(void** out, size_t nbytes);
int pool_free(void* ptr);
void pool_trim();                      // gives every cached block back
void capture_begun(hipStream_t s);                       // the calling thread is about to open a capture of s ...
void capture_ended(hipStream_t s, bool destroyed);       // ... and has ended it or failed to, or (any thread) the stream goes; nothing if it is another thread's
bool thread_captures();                                  // the calling thread has a capture open (of those)
bool runtime_allocates();                                // the runtime permits the calling thread to allocate and to wait: it has no capture open at all
bool pool_range(const void* ptr, uintptr_t* base, uintptr_t* end);   // the block in use that ptr lies in, as far as it was asked for
// n bytes from ptr on: inside one block in use of device dev; outside: they start in a block of fhip_malloc, but it is free, or they run past what was
// asked for (and the slack); elsewhere: nothing of fhip_malloc's, or another device's
enum class Place { inside, outside, elsewhere };
Place pool_place(const void* ptr, size_t n, int dev);
int device_malloc(void** out, size_t n, const char* what);           // hipMalloc; with no memory left, once more after pool_trim
void* device_malloc_beside_captures(size_t n);                       // hipMalloc also while threads have captures open, which it leaves as they are; null: no memory

// transfer.hip: copies through pinned memory of the library's own; both directions and the host-to-host unpackers
constexpr size_t H2D_STAGED = (size_t)640 << 10;   // up to here copy_h2d has read its source when it returns
int copy_h2d(void* d, const void* h, size_t n, hipStream_t s);
int upload(void* d, const void* h, size_t n, hipStream_t s);     // copy_h2d that has read its source when it returns, and from H2D_STAGED on brought it over; refused in a capture
int copy_d2h(void* h, const void* d, size_t n, hipStream_t s);   // synchronises; refused in a capture
int dequant_host(uint32_t type, const uint8_t* h_raw, size_t nblocks, size_t block_values, size_t block_bytes, float* h_out);   // synchronises

// dequant.hip: nblocks blocks of pinned host memory, which is read up to the next 16 bytes, to floats of pinned host memory; workgroup w < *wgs stores seq in done[w] when what it
// writes has arrived. Both 16-byte aligned, at most 4096 values a word of `done`.
int launch_dequant_through(uint32_t type, const uint8_t* pinned_raw, size_t nblocks, float* pinned_out, uint32_t* done, uint32_t seq, hipStream_t s, int* wgs);

}  // namespace fhip
