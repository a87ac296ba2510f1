// nuosc_xfer.h -- host <-> device transfers of fields through pinned slots.
//
// A caller's arrays are ordinary (pageable) memory.  Copied by the runtime
// they cost a device staging buffer of the same size and pass one bounce
// buffer on one thread, 10-13 GB/s into freshly allocated arrays, whose pages
// are first touched there.  Here the pack kernel writes FP64 values straight
// into a pinned slot over the bus (measured 50-54 GB/s in 2-8 MB pieces; a
// slot read by the unpack kernel: 49-53 GB/s), and several threads, one slot
// each, move the slots to or from the caller's array meanwhile.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <functional>

namespace nuosc {

constexpr size_t kSlotBytes = 4u << 20;
constexpr int kXferThreads = 8;   // of the 16 slots a device may hold: two large transfers at once

// Handles that may transfer: the slots are freed when the last one goes.
void xfer_retain();
void xfer_release();

// Threads for a transfer of this many bytes, the caller's included.  Each one
// more may have to wait its turn of the scheduler (about 3 ms) where the caller's
// program keeps every core busy, and the transfer ends with its last thread; into
// new pages they also get in each other's way.  8 MB with the workers of a thread
// pool spinning: 2.8 ms with eight threads, 0.60 with two, 0.47 with one (0.69 by
// the runtime's copy); nine of 3-8 MB into new arrays: 8.6 ms with two, 2.9 with
// one (5.9).  92 MB: 10.5 ms with one, 7.3 with two, 4.3 with eight.
inline int xfer_threads(long long bytes) { return bytes < (32 << 20) ? 1 : kXferThreads; }

// Moves nchunks chunks, on up to this many threads.  down: enqueue(c, slot) queues work on s that fills
// slot, then host(c, slot) runs once it is done; up: host(c, slot) fills the
// slot, then enqueue(c, slot) queues the work that reads it.  Returns when
// all of it is done; an error (also of a chunk not started because of it) is
// returned, hipErrorOutOfMemory if no slot can be had, with nothing left queued on s.
hipError_t xfer_run(int device, hipStream_t s, long long nchunks, int nthreads, bool down,
                    const std::function<hipError_t(long long, void*)>& enqueue,
                    const std::function<void(long long, void*)>& host);

}  // namespace nuosc
