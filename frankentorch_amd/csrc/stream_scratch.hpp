// Optional scratch memory for kernels that hand data to the next launch on the same stream.
#pragma once

#include <mutex>

#include "common.hpp"

namespace fth {

enum class ScratchUse { SplitPlanes, DecodeShares };

constexpr size_t kStreamScratchMost = (size_t)1 << 30;    // one request, and one block
constexpr size_t kCaptureScratchMost = (size_t)4 << 30;   // all blocks that captured graphs hold

// Held from the request for scratch until the last launch that uses it: another thread's launches on the same stream do not
// come between the writer and its readers.
class StreamScratch {
   public:
    StreamScratch();
    // A block of at least `bytes` for launches on `st`, or NULL when it cannot be had: more than kStreamScratchMost, no memory
    // (the device is not drained for it and no error is left behind), hipStreamPerThread (one handle for another stream in
    // every thread). Outside a capture the block is the stream's own, kept and grown. A capture gets a block that nothing else
    // uses, since its graph may be replayed on any stream beside anything: kept until release_capture_scratch, otherwise for
    // good, and NULL once kCaptureScratchMost is held.
    void *get(hipStream_t st, ScratchUse use, size_t bytes);

   private:
    std::lock_guard<std::mutex> lock_;
};

// While it lives, this thread may allocate beside and inside its own stream captures.
class AllocateInCapture {
   public:
    AllocateInCapture();
    ~AllocateInCapture();
    AllocateInCapture(const AllocateInCapture &) = delete;
    AllocateInCapture &operator=(const AllocateInCapture &) = delete;

   private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool changed_;
};

// The capture that `st` is recording, 0 for none.
unsigned long long capture_id(hipStream_t st);
// Frees what the capture was given. Its graph and executables are gone and none of their replays is running.
void release_capture_scratch(unsigned long long id);
// Frees every stream's own blocks (drains the device first); captured graphs keep theirs.
void release_stream_scratch();
void stream_scratch_stats(uint64_t *live, uint64_t *retired);

}  // namespace fth
