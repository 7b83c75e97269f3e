// Scratch blocks of streams and of captured graphs (stream_scratch.hpp). Host code.
//
// A stream's own block serves every launch on that stream: launches on a stream run one after another, so a block is free for
// the next user as soon as the previous user's last launch has been queued. It is never recorded into a graph. An outgrown
// block may still be read by queued kernels and is kept until release_stream_scratch; blocks double, so what is kept of them
// adds up to less than the bound on one block again.

#include <cstdlib>
#include <map>
#include <new>
#include <tuple>
#include <vector>

#include "stream_scratch.hpp"

namespace fth {
namespace {

struct Block {
    void *ptr = nullptr;
    size_t bytes = 0;
};
using CaptureKey = std::tuple<unsigned long long, hipStream_t, int>;  // launches of one capture on one stream are ordered

struct State {
    std::mutex mu;
    std::map<std::pair<hipStream_t, int>, Block> own;
    std::vector<Block> outgrown;
    std::map<CaptureKey, Block> captured;                           // the block to use next
    std::multimap<unsigned long long, Block> capture_blocks;        // every block of a capture
    uint64_t own_bytes = 0, outgrown_bytes = 0, capture_bytes = 0;
};
State &state() {
    static State *s = new State();  // never destroyed: streams outlive static destructors
    return *s;
}

// FT_HIP_STREAM_SCRATCH (testing): 0 = no scratch is ever given, 2 = every allocation is refused by the driver, 3 = none is given
// inside captures.
int knob() {
    static const int v = [] {
        const char *e = std::getenv("FT_HIP_STREAM_SCRATCH");
        return e ? std::atoi(e) : 1;
    }();
    return v;
}

// hipMalloc that leaves no error behind.
void *try_malloc(size_t bytes) {
    const AllocateInCapture allow;
    void *p = nullptr;
    if (hipMalloc(&p, knob() == 2 ? (size_t)1 << 50 : bytes) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
    }
    return p;
}

// The capture state of `st`; false when it cannot be told or the capture is broken.
bool capture_of(hipStream_t st, unsigned long long *id) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    *id = 0;
    if (hipStreamGetCaptureInfo_v2(st, &status, id, nullptr, nullptr, nullptr) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (status == hipStreamCaptureStatusNone) *id = 0;
    return status != hipStreamCaptureStatusInvalidated;
}

}  // namespace

AllocateInCapture::AllocateInCapture() : changed_(hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess) {
    if (!changed_) (void)hipGetLastError();
}
AllocateInCapture::~AllocateInCapture() {
    if (changed_ && hipThreadExchangeStreamCaptureMode(&mode_) != hipSuccess) (void)hipGetLastError();
}

StreamScratch::StreamScratch() : lock_(state().mu) {}

void *StreamScratch::get(hipStream_t st, ScratchUse use, size_t bytes) try {
    State &s = state();
    unsigned long long id = 0;
    if (knob() == 0 || bytes > kStreamScratchMost || st == hipStreamPerThread || !capture_of(st, &id) || (id && knob() == 3)) return nullptr;
    Block &b = id ? s.captured[CaptureKey(id, st, (int)use)] : s.own[std::make_pair(st, (int)use)];
    if (b.bytes >= bytes) return b.ptr;
    size_t want = 2 * b.bytes < kStreamScratchMost ? 2 * b.bytes : kStreamScratchMost;
    if (want < bytes) want = bytes;
    if (id && s.capture_bytes + want > kCaptureScratchMost) want = bytes;
    if (id && s.capture_bytes + want > kCaptureScratchMost) return nullptr;
    // room for the book-keeping first, so that nothing is lost if the host has none
    if (!id) s.outgrown.reserve(s.outgrown.size() + 1);
    auto it = id ? s.capture_blocks.emplace(id, Block{}) : s.capture_blocks.end();
    void *p = try_malloc(want);
    if (!p && want != bytes) p = try_malloc(want = bytes);
    if (!p) {
        if (id) s.capture_blocks.erase(it);
        return nullptr;
    }
    if (id) {
        it->second = Block{p, want};
        s.capture_bytes += want;
    } else {
        if (b.ptr) {
            s.outgrown.push_back(b);  // (reserved above)
            s.outgrown_bytes += b.bytes;
            s.own_bytes -= b.bytes;
        }
        s.own_bytes += want;
    }
    b = Block{p, want};
    return p;
} catch (const std::bad_alloc &) {
    return nullptr;
}

unsigned long long capture_id(hipStream_t st) {
    unsigned long long id = 0;
    return capture_of(st, &id) ? id : 0;
}

void release_capture_scratch(unsigned long long id) {
    State &s = state();
    std::lock_guard<std::mutex> lock(s.mu);
    const auto range = s.capture_blocks.equal_range(id);
    for (auto it = range.first; it != range.second; ++it) {
        (void)hipFree(it->second.ptr);
        s.capture_bytes -= it->second.bytes;
    }
    s.capture_blocks.erase(range.first, range.second);
    s.captured.erase(s.captured.lower_bound(CaptureKey(id, nullptr, 0)), s.captured.lower_bound(CaptureKey(id + 1, nullptr, 0)));
}

void release_stream_scratch() {
    State &s = state();
    std::lock_guard<std::mutex> lock(s.mu);
    if (s.own.empty() && s.outgrown.empty()) return;
    if (hipDeviceSynchronize() != hipSuccess) {  // a capture forbids it, for instance: keep everything
        (void)hipGetLastError();
        return;
    }
    for (auto &kv : s.own) (void)hipFree(kv.second.ptr);
    for (Block &b : s.outgrown) (void)hipFree(b.ptr);
    s.own.clear();
    s.outgrown.clear();
    s.own_bytes = s.outgrown_bytes = 0;
}

void stream_scratch_stats(uint64_t *live, uint64_t *retired) {
    State &s = state();
    std::lock_guard<std::mutex> lock(s.mu);
    *live = s.own_bytes + s.capture_bytes;
    *retired = s.outgrown_bytes;
}

}  // namespace fth
