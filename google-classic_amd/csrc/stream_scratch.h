// stream_scratch.h -- scratch of a call on the library stream.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

namespace holo {

// Scratch for the launches of one call, from its construction to its
// destruction, in stream order.  Kept per stream, so calls on several streams
// never share it: up to 512 KiB a part of an arena that cuda_init allocates (so
// a decode attention allocates nothing, also while another stream is captured),
// above that a buffer, for up to 8 streams; a further stream takes over the
// least recently used buffer once the device is idle.  The pool's lock
// is held meanwhile, so calls of several threads on one stream run one after
// the other.  (Stream-ordered allocations instead cost about 10 us of host time
// a call.)  Under capture a part of the arena that is the graph's own (a
// graph must not hold the stream's scratch, which eager calls use too and
// another stream may take over), or, past 1 MiB or with the arena full, a
// stream-ordered allocation (whose nodes cost a replay about 15 us a call: 32
// decode attentions at 600 positions 196 us, with them 673).
class StreamScratch {
public:
    explicit StreamScratch(size_t bytes);
    ~StreamScratch();
    StreamScratch(const StreamScratch &) = delete;
    StreamScratch &operator=(const StreamScratch &) = delete;
    void *get() const { return buf_; }  // nullptr: no memory

private:
    std::unique_lock<std::mutex> lock_;
    void *buf_ = nullptr;
    bool free_ = false;  // a stream-ordered allocation
};

bool stream_scratch_init();  // the arena
void stream_scratch_release();  // all of it
void stream_scratch_drop(hipStream_t st);  // a stream's, before it is destroyed
// A graph's parts of the arena, by the id of its capture: captures that end in
// holo_graph_destroy give them back; of others they stay taken.
void stream_scratch_drop_capture(unsigned long long id);
void stream_scratch_reclaim();  // what a drop under an open capture left

}  // namespace holo
