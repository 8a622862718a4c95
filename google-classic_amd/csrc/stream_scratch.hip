// stream_scratch.hip -- the kept scratch buffers of stream_scratch.h.
#include "stream_scratch.h"
#include "common.h"

#include <algorithm>
#include <vector>

namespace holo {

namespace {

struct Slot {
    hipStream_t stream;
    int dev;
    void *buf;
    size_t bytes;
    uint64_t used;  // 0: free
};
constexpr int kSlots = 8;
std::mutex g_mu;
Slot g_slots[kSlots];
uint64_t g_clock = 0;

// A buffer of at least `bytes` for the library stream; nullptr when there is
// no memory.  g_mu is held.
void *slot(size_t bytes)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    Slot *s = nullptr, *old = &g_slots[0];
    for (Slot &t : g_slots) {
        if (t.used && t.stream == stream() && t.dev == dev) s = &t;
        if (t.used < old->used) old = &t;
    }
    if (!s) {
        s = old;
        if (s->used && hipDeviceSynchronize() != hipSuccess) {  // another thread captures
            (void)hipGetLastError();
            return nullptr;
        }
        if (s->used && s->dev != dev) {  // a buffer of another device
            (void)hipFree(s->buf);
            s->buf = nullptr;
            s->bytes = 0;
        }
        s->stream = stream();
        s->dev = dev;
    }
    s->used = ++g_clock;
    if (s->bytes >= bytes) return s->buf;
    if (s->buf) {
        if (hipStreamSynchronize(stream()) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        (void)hipFree(s->buf);
    }
    s->buf = nullptr;
    s->bytes = 0;
    const size_t grown = std::max(bytes, (size_t)1 << 20);
    if (hipMalloc(&s->buf, grown) != hipSuccess) {
        (void)hipGetLastError();
        s->buf = nullptr;
        return nullptr;
    }
    s->bytes = grown;
    return s->buf;
}

// The arena's parts in order of address.  The calls of one capture on one stream
// run in order and share a part, and so do the small eager calls of a stream.
struct Part {
    size_t at, bytes;
    unsigned long long id;  // of the capture; 0: eager calls
    hipStream_t stream;
    bool dropped;  // its graph is gone
};
constexpr size_t kArena = (size_t)16 << 20, kMaxPart = (size_t)1 << 20, kSmallPart = (size_t)512 << 10;
uint8_t *g_arena = nullptr;
std::vector<Part> g_parts;
bool g_dropped = false;  // some part is

// At least `bytes` for capture `id` (or eager calls) on the library stream; nullptr when they
// do not fit.  g_mu is held.
void *arena_part(size_t bytes, unsigned long long id)
{
    if (!g_arena || bytes > kMaxPart) return nullptr;
    for (const Part &p : g_parts)
        if (p.id == id && p.stream == stream() && p.bytes >= bytes) return g_arena + p.at;
    bytes = (bytes + 4095) & ~(size_t)4095;
    size_t at = 0;
    auto it = g_parts.begin();
    for (; it != g_parts.end() && it->at - at < bytes; ++it) at = it->at + it->bytes;
    if (at + bytes > kArena) return nullptr;
    g_parts.insert(it, Part{at, bytes, id, stream(), false});
    return g_arena + at;
}

// Gives the dropped parts back, once the device is idle: a last replay may be
// under way.  Not while a capture is open, which waiting would end: the next
// holo_graph_begin or _destroy does it then.  g_mu is held.
void reclaim()
{
    if (!g_dropped || stream_capturing()) return;
    if (hipDeviceSynchronize() != hipSuccess) {  // another thread captures
        (void)hipGetLastError();
        return;
    }
    g_parts.erase(std::remove_if(g_parts.begin(), g_parts.end(), [](const Part &p) { return p.dropped; }), g_parts.end());
    g_dropped = false;
}

}  // namespace

StreamScratch::StreamScratch(size_t bytes) : lock_(g_mu)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(stream(), &st, &id) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    if (st == hipStreamCaptureStatusNone) {
        if (bytes > kSmallPart || (buf_ = arena_part(bytes, 0)) == nullptr) buf_ = slot(bytes);
    } else if ((buf_ = arena_part(bytes, id)) == nullptr) {
        free_ = hipMallocAsync(&buf_, bytes, stream()) == hipSuccess;
        if (!free_) {
            (void)hipGetLastError();
            buf_ = nullptr;
        }
    }
}

StreamScratch::~StreamScratch()
{
    if (free_) HOLO_CHECK(hipFreeAsync(buf_, stream()));
}

bool stream_scratch_init()
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_arena) return true;
    if (hipMalloc((void **)&g_arena, kArena) == hipSuccess) return true;
    (void)hipGetLastError();
    g_arena = nullptr;
    return false;
}

void stream_scratch_drop_capture(unsigned long long id)
{
    std::lock_guard<std::mutex> lk(g_mu);
    for (Part &p : g_parts)
        if (p.id == id) p.dropped = g_dropped = true;
    reclaim();
}

void stream_scratch_reclaim()
{
    std::lock_guard<std::mutex> lk(g_mu);
    reclaim();
}

void stream_scratch_release()
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_arena) (void)hipFree(g_arena);
    g_arena = nullptr;
    g_parts.clear();
    g_dropped = false;
    for (Slot &s : g_slots) {
        if (s.buf) (void)hipFree(s.buf);
        s = Slot{};
    }
}

void stream_scratch_drop(hipStream_t st)
{
    std::lock_guard<std::mutex> lk(g_mu);
    for (Slot &s : g_slots)
        if (s.used && s.stream == st) {
            (void)hipStreamSynchronize(st);
            if (s.buf) (void)hipFree(s.buf);
            s = Slot{};
        }
    auto small = [&](const Part &p) { return p.id == 0 && p.stream == st; };
    if (std::any_of(g_parts.begin(), g_parts.end(), small)) {
        (void)hipStreamSynchronize(st);
        g_parts.erase(std::remove_if(g_parts.begin(), g_parts.end(), small), g_parts.end());
    }
}

}  // namespace holo
