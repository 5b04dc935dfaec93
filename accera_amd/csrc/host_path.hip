// Host-pointer path of the package functions: what `functions[name](A, B, C)` of a HAT package runs
// (/root/reference/README.md:118-136, /root/reference/accera/python/accera/Package.py:776-784: a function of a HOST
// package takes NumPy arrays, i.e. pageable host memory).
//
// The caller's arrays are pageable, and this system does not let existing memory be pinned after the fact, so every
// byte goes through pinned staging buffers that the library allocates itself (hipHostMalloc):
//   * one context per call in flight -- device buffers for A, B, C, a ring of pinned staging slots, a stream and one
//     event per slot -- taken from a pool for the duration of the call, so calls from different host threads do not
//     wait for each other (each brings or reuses its own context);
//   * host to device: the caller's bytes are copied into a staging slot by a few worker threads, the slot is sent with
//     an asynchronous copy, and the next slot is filled meanwhile (a slot is reused once its copy's event has passed);
//   * the kernel runs on the context's stream behind the copies;
//   * a large product in several parts (rows of A and C): kernels and copies back have streams and a ring of their own, so that a part
//     is computed as soon as B and its rows of A are there, and travels back while the next rows travel in;
//   * device to host: the same ring the other way round -- the copies of the first slots are queued at once, each slot is
//     copied out to the caller's array when its event has passed and then queued again for a later piece.
#include "host_path.h"
#include "copy_pool.h"

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <vector>

namespace acc950 {

namespace {

// One staging slot, and how many a ring has.  (A copy costs its call about 10 us besides the bytes; 134 MB in parts: 2.44 ms with
// three slots of 8 MB, 2.65 with four of 4, 2.95 with eight of 2.)
constexpr size_t kSlotBytes = (size_t)8 << 20;
constexpr int kSlots = 3;
// A result of up to this size -- half of the last-level cache it was measured with, 32 MB -- is stored through the caches, where the caller, who reads it next,
// finds it.  (The call and then C.sum(), us, stores past the caches / through them: fp16 to fp32 1024^3, 4 MB, 483 to 500 / 460 to 465, 1024x2048x1024, 8 MB,
// 792 / 745, 2048x2048x1024, 16 MB, 1281 to 1325 / 1195 to 1270; 4096x2048x512, 32 MB, 2155 / 2238 and on another day 2248 / 2073, 4096x4096x512, 64 MB, 4157 / 4124;
// the call alone 311 / 313, 469 / 475, 670 / 678, 937 / 962, 1641 / 1667.)
constexpr size_t kCachedResult = (size_t)16 << 20;

CopyPool& copy_pool()
{
    static CopyPool* pool = new CopyPool; // (never destroyed: its threads may still be parked when the process ends)
    return *pool;
}

// ---- contexts ------------------------------------------------------------------------------
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

struct HostContext {
    int device = 0;
    hipStream_t stream = nullptr;
    DevBuf a, b, c;
    char* slot[kSlots] = {};
    hipEvent_t event[kSlots] = {};
    // calls in several parts only (made by the first of them)
    hipStream_t compute = nullptr, back = nullptr;
    char* back_slot[kSlots] = {};
    hipEvent_t back_event[kSlots] = {}, arrived = nullptr, computed = nullptr;
};

std::mutex g_pool_mutex;
std::vector<HostContext*> g_idle; // contexts not in use, any device
std::atomic<unsigned long long>* g_allocations = nullptr;

hipError_t make_context(int device, HostContext** out)
{
    HostContext* c = new HostContext;
    c->device = device;
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    for (int i = 0; i < kSlots && e == hipSuccess; ++i) {
        e = hipHostMalloc((void**)&c->slot[i], kSlotBytes, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&c->event[i], hipEventDisableTiming);
    }
    if (e != hipSuccess) {
        for (int i = 0; i < kSlots; ++i) {
            if (c->event[i]) (void)hipEventDestroy(c->event[i]);
            if (c->slot[i]) (void)hipHostFree(c->slot[i]);
        }
        if (c->stream) (void)hipStreamDestroy(c->stream);
        delete c;
        return e;
    }
    *out = c;
    return hipSuccess;
}

hipError_t prepare_parts(HostContext& c)
{
    hipError_t e = hipSuccess;
    for (hipStream_t* s : {&c.compute, &c.back})
        if (e == hipSuccess && !*s) e = hipStreamCreateWithFlags(s, hipStreamNonBlocking);
    for (hipEvent_t* ev : {&c.arrived, &c.computed})
        if (e == hipSuccess && !*ev) e = hipEventCreateWithFlags(ev, hipEventDisableTiming);
    for (int i = 0; i < kSlots; ++i) {
        if (e == hipSuccess && !c.back_slot[i]) e = hipHostMalloc((void**)&c.back_slot[i], kSlotBytes, hipHostMallocDefault);
        if (e == hipSuccess && !c.back_event[i]) e = hipEventCreateWithFlags(&c.back_event[i], hipEventDisableTiming);
    }
    return e; // (what was made stays with the context, and goes with it)
}

hipError_t acquire(HostContext** out)
{
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        for (size_t i = 0; i < g_idle.size(); ++i)
            if (g_idle[i]->device == device) {
                *out = g_idle[i];
                g_idle.erase(g_idle.begin() + (long)i);
                return hipSuccess;
            }
    }
    return make_context(device, out);
}

void release(HostContext* c)
{
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    g_idle.push_back(c);
}

hipError_t reserve(DevBuf& b, size_t bytes)
{
    if (bytes <= b.bytes) return hipSuccess;
    if (b.p) {
        hipError_t e = hipFree(b.p);
        if (e != hipSuccess) return e;
        b.p = nullptr;
        b.bytes = 0;
    }
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e == hipSuccess) {
        b.bytes = bytes;
        if (g_allocations) ++*g_allocations;
    }
    return e;
}

// Bytes of a piece of a transfer: four pieces, so that one is copied on the host while another is on the bus, but
// not less than two megabytes (1024^3 fp16 with an fp32 result 367 us with one), and never more than a slot; below four megabytes one
// piece, as a second one wakes the copying threads and calls the copy again (23x2366x321 fp32, a B of 3 MB, 201 us in two, 163 so; 234x1536x1024 fp16 240 / 199).
size_t piece_bytes(size_t bytes)
{
    if (bytes < (size_t)4 << 20) return bytes;
    const size_t quarter = (bytes / 4 + 65535) & ~(size_t)65535;
    return std::min(std::max(quarter, (size_t)2 << 20), kSlotBytes);
}

// caller's array -> device buffer, through the staging ring
hipError_t upload(HostContext& c, void* dev, const void* host, size_t bytes)
{
    const char* src = (const char*)host;
    const size_t step = piece_bytes(bytes);
    size_t piece = 0;
    for (size_t off = 0; off < bytes; off += step, ++piece) {
        const int s = (int)(piece % kSlots);
        const size_t n = std::min(bytes - off, step);
        // (the slot's last copy to the device -- of this call or an earlier one -- has read it)
        hipError_t e = hipEventSynchronize(c.event[s]);
        if (e != hipSuccess) return e;
        copy_pool().copy(c.slot[s], src + off, n, true);
        e = hipMemcpyAsync((char*)dev + off, c.slot[s], n, hipMemcpyHostToDevice, c.stream);
        if (e == hipSuccess) e = hipEventRecord(c.event[s], c.stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// device buffer -> caller's array
hipError_t download(HostContext& c, void* host, const void* dev, size_t bytes)
{
    char* dst = (char*)host;
    const size_t step = piece_bytes(bytes);
    const size_t pieces = (bytes + step - 1) / step;
    auto queue = [&](size_t piece) {
        const size_t off = piece * step, n = std::min(bytes - off, step);
        const int s = (int)(piece % kSlots);
        hipError_t e = hipMemcpyAsync(c.slot[s], (const char*)dev + off, n, hipMemcpyDeviceToHost, c.stream);
        if (e == hipSuccess) e = hipEventRecord(c.event[s], c.stream);
        return e;
    };
    // (stream order puts these behind the kernel, and behind the uploads that last read the slots)
    for (size_t piece = 0; piece < pieces && piece < (size_t)kSlots; ++piece)
        if (hipError_t e = queue(piece); e != hipSuccess) return e;
    for (size_t piece = 0; piece < pieces; ++piece) {
        const size_t off = piece * step, n = std::min(bytes - off, step);
        const int s = (int)(piece % kSlots);
        hipError_t e = hipEventSynchronize(c.event[s]);
        if (e != hipSuccess) return e;
        copy_pool().copy(dst + off, c.slot[s], n, bytes > kCachedResult);
        if (piece + kSlots < pieces)
            if (e = queue(piece + kSlots); e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Has the event passed?  (A query that answers "not yet" also leaves that as the thread's last error, which the next
// kernel launch would report.)
hipError_t passed(hipEvent_t event, bool* yes)
{
    const hipError_t e = hipEventQuery(event);
    *yes = e == hipSuccess;
    if (e != hipErrorNotReady) return e;
    (void)hipGetLastError();
    return hipSuccess;
}

// A call in several parts: all of B and the first part's bytes of A go in; then every part is launched as its bytes of A have
// arrived, and its bytes of C come back on a stream of their own while later bytes of A go in.  One thread deals out the copies between
// the caller's arrays and both rings: whatever slot is ready next, results first.  fp16 4096^3 with an fp32 result, 134 MB over the
// bus: 3.1 ms one after the other, 2.45 in eight parts.
hipError_t run_parts(HostContext& c, const HostOperands& h, const std::vector<HostPart>& parts, const HostLaunchFn& launch, int* launch_status)
{
    struct Piece { char* dev; char* host; size_t bytes; int part; bool last; };
    std::vector<Piece> in, back;
    const auto cut = [](std::vector<Piece>& to, char* dev, char* host, size_t bytes, int part) {
        const size_t pieces = (bytes + kSlotBytes - 1) / kSlotBytes, step = ((bytes + pieces - 1) / pieces + 4095) & ~(size_t)4095; // (equal ones)
        for (size_t off = 0; off < bytes; off += step) {
            const size_t n = std::min(bytes - off, step);
            to.push_back(Piece{dev + off, host + off, n, part, off + n == bytes});
        }
    };
    cut(in, (char*)c.b.p, (char*)h.B, h.b_bytes, -1);
    for (int i = 0; i < (int)parts.size(); ++i) {
        cut(in, (char*)c.a.p + parts[i].a_off, (char*)h.A + parts[i].a_off, parts[i].a_bytes, i);
        cut(back, (char*)c.c.p + parts[i].c_off, (char*)h.C + parts[i].c_off, parts[i].c_bytes, i);
    }
    size_t sent = 0, queued = 0, drained = 0;
    int launched = 0;
    hipError_t e = hipSuccess;
    while (drained < back.size()) {
        bool ready = false;
        if (drained < queued) {
            if ((e = passed(c.back_event[drained % kSlots], &ready)) != hipSuccess) return e;
            // (nothing left to send: there is nothing else to do than wait)
            if (!ready && sent == in.size()) {
                if ((e = hipEventSynchronize(c.back_event[drained % kSlots])) != hipSuccess) return e;
                ready = true;
            }
            if (ready) {
                const Piece& p = back[drained];
                copy_pool().copy(p.host, c.back_slot[drained % kSlots], p.bytes, h.c_bytes > kCachedResult);
                ++drained;
            }
        }
        if (!ready && sent < in.size()) {
            const Piece& p = in[sent];
            const int s = (int)(sent % kSlots);
            bool free_slot = false;
            if ((e = passed(c.event[s], &free_slot)) != hipSuccess) return e;
            // (neither ring has a slot ready: every slot of the way in is on the bus, the oldest is next)
            if (!free_slot && (e = hipEventSynchronize(c.event[s])) != hipSuccess) return e;
            copy_pool().copy(c.slot[s], p.host, p.bytes, true);
            if ((e = hipMemcpyAsync(p.dev, c.slot[s], p.bytes, hipMemcpyHostToDevice, c.stream)) != hipSuccess) return e;
            if ((e = hipEventRecord(c.event[s], c.stream)) != hipSuccess) return e;
            ++sent;
            if (p.part >= 0 && p.last) {
                // (a wait takes the event as it was last recorded when the wait is queued: one event serves all parts)
                if ((e = hipEventRecord(c.arrived, c.stream)) != hipSuccess) return e;
                if ((e = hipStreamWaitEvent(c.compute, c.arrived, 0)) != hipSuccess) return e;
                if ((*launch_status = launch(p.part, c.a.p, c.b.p, c.c.p, c.compute)) != 0) return hipSuccess;
                if ((e = hipEventRecord(c.computed, c.compute)) != hipSuccess) return e;
                if ((e = hipStreamWaitEvent(c.back, c.computed, 0)) != hipSuccess) return e;
                ++launched;
            }
        }
        for (; queued < back.size() && queued < drained + kSlots && back[queued].part < launched; ++queued) {
            const Piece& p = back[queued];
            const int s = (int)(queued % kSlots);
            if ((e = hipMemcpyAsync(c.back_slot[s], p.dev, p.bytes, hipMemcpyDeviceToHost, c.back)) != hipSuccess) return e;
            if ((e = hipEventRecord(c.back_event[s], c.back)) != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

} // namespace

void host_path_count_allocations(std::atomic<unsigned long long>* counter) { g_allocations = counter; }

hipError_t host_path_release_idle(int device)
{
    std::vector<HostContext*> mine;
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        for (size_t i = 0; i < g_idle.size();) {
            if (g_idle[i]->device != device) { ++i; continue; }
            mine.push_back(g_idle[i]);
            g_idle.erase(g_idle.begin() + (long)i);
        }
    }
    // (a context goes back to the pool with its stream idle: nothing of it is in use any more)
    hipError_t first = hipSuccess;
    auto note = [&](hipError_t e) { if (e != hipSuccess && first == hipSuccess) first = e; };
    for (HostContext* c : mine) {
        for (DevBuf* b : {&c->a, &c->b, &c->c})
            if (b->p) note(hipFree(b->p));
        for (int i = 0; i < kSlots; ++i) {
            for (hipEvent_t ev : {c->event[i], c->back_event[i]})
                if (ev) note(hipEventDestroy(ev));
            for (char* p : {c->slot[i], c->back_slot[i]})
                if (p) note(hipHostFree(p));
        }
        for (hipEvent_t ev : {c->arrived, c->computed})
            if (ev) note(hipEventDestroy(ev));
        for (hipStream_t s : {c->stream, c->compute, c->back})
            if (s) note(hipStreamDestroy(s));
        delete c;
    }
    return first;
}

hipError_t host_path_run(const HostOperands& h, const std::vector<HostPart>& parts, const HostLaunchFn& launch, int* launch_status)
{
    HostContext* c = nullptr;
    hipError_t e = acquire(&c);
    if (e != hipSuccess) return e;
    *launch_status = 0;
    bool in_parts = false;
    CopyPool::Busy awake(copy_pool(), h.a_bytes + h.b_bytes + h.c_bytes >= ((size_t)4 << 20));
    try {
    do {
        if ((e = reserve(c->a, h.a_bytes ? h.a_bytes : 16)) != hipSuccess) break;
        if ((e = reserve(c->b, h.b_bytes ? h.b_bytes : 16)) != hipSuccess) break;
        if ((e = reserve(c->c, h.c_bytes ? h.c_bytes : 16)) != hipSuccess) break;
        if (parts.size() > 1) {
            if (prepare_parts(*c) == hipSuccess) {
                in_parts = true;
                e = run_parts(*c, h, parts, launch, launch_status);
                break;
            }
            (void)hipGetLastError(); // (no second ring to be had: in one piece then)
        }
        if ((e = upload(*c, c->a.p, h.A, h.a_bytes)) != hipSuccess) break;
        if ((e = upload(*c, c->b.p, h.B, h.b_bytes)) != hipSuccess) break;
        if (h.send_c && (e = upload(*c, c->c.p, h.C, h.c_bytes)) != hipSuccess) break;
        *launch_status = launch(-1, c->a.p, c->b.p, c->c.p, c->stream);
        if (*launch_status != 0) break;
        if ((e = download(*c, h.C, c->c.p, h.c_bytes)) != hipSuccess) break;
    } while (false);
    } catch (const std::exception&) { // (the lists of pieces, or a copying thread: no memory for them)
        e = hipErrorOutOfMemory;
    }
    // whatever happened, the streams are idle and the slots are free when the context goes back
    hipError_t e2 = hipStreamSynchronize(c->stream);
    if (in_parts)
        for (hipStream_t s : {c->compute, c->back}) {
            const hipError_t e3 = hipStreamSynchronize(s);
            if (e2 == hipSuccess) e2 = e3;
        }
    release(c);
    return e != hipSuccess ? e : e2;
}

} // namespace acc950
