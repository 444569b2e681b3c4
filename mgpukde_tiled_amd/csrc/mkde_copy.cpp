// mkde_copy.cpp -- large copies between pageable host memory and the device.
//
// hipMemcpyAsync on pageable memory moves it through the runtime's staging
// buffers with one thread: a 268 MB raster came back at 10 GB/s (26 ms, of
// which the link needed 5), because that thread also takes every page fault of
// the caller's fresh buffer.  Here a copy is cut into chunks that several
// lanes take in turn; a lane is a stream, two pinned chunk buffers and a thread,
// so its transfer of one chunk runs beside the host copy of the other, and the
// host copies (and page faults) of the lanes run in parallel.  The raster takes
// 6 ms; chunks of 0.5 / 1 / 2 / 4 MB: 8.5 / 8.2 / 7.9 / 8.7 ms for the whole call
// (a 4 MB raster is best at 1 MB), four lanes instead of eight 9.6 ms.
//
// Where other contexts' kernels run at the same time (the job server's slots),
// the lanes' streams would share the few hardware queues with them and wait
// behind them (a burst of 16 jobs: 14.9 ms against 13.6 ms): there the transfers
// go through the context's own stream, and only for copies of MIN_SHARED and more.
//
// A device has at most MAX_LANES lanes, made when copies have earned them; a copy
// borrows the free ones it can use and gives them back.  They outlast the contexts: a
// program with a context per call and a 16 MB raster, whose lanes went with its
// context, spent 6.6 of 9.7 ms a call on destroying their streams (2.4 ms a call without
// lanes, 0.9 now).  mkde_ctx_release frees the idle ones, and so does a job server
// when it starts: their streams would keep a share of the hardware queues from its
// slots (its burst 4% longer).  Helper threads live for one copy.
#include "mkde_copy.h"

#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <utility>

namespace mkde_copy {
namespace {

constexpr size_t CHUNK = (size_t)1 << 20;   // bytes of one pinned buffer
constexpr int MAX_LANES = 12;               // a device's; 24 MB pinned
constexpr int LANES_PER_COPY = 8;
constexpr size_t BYTES_PER_LANE = (size_t)2 << 20;
constexpr int MAX_DEVICES = 64;

struct Lane {
    int device = 0;
    Lane *next = nullptr;   // of the idle ones
    hipStream_t stream = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    unsigned char *buf[2] = {nullptr, nullptr};

    hipError_t make(int dev)
    {
        device = dev;
        hipError_t e = hipSuccess;
        for (int k = 0; k < 2 && e == hipSuccess; ++k) {
            e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
            if (e == hipSuccess) e = hipHostMalloc((void **)&buf[k], CHUNK, hipHostMallocDefault);
        }
        return e;
    }
    // Its own stream, made at the first copy that does not bring one.
    hipError_t own_stream()
    {
        const hipError_t e = stream ? hipSuccess : hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
        if (e != hipSuccess) stream = nullptr;
        return e;
    }
    ~Lane()
    {
        for (int k = 0; k < 2; ++k) {
            if (buf[k]) (void)hipHostFree(buf[k]);
            if (ev[k]) (void)hipEventDestroy(ev[k]);
        }
        if (stream) (void)hipStreamDestroy(stream);
    }
};

struct Device {
    Lane *idle = nullptr;
    int lanes = 0;      // that exist or are being made, borrowed ones included
    size_t moved = 0;   // bytes of copies that were ones for lanes
};

std::mutex g_mu;
Device g_dev[MAX_DEVICES];

// Up to `want` lanes of the device, with streams of their own if asked for: idle ones
// first, then new ones.  What has to be made is made outside the lock.
int borrow(int device, int want, size_t bytes, bool own, Lane **got)
{
    Device &d = g_dev[device];
    int n = 0, fresh = 0;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (d.moved < MIN_MOVED) d.moved += bytes;
        for (; n < want && d.idle; ++n) {
            got[n] = d.idle;
            d.idle = d.idle->next;
        }
        if (d.moved >= MIN_MOVED) fresh = want - n < MAX_LANES - d.lanes ? want - n : MAX_LANES - d.lanes;
        d.lanes += fresh;
    }
    int lost = 0;
    for (int i = 0; i < fresh; ++i) {
        Lane *l = lost ? nullptr : new (std::nothrow) Lane();
        if (l && l->make(device) == hipSuccess) {
            got[n++] = l;
            continue;
        }
        delete l;
        ++lost;
    }
    int use = 0;   // those that can be used stand first
    for (int i = 0; i < n; ++i)
        if (!own || got[i]->own_stream() == hipSuccess) std::swap(got[use++], got[i]);
    if (lost || use < n) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lk(g_mu);
        d.lanes -= lost;
        for (; n > use; --n) {
            got[n - 1]->next = d.idle;
            d.idle = got[n - 1];
        }
    }
    return use;
}

void unborrow(int device, Lane **lanes, int n)
{
    std::lock_guard<std::mutex> lk(g_mu);
    for (int i = 0; i < n; ++i) {
        lanes[i]->next = g_dev[device].idle;
        g_dev[device].idle = lanes[i];
    }
}

struct Copy {
    unsigned char *dst;
    const unsigned char *src;
    size_t bytes;
    bool to_host;
    hipStream_t shared;   // every transfer's stream, or null: the lanes' own
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};

    size_t len(size_t off) const { return bytes - off < CHUNK ? bytes - off : CHUNK; }

    // One lane's share: chunks off the common counter until none is left.
    // Every chunk's transfer has ended when this returns.
    void work(Lane &l)
    {
        hipError_t e = hipSetDevice(l.device);
        const hipStream_t stream = shared ? shared : l.stream;
        size_t at[2] = {0, 0};
        bool busy[2] = {false, false};
        auto settle = [&](int k) {   // slot k's transfer ends; a chunk for the host moves on
            if (!busy[k]) return;
            busy[k] = false;
            const hipError_t w = hipEventSynchronize(l.ev[k]);
            if (e == hipSuccess) e = w;
            if (e == hipSuccess && to_host) memcpy(dst + at[k], l.buf[k], len(at[k]));
        };
        int k = 0;
        while (e == hipSuccess && err.load(std::memory_order_relaxed) == (int)hipSuccess) {
            const size_t off = next.fetch_add(CHUNK);
            if (off >= bytes) break;
            if (!to_host) {
                settle(k);   // slot k's last chunk has left its buffer
                if (e != hipSuccess) break;
                memcpy(l.buf[k], src + off, len(off));
                e = hipMemcpyAsync(dst + off, l.buf[k], len(off), hipMemcpyHostToDevice, stream);
            } else {
                e = hipMemcpyAsync(l.buf[k], src + off, len(off), hipMemcpyDeviceToHost, stream);
            }
            if (e == hipSuccess) e = hipEventRecord(l.ev[k], stream);
            if (e != hipSuccess) break;
            at[k] = off;
            busy[k] = true;
            k ^= 1;
            if (to_host) settle(k);   // the other slot's chunk, beside this one's transfer
        }
        settle(k);
        settle(k ^ 1);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(stream);   // nothing of this copy is left in flight
            err.store((int)e);
        }
    }
};

}  // namespace

void give_back(int device)
{
    if (device < 0 || device >= MAX_DEVICES) return;
    Lane *l;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        l = g_dev[device].idle;
        g_dev[device].idle = nullptr;
        for (Lane *i = l; i; i = i->next) --g_dev[device].lanes;
    }
    while (l) {
        Lane *next = l->next;
        delete l;
        l = next;
    }
}

hipError_t run(int device, hipStream_t shared, void *dst, const void *src, size_t bytes, bool to_host, bool *done)
{
    *done = false;
    if (bytes < least(shared != nullptr, to_host) || device < 0 || device >= MAX_DEVICES) return hipSuccess;
    const size_t by_size = (bytes + BYTES_PER_LANE - 1) / BYTES_PER_LANE;
    Lane *lanes[LANES_PER_COPY];
    const int n = borrow(device, by_size < (size_t)LANES_PER_COPY ? (int)by_size : LANES_PER_COPY, bytes, !shared, lanes);
    if (n == 0) return hipSuccess;
    Copy c;
    c.dst = (unsigned char *)dst;
    c.src = (const unsigned char *)src;
    c.bytes = bytes;
    c.to_host = to_host;
    c.shared = shared;
    std::thread helpers[LANES_PER_COPY];
    int started = 1;
    try {
        for (; started < n; ++started) helpers[started] = std::thread([&c, l = lanes[started]] { c.work(*l); });
    } catch (...) {
        // fewer helpers: the lanes that run take every chunk
    }
    c.work(*lanes[0]);
    for (int i = 1; i < started; ++i) helpers[i].join();
    unborrow(device, lanes, n);
    *done = true;
    return (hipError_t)c.err.load();
}

}  // namespace mkde_copy
