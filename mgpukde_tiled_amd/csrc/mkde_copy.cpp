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
// go through the context's own stream (the same raster call: 11.3 ms), and only
// for copies of MIN_SHARED and more.
//
// Lanes belong to the process: at most MAX_LANES exist, a copy borrows the free
// ones it can use and gives them back, and all are freed when the last context
// is destroyed.  Helper threads live for one copy.
#include "mkde_copy.h"

#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace mkde_copy {
namespace {

constexpr size_t CHUNK = (size_t)1 << 20;   // bytes of one pinned buffer
constexpr int MAX_LANES = 12;               // 24 MB pinned in all
constexpr int LANES_PER_COPY = 8;
constexpr size_t BYTES_PER_LANE = (size_t)2 << 20;

struct Lane {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    unsigned char *buf[2] = {nullptr, nullptr};

    hipError_t make(int dev)
    {
        device = dev;
        hipError_t e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
        for (int k = 0; k < 2 && e == hipSuccess; ++k) {
            e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
            if (e == hipSuccess) e = hipHostMalloc((void **)&buf[k], CHUNK, hipHostMallocDefault);
        }
        return e;
    }
    void drop()
    {
        for (int k = 0; k < 2; ++k) {
            if (buf[k]) (void)hipHostFree(buf[k]);
            if (ev[k]) (void)hipEventDestroy(ev[k]);
        }
        if (stream) (void)hipStreamDestroy(stream);
    }
};

std::mutex g_mu;
int g_users = 0;
int g_lanes = 0;                    // lanes that exist, borrowed ones included
std::vector<Lane *> &idle()
{
    static std::vector<Lane *> *v = new std::vector<Lane *>();   // outlives every static destructor
    return *v;
}

// Up to `want` lanes of the device: idle ones first, then new ones.
std::vector<Lane *> borrow(int device, int want)
{
    std::vector<Lane *> got;
    std::lock_guard<std::mutex> lk(g_mu);
    std::vector<Lane *> &v = idle();
    for (size_t i = v.size(); i-- > 0 && (int)got.size() < want;)
        if (v[i]->device == device) {
            got.push_back(v[i]);
            v.erase(v.begin() + (std::ptrdiff_t)i);
        }
    while ((int)got.size() < want && g_lanes < MAX_LANES) {
        Lane *l = new Lane();
        if (l->make(device) != hipSuccess) {
            (void)hipGetLastError();
            l->drop();
            delete l;
            break;
        }
        ++g_lanes;
        got.push_back(l);
    }
    return got;
}

void give_back(std::vector<Lane *> &lanes)
{
    std::lock_guard<std::mutex> lk(g_mu);
    for (Lane *l : lanes) idle().push_back(l);
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

void retain()
{
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_users;
}

void release()
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_users > 0) return;
    for (Lane *l : idle()) {
        l->drop();
        delete l;
        --g_lanes;
    }
    idle().clear();
}

hipError_t run(int device, hipStream_t shared, void *dst, const void *src, size_t bytes, bool to_host, bool *done)
{
    *done = false;
    const size_t by_size = (bytes + BYTES_PER_LANE - 1) / BYTES_PER_LANE;
    const int want = by_size < (size_t)LANES_PER_COPY ? (int)by_size : LANES_PER_COPY;
    std::vector<Lane *> lanes = borrow(device, want);
    if (lanes.empty()) return hipSuccess;
    Copy c;
    c.dst = (unsigned char *)dst;
    c.src = (const unsigned char *)src;
    c.bytes = bytes;
    c.to_host = to_host;
    c.shared = shared;
    std::vector<std::thread> helpers;
    try {
        helpers.reserve(lanes.size());
        for (size_t i = 1; i < lanes.size(); ++i) helpers.emplace_back([&c, l = lanes[i]] { c.work(*l); });
    } catch (const std::exception &) {
        // fewer helpers: the lanes that run take every chunk
    }
    c.work(*lanes[0]);
    for (std::thread &t : helpers) t.join();
    give_back(lanes);
    *done = true;
    return (hipError_t)c.err.load();
}

}  // namespace mkde_copy
