/*
 * idle_kits.h -- what a handle without a caller's stream takes from the driver whatever its volume: a stream
 * and a pinned page for the totals. Making and destroying them took 80 us, as long as everything that a
 * 128^3 volume needs on the device, so a destroyed handle leaves them, idle, to the next one on its device: at
 * most kIdleKits per device wait here, the rest are destroyed. Any thread may take or leave one. Idle, they cost
 * work on the null stream, which orders itself after blocking streams, nothing that could be measured (a small
 * kernel on it 4.9 us, with a wait 15.3, none to four of them idle).
 *
 * hipDeviceReset takes a device's streams and allocations away, and what is made after it may have the same
 * handles and addresses. An allocation's buffer id is never given twice in a process, so each kit holds a small
 * allocation on its device and is only handed on while that address still names the allocation (62 ns).
 * The same test tells whether the pinned page of miso_fe_run_noalloc is still there (KeptPage).
 */
#ifndef MINIISO_IDLE_KITS_H
#define MINIISO_IDLE_KITS_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>

namespace miso {

constexpr size_t kPinnedTotals = 2 * sizeof(uint64_t);

/* the id of the allocation that holds p; 0 if there is none, or the driver gives no ids */
inline unsigned long long buffer_id(const void* p)
{
    unsigned long long id = 0;
    if (!p) return 0;
    if (hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return id;
}

struct Kit {
    hipStream_t stream = nullptr;
    uint64_t* totals = nullptr;
    void* mark = nullptr;               // an allocation of the device, which goes where the stream goes
    unsigned long long mark_id = 0;
    int dev = 0;

    bool there() const { return mark_id && buffer_id(mark) == mark_id; }
};

inline void destroy_kit(Kit& k)
{
    if (k.totals) (void)hipHostFree(k.totals);
    if (k.mark) (void)hipFree(k.mark);
    if (k.stream) (void)hipStreamDestroy(k.stream);
    k = Kit();
}

/* a new kit for the current device dev, or the driver's error and nothing made */
inline hipError_t make_kit(Kit* out, int dev)
{
    Kit k;
    k.dev = dev;
    // a blocking stream: ordered after work on the null stream (where callers that produce a
    // device volume without naming a stream usually ran)
    hipError_t e = hipStreamCreateWithFlags(&k.stream, hipStreamDefault);
    if (e != hipSuccess) k.stream = nullptr;
    if (e == hipSuccess) {
        e = hipHostMalloc((void**)&k.totals, kPinnedTotals, hipHostMallocDefault);
        if (e != hipSuccess) k.totals = nullptr;
    }
    if (e == hipSuccess) {
        e = hipMalloc(&k.mark, 1);
        if (e != hipSuccess) k.mark = nullptr;
    }
    if (e != hipSuccess) {
        destroy_kit(k);
        return e;
    }
    k.mark_id = buffer_id(k.mark);
    *out = k;
    return hipSuccess;
}

constexpr int kIdleKits = 4;            // per device
constexpr int kIdleDevices = 64;        // of the first so many devices

/* Fixed places, so that neither taking nor leaving a kit allocates: a handle's end cannot fail. */
class IdleKits {
    std::mutex lock;
    Kit kits[kIdleDevices][kIdleKits];
    int count[kIdleDevices] = {};

public:
    hipError_t take(Kit* out)
    {
        int dev = 0;
        if (const hipError_t e = hipGetDevice(&dev)) return e;
        while (dev >= 0 && dev < kIdleDevices) {
            Kit k;
            {
                std::lock_guard<std::mutex> hold(lock);
                if (!count[dev]) break;
                k = kits[dev][--count[dev]];
            }
            if (k.there()) {
                *out = k;
                return hipSuccess;
            }
            // the device was reset: what the kit names is gone, or may be someone else's by now
        }
        return make_kit(out, dev);
    }

    /* the stream's work is done, without an error if `clean` */
    void leave(Kit& k, bool clean)
    {
        if (!k.there() && k.mark_id) {
            k = Kit();                  // a device reset while the handle lived
            return;
        }
        if (clean && k.mark_id && k.dev >= 0 && k.dev < kIdleDevices) {
            std::lock_guard<std::mutex> hold(lock);
            int& n = count[k.dev];
            if (n < kIdleKits) {
                kits[k.dev][n++] = k;
                k = Kit();
                return;
            }
        }
        destroy_kit(k);
    }
};

inline IdleKits& idle_kits()
{
    static IdleKits k;
    return k;
}

/* A pinned page for two totals, made on the first call and kept. */
class KeptPage {
    uint64_t* page = nullptr;
    unsigned long long id = 0;

public:
    /* NULL where the host has none left; the next call tries again. The call may come while the thread captures a
     * graph, which the allocation does not touch. */
    uint64_t* get()
    {
        if (page && buffer_id(page) == id) return page;
        page = nullptr;                 // none yet, or it went with a device reset
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (hipHostMalloc((void**)&page, kPinnedTotals, hipHostMallocDefault) != hipSuccess) {
            page = nullptr;
            (void)hipGetLastError();
        }
        id = buffer_id(page);
        if (page && !id) {
            (void)hipHostFree(page);
            page = nullptr;
        }
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        return page;
    }
};

}  // namespace miso

#endif
