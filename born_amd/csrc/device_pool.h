// Device buffers handed out and taken back by born_rocm_alloc and born_rocm_free.  The backend's operations return a new
// buffer each: an MNIST network's forward pass makes eleven, and hipMalloc and hipFree (which waits
// for the device) took most of its time (64 images: 339 us, 170 like this).  A freed buffer of up to POOL_BUFFER_MAX bytes is kept, up to
// POOL_TOTAL_MAX bytes and POOL_COUNT_MAX buffers in all, the oldest given back first; all of them where the library finds memory
// short (device_malloc, which its other allocations go through too); and all but the last POOL_IDLE_MAX bytes when the last buffer
// handed out has come back.  (Not all of them then: a loss over torch's tensors has one small buffer at a time, and to free it at once
// made an MNIST evaluation step 119 us, which is 111.)
//
// A kept buffer may still be in use by work on any stream of its device.  It is handed out again only once the whole device
// has been waited for after it was freed.  hipFree does that wait: the smallest kept buffer goes back to the device, and every
// buffer freed before that call is idle from then on.  (hipDeviceSynchronize would spare that buffer, but it is refused and ends the
// capture where a stream is being captured in relaxed mode, in which hipMalloc and hipFree are allowed.)  Where the program has waited
// for the device's results since the free (the usual end of a pass) the wait finds the device idle; else a fresh buffer costs less
// than draining the device, until the pool is full.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <list>
#include <mutex>
#include <unordered_map>

namespace born {

class DevicePool {
    static constexpr size_t POOL_BUFFER_MAX = (size_t)32 << 20, POOL_TOTAL_MAX = (size_t)256 << 20, POOL_IDLE_MAX = (size_t)16 << 20, POOL_COUNT_MAX = 256, GRAIN = 512;
    static constexpr int DEVICES = 64;

    struct Live {
        size_t bytes;                         // 0: too large to be kept
        int dev;
    };
    struct Kept {
        void *p;
        size_t bytes;
        int dev;
        uint64_t freed, waits;                // the free's number; how often the program had waited by then
    };
    std::mutex mu;
    std::unordered_map<void *, Live> live;    // buffers handed out
    std::list<Kept> kept;                     // oldest first
    size_t total = 0;
    uint64_t frees = 0, waits = 0, idle[DEVICES] = {};   // idle[d]: frees up to this number have been waited for on device d

public:
    // The program has waited for a stream.
    void waited() {
        std::lock_guard<std::mutex> g(mu);
        waits++;
    }

    hipError_t alloc(size_t bytes, void **out) {
        int dev = 0;
        const bool keeps = bytes <= POOL_BUFFER_MAX && hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < DEVICES;
        const size_t size = keeps ? (bytes + GRAIN - 1) / GRAIN * GRAIN : bytes;
        if (keeps) {
            if (take(dev, size, out)) return hipSuccess;
            std::list<Kept> back;
            uint64_t upto;
            if (give_back(dev, size, back, &upto)) {
                const hipError_t e = hipFree(back.front().p);        // (outside the lock: other threads go on)
                std::unique_lock<std::mutex> g(mu);
                if (e == hipSuccess) {
                    if (upto > idle[dev]) idle[dev] = upto;
                } else {                                             // (not now: kept on, in its place)
                    (void)hipGetLastError();
                    total += back.front().bytes;
                    auto at = kept.begin();
                    while (at != kept.end() && at->freed < back.front().freed) ++at;
                    kept.splice(at, back);
                }
                g.unlock();
                if (take(dev, size, out)) return hipSuccess;
            }
        }
        const hipError_t e = malloc_or_release(size, out);
        if (e == hipSuccess) {
            try {
                std::lock_guard<std::mutex> g(mu);
                live[*out] = Live{keeps ? size : 0, dev};
            } catch (...) {
                (void)hipFree(*out);
                throw;
            }
        }
        return e;
    }

    hipError_t free(void *p) {
        std::list<Kept> out;
        {
            std::lock_guard<std::mutex> g(mu);
            const auto it = live.find(p);
            if (it == live.end()) {
                for (const Kept &k : kept)
                    if (k.p == p) return hipErrorInvalidValue;       // freed before
            } else {
                if (it->second.bytes) {
                    kept.push_back(Kept{p, it->second.bytes, it->second.dev, ++frees, waits});
                    total += it->second.bytes;
                    p = nullptr;
                }
                live.erase(it);
                while (total > (live.empty() ? POOL_IDLE_MAX : POOL_TOTAL_MAX) || kept.size() > POOL_COUNT_MAX) {
                    total -= kept.front().bytes;
                    out.splice(out.end(), kept, kept.begin());
                }
            }
        }
        hipError_t e = p ? hipFree(p) : hipSuccess;
        for (const Kept &k : out) {
            const hipError_t f = hipFree(k.p);
            if (e == hipSuccess) e = f;
        }
        if (e != hipSuccess) (void)hipGetLastError();                // (returned: the next launch does not report it again)
        return e;
    }

    // hipMalloc; where memory is short, again without what is kept here.
    hipError_t malloc_or_release(size_t bytes, void **out) {
        const hipError_t e = hipMalloc(out, bytes);
        if (e != hipErrorOutOfMemory) return e;
        std::list<Kept> give;
        {
            std::lock_guard<std::mutex> g(mu);
            give.swap(kept);
            total = 0;
        }
        if (give.empty()) return e;
        (void)hipGetLastError();
        for (const Kept &k : give) (void)hipFree(k.p);
        return hipMalloc(out, bytes);
    }

private:
    // The oldest kept buffer of the size, where it is idle.
    bool take(int dev, size_t size, void **out) {
        std::lock_guard<std::mutex> g(mu);
        for (auto it = kept.begin(); it != kept.end(); ++it) {
            if (it->dev != dev || it->bytes != size) continue;
            if (it->freed > idle[dev]) return false;                 // (so are the later ones)
            live[it->p] = Live{size, dev};
            *out = it->p;
            total -= size;
            kept.erase(it);
            return true;
        }
        return false;
    }

    // Takes the smallest kept buffer of the device out, to be freed for the wait, where a buffer of the size is kept and the wait is
    // worth it.
    bool give_back(int dev, size_t size, std::list<Kept> &back, uint64_t *upto) {
        std::lock_guard<std::mutex> g(mu);
        auto found = kept.end(), least = kept.end();
        for (auto it = kept.begin(); it != kept.end(); ++it) {
            if (it->dev != dev) continue;
            if (it->bytes == size && found == kept.end()) found = it;
            if (least == kept.end() || it->bytes < least->bytes) least = it;
        }
        if (found == kept.end()) return false;
        if (found->waits >= waits && total + size <= POOL_TOTAL_MAX && kept.size() < POOL_COUNT_MAX) return false;
        *upto = frees;
        total -= least->bytes;
        back.splice(back.end(), kept, least);
        return true;
    }
};

// (never destroyed: a buffer may come back while the process ends)
inline DevicePool &device_pool() {
    static DevicePool *const pool = new DevicePool;
    return *pool;
}
// The library's own buffers: not kept, but allocated like the others where memory is short.
template <class T>
inline hipError_t device_malloc(T **out, size_t bytes) {
    return device_pool().malloc_or_release(bytes, (void **)out);
}

}  // namespace born
