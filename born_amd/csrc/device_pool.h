// Device buffers handed out and taken back by born_rocm_alloc and born_rocm_free.  The backend's operations return a new
// buffer each: an MNIST network's forward pass makes eleven, and hipMalloc and hipFree (which waits
// for the device) took most of its time (64 images: 347 us, 154 like this).  A freed buffer of up to POOL_BUFFER_MAX bytes is kept, up to
// POOL_TOTAL_MAX bytes and POOL_COUNT_MAX buffers in all, the oldest given back first, all of them where memory runs out.
//
// A kept buffer may still be in use by work on any stream of its device.  It is handed out again only once the whole device
// has been waited for after it was freed: what hipFree promises.  One wait serves every buffer freed before it.  Where
// the program has waited for the device's results since the free (the usual end of a pass) that wait finds the device idle; else a
// fresh buffer costs less than draining the device, until the pool is full.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <list>
#include <mutex>
#include <unordered_map>

namespace born {

class DevicePool {
    static constexpr size_t POOL_BUFFER_MAX = (size_t)32 << 20, POOL_TOTAL_MAX = (size_t)256 << 20, POOL_COUNT_MAX = 256, GRAIN = 512;
    static constexpr int DEVICES = 64;

    struct Live {
        size_t bytes;
        int dev;
    };
    struct Kept {
        void *p;
        size_t bytes;
        int dev;
        uint64_t freed, waits;                // the free's number; how often the program had waited by then
    };
    std::mutex mu;
    std::unordered_map<void *, Live> live;    // buffers the pool may keep when they come back
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
        if (bytes > POOL_BUFFER_MAX || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= DEVICES) return fresh_or_release(bytes, out);
        const size_t size = (bytes + GRAIN - 1) / GRAIN * GRAIN;
        Kept got = {nullptr, 0, 0, 0, 0};
        bool wait = false;
        uint64_t upto = 0;
        {
            std::lock_guard<std::mutex> g(mu);
            auto best = kept.end();
            for (auto it = kept.begin(); it != kept.end(); ++it) {   // the oldest of the size: the first to have been waited for
                if (it->dev == dev && it->bytes == size) {
                    best = it;
                    break;
                }
            }
            if (best != kept.end()) {
                wait = best->freed > idle[dev];
                if (!wait || best->waits < waits || total + size > POOL_TOTAL_MAX || kept.size() >= POOL_COUNT_MAX) {
                    got = *best;
                    kept.erase(best);
                    total -= size;
                    upto = frees;
                    if (!wait) live[got.p] = Live{size, dev};
                }
            }
        }
        if (got.p && wait) {
            const hipError_t e = hipDeviceSynchronize();             // (outside the lock: other threads go on)
            std::lock_guard<std::mutex> g(mu);
            if (e == hipSuccess) {
                if (upto > idle[dev]) idle[dev] = upto;
                live[got.p] = Live{size, dev};
            } else {                                                 // (not now, for instance while a stream is captured: kept on)
                (void)hipGetLastError();
                kept.push_back(got);
                total += size;
                got.p = nullptr;
            }
        }
        if (got.p) {
            *out = got.p;
            return hipSuccess;
        }
        const hipError_t e = fresh_or_release(size, out);
        if (e == hipSuccess) {
            std::lock_guard<std::mutex> g(mu);
            live[*out] = Live{size, dev};
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
                kept.push_back(Kept{p, it->second.bytes, it->second.dev, ++frees, waits});
                total += it->second.bytes;
                live.erase(it);
                while (total > POOL_TOTAL_MAX || kept.size() > POOL_COUNT_MAX) {
                    total -= kept.front().bytes;
                    out.splice(out.end(), kept, kept.begin());
                }
                p = nullptr;
            }
        }
        hipError_t e = p ? hipFree(p) : hipSuccess;
        for (const Kept &k : out) {
            const hipError_t f = hipFree(k.p);
            if (e == hipSuccess) e = f;
        }
        return e;
    }

private:
    hipError_t fresh_or_release(size_t bytes, void **out) {
        hipError_t e = hipMalloc(out, bytes);
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
};

}  // namespace born
