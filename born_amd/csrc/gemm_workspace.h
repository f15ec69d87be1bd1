// Workspaces of the matrix products: packed operands and partial products, written by one launch of a product and read by the
// next.  A product holds its workspace from before its first launch until after its last (the lease below), so that no other host
// thread's product on the same stream comes between them; the stream's own order does the rest.
//
//   * A stream's products share one buffer of the stream, of GEMM_WS_MIN or GEMM_WS_MAX bytes, kept for its next ones; at most
//     MAX_STREAMS of them, the one unused longest goes for a new one (hipFree waits for the device).  hipStreamPerThread is a stream of
//     each thread under one handle: a buffer for each.
//   * Products recorded into a graph have a buffer of that capture, and of the stream they were recorded on: replays overlap neither
//     eager products nor other graphs' replays.  It belongs to the graph (a user object) and comes back when the graph and all
//     that was instantiated from it are gone; its memory is given back when the next buffer is wanted.
//   * Buffers are allocated with this thread's capture mode relaxed: an allocation here ends no capture, this thread's or another's.
//
// No buffer (out of memory, or a stream whose capture state cannot be asked): the product is computed without.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <exception>
#include <list>
#include <memory>
#include <mutex>
#include <vector>

#include "device_pool.h"
#include "gemm_plan.h"

namespace born {

class GemmWorkspaces {
    struct Buffer {
        std::mutex busy;                      // held while launches that use the buffer are being enqueued
        void *p = nullptr;
        size_t bytes = 0;
        bool gone = false;                    // taken from its stream: ask again
    };
    struct Entry {
        int dev;
        hipStream_t st;
        uint64_t thread;                      // hipStreamPerThread: whose; else 0
        unsigned long long capture;           // the capture's number; 0 outside
        std::shared_ptr<Buffer> buffer;
    };
    std::mutex mu;                            // the lists; never held while a graph is touched
    std::list<Entry> streams, captures;       // streams: the one used last in front
    std::mutex dead_mu;                       // (of its own: a graph's end may come from within the runtime)
    std::vector<void *> dead;                 // memory of graphs that are gone

    // The buffer of a graph, as its user object.
    struct Owned {
        GemmWorkspaces *home;
        std::shared_ptr<Buffer> buffer;
    };
    static void graph_gone(void *x) {         // (no HIP call is allowed here)
        std::unique_ptr<Owned> o((Owned *)x);
        GemmWorkspaces &w = *o->home;
        std::lock_guard<std::mutex> g(w.dead_mu);
        try {
            w.dead.push_back(o->buffer->p);
        } catch (const std::exception &) {
        }
        o->buffer->gone = true;
    }

    // Allocations and frees between this and its end leave captures alone.
    struct Relaxed {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        bool on = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
        ~Relaxed() {
            if (on) (void)hipThreadExchangeStreamCaptureMode(&mode);
        }
    };
    void give_back() {
        std::vector<void *> out;
        {
            std::lock_guard<std::mutex> g(dead_mu);
            out.swap(dead);
        }
        for (void *p : out) (void)hipFree(p);
    }
    void *allocate(size_t bytes) {
        Relaxed relaxed;
        give_back();
        void *p = nullptr;
        if (device_malloc(&p, bytes) == hipSuccess) return p;
        (void)hipGetLastError();
        return nullptr;
    }
    static size_t size_of(size_t bytes) { return bytes > GEMM_WS_MIN ? GEMM_WS_MAX : GEMM_WS_MIN; }
    static uint64_t this_thread() {
        static std::atomic<uint64_t> threads{0};
        thread_local const uint64_t mine = ++threads;
        return mine;
    }

public:
    static constexpr size_t MAX_STREAMS = 16;

    // A workspace in use: p is null where there is none.
    struct Lease {
        std::shared_ptr<Buffer> buffer;
        std::unique_lock<std::mutex> lock;
        float *p = nullptr;
    };

    Lease take(hipStream_t st, size_t bytes) {
        try {
            int dev = 0;
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
            if (bytes > GEMM_WS_MAX || hipGetDevice(&dev) != hipSuccess) return Lease();
            if (st && hipStreamIsCapturing(st, &status) != hipSuccess) {   // (the null stream is never captured)
                (void)hipGetLastError();
                return Lease();
            }
            if (status == hipStreamCaptureStatusInvalidated) return Lease();
            return status == hipStreamCaptureStatusActive ? of_capture(dev, st, bytes) : of_stream(dev, st, bytes);
        } catch (const std::exception &) {    // out of host memory
            return Lease();
        }
    }

private:
    static Lease lease(const std::shared_ptr<Buffer> &b, std::unique_lock<std::mutex> &&lock) {
        Lease l;
        l.buffer = b;
        l.lock = std::move(lock);
        l.p = (float *)b->p;
        return l;
    }

    Lease of_stream(int dev, hipStream_t st, size_t bytes) {
        const uint64_t thread = st == hipStreamPerThread ? this_thread() : 0;
        for (;;) {
            std::shared_ptr<Buffer> b, old;
            {
                std::lock_guard<std::mutex> g(mu);
                auto it = streams.begin();
                while (it != streams.end() && !(it->dev == dev && it->st == st && it->thread == thread)) ++it;
                if (it != streams.end()) {
                    streams.splice(streams.begin(), streams, it);
                } else {
                    streams.push_front(Entry{dev, st, thread, 0, std::make_shared<Buffer>()});
                    if (streams.size() > MAX_STREAMS) {
                        old = streams.back().buffer;
                        streams.pop_back();
                    }
                }
                b = streams.front().buffer;
            }
            if (old) {                                               // (its product's launches are enqueued by then; hipFree waits for them)
                std::lock_guard<std::mutex> o(old->busy);
                Relaxed relaxed;
                if (old->p) (void)hipFree(old->p);
                old->p = nullptr;
                old->gone = true;
            }
            std::unique_lock<std::mutex> lock(b->busy);
            if (b->gone) continue;
            if (b->bytes < bytes || !b->p) {
                if (b->p) {                                          // a larger one (hipFree waits for what still uses the old one)
                    Relaxed relaxed;
                    (void)hipFree(b->p);
                }
                b->p = allocate(size_of(bytes));
                b->bytes = b->p ? size_of(bytes) : 0;
            }
            return b->p ? lease(b, std::move(lock)) : Lease();
        }
    }

    Lease of_capture(int dev, hipStream_t st, size_t bytes) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        hipGraph_t graph = nullptr;
        if (hipStreamGetCaptureInfo_v2(st, &status, &id, &graph, nullptr, nullptr) != hipSuccess || !graph) {
            (void)hipGetLastError();
            return Lease();
        }
        std::shared_ptr<Buffer> b;
        {
            std::lock_guard<std::mutex> g(mu), d(dead_mu);
            for (auto it = captures.begin(); it != captures.end();) {
                if (it->buffer->gone) {
                    it = captures.erase(it);
                    continue;
                }
                if (it->dev == dev && it->st == st && it->capture == id && it->buffer->bytes >= bytes) b = it->buffer;
                ++it;
            }
        }
        if (!b) {
            b = std::make_shared<Buffer>();
            std::unique_ptr<Owned> owned(new Owned{this, b});
            std::list<Entry> entry{Entry{dev, st, 0, id, b}};
            b->p = allocate(size_of(bytes));
            b->bytes = size_of(bytes);
            if (!b->p) return Lease();
            hipUserObject_t object = nullptr;
            if (hipUserObjectCreate(&object, owned.get(), graph_gone, 1, hipUserObjectNoDestructorSync) != hipSuccess) {
                (void)hipGetLastError();
                Relaxed relaxed;
                (void)hipFree(b->p);
                return Lease();
            }
            owned.release();
            if (hipGraphRetainUserObject(graph, object, 1, hipGraphUserObjectMove) != hipSuccess) {
                (void)hipGetLastError();
                (void)hipUserObjectRelease(object, 1);               // (graph_gone: given back with the next one)
                return Lease();
            }
            std::lock_guard<std::mutex> g(mu);
            captures.splice(captures.begin(), entry);
        }
        return lease(b, std::unique_lock<std::mutex>(b->busy));
    }
};

}  // namespace born
