// zq3d_hostcopy.h -- copies between a caller's ordinary (pageable) arrays and device memory for the host-
// pointer entry points, staged through pinned slots by several threads.
//
// A plain hipMemcpy of pageable memory moves 28 GB/s to the device and 17 GB/s back here: one thread fills
// or drains the runtime's staging buffer.  The link does 57 GB/s from pinned memory, so a call's arrays
// are cut into batches of up to a slot, and each thread copies a batch between the caller's memory and
// its own pinned slots (two, so that the link works on one while the thread works on the other) and
// enqueues the device copy on the null stream, in whose order the kernels follow.  A call of one batch
// (small grids) stays on the calling thread: its arrays share a slot and a single wait.  Memory that the
// runtime knows (pinned by the caller: the link reads it without a slot; or device memory, which the host
// may not be able to read) is left to hipMemcpy.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <thread>
#include <vector>

namespace zq3d {

// One array of a copy.
struct HostSpan {
    void* dev;
    const void* host;  // written to by to_host
    size_t bytes;
};

// Calls are serialised by the owner (the workspace's mutex).
class HostCopy {
public:
    hipError_t to_device(std::initializer_list<HostSpan> a) { return run(a, true); }
    // (waits for the work before it on the null stream)
    hipError_t to_host(std::initializer_list<HostSpan> a) { return run(a, false); }

    // gives the pinned slots back and ends the threads
    void release() {
        if (pool_ && pool_->pid == getpid()) {
            std::unique_lock<std::mutex> lk(pool_->mu);
            pool_->stop = true;
            pool_->wake.notify_all();
            pool_->done.wait(lk, [&] { return pool_->alive == 0; });
            lk.unlock();
            delete pool_;
        }
        pool_ = nullptr;
        for (Lane& l : lane_) {
            for (int i = 0; i < 2; i++) {
                if (l.used[i]) (void)hipEventSynchronize(l.ev[i]);
                if (l.ev[i]) (void)hipEventDestroy(l.ev[i]);
                if (l.slot[i]) (void)hipHostFree(l.slot[i]);
            }
            l = Lane{};
        }
    }

private:
    static constexpr size_t kSlot = 2u << 20;
    static constexpr int kLanes = 6;  // the calling thread and five more: 24 MiB of slots at most

    struct Piece {
        char* dev;
        char* host;
        size_t bytes, at;  // at: offset in the slot
    };
    struct Batch {
        size_t first, count;  // pieces
    };
    struct Lane {
        char* slot[2] = {};
        hipEvent_t ev[2] = {};
        bool used[2] = {};  // the device may still read the slot until its event
    };
    // Threads wait here between calls.  Never destroyed while they live: at process exit they just end.
    struct Pool {
        std::mutex mu;
        std::condition_variable wake, done;
        HostCopy* job = nullptr;
        unsigned turn = 0;
        int alive = 0, busy = 0;
        bool stop = false;
        pid_t pid = getpid();
    };

    static void serve(Pool* p, int lane) {
        unsigned seen = 0;
        std::unique_lock<std::mutex> lk(p->mu);
        for (;;) {
            p->wake.wait(lk, [&] { return p->stop || p->turn != seen; });
            if (p->stop) break;
            seen = p->turn;
            HostCopy* c = p->job;
            lk.unlock();
            c->work(lane);
            lk.lock();
            if (--p->busy == 0) p->done.notify_all();
        }
        if (--p->alive == 0) p->done.notify_all();
    }

    hipError_t ready(Lane& l, int i) {
        if (l.slot[i]) return hipSuccess;
        hipError_t e = hipSuccess;
        if (!l.ev[i]) e = hipEventCreateWithFlags(&l.ev[i], hipEventDisableTiming);
        void* p = nullptr;
        if (e == hipSuccess) e = hipHostMalloc(&p, kSlot, hipHostMallocDefault);
        if (e == hipSuccess) l.slot[i] = (char*)p;
        return e;
    }

    void work(int lane) {
        hipError_t e = hipSetDevice(device_);
        if (e == hipSuccess) e = to_dev_ ? push(lane_[lane]) : pull(lane_[lane]);
        if (e != hipSuccess) {
            hipError_t none = hipSuccess;
            err_.compare_exchange_strong(none, e);
        }
    }

    // without a slot (no pinned memory to be had): the batch by plain copies
    hipError_t plain(size_t b) {
        (void)hipGetLastError();
        hipError_t e = hipSuccess;
        for (size_t k = batches_[b].first; k < batches_[b].first + batches_[b].count && e == hipSuccess; k++) {
            const Piece& q = pieces_[k];
            e = to_dev_ ? hipMemcpy(q.dev, q.host, q.bytes, hipMemcpyHostToDevice)
                        : hipMemcpy(q.host, q.dev, q.bytes, hipMemcpyDeviceToHost);
        }
        return e;
    }

    hipError_t push(Lane& l) {
        hipError_t e = hipSuccess;
        for (int i = 0; e == hipSuccess; i ^= 1) {
            const size_t b = next_.fetch_add(1);
            if (b >= batches_.size()) break;
            if (ready(l, i) != hipSuccess) {
                e = plain(b);
                continue;
            }
            if (l.used[i] && (e = hipEventSynchronize(l.ev[i])) != hipSuccess) break;
            l.used[i] = false;
            for (size_t k = batches_[b].first; k < batches_[b].first + batches_[b].count && e == hipSuccess; k++) {
                const Piece& q = pieces_[k];
                std::memcpy(l.slot[i] + q.at, q.host, q.bytes);
                e = hipMemcpyAsync(q.dev, l.slot[i] + q.at, q.bytes, hipMemcpyHostToDevice, 0);
                l.used[i] = true;
            }
            if (l.used[i]) {
                const hipError_t r = hipEventRecord(l.ev[i], 0);
                if (e == hipSuccess) e = r;
            }
        }
        return e;
    }

    hipError_t pull(Lane& l) {
        hipError_t e = hipSuccess;
        const size_t none = ~(size_t)0;
        size_t in_slot[2] = {none, none};
        for (int i = 0;; i ^= 1) {
            size_t b = none;
            if (e == hipSuccess && (b = next_.fetch_add(1)) >= batches_.size()) b = none;
            bool copied = false;
            if (b != none && ready(l, i) != hipSuccess) {
                e = plain(b);
                copied = true;
            } else if (b != none) {
                if (l.used[i]) e = hipEventSynchronize(l.ev[i]);
                for (size_t k = batches_[b].first; k < batches_[b].first + batches_[b].count && e == hipSuccess; k++) {
                    const Piece& q = pieces_[k];
                    e = hipMemcpyAsync(l.slot[i] + q.at, q.dev, q.bytes, hipMemcpyDeviceToHost, 0);
                    l.used[i] = true;
                }
                if (e == hipSuccess) e = hipEventRecord(l.ev[i], 0);
                if (e == hipSuccess) in_slot[i] = b;
            }
            const int o = i ^ 1;  // the batch before, while this one is on its way
            if (in_slot[o] != none) {
                const hipError_t r = hipEventSynchronize(l.ev[o]);
                l.used[o] = false;
                const Batch& done = batches_[in_slot[o]];
                if (r == hipSuccess)
                    for (size_t k = done.first; k < done.first + done.count; k++)
                        std::memcpy(pieces_[k].host, l.slot[o] + pieces_[k].at, pieces_[k].bytes);
                else if (e == hipSuccess) e = r;
                in_slot[o] = none;
            } else if (in_slot[i] == none && !copied) {
                return e;
            }
        }
    }

    // whether the host array is ordinary memory (a query is about a microsecond)
    static bool pageable(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // (runtimes that report such memory as an error)
        return true;
    }

    static hipError_t copy(const HostSpan& s, bool to_dev) {
        return to_dev ? hipMemcpy(s.dev, s.host, s.bytes, hipMemcpyHostToDevice)
                      : hipMemcpy(const_cast<void*>(s.host), s.dev, s.bytes, hipMemcpyDeviceToHost);
    }

    // the ordinary arrays as batches of a slot each, small arrays sharing one
    void plan(std::initializer_list<HostSpan> a) {
        pieces_.clear();
        batches_.clear();
        direct_.clear();
        size_t at = kSlot;
        for (const HostSpan& s : a) {
            if (s.bytes && !pageable(s.host)) {
                direct_.push_back(s);
                continue;
            }
            for (size_t o = 0; o < s.bytes;) {
                if (at >= kSlot) {
                    batches_.push_back(Batch{pieces_.size(), 0});
                    at = 0;
                }
                const size_t n = std::min(s.bytes - o, kSlot - at);
                pieces_.push_back(Piece{(char*)s.dev + o, (char*)const_cast<void*>(s.host) + o, n, at});
                batches_.back().count++;
                o += n;
                at = (at + n + 255) & ~(size_t)255;
            }
        }
    }

    void start() {
        if (pool_ && pool_->pid == getpid()) return;
        pool_ = new Pool;  // (after a fork the threads are the parent's: that pool is left alone)
        for (int i = 1; i < kLanes; i++) {
            {
                std::lock_guard<std::mutex> lk(pool_->mu);
                pool_->alive++;
            }
            try {
                std::thread(serve, pool_, i).detach();
            } catch (...) {  // fewer threads
                std::lock_guard<std::mutex> lk(pool_->mu);
                pool_->alive--;
                break;
            }
        }
    }

    // the arrays one after the other
    static hipError_t in_turn(std::initializer_list<HostSpan> a, bool to_dev) {
        hipError_t e = hipSuccess;
        for (const HostSpan& s : a)
            if (s.bytes && e == hipSuccess) e = copy(s, to_dev);
        return e;
    }

    // whether two of the host arrays share memory
    static bool overlap(std::initializer_list<HostSpan> a) {
        for (const HostSpan* s = a.begin(); s != a.end(); s++)
            for (const HostSpan* t = a.begin(); t != s; t++) {
                const uintptr_t x = (uintptr_t)s->host, y = (uintptr_t)t->host;
                if (s->bytes && t->bytes && x < y + t->bytes && y < x + s->bytes) return true;
            }
        return false;
    }

    hipError_t run(std::initializer_list<HostSpan> a, bool to_dev) {
        // an error of earlier work on this thread (a launch that failed): the copies may clear it
        const hipError_t before = hipPeekAtLastError();
        const hipError_t e = copy_all(a, to_dev);
        return e != hipSuccess ? e : before;
    }

    hipError_t copy_all(std::initializer_list<HostSpan> a, bool to_dev) {
        // results for one array (a caller's single scalar field as temperature and density): the last one stays
        if (!to_dev && overlap(a)) return in_turn(a, to_dev);
        try {
            plan(a);
            if (batches_.size() > 1) start();
        } catch (...) {  // no memory for the plan: the plain copies
            return in_turn(a, to_dev);
        }
        hipError_t e = hipSuccess;
        for (size_t k = 0; k < direct_.size() && e == hipSuccess; k++) e = copy(direct_[k], to_dev);
        if (e != hipSuccess || batches_.empty()) return e;
        to_dev_ = to_dev;
        next_ = 0;
        err_.store(hipSuccess);
        e = hipGetDevice(&device_);
        if (e != hipSuccess) return e;
        const bool many = batches_.size() > 1 && pool_;
        if (many) {
            std::lock_guard<std::mutex> lk(pool_->mu);
            pool_->job = this;
            pool_->busy = pool_->alive;
            pool_->turn++;
            pool_->wake.notify_all();
        }
        work(0);
        if (many) {
            std::unique_lock<std::mutex> lk(pool_->mu);
            pool_->done.wait(lk, [&] { return pool_->busy == 0; });
        }
        return err_;
    }

    std::vector<Piece> pieces_;
    std::vector<Batch> batches_;
    std::vector<HostSpan> direct_;  // arrays that hipMemcpy takes
    std::atomic<size_t> next_{0};
    std::atomic<hipError_t> err_{hipSuccess};
    bool to_dev_ = false;
    int device_ = 0;
    Lane lane_[kLanes];
    Pool* pool_ = nullptr;
};

}  // namespace zq3d
