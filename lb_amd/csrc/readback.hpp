// readback.hpp -- planes of a context to the caller's FP64 arrays.
//
// A copy into the caller's ordinary memory runs at 10 to 17 GB/s: the runtime
// stages it through one thread, which also takes the page faults of a fresh
// array.  Here chunks go through a ring of pinned slots, and several threads
// move them on, so that the link, the page faults and the copies overlap; the
// planes cross the link in the arithmetic type (the widening to FP64 is exact).
// Four fields: 256^3 FP32 41-53 -> 11 ms (the link's 28 GB/s), 32^3 FP32 (one slot,
// one thread) 0.11 -> 0.08.
#pragma once

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

#include "context.hpp"

// Pinned blocks between the reads of all contexts: allocating one takes longer than
// a small read saves, and a program makes many lattices (32^3, first read of a
// lattice: 0.41 ms against 0.31 with the plain copies).  At most KEEP blocks stay, and
// none after the last context.
class PinnedBlocks {
public:
    char* take(size_t bytes)
    {
        {
            std::lock_guard<std::mutex> lock(m);
            for (int k = 0; k < n; ++k)
                if (free_[k].bytes == bytes) {
                    char* p = free_[k].p;
                    free_[k] = free_[--n];
                    return p;
                }
        }
        char* p = nullptr;
        if (hipHostMalloc((void**)&p, bytes, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        return p;
    }
    void give(char* p, size_t bytes)
    {
        {
            std::lock_guard<std::mutex> lock(m);
            if (contexts > 0 && n < KEEP) {
                free_[n++] = {p, bytes};
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void opened()
    {
        std::lock_guard<std::mutex> lock(m);
        ++contexts;
    }
    void closed()
    {
        Block drop[KEEP];
        int k = 0;
        {
            std::lock_guard<std::mutex> lock(m);
            if (--contexts == 0)
                while (n) drop[k++] = free_[--n];
        }
        while (k) (void)hipHostFree(drop[--k].p);
    }

private:
    static constexpr int KEEP = 4;
    struct Block {
        char* p;
        size_t bytes;
    };
    std::mutex m;
    Block free_[KEEP];
    int n = 0, contexts = 0;
};

static inline PinnedBlocks& pinned_blocks()
{
    static PinnedBlocks b;
    return b;
}

// Outputs of at least RB_MANY bytes take the ring, and those that one slot holds,
// which takes no other thread.  Between, the copies into the caller's memory stay: with
// a caller's own thread pool that spins on every CPU between its uses (OpenMP's
// default, the process's share of the CPUs no larger than the pool), one pass in ten
// or more stalled for 10 to 30 ms after such a read.  ms a read and the pool's next use,
// median and 90 % line, copies / ring: 256x128x128 FP32 (128 MiB) 8.5, 8.7 / 4.2, 29.8;
// 192^3 FP32 (216) 23.4, 26.5 / 7.0, 32.2; 208^3 FP32 (275) 36.6, 37.6 / 13.9, 15.8, FP16
// 32.4, 33.2 / 8.0, 8.4; 256^3 FP32 (512) 65.6, 69.0 / 25.0, 27.2.  The line is between the
// largest output that stalled and the smallest that did not, at 30 to 300 steps between
// the reads; why larger ones do not was not found.
class Ring {
public:
    // wanted planes: dst[k] not null.  Planes that share memory keep the order of the
    // copies, the last one's values.
    Ring(lbm_ctx* c, double* const* dst, int np)
    {
        size_t wanted = 0;
        for (int k = 0; k < np; ++k) {
            if (!dst[k]) continue;
            ++wanted;
            for (int l = 0; l < k; ++l)
                if (dst[l] && dst[l] < dst[k] + c->NU && dst[k] < dst[l] + c->NU) return;
        }
        const size_t bytes = wanted * c->NU * sizeof(double);
        if (bytes > RB_SLOT && bytes < RB_MANY) return;
        slots = bytes <= RB_SLOT ? 1 : RB_SLOTS;
        for (int k = 0; k < slots; ++k)
            if (!c->rb_ev[k] && hipEventCreateWithFlags(&c->rb_ev[k], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                c->rb_ev[k] = nullptr;
                return;
            }
        mem = pinned_blocks().take(slots * RB_SLOT);
    }
    ~Ring()
    {
        if (mem) pinned_blocks().give(mem, slots * RB_SLOT);
    }
    Ring(const Ring&) = delete;
    Ring& operator=(const Ring&) = delete;
    explicit operator bool() const { return mem != nullptr; }

    char* mem = nullptr;
    int slots = 0;
};

// np planes of c->NU values each, consecutive at src, divided by div, to dst[k]
// (null: not wanted).  Returns when they have arrived.
template <class S>
static lbm_status read_planes(lbm_ctx* c, const Ring& ring, const S* src, double* const* dst, int np, double div = 1.0)
{
    // a chunk: values [i, i + n) of the planes' run, which may be of several planes
    struct Chunk {
        size_t i, n;
    };
    std::vector<Chunk> ch;
    const size_t per = RB_SLOT / sizeof(S), NU = c->NU;
    std::unique_ptr<std::atomic<bool>[]> done;
    try {
        for (int k = 0, l; k < np; k = l + 1) {   // runs [k, l) of wanted planes
            for (l = k; l < np && dst[l]; ++l) {}
            for (size_t i = (size_t)k * NU; i < (size_t)l * NU; i += per)
                ch.push_back({i, std::min(per, (size_t)l * NU - i)});
        }
        done.reset(new std::atomic<bool>[ch.size()]);
    } catch (const std::bad_alloc&) {
        return LBM_E_OOM;
    }
    const int n = (int)ch.size();
    for (int j = 0; j < n; ++j) done[j] = false;
    std::atomic<int> issued{0}, claimed{0};
    std::atomic<bool> failed{false};

    const int K = ring.slots;
    auto slot = [&](int j) { return (S*)(ring.mem + (size_t)(j % K) * RB_SLOT); };
    auto move = [&](int j) {
        if (hipEventSynchronize(c->rb_ev[j % K]) != hipSuccess) {
            failed = true;
            return;
        }
        const S* s = slot(j);
        for (size_t i = ch[j].i, e = i + ch[j].n; i < e;) {
            const size_t k = i / NU, m = std::min(e, (k + 1) * NU) - i;
            double* d = dst[k] + (i - k * NU);
            if (div == 1.0)
                for (size_t t = 0; t < m; ++t) d[t] = (double)s[t];
            else
                for (size_t t = 0; t < m; ++t) d[t] = (double)s[t] / div;
            s += m;
            i += m;
        }
        done[j].store(true, std::memory_order_release);
    };
    auto worker = [&] {
        for (;;) {
            const int j = claimed.fetch_add(1);
            if (j >= n) return;
            while (issued.load(std::memory_order_acquire) <= j) {
                if (failed) return;
                std::this_thread::yield();
            }
            move(j);
        }
    };
    // a small output takes no other thread, a large one up to 7
    std::vector<std::thread> team;
    const int nt = K == 1 ? 0 : (int)std::min<size_t>({7, std::max(4u, std::thread::hardware_concurrency()) / 2 - 1, (size_t)n - 1});
    try {
        team.reserve(nt);
        for (int t = 0; t < nt; ++t) team.emplace_back(worker);
    } catch (...) {   // fewer threads: this one takes what is left
    }
    int next = 0;
    while (!failed) {
        for (; next < n && (next < K || done[next - K].load(std::memory_order_acquire)); ++next) {
            if (hipMemcpyAsync(slot(next), src + ch[next].i, ch[next].n * sizeof(S), hipMemcpyDeviceToHost, c->stream) !=
                    hipSuccess ||
                hipEventRecord(c->rb_ev[next % K], c->stream) != hipSuccess) {
                failed = true;
                break;
            }
            issued.store(next + 1, std::memory_order_release);
        }
        int j = claimed.load();
        if (j < next && claimed.compare_exchange_strong(j, j + 1))
            move(j);
        else if (j >= n && next == n)   // claimed chunks wait to be issued
            break;
        else
            std::this_thread::yield();
    }
    for (std::thread& t : team) t.join();
    HIPCHK(hipStreamSynchronize(c->stream));
    return failed ? LBM_E_HIP : LBM_OK;
}
