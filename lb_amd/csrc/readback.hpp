// readback.hpp -- planes of a context to the caller's FP64 arrays.
//
// A copy into the caller's ordinary memory runs at 10 to 17 GB/s: the runtime
// stages it through one thread, which also takes the page faults of a fresh
// array.  Here chunks go through a ring of pinned slots, and several threads
// move them on, so that the link, the page faults and the copies overlap; the
// planes cross the link in the arithmetic type (the widening to FP64 is exact).
// Four fields: 256^3 FP32 53.6 -> 10.4 ms, 192^3 FP16 21 -> 5.0, 160 x 144 x 160
// FP64 6.7 -> 4.2 (the link's 28 GB/s), 32^3 FP32 (one slot, one thread) 0.19 -> 0.08.
#pragma once

#include <algorithm>
#include <atomic>
#include <memory>
#include <new>
#include <thread>

#include "context.hpp"

// True where np planes go through the ring, which the first such read of a
// context allocates (false too if there is no pinned memory): where one slot holds
// them, which takes no other thread, and from 96 MiB on.  Between, the copies into
// the caller's memory stay: a caller's own thread pool that spins on every CPU
// between its uses (OpenMP's default) was held up for some 10 ms after the ring's
// threads had run.  With such a pool, a pass of the 130x98x114 cavity (46 MB)
// took 17.8 ms without the ring and 20.5 with it, the 203x97x131 box (82 MB) 16.3 and
// 24.6; the 256^3 box (537 MB) 251 and 227, the 160x144x160 FP64 box (118 MB) 52.5 and
// 47.1.
static inline bool ring_ready(lbm_ctx* c, double* const* dst, int np)
{
    // planes that share memory keep the order of the copies, the last one's values:
    // the ring's threads would write them in any order
    for (int k = 0; k < np; ++k)
        for (int l = 0; l < k; ++l)
            if (dst[k] && dst[l] && dst[l] < dst[k] + c->NU && dst[k] < dst[l] + c->NU) return false;
    const size_t bytes = (size_t)np * c->NU * sizeof(double);
    if (bytes > RB_SLOT && bytes < RB_MANY) return false;
    if (c->rb_host) return true;
    // no more slots than five FP64 planes fill
    c->rb_slots = (int)std::min<size_t>(RB_SLOTS, (5 * c->NU * sizeof(double) + RB_SLOT - 1) / RB_SLOT);
    for (int k = 0; k < c->rb_slots; ++k)
        if (!c->rb_ev[k] && hipEventCreateWithFlags(&c->rb_ev[k], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            c->rb_ev[k] = nullptr;
            return false;
        }
    if (hipHostMalloc((void**)&c->rb_host, RB_SLOT * c->rb_slots, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        c->rb_host = nullptr;
        return false;
    }
    return true;
}

// np planes of c->NU values each, consecutive at src, divided by div, to dst[k]
// (null: not wanted).  Returns when they have arrived.
template <class S>
static lbm_status read_planes(lbm_ctx* c, const S* src, double* const* dst, int np, double div = 1.0)
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

    const int K = c->rb_slots;
    auto slot = [&](int j) { return (S*)(c->rb_host + (size_t)(j % K) * RB_SLOT); };
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
    // one thread more for every 2 MB, up to 7
    std::vector<std::thread> team;
    const int nt = (int)std::min<size_t>({7, std::max(2u, std::thread::hardware_concurrency()) / 2 - 1,
                                          (size_t)n * RB_SLOT / RB_PER_THREAD});
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
