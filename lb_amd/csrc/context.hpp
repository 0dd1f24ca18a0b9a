// context.hpp -- one lattice context: its device buffers, the kernel arguments
// formed from it and the launches shared by the core's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/lbm_closure.h"
#include "lbm_kernels.hpp"

using namespace lbm;

// pinned ring of the read-backs (readback.hpp): its slots, bytes of a slot
static constexpr int RB_SLOTS = 16;
static constexpr size_t RB_SLOT = 1 << 20;
static constexpr size_t RB_MANY = 256 << 20;   // the ring's threads are used from here on

struct lbm_ctx {
    lbm_desc d;
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    size_t N = 0;              // padded cells
    size_t NP = 0;             // population plane stride: N up to a whole cache line
    bool turn = false;         // odd steps take the tiles from the last to the first
    bool nt_even = false, nt_odd = false;   // the step takes the streaming hint
    size_t NU = 0;             // caller's cells
    size_t elem = 0;           // bytes per stored population
    size_t rbytes = 0;         // bytes per arithmetic value
    Geo g{};
    bool flags_needed = false; // any non-fluid cell (halo included)
    int n_inlet = 0, n_eq = 0, n_outlet = 0, n_ghost = 0, n_pub = 0;
    int n_interp = 0;             // interpolated outlet entries
    int n_upd = 0;                // moving-wall and Zou-He inlet entries
    std::vector<int> ghost_off;  // launch boundaries of the ghost list (dependency levels)
    void* pops = nullptr;
    uint8_t* cls = nullptr;
    uint64_t* node = nullptr;
    int32_t* bcidx = nullptr;
    void* inl_state = nullptr;
    NodeDev* inl = nullptr;
    NodeDev* outl = nullptr;
    NodeDev* ghost = nullptr;
    void* pub_mac = nullptr;
    void* inl_post = nullptr;     // hand-over to the inlet rule (k_inlet_state, or deferred): f* and rho, u
    void* inl_mac = nullptr;
    void* pub_post = nullptr;
    void* macro = nullptr;     // 4 planes, arithmetic type, padded layout
    double* stage = nullptr;   // 5 planes FP64, caller layout
    double* partials = nullptr;
    std::vector<double> h_partials;
    int64_t steps = 0;
    bool initialized = false;
    bool first = false;
    bool nan_seen = false;
    bool diag_next = false;    // the next launched step reduces mass, momentum and wall force
    double last_ms = 0.0;
    size_t dev_bytes = 0;
    // learned closure
    bool mlp_ready = false;
    float* cl_params = nullptr;   // FP32 parameters
    uint16_t* cl_wb = nullptr;    // BF16 W1 [64][16] + W2 [64][64]
    float cl_b3 = 0.0f;
    float* cl_norm = nullptr;     // [4][12] mean, 1/sd, envelope low, high
    float* ccache = nullptr;      // coefficient per cell held between network evaluations
    int cl_every = 1;             // evaluate the network every cl_every steps
    int64_t cl_count = 0;         // steps since the last (re)start of the refresh cycle
    // time averaging (MomentTimeAvg)
    double* avg = nullptr;        // 4 FP64 planes, caller layout: sums of rho, ux, uy, uz
    int64_t avg_count = 0;        // states added
    bool avg_pending = false;     // the current state is counted but not yet added
    bool avg_each = false;        // launch_steps: count the state after every step
    // probe records taken without a synchronisation
    double* probe_buf = nullptr;  // [PROBE_CAP][4] on the device
    int probe_n = 0;              // records in probe_buf
    std::vector<double> probe_host;  // records drained from the device, oldest first
    // outlet omega damping
    int sp_axis = -1, sp_begin = 0, sp_interval = 1;
    // ErrorQuadratic on the device
    std::vector<uint8_t> h_flag1;   // flag == 1 per caller cell (the cells the norm sums over)
    uint8_t* flag1 = nullptr;       // the same on the device, uploaded by the first evaluation
    void* uerr = nullptr;           // previous velocity, 3 planes of the arithmetic type, caller layout
    // per-block partials of a diagnostics step go here instead of `partials` when set
    double* diag_dst = nullptr;
    // read-backs
    hipEvent_t rb_ev[RB_SLOTS] = {};
    // asynchronous snapshots: rho, u, omega into snap_dev on the context stream,
    // then a copy to pinned host memory on copy_stream while steps go on
    double* snap_dev = nullptr;       // 5 planes FP64, caller layout
    double* snap_host = nullptr;      // pinned, 5 planes
    hipStream_t copy_stream = nullptr;
    hipEvent_t ev_snap = nullptr, ev_snap_copy = nullptr;
    bool snap_pending = false;
    int64_t snap_step = 0;
    // Deferred interpolated outlet: the rule runs in the next reader of an
    // outlet cell, with the post-collision records of the step that produced
    // the state.  Records alternate between pub_post (even steps) and
    // pub_post2 (odd steps), so a step can read the previous step's while
    // writing its own.
    bool outl_deferred = false;
    bool outl_pending = false;      // the current state's outlet cells still need the rule
    void* pub_post2 = nullptr;
    // Deferred inlet: the moving-wall and Zou-He rules run in the next
    // step's kernel from the records (inl_post, inl_mac) of the step that
    // produced the state.
    bool inl_deferred = false;
    bool inl_pending = false;       // the inlet cells' stored state still needs its rule
};

static constexpr int PROBE_CAP = 4096;

// The interpolated outlet's weight c_s = 1/sqrt(3) (OutletDensityInterpolated.h:226)
// in the constants' precision.
template <class R>
static inline R outlet_cs(const lbm_ctx* c)
{
    return (c->d.compat & LBM_COMPAT_F32CONST) ? (R)(1.f / sqrtf(3.f)) : (R)(1.0 / std::sqrt(3.0));
}

// Post-collision records written by step t (deferred outlet: alternating buffers).
static inline void* pub_records(const lbm_ctx* c, int64_t t)
{
    return (c->outl_deferred && (t & 1)) ? c->pub_post2 : c->pub_post;
}

#define HIPCHK(x)                                   \
    do {                                            \
        hipError_t e_ = (x);                        \
        if (e_ != hipSuccess) return LBM_E_HIP;     \
    } while (0)

static inline lbm_status dev_alloc(lbm_ctx* c, void** p, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return LBM_E_OOM;
    }
    c->dev_bytes += bytes;
    return LBM_OK;
}

template <class ST>
static inline void fill_common(const lbm_ctx* c, typename ST::T** p, typename ST::R* rest, Consts<typename ST::R>& K)
{
    using R = typename ST::R;
    K = make_consts<R>(c->d.compat);
    for (int k = 0; k < 4; ++k) rest[k] = ST::dev ? (R)(K.w[k] * (R)c->d.rho0) : R(0);
    typename ST::T* base = (typename ST::T*)c->pops;
    for (int q = 0; q < Q; ++q) p[q] = base + (size_t)q * c->NP;
}

static inline MlpWeights closure_weights(const lbm_ctx* c)
{
    MlpWeights W;
    W.w1 = c->cl_wb;
    W.w2 = c->cl_wb ? c->cl_wb + NHID * 16 : nullptr;
    W.b1 = c->cl_params ? c->cl_params + OFF_B1 : nullptr;
    W.b2 = c->cl_params ? c->cl_params + OFF_B2 : nullptr;
    W.w3 = c->cl_params ? c->cl_params + OFF_W3 : nullptr;
    W.norm = c->cl_norm;
    W.b3 = c->cl_b3;
    W.c = (float)c->d.c_les;
    return W;
}

template <class ST>
static inline AuxArgs<ST> aux_args(const lbm_ctx* c)
{
    using R = typename ST::R;
    AuxArgs<ST> a;
    std::memset(&a, 0, sizeof(a));
    fill_common<ST>(c, a.p, a.rest, a.K);
    a.cls = c->cls;
    a.bcidx = c->bcidx;
    a.inl_state = (R*)c->inl_state;
    a.macro = (R*)c->macro;
    a.g = c->g;
    a.tau = (R)c->d.tau;
    a.cles = (R)c->d.c_les;
    a.omega0 = R(1) / (R)c->d.tau;
    a.closure = c->d.closure;
    a.lit = c->d.arith == LBM_ARITH_LITERAL;
    a.odd = (int)(c->steps & 1);
    a.first = c->first ? 1 : 0;
    a.io = c->stage;
    a.sp_axis = c->sp_axis;
    a.sp_begin = c->sp_begin;
    a.sp_deriv = ((R)c->d.sponge_high - (R)c->d.sponge_low) / (R)c->sp_interval;
    a.outl_pending = c->outl_pending ? 1 : 0;
    a.outl = c->outl;
    a.pub_prev = (const R*)pub_records(c, c->steps - 1);
    a.cs = outlet_cs<R>(c);
    a.crev20 = (c->d.compat & LBM_COMPAT_CREV20) ? 1 : 0;
    a.inl_pending = c->inl_pending ? 1 : 0;
    a.inl = c->inl;
    a.inl_post = (const R*)c->inl_post;
    a.inl_mac = (const R*)c->inl_mac;
    return a;
}

static inline unsigned blocks_for(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

template <class ST>
static inline PatchArgs<ST> patch_args(const lbm_ctx* c)
{
    using R = typename ST::R;
    PatchArgs<ST> a;
    std::memset(&a, 0, sizeof(a));
    fill_common<ST>(c, a.p, a.rest, a.K);
    a.cls = c->cls;
    a.bcidx = c->bcidx;
    a.inl_state = (R*)c->inl_state;
    a.pub_mac = (const R*)c->pub_mac;
    a.pub_post = (const R*)c->pub_post;
    a.g = c->g;
    a.nu = (R)c->d.nu;
    // the outlet's interpolation weight (OutletDensityInterpolated.h:226) is
    // 1/sqrt(3) in the constants' precision
    a.cs = outlet_cs<R>(c);
    a.inletrho = (c->d.compat & LBM_COMPAT_INLETRHO) ? 1 : 0;
    a.crev20 = (c->d.compat & LBM_COMPAT_CREV20) ? 1 : 0;
    return a;
}

// Boundary rules that read what other cells produced in the same step, in
// the reference's order: inlet, outlet, periodic.
template <class ST>
static inline lbm_status launch_patches(lbm_ctx* c, int odd_next)
{
    PatchArgs<ST> a = patch_args<ST>(c);
    a.odd = odd_next;
    a.pub_post = (const typename ST::R*)pub_records(c, c->steps);   // this step's records
    if (c->n_upd && !c->inl_deferred) {
        PatchArgs<ST> u = a;
        u.nodes = c->inl;
        u.n = c->n_inlet;
        u.pub_mac = (const typename ST::R*)c->inl_mac;
        u.pub_post = (const typename ST::R*)c->inl_post;
        k_inlet_state<ST><<<blocks_for(u.n), TPB, 0, c->stream>>>(u);
    }
    const int n_interp = c->outl_deferred ? 0 : c->n_interp;
    if (c->n_eq || n_interp) {
        a.nodes = c->inl;
        a.n = c->n_eq ? c->n_inlet : 0;
        const int bi = (a.n + NODES_PER_BLOCK - 1) / NODES_PER_BLOCK;
        const int no = n_interp ? c->n_outlet : 0;
        k_inlet_outlet<ST><<<bi + (no + NODES_PER_BLOCK - 1) / NODES_PER_BLOCK, TPB, 0, c->stream>>>(a, c->outl, no, bi);
    }
    if (c->n_outlet > c->n_interp) {
        a.nodes = c->outl;
        a.n = c->n_outlet;
        k_outlet_eq<ST><<<blocks_for(a.n), TPB, 0, c->stream>>>(a);
    }
    for (size_t l = 0; l + 1 < c->ghost_off.size(); ++l) {
        a.nodes = c->ghost + c->ghost_off[l];
        a.n = c->ghost_off[l + 1] - c->ghost_off[l];
        k_periodic<ST><<<blocks_for(a.n), TPB, 0, c->stream>>>(a);
    }
    HIPCHK(hipGetLastError());
    return LBM_OK;
}

// Add the pending state to the time-average sums with its own pass.
template <class ST>
static inline lbm_status avg_flush_st(lbm_ctx* c)
{
    if (!c->avg_pending) return LBM_OK;
    AuxArgs<ST> a = aux_args<ST>(c);
    a.io = c->avg;
    k_moment_add<ST><<<blocks_for(c->NU), TPB, 0, c->stream>>>(a);
    HIPCHK(hipGetLastError());
    c->avg_pending = false;
    return LBM_OK;
}

// Seed of the stochastic-rounding stores of step t (any fixed bijective mix
// of the step counter: runs with the same inputs give the same results).
static inline uint32_t step_seed(uint64_t t)
{
    uint64_t x = t * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    x ^= x >> 31;
    x *= 0xBF58476D1CE4E5B9ull;
    x ^= x >> 27;
    return (uint32_t)(x >> 32);
}

// Queue nsteps steps of a context in storage format ST (steps.hip, compiled
// once per format).
template <class ST>
lbm_status launch_by_coll(lbm_ctx* c, int nsteps);
