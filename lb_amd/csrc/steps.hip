// steps.hip -- the launches of the collide-stream step for one storage format,
// LBM_STORE (StoreF64, StoreF32, ...); compiled once per format.
#include "context.hpp"

#ifndef LBM_STORE
#error "LBM_STORE names the storage policy of this translation unit"
#endif

// One step of either parity, with the streaming hint (nt) or without.
template <class ST, int COLL, bool LIT, bool FLAGS, bool CC, bool INL>
static void launch_step(bool odd, bool nt, dim3 grid, hipStream_t s, const StepArgs<ST>& a)
{
    if (!nt) {
        if (odd) k_step<ST, COLL, LIT, true, FLAGS, CC, INL, false><<<grid, TPB, 0, s>>>(a);
        else k_step<ST, COLL, LIT, false, FLAGS, CC, INL, false><<<grid, TPB, 0, s>>>(a);
    } else if constexpr (sizeof(typename ST::T) == 2 && COLL == LBM_COLLISION_CUM2015 && FLAGS && !CC && !INL) {
        if (odd) k_step_w7<ST, true><<<grid, TPB, 0, s>>>(a);
        else k_step_w7<ST, false><<<grid, TPB, 0, s>>>(a);
    } else {
        if (odd) k_step<ST, COLL, LIT, true, FLAGS, CC, INL, true><<<grid, TPB, 0, s>>>(a);
        else k_step<ST, COLL, LIT, false, FLAGS, CC, INL, true><<<grid, TPB, 0, s>>>(a);
    }
}

template <class ST, int COLL, bool FLAGS>
static void launch_mlp(bool odd, bool nt, dim3 grid, hipStream_t s, const MlpStepArgs<ST>& a)
{
    if (odd && nt) k_step_mlp<ST, COLL, true, FLAGS, true><<<grid, TPB, 0, s>>>(a);
    else if (odd) k_step_mlp<ST, COLL, true, FLAGS, false><<<grid, TPB, 0, s>>>(a);
    else if (nt) k_step_mlp<ST, COLL, false, FLAGS, true><<<grid, TPB, 0, s>>>(a);
    else k_step_mlp<ST, COLL, false, FLAGS, false><<<grid, TPB, 0, s>>>(a);
}

template <class ST, int COLL, bool LIT>
static lbm_status launch_steps(lbm_ctx* c, int nsteps)
{
    using R = typename ST::R;
    StepArgs<ST> a;
    std::memset(&a, 0, sizeof(a));
    fill_common<ST>(c, a.p, a.rest, a.K);
    a.cls = c->cls;
    a.node = c->node;
    a.bcidx = c->bcidx;
    a.inl_state = (R*)c->inl_state;
    a.inl = c->inl;
    a.pub_mac = (R*)c->pub_mac;
    a.pub_post = (R*)c->pub_post;
    a.inl_post = (R*)c->inl_post;
    a.inl_mac = (R*)c->inl_mac;
    a.macro = (const R*)c->macro;
    a.partials = c->diag_dst ? c->diag_dst : c->partials;
    a.ccache = c->ccache;
    a.g = c->g;
    a.sp_axis = c->sp_axis;
    a.sp_begin = c->sp_begin;
    a.sp_deriv = ((R)c->d.sponge_high - (R)c->d.sponge_low) / (R)c->sp_interval;
    a.outl = c->outl;
    a.cs = outlet_cs<R>(c);
    a.omega0 = R(1) / (R)c->d.tau;   // 1.f / tau (OmegaNo.h:44, NonDim...h:114)
    a.tau = (R)c->d.tau;
    a.cles = (R)c->d.c_les;
    a.crev20 = (c->d.compat & LBM_COMPAT_CREV20) ? 1 : 0;
    a.closure = c->d.closure;
    const bool mlp = c->d.closure == LBM_CLOSURE_MLP;
    MlpStepArgs<ST> ma;
    if (mlp) {
        if (!c->mlp_ready) return LBM_E_STATE;
        ma.mlp = closure_weights(c);
    }
    const bool patches = (c->n_upd && !c->inl_deferred) || c->n_eq || (c->n_outlet && !c->outl_deferred) ||
                         c->n_ghost;
    const dim3 grid((unsigned)c->g.ntiles);
    HIPCHK(hipEventRecord(c->ev0, c->stream));
    for (int s = 0; s < nsteps; ++s) {
        a.first = c->first ? 1 : 0;
        // a counted state is added by the step that reads it; the network step
        // does not fuse the add, so it gets its own pass first
        if (mlp && c->avg_pending && c->cl_count % c->cl_every == 0) {
            lbm_status st = avg_flush_st<ST>(c);
            if (st != LBM_OK) return st;
        }
        a.avg = c->avg_pending ? c->avg : nullptr;
        c->avg_pending = false;
        a.diag = (s == 0 && c->diag_next) ? 1 : 0;
        a.pub_post = (R*)pub_records(c, c->steps);
        a.pub_prev = (const R*)pub_records(c, c->steps - 1);
        a.outl_pending = c->outl_pending ? 1 : 0;
        a.inl_pending = c->inl_pending ? 1 : 0;
        if constexpr (ST::sr) a.seed = step_seed((uint64_t)c->steps);
        const bool odd = (c->steps & 1) != 0;
        a.g.back = odd && c->turn;
        const bool nt = odd ? c->nt_odd : c->nt_even;
        if constexpr (sizeof(R) == 4 && !LIT && COLL <= LBM_COLLISION_CUM2015) {
            if (mlp && c->cl_count % c->cl_every == 0) {
                // network evaluated in this step; coefficients kept for the next ones
                ma.s = a;
                if (c->flags_needed) launch_mlp<ST, COLL, true>(odd, nt, grid, c->stream, ma);
                else launch_mlp<ST, COLL, false>(odd, nt, grid, c->stream, ma);
            } else if (mlp) {
                if (c->flags_needed) launch_step<ST, COLL, false, true, true, false>(odd, nt, grid, c->stream, a);
                else launch_step<ST, COLL, false, false, true, false>(odd, nt, grid, c->stream, a);
            }
            if (mlp) c->cl_count++;
        }
        if (!mlp) {
            if (!c->flags_needed) launch_step<ST, COLL, LIT, false, false, false>(odd, nt, grid, c->stream, a);
            else if (c->inl_deferred) launch_step<ST, COLL, LIT, true, false, true>(odd, nt, grid, c->stream, a);
            else launch_step<ST, COLL, LIT, true, false, false>(odd, nt, grid, c->stream, a);
        }
        HIPCHK(hipGetLastError());
        if (patches) {
            lbm_status st = launch_patches<ST>(c, odd ? 0 : 1);
            if (st != LBM_OK) return st;
        }
        c->first = false;
        c->steps++;
        c->outl_pending = c->outl_deferred;
        c->inl_pending = c->inl_deferred;
        if (c->avg_each) {
            c->avg_pending = true;
            c->avg_count++;
        }
    }
    HIPCHK(hipEventRecord(c->ev1, c->stream));
    return LBM_OK;
}

template <class ST, bool LIT>
static lbm_status launch_coll(lbm_ctx* c, int nsteps)
{
    switch (c->d.collision) {
    case LBM_COLLISION_CUM2015: return launch_steps<ST, LBM_COLLISION_CUM2015, LIT>(c, nsteps);
    case LBM_COLLISION_CUM2017: return launch_steps<ST, LBM_COLLISION_CUM2017, LIT>(c, nsteps);
    case LBM_COLLISION_COMBINED: return launch_steps<ST, LBM_COLLISION_COMBINED, LIT>(c, nsteps);
    default: return launch_steps<ST, LBM_COLLISION_SRT, LIT>(c, nsteps);
    }
}

template <class ST>
lbm_status launch_by_coll(lbm_ctx* c, int nsteps)
{
    // 16-bit storage runs the fast arithmetic only (checked when the lattice is created)
    if constexpr (sizeof(typename ST::T) > 2) {
        if (c->d.arith == LBM_ARITH_LITERAL) return launch_coll<ST, true>(c, nsteps);
    }
    return launch_coll<ST, false>(c, nsteps);
}

template lbm_status launch_by_coll<LBM_STORE>(lbm_ctx*, int);
