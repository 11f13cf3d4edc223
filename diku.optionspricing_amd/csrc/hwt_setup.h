// hwt_setup.h -- what prepares one option for FP64 pricing (hwt_tri.h): its constants,
// its two discount bonds and the way it is priced.  Run a thread per option by k_setup
// and a wave per option by k_price_small.
#pragma once

#include "hwt_tri.h"

namespace hwt {

// An option's fields in a batch.
struct OptFields {
    double strike, maturity, length, a, sigma;
    uint16_t term_unit, term_steps;
    int8_t type;
};
__device__ __forceinline__ OptFields option_fields(const DevOpts &o, int i)
{
    return OptFields{o.strike[i], o.maturity[i], o.length[i], o.a[i], o.sigma[i], o.term_unit[i], o.term_steps[i], o.type[i]};
}

// Option i's constants, from its fields f or from the constants the caller gave;
// returns ST_*.
__device__ __forceinline__ int32_t option_record(const DevOpts &o, int i, OptFields &f, int32_t maxWidth, OptConst &c)
{
    int32_t st;
    if (o.consts) {
        const hwt_option_constants_f64 k = o.consts[i];
        f.term_unit = k.term_unit;
        st = constants_given(k.t, k.dt, k.dr, k.X, k.M, k.jmax, k.n, k.width, k.term_unit, k.type, maxWidth,
                             o.consts_f32 != 0, c);
    } else {
        st = option_constants(f.strike, f.maturity, f.length, f.term_unit, f.term_steps, f.a, f.sigma, f.type, maxWidth, c);
    }
    c.status = st;
    return st;
}

enum TriKind { TRI_DONE, TRI_GROUPED, TRI_WINDOWED, TRI_GENERAL };

// The price of an option that needs no tree (TRI_DONE), or how its tree is priced,
// with the edge record and the windows' sort key.
template <class Yield>
__device__ __forceinline__ TriKind tri_setup(OptConst &c, int tu, Yield &&yield, bool spread, double unit_dmin,
                                             TriEdge &edges, int64_t &key, double &value)
{
    if (c.status != ST_OK) {
        value = NAN;
        return TRI_DONE;
    }
    value = 100.0;  // no steps: the face value (seq/Seq.hpp:119,171)
    if (c.n == 0) return TRI_DONE;
    const double tn = c.n * c.dt;
    c.Pn = exp(-yield(tn, tu) * tn);
    value = 100.0 * c.Pn;  // exercise outside the tree: the zero-coupon bond
    if (c.e < 0) return TRI_DONE;
    const double te = c.e * c.dt;
    c.Pe = exp(-yield(te, tu) * te);
    TreeShape t{c.w, c.jmax, c.M, c.dr, c.dt, 0.0, 0.0};
    const EdgeDiscounts ed = edge_discounts(t);
    edge_factors(t, ed);
    edges = tri_edge(t, ed);
    c.rho = t.rho;
    c.rhop = t.rhop;
    const bool grouped = c.w <= (spread ? TRI_SPREAD_WIDTH : TRI_GROUP_WIDTH);
    int lo = c.jmax, up = c.jmax, half = c.jmax;
    if (!grouped) {
        // priced over the nodes that carry weight, most at step n
        c.sigmas = window_sigmas(c);
        const Reach reach = make_reach(c.sigmas, c.M, c.dr, c.dt, c.n, c.jmax);
        key = (int64_t)reach_updates(reach, c.n, c.e);
        reach_at(reach, c.n, min(c.e, c.jmax) + (c.n - c.e), lo, up);
        // a window's other nodes have scales too: whole lanes' spare nodes lie up to
        // WAVE - 1 beyond those kept, and the smallest window is MIN_WINDOW nodes a lane
        half = min(max(max(lo, up) + WAVE - 1, MIN_WINDOW * WAVE - 1), c.jmax);
    }
    if (tri_ok(t, edges, c.n, half, grouped ? 100.0f : 200.0f) && (grouped || lo + up + 17 <= TRI_MAX_NODES))
        return grouped ? TRI_GROUPED : TRI_WINDOWED;
    // the general kernel's scales (unit_form_ok)
    double etab[EDGE_TAB];
    edge_table(t, etab);
    c.unit = unit_form_ok(t, etab, unit_dmin) ? 1 : 0;
    c.sigmas = window_sigmas(c);
    return TRI_GENERAL;
}

} // namespace hwt
