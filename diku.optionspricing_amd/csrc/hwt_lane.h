// hwt_lane.h -- form 1 device code: one lane prices one option.
//
// Each lane owns its option's two tree columns (forward state y, backward
// state b) in global memory, interleaved across the 64 lanes of its wave:
// node k of column c of lane l lives at  base_wave + (c*W + k)*64 + l, so the
// nodes a wave touches in one sweep position form one contiguous 512-byte row
// and every load and store is coalesced.  A step sweeps the active region with
// a three-value sliding window (previous, current, next) in registers and
// recomputes the stencil coefficients on the fly (closed forms, node discounts
// advanced by one multiplication per node, edge nodes from the option's edge
// table).  The same duality as the wave form gives the price from the two
// columns at the exercise step.
//
// Trees the tridiagonal form holds (tri_ok) step in it (lane_price_tri), eight steps
// to a sweep: a sweep is a dependent walk through memory, so what bounds the form
// is its latency and the coefficients formed on the way, and both are paid once
// for the eight steps.  16,384 options on 47-node trees of 108 steps: 1,170 us node
// by node, 266 at four steps to a sweep, 216 with the reads a chunk ahead of use
// and the inner chunks free of branches, 150 at eight steps.
#pragma once

#include "hwt_scale.h"
#include "hwt_tri.h"

namespace hwt {

constexpr int LANE_MAX_WIDTH = WAVE_MAX_WIDTH;
constexpr int LANE_BLOCK = 64;  // lanes per workgroup by default: spreads a small batch's waves over the CUs

struct LaneColumn {
    double *p;  // node 0 of this lane's column
    __device__ double &operator[](int k) const { return p[(size_t)k * WAVE]; }
};

// Sweep one step over [lo, hi] (new region), reading the old state (nonzero
// only on [olo, ohi]) in place.  FWD: forward operator G, else G^T.
template <bool FWD>
__device__ __forceinline__ void lane_sweep(const TreeShape &t, const double *etab, LaneColumn col, int lo, int hi,
                                           int olo, int ohi)
{
    const double q = exp(-t.dr * t.dt);
    double Em = node_disc(lo - 1, t.jmax, t.dr, t.dt);  // E_{k-1}
    double E0 = Em * q, Ep = E0 * q;
    // old value at lo-1: inside the old region when the backward light cone
    // narrows, zero when it lies outside the old region or the tree
    double prev = (lo - 1 >= olo && lo - 1 <= ohi && lo >= 1) ? col[lo - 1] : 0.0;
    double cur = (lo >= olo && lo <= ohi) ? col[lo] : 0.0;
    for (int k = lo; k <= hi; ++k) {
        const double nxt = (k + 1 >= olo && k + 1 <= ohi) ? col[k + 1] : 0.0;
        const int j = k - t.jmax;
        double cl, cm, cr;
        if (k < 3 || k > t.w - 4) {
            const double *e = etab + (FWD ? 0 : 18) + 3 * edge_slot_of(k, t.w);
            cl = e[0];
            cm = e[1];
            cr = e[2];
        } else if (FWD) {
            cl = pu_std(j - 1, t.M) * Em;
            cm = pm_std(j, t.M) * E0;
            cr = pd_std(j + 1, t.M) * Ep;
        } else {
            cl = pd_std(j, t.M) * E0;
            cm = pm_std(j, t.M) * E0;
            cr = pu_std(j, t.M) * E0;
        }
        col[k] = fma(cr, nxt, fma(cl, prev, cm * cur));
        prev = cur;
        cur = nxt;
        Em = E0;
        E0 = Ep;
        Ep *= q;
    }
}

// Prices one option; columns at Y (forward) and B (backward).
__device__ __forceinline__ double lane_price(const OptConst &c, const double *etab, LaneColumn Y, LaneColumn B)
{
    const TreeShape t{c.w, c.jmax, c.M, c.dr, c.dt, c.rho, c.rhop};
    const int J = c.jmax, n = c.n, e = c.e;
    // forward: delta at the root, e steps
    Y[J] = 1.0;
    for (int i = 0; i < e; ++i) {
        const int ho = min(i, J), hn = min(i + 1, J);
        lane_sweep<true>(t, etab, Y, J - hn, J + hn, J - ho, J + ho);
    }
    // backward: face value at step n over the nodes that reach the exercise
    // region, then n - e steps, each one node narrower per side
    const int ep = min(e, J);
    auto need = [&](int s) { return min(J, ep + (s - e)); };
    {
        const int h = need(n);
        for (int k = J - h; k <= J + h; ++k) {
            double v = 100.0;
            if (k == 0) v -= t.rho * 100.0;
            if (k == t.w - 1) v -= t.rhop * 100.0;
            B[k] = v;
        }
    }
    for (int s = n; s > e; --s) {
        const int ho = need(s), hn = need(s - 1);
        lane_sweep<false>(t, etab, B, J - hn, J + hn, J - ho, J + ho);
    }
    // combine at the exercise step
    const int lo = J - ep, hi = J + ep;
    auto yk = [&](int k) {
        double v = Y[k];
        if (k == 1) v -= t.rho * (0 >= lo ? Y[0] : 0.0);
        if (k == t.w - 2) v -= t.rhop * (t.w - 1 <= hi ? Y[t.w - 1] : 0.0);
        return v;
    };
    auto bk = [&](int k) {
        double v = B[k];
        if (k == 0) v += t.rho * B[1];
        if (k == t.w - 1) v += t.rhop * B[t.w - 2];
        return v;
    };
    double s1 = 0.0, s2 = 0.0;
    for (int k = lo; k <= hi; ++k) {
        const double yv = yk(k);
        s1 += yv;
        s2 += yv * bk(k);
    }
    const double scale = 100.0 * s1 * c.Pn / (s2 * c.Pe);
    double s3 = 0.0;
    for (int k = lo; k <= hi; ++k) {
        const double Bv = scale * bk(k);
        double v = (c.type == 1) ? c.X - Bv : Bv - c.X;  // PUT : CALL
        v = (v < 0.0) ? 0.0 : v;
        if (v == INFINITY) v = DBL_MAX;
        s3 += yk(k) * v;
    }
    return c.Pe / s1 * s3;
}


// ------------------------------------------------- the tridiagonal form
// S steps of u'_k = u_{k-1} + m_k u_k + r_k u_{k+1} in one sweep over nodes
// [lo, hi], in place; the old state is nonzero on [olo, ohi] inside it and the
// result scaled by `down` (hwt_scale.h).
// Level l of the sweep trails the one before by a node: with u_0[k] just read,
// level l makes node k - l.  Nodes are read a chunk at a time, a chunk ahead of use.
constexpr int LANE_CHUNK = 8;

template <int S>
__device__ __forceinline__ void lane_tri_sweep(const TreeShape &t, const TriEdge &e, LaneColumn col, int lo, int hi,
                                               int olo, int ohi, double down)
{
    static_assert(S == 1 || S == 2 || S == 4 || S == 8, "levels");
    double a[S], b[S], m[S], r[S];  // level l's last two nodes; the coefficients level l + 1 uses
#pragma unroll
    for (int l = 0; l < S; ++l) a[l] = b[l] = m[l] = r[l] = 0.0;
    // node lo's closed forms
    double x = (double)(lo - t.jmax) * t.M, E = exp(-(double)(lo - t.jmax) * e.h);
    // one node: c is level 0's; levels from `first` on still make a node
    auto node = [&](int k, double c, int first, bool store) {
#pragma unroll
        for (int l = 0; l < S; ++l) {
            double v = 0.0;
            if (l >= first) v = fma(r[l], c, fma(m[l], b[l], a[l]));
            a[l] = b[l];
            b[l] = c;
            c = v;
        }
        if (store) col[k - S] = c * down;
    };
    // the coefficients of node k, made after its level-0 value is in, move up a level
    auto coefs = [&](int k, bool edges) {
#pragma unroll
        for (int l = S - 1; l > 0; --l) {
            m[l] = m[l - 1];
            r[l] = r[l - 1];
        }
        const double xn = x + t.M, En = E * e.q;
        m[0] = fma(-6.0 * x, x, 4.0) * E;
        r[0] = (pu6(x) * E) * (pd6(xn) * En);
        if (edges && (k < 2 || k >= t.w - 2)) {
            if (k == 1) m[0] = e.m1;
            if (k == t.w - 2) {
                m[0] = e.mt1;
                r[0] = e.rt;
            }
            if (k == 0) {
                m[0] = e.m0;
                r[0] = e.r0;
            }
            if (k == t.w - 1) {
                m[0] = e.mt;
                r[0] = 0.0;
            }
        }
        x = xn;
        E = En;
    };
    auto load = [&](int k0, double (&c)[LANE_CHUNK]) {
        if (k0 >= olo && k0 + LANE_CHUNK - 1 <= ohi) {
#pragma unroll
            for (int i = 0; i < LANE_CHUNK; ++i) c[i] = col[k0 + i];
        } else {
#pragma unroll
            for (int i = 0; i < LANE_CHUNK; ++i) c[i] = (k0 + i >= olo && k0 + i <= ohi) ? col[k0 + i] : 0.0;
        }
    };
    double c[LANE_CHUNK], next[LANE_CHUNK];
    load(lo, c);
    for (int k0 = lo; k0 <= hi; k0 += LANE_CHUNK) {
        load(k0 + LANE_CHUNK, next);  // in flight while this chunk steps
        if (k0 >= lo + S && k0 >= 2 && k0 + LANE_CHUNK - 1 <= min(hi, t.w - 3)) {
            // straight through, so that the levels of neighbouring nodes overlap
#pragma unroll
            for (int i = 0; i < LANE_CHUNK; ++i) {
                node(k0 + i, c[i], 0, true);
                coefs(k0 + i, false);
            }
        } else {
#pragma unroll
            for (int i = 0; i < LANE_CHUNK; ++i)
                if (k0 + i <= hi) {
                    node(k0 + i, c[i], 0, k0 + i - S >= lo);
                    coefs(k0 + i, true);
                }
        }
#pragma unroll
        for (int i = 0; i < LANE_CHUNK; ++i) c[i] = next[i];
    }
    // the last S nodes: level l makes node hi while level 0 is l + 1 past it
#pragma unroll
    for (int i = 0; i < S; ++i) {
        node(hi + 1 + i, 0.0, i, hi + 1 + i - S >= lo);
#pragma unroll
        for (int l = S - 1; l > 0; --l) {
            m[l] = m[l - 1];
            r[l] = r[l - 1];
        }
    }
}

// `steps` steps over a region that `range(i)` gives after i of them, up to
// eight to a sweep.
template <class Range>
__device__ __forceinline__ void lane_tri_steps(const TreeShape &t, const TriEdge &e, LaneColumn col, int steps,
                                               bool grows, Range &&range)
{
    const int J = t.jmax;
    SixfoldScale scale;
    for (int i = 0; i < steps;) {
        const int left = steps - i, c = left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1;
        const int from = range(i), to = range(i + c), h = grows ? to : from;
        const double down = pow2_down(scale.bits(c));
        switch (c) {
        case 8: lane_tri_sweep<8>(t, e, col, J - h, J + h, J - from, J + from, down); break;
        case 4: lane_tri_sweep<4>(t, e, col, J - h, J + h, J - from, J + from, down); break;
        case 2: lane_tri_sweep<2>(t, e, col, J - h, J + h, J - from, J + from, down); break;
        default: lane_tri_sweep<1>(t, e, col, J - h, J + h, J - from, J + from, down); break;
        }
        i += c;
    }
}

// f(k, d1_k, d2_k) for nodes root .. root + h upwards, then root - 1 .. root - h
// downwards, both scales 1 at the root and by the closed forms.
template <class F>
__device__ __forceinline__ void lane_tri_scales(const TreeShape &t, const TriEdge &e, int h, F &&f)
{
    const double qi = 1.0 / e.q;
    double x = 0.0, E = 1.0, d1 = 1.0, d2 = 1.0;
    f(t.jmax, d1, d2);
    for (int j = 1; j <= h; ++j) {
        d1 *= pu6(x) * E;
        x += t.M;
        E *= e.q;
        d2 *= pd6(x) * E;
        f(t.jmax + j, d1, d2);
    }
    x = 0.0, E = 1.0, d1 = 1.0, d2 = 1.0;
    for (int j = 1; j <= h; ++j) {
        d2 /= pd6(x) * E;
        x -= t.M;
        E *= qi;
        d1 /= pu6(x) * E;
        f(t.jmax - j, d1, d2);
    }
}

__device__ __forceinline__ double lane_price_tri(const OptConst &c, const TreeShape &t, const TriEdge &ed, LaneColumn Y,
                                                 LaneColumn B)
{
    const int J = c.jmax, n = c.n, e = c.e, top = c.w - 1;
    Y[J] = 1.0;
    lane_tri_steps(t, ed, Y, e, true, [&](int i) { return min(i, J); });
    const int ep = min(e, J);
    auto need = [&](int s) { return min(J, ep + (s - e)); };
    lane_tri_scales(t, ed, need(n), [&](int k, double, double d2) {
        double v = 1.0;
        if (k == 0) v -= t.rho;
        if (k == top) v = (v - t.rhop) / ed.d2_t;
        B[k] = v / d2;
    });
    lane_tri_steps(t, ed, B, n - e, false, [&](int i) { return need(n - i); });
    // both states scaled back, node 0's d1 and node w-1's d2 by their factors
    lane_tri_scales(t, ed, ep, [&](int k, double d1, double d2) {
        if (k == 0) d1 *= ed.d1_0;
        if (k == top) d2 *= ed.d2_t;
        Y[k] = Y[k] * d1;
        B[k] = B[k] * d2;
    });
    // the edge transform undone (both edges are inside or both outside)
    if (ep == J) {
        Y[1] -= t.rho * Y[0];
        Y[top - 1] -= t.rhop * Y[top];
        B[0] += t.rho * B[1];
        B[top] += t.rhop * B[top - 1];
    }
    const int lo = J - ep, hi = J + ep;
    double s1 = 0.0, s2 = 0.0;
    for (int k = lo; k <= hi; ++k) {
        const double yv = Y[k];
        s1 += yv;
        s2 = fma(yv, B[k], s2);
    }
    const double scale = 100.0 * s1 * c.Pn / (s2 * c.Pe);
    double s3 = 0.0;
    for (int k = lo; k <= hi; ++k) {
        const double Bv = scale * B[k];
        double v = (c.type == 1) ? c.X - Bv : Bv - c.X;  // PUT : CALL
        v = (v < 0.0) ? 0.0 : v;
        if (v == INFINITY) v = DBL_MAX;
        s3 = fma(Y[k], v, s3);
    }
    return c.Pe / s1 * s3;
}

} // namespace hwt
