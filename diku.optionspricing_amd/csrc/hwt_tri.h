// hwt_tri.h -- FP64 pricing of form 2: every tree as powers of one tridiagonal
// matrix with a unit sub-diagonal.
//
// The matrix.  With a_k = G[k][k-1], m_k = G[k][k], c_k = G[k][k+1] the
// edge-corrected forward operator (hwt_math.h), the diagonal similarities
//     y = D1 u,  d1_k = 6 a_k d1_{k-1},      b = D2 v,  d2_k = 6 c_{k-1} d2_{k-1}
// turn BOTH passes, y' = G y and b' = G^T b, into the same step (up to a
// factor 6 per step)
//     u'_k = u_{k-1} + 6 m_k u_k + 36 a_{k+1} c_k u_{k+1},
// two FMAs per node: a tridiagonal matrix is known by its diagonal and the
// products across it, and those of G and G^T are equal.  So a tree has one
// set of coefficients for both passes, D1 and D2 are needed only where the
// backward pass starts and where the two states meet, and every factor that
// is common to a whole state cancels in the price (states are scaled by
// powers of two on the way, and D1, D2 are normalised anywhere).  6 a_k, 6 m_k
// and 6 c_k are the branching probabilities times 6 (1 + 3(x^2 + x), 4 - 6x^2,
// 1 + 3(x^2 - x), x = jM) and the node discount; only six entries differ
// (TriEdge).  Trees whose scales could leave the range (tri_ok: a volatility or
// a width far beyond the usual) are priced by the general wide kernel.
//
// The layout.  A group of L lanes holds one tree, K consecutive nodes per
// lane, 64 / L trees side by side in a wave; values cross lanes by DPP shifts.
// A step costs 2K FMAs and 4 DPP moves per lane whatever L is, so fewer lanes
// and more nodes per lane spend less of it on moves (and on padding): K is 6
// to 11 (168 VGPRs, three waves per SIMD), L the least power of two that holds
// the tree up to 175 nodes.  Wider trees run alone in a wave (L = 64) in
// windows that follow their weight (Reach).
#pragma once

#include "hwt_flat.h"
#include "hwt_pipeline.h"
#include "hwt_scale.h"

namespace hwt {

// What the edges change, and the discount per node.  Six entries of G differ
// from the closed forms: G[0][0], G[1][1], G[1][0] and G[w-1][w-1], G[w-2][w-2],
// G[w-2][w-1] (edge_table_closed; in a 3-node tree, whose middle node borders both
// edges, G[1][1] takes both corrections).  So do, times 6: the diagonal at nodes 0,
// 1, w-2, w-1, the products across it r_0, r_{w-2}, and the scales of node 0 (d1)
// and node w-1 (d2), by a factor each.
struct TriEdge {
    double m0, m1, r0, d1_0, mt1, mt, rt, d2_t, h, q;  // h = dr dt, q = e^{-h}
};
static_assert(sizeof(TriEdge) == TRI_EDGE * sizeof(double), "edge record");

__device__ __forceinline__ TriEdge tri_edge(const TreeShape &t, const EdgeDiscounts &e)
{
    const double M = t.M;
    const int J = t.jmax;
    const double F00 = pd_bot(-J, M) * e.E0, F10 = pm_bot(-J, M) * e.E0;
    const double F01 = pd_std(1 - J, M) * e.E1, F11 = pm_std(1 - J, M) * e.E1;
    const double Faa = pu_top(J, M) * e.Ea, Fba = pm_top(J, M) * e.Ea;
    const double Fab = pu_std(J - 1, M) * e.Eb, Fbb = pm_std(J - 1, M) * e.Eb;
    const double G00 = F00 - t.rho * F01, Gaa = Faa - t.rhop * Fab;
    const double G10 = F10 - t.rho * F11 + t.rho * G00, Gba = Fba - t.rhop * Fbb + t.rhop * Gaa;
    double G11 = F11 + t.rho * F01, Gbb = Fbb + t.rhop * Fab;
    if (J == 1) G11 = Gbb = F11 + t.rho * F01 + t.rhop * Fab;
    // d1 from node 0 to 1 by 6 G10, by the closed form pu(-J) E0; d2 to node w-1
    // by 6 Gba, by the closed form pd(J) Ea
    return TriEdge{6.0 * G00, 6.0 * G11, 36.0 * (F01 * G10), pu_std(-J, M) * e.E0 / G10,
                   6.0 * Gbb, 6.0 * Gaa, 36.0 * (Fab * Gba), Gba / (pd_std(J, M) * e.Ea), t.dr * t.dt, e.q};
}

// Whether a tree stepped over `half` nodes either side of the root stays in
// range.  Going out, ln d1 and ln d2 change per node by at most -ln(1 - 3x + 3x^2)
// at x = j |M|, which is convex up to x = 1/4 (so at most half of its last value on
// average), and by the discount's j h; the state by 6 e^{h half} per step, scaled back
// as it goes.  The scales have to exist (entries away from zero) where the edges
// are inside.  `lim` bounds |ln d|: 200 where the scales are normalised at the root,
// 100 for groups, which normalise at node 0, so that products of two scales and
// a state stay below e^700.
__device__ __forceinline__ bool tri_ok(const TreeShape &t, const TriEdge &e, int n, int half, float lim)
{
    const float x = (float)half * (float)-t.M, h = (float)(t.dr * t.dt), mean = x <= 0.25f ? 0.5f : 1.0f;
    const float per = -0.69314718f * log2_f(fminf(1.0f, 1.0f - 3.0f * x + 3.0f * x * x));
    bool ok = (float)half * (mean * per + 0.5f * h * (float)(half + 1)) <= lim && h * (float)half <= 0.5f &&
              (float)n * h * (float)half <= 300.0f && x < 0.75f;
    if (half >= t.jmax)
        ok = ok && fabs(e.d1_0) > 1e-6 && fabs(e.d1_0) < 1e6 && fabs(e.d2_t) > 1e-6 && fabs(e.d2_t) < 1e6 &&
             fabs(e.m0) < 1e6 && fabs(e.mt) < 1e6 && fabs(e.m1) < 1e6 && fabs(e.mt1) < 1e6 && fabs(e.r0) < 1e6 &&
             fabs(e.rt) < 1e6 && fabs(t.rho) < 1e6 && fabs(t.rhop) < 1e6;
    return ok;
}

// -------------------------------------------------------------------- lanes
// The value of the lane below / above inside a group of L lanes.  Zero comes in
// at the ends of a wave (64) and of a row (16); narrower groups get a
// neighbour's or their own value there, which they must not use.
template <int L>
__device__ __forceinline__ double group_lower(double x)
{
    if constexpr (L == 64) return dpp_mov<0x138>(x);
    else if constexpr (L >= 8) return dpp_mov<0x111>(x);
    else if constexpr (L == 4) return dpp_mov<0x90>(x);   // quad_perm [0,0,1,2]
    else if constexpr (L == 2) return dpp_mov<0xA0>(x);   // quad_perm [0,0,2,2]
    else return 0.0;
}
template <int L>
__device__ __forceinline__ double group_upper(double x)
{
    if constexpr (L == 64) return dpp_mov<0x130>(x);
    else if constexpr (L >= 8) return dpp_mov<0x101>(x);
    else if constexpr (L == 4) return dpp_mov<0xF9>(x);   // quad_perm [1,2,3,3]
    else if constexpr (L == 2) return dpp_mov<0xF5>(x);   // quad_perm [1,1,3,3]
    else return 0.0;
}

// Sum over the group, the same in each of its lanes.
template <int L>
__device__ __forceinline__ double group_sum(double v)
{
    if constexpr (L == 64) return wave_sum(v);
    if constexpr (L >= 2) v += dpp_mov<0xB1>(v);
    if constexpr (L >= 4) v += dpp_mov<0x4E>(v);
    if constexpr (L >= 8) v += dpp_mov<0x141>(v);
    if constexpr (L >= 16) v += dpp_mov<0x140>(v);
    return v;
}

// Product over the lanes of the group below this one.
template <int L>
__device__ __forceinline__ double group_product_below(double p, int l)
{
#pragma unroll
    for (int off = 1; off < L; off <<= 1) {
        const double t = __shfl_up(p, off, WAVE);
        if (l >= off) p *= t;
    }
    const double t = __shfl_up(p, 1, WAVE);
    return (L == 1 || l == 0) ? 1.0 : t;
}

// ------------------------------------------------------------- coefficients
__device__ __forceinline__ double pu6(double x) { return fma(3.0, fma(x, x, x), 1.0); }
__device__ __forceinline__ double pd6(double x) { return fma(3.0, fma(x, x, -x), 1.0); }

// The closed forms along this lane's nodes k = k0 + s, upwards: f(s, a, c, E, x)
// with a = 6 a_k and c = 6 c_{k-1} (what d1 and d2 grow by from node k-1 to
// k), the node's discount E and x = jM.  The entries at the edges differ; what
// depends on them is put right in LDS (edit_nodes).
template <int K, class F>
__device__ __forceinline__ void tri_walk(const TreeShape &t, const TriEdge &e, int k0, F &&f)
{
    double x = (double)(k0 - 1 - t.jmax) * t.M, E = exp(-(double)(k0 - 1 - t.jmax) * e.h);
#pragma unroll
    for (int s = 0; s < K; ++s) {
        const double a = pu6(x) * E;
        x += t.M;
        E *= e.q;
        f(s, a, pd6(x) * E, E, x);
    }
}

// Nodes of a group through LDS: every lane's K values go out (slot 64 s + lane,
// no bank conflicts), the group's first lane edits single nodes, and they come
// back.  Cheaper than comparing every node's index against the edges': the
// selects took a third of a group's set-up and sums.
template <int L, int K, class F>
__device__ __forceinline__ void edit_nodes(double (&z)[K], int lane, int l, lds_f64 *lds, F &&edit)
{
#pragma unroll
    for (int s = 0; s < K; ++s) lds[s * WAVE + lane] = z[s];
    __syncthreads();
    if (l == 0) {
        auto node = [&](int k) -> lds_f64 & { return lds[(k % K) * WAVE + lane + k / K]; };  // k counts from k0
        edit(node);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < K; ++s) z[s] = lds[s * WAVE + lane];
    __syncthreads();
}

// m[s] = 6 m_k and r[s] = 36 a_{k+1} c_k of nodes k = base + l K + s; zero on
// padding.  `edges` (wave-uniform): the window reaches an edge of the tree.
// With v also the backward pass's start in v-units, T^{-T} 1 / d2 (the face value's
// 100 cancels), d2 normalised over the group.
template <int L, int K, bool START>
__device__ __forceinline__ void tri_coefs(const TreeShape &t, const TriEdge &e, bool edges, int base, int lane, int l,
                                          double (&m)[K], double (&r)[K], double (&v)[K], lds_f64 *lds)
{
    const int k0 = base + l * K, in = t.w - k0;  // the lane's tree nodes are s < in
    double p = 1.0;
    tri_walk<K>(t, e, k0, [&](int s, double a, double c, double E, double x) {
        const double Ez = s < in ? E : 0.0;
        m[s] = fma(-6.0 * x, x, 4.0) * Ez;
        // r of the node below is this node's a c; r of the last one needs the next
        if (s > 0) r[s - 1] = a * (pd6(x) * Ez);
        if (s == K - 1) {
            const double xn = x + t.M;
            r[s] = K < in ? (pu6(x) * E) * (pd6(xn) * (E * e.q)) : 0.0;
        }
        if (START) {
            v[s] = c;
            p *= (s == 0 && l == 0) ? 1.0 : c;
        }
    });
    if (START) {
        double below = group_product_below<L>(p, l);
        if constexpr (L == 64) {
            const int root = uni((t.jmax - base) / K);  // the lane that holds the root
            below /= readlane_f64(below, root);
        }
        double inv = 1.0 / (below * p);
#pragma unroll
        for (int s = K - 1; s >= 0; --s) {
            const double c = v[s];
            v[s] = inv;
            inv *= c;
        }
    }
    if (edges) {
        const int top = t.w - 1 - base;  // node w-1's place in the window
        const bool lowest = base == 0, low1 = base <= 1, high = top < L * K, high1 = top - 1 < L * K;
        edit_nodes<L, K>(m, lane, l, lds, [&](auto node) {
            if (low1) node(1 - base) = e.m1;
            if (high1) node(top - 1) = e.mt1;
            if (lowest) node(0) = e.m0;
            if (high) node(top) = e.mt;
        });
        edit_nodes<L, K>(r, lane, l, lds, [&](auto node) {
            if (lowest) node(0) = e.r0;
            if (high1) node(top - 1) = e.rt;
        });
        if (START)
            edit_nodes<L, K>(v, lane, l, lds, [&](auto node) {
                if (lowest) node(0) *= 1.0 - t.rho;
                if (high) node(top) *= (1.0 - t.rhop) / e.d2_t;
            });
    }
}

// ------------------------------------------------------------------- steps
// One step from src into dst.  in_lane0 is 0 on a group's first lane where the
// shift brings in a foreign value (L = 2, 4, 8), else unused.
template <int L, int K>
__device__ __forceinline__ void tri_step(const double (&src)[K], double (&dst)[K], const double (&m)[K],
                                         const double (&r)[K], double in_lane0)
{
    const double left = group_lower<L>(src[K - 1]);
    const double right = group_upper<L>(src[0]);
#pragma unroll
    for (int s = 0; s < K; ++s) {
        double v;
        if (s > 0) v = fma3(m[s], src[s], src[s - 1]);
        else if (L == 64 || L == 16) v = fma3(m[0], src[0], left);
        else if (L == 1) v = m[0] * src[0];
        else v = fma(in_lane0, left, m[0] * src[0]);
        if (L == 1 && s + 1 == K) dst[s] = v;
        else dst[s] = fma(r[s], s + 1 < K ? src[s + 1] : right, v);
    }
}

// nsteps steps in place, scaled on the way (hwt_scale.h).
template <int L, int K>
__device__ __forceinline__ void tri_steps(double (&z)[K], const double (&m)[K], const double (&r)[K], double in_lane0,
                                          int nsteps, SixfoldScale &scale)
{
    double t[K];
    scaled_steps(
        scale, nsteps,
        [&](int c) {
            for (int it = 0; it + 1 < c; it += 2) {
                tri_step<L, K>(z, t, m, r, in_lane0);
                tri_step<L, K>(t, z, m, r, in_lane0);
            }
            if (c & 1) {
                tri_step<L, K>(z, t, m, r, in_lane0);
#pragma unroll
                for (int s = 0; s < K; ++s) z[s] = t[s];
            }
        },
        [&](double f) {
#pragma unroll
            for (int s = 0; s < K; ++s) z[s] *= f;
        });
}

// Price from the two states at the exercise step, u (forward) and v
// (backward), in the same window:
//   S1 = sum y, S2 = sum y b (equal in edge-transformed and plain states),
//   scale = 100 S1 Pn / (S2 Pe), price = Pe / S1 sum y payoff(scale b).
// What the scaling left of the states' growth (sixfold_left) goes with d1 and d2, so that
// any bond price in FP64's range fits.
template <int L, int K>
__device__ __forceinline__ double tri_price(const TreeShape &t, const TriEdge &e, bool edges, int base, int lane, int l,
                                            double (&u)[K], double (&v)[K], int left_u, int left_v, double X, double Pe,
                                            double Pn, int type, lds_f64 *lds)
{
    // u and v times the scales' products along the lane, then times the lane's own
    double p1 = 1.0, p2 = 1.0;
    const int in = t.w - (base + l * K);
    tri_walk<K>(t, e, base + l * K, [&](int s, double a, double c, double, double) {
        if (s > 0 || l > 0) {
            p1 *= s < in ? a : 0.0;  // padding: no weight, and a bond value above 0, which an
            p2 *= s < in ? c : 1.0;  // infinite scale does not turn into a NaN
        }
        u[s] *= p1;
        v[s] *= p2;
    });
    double d1 = group_product_below<L>(p1, l), d2 = group_product_below<L>(p2, l);
    if constexpr (L == 64) {
        const int root = uni((t.jmax - base) / K);
        d1 /= readlane_f64(d1, root);
        d2 /= readlane_f64(d2, root);
    }
    d1 = ldexp(d1, -left_u);
    d2 = ldexp(d2, -left_v);
#pragma unroll
    for (int s = 0; s < K; ++s) {
        u[s] *= d1;
        v[s] *= d2;
    }
    if (edges) {
        // node 0's d1 and node w-1's d2, then the edge transform undone: y = T^{-1} z,
        // b = T^T z
        const int top = t.w - 1 - base;
        const bool lowest = base == 0, high = top < L * K;
        edit_nodes<L, K>(u, lane, l, lds, [&](auto node) {
            if (lowest) {
                const double y0 = node(0) * e.d1_0;
                node(0) = y0;
                node(1) -= t.rho * y0;
            }
            if (high) node(top - 1) -= t.rhop * node(top);
        });
        edit_nodes<L, K>(v, lane, l, lds, [&](auto node) {
            if (lowest) node(0) += t.rho * node(1);
            if (high) node(top) = fma(t.rhop, node(top - 1), node(top) * e.d2_t);
        });
    }
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int s = 0; s < K; ++s) {
        s1 += u[s];
        s2 = fma(u[s], v[s], s2);
    }
    s1 = group_sum<L>(s1);
    s2 = group_sum<L>(s2);
    const double scale = 100.0 * s1 * Pn / (s2 * Pe);
    double s3 = 0.0;
#pragma unroll
    for (int s = 0; s < K; ++s) {
        const double B = scale * v[s];
        double f = (type == 1) ? X - B : B - X;  // PUT : CALL
        f = (f < 0.0) ? 0.0 : f;
        f = (f > RealMax<double>::value) ? RealMax<double>::value : f;
        s3 = fma(u[s], f, s3);
    }
    return Pe / s1 * group_sum<L>(s3);
}

// ------------------------------------------------------------------- groups
// Prices the 64 / L trees of one group of tasks; returns each tree's price in
// every lane of its L lanes.  The trees end together: with N the tallest one's
// height, tree i starts its forward pass at step N - n_i (its state is zero
// before) and swaps to the backward state at N - n_i + e_i, through LDS (64 K
// slots: the backward start goes in first, the forward state takes its place).
// The wave stops at each step where some tree starts or swaps.
template <int L, int K>
__device__ __forceinline__ double price_tri_group(const OptConst *__restrict__ cst, const TriEdge *__restrict__ edge,
                                                  int o, bool active, lds_f64 *lds)
{
    // opaque, so that what every (L, K) derives from it is not hoisted out of
    // the caller's loop and spilled
    int lane = threadIdx.x;
    asm volatile("" : "+v"(lane));
    const int l = lane % L, k0 = l * K;
    int n, e, root;  // root: the root's place among the lane's nodes
    double m[K], r[K], z[K];
    {
        const OptConst c = cst[o];
        const TreeShape t{c.w, c.jmax, c.M, c.dr, c.dt, c.rho, c.rhop};
        const TriEdge ed = edge[o];
        n = active ? c.n : 0;
        e = active ? c.e : 0;
        root = c.jmax - k0;
        tri_coefs<L, K, true>(t, ed, true, 0, lane, l, m, r, z, lds);
#pragma unroll
        for (int s = 0; s < K; ++s) lds[s * WAVE + lane] = z[s];
    }
#pragma unroll
    for (int s = 0; s < K; ++s) z[s] = 0.0;
    const double in_lane0 = l == 0 ? 0.0 : 1.0;
    const int N = -wave_min_i32(-n);
    const int start = N - n, swap = start + e;
    int i = 0;
    SixfoldScale scale;
    for (;;) {
        if (i == start) {
#pragma unroll
            for (int s = 0; s < K; ++s) z[s] = (s == root) ? 1.0 : 0.0;
        }
        if (i == swap) {
#pragma unroll
            for (int s = 0; s < K; ++s) {
                const double v = lds[s * WAVE + lane];
                lds[s * WAVE + lane] = z[s];
                z[s] = v;
            }
        }
        if (i >= N) break;
        const int next = wave_min_i32(start > i ? start : (swap > i ? swap : N));
        tri_steps<L, K>(z, m, r, in_lane0, next - i, scale);
        i = next;
    }
    double u[K];
#pragma unroll
    for (int s = 0; s < K; ++s) u[s] = lds[s * WAVE + lane];
    asm volatile("" : "+v"(o));  // read the option's constants again rather than hold them through the steps
    const OptConst c = cst[o];
    const TreeShape t{c.w, c.jmax, c.M, c.dr, c.dt, c.rho, c.rhop};
    __syncthreads();
    return tri_price<L, K>(t, edge[o], true, 0, lane, l, u, z, sixfold_left(start, swap), sixfold_left(swap, N), c.X, c.Pe,
                           c.Pn, c.type, lds);
}

// ------------------------------------------------------------------ windows
// One phase of a wide tree: bring the window in (the pass's start values, or the
// previous window's nodes from LDS, zeros elsewhere), run its steps, and leave
// it in LDS -- or, at the end of the forward pass, in `park`, and at the end of
// the backward pass return the price.
struct TriPhase {
    int K, base, steps;
    bool first, last, back;
    int in_base, in_n;  // the previous window's nodes in LDS
    int f_base, f_n;    // the parked forward state's
    int left_u, left_v; // what the scaling leaves of either state's growth
};

// The tree's records are read again in each phase (scalar loads) rather than
// held in registers through the steps.
template <int K>
__device__ __forceinline__ double tri_phase(const OptConst *__restrict__ cst, const TriEdge *__restrict__ edge, int o,
                                            const TriPhase &p, int lane, lds_f64 *lds, double *park,
                                            SixfoldScale &scale)
{
    asm volatile("" : "+s"(o), "+v"(lane));
    const OptConst c = cst[o];
    const TriEdge ed = edge[o];
    const TreeShape t = uni(TreeShape{c.w, c.jmax, c.M, c.dr, c.dt, c.rho, c.rhop});
    const int k0 = p.base + lane * K;
    double z[K], m[K], r[K];
    const bool edges = p.base < 2 || p.base + WAVE * K > t.w - 3;
    if (p.first && p.back) {
        tri_coefs<WAVE, K, true>(t, ed, edges, p.base, lane, lane, m, r, z, lds);
    } else {
#pragma unroll
        for (int s = 0; s < K; ++s) {
            const int k = k0 + s - p.in_base;
            z[s] = p.first ? (k0 + s == t.jmax ? 1.0 : 0.0) : (k >= 0 && k < p.in_n) ? lds[k] : 0.0;
        }
        __syncthreads();
        double none[K];
        tri_coefs<WAVE, K, false>(t, ed, edges, p.base, lane, lane, m, r, none, lds);
    }
    tri_steps<WAVE, K>(z, m, r, 1.0, p.steps, scale);
    if (!p.last) {
#pragma unroll
        for (int s = 0; s < K; ++s) lds[lane * K + s] = (k0 + s < t.w) ? z[s] : 0.0;
        __syncthreads();
        return 0.0;
    }
    if (!p.back) {
#pragma unroll
        for (int s = 0; s < K; ++s) park[lane * K + s] = z[s];
        return 0.0;
    }
    double u[K];
#pragma unroll
    for (int s = 0; s < K; ++s) {
        const int k = k0 + s - p.f_base;
        u[s] = (k >= 0 && k < p.f_n) ? park[k] : 0.0;
    }
    asm volatile("" : "+s"(o));
    const OptConst ce = cst[o];
    const TreeShape te = uni(TreeShape{ce.w, ce.jmax, ce.M, ce.dr, ce.dt, ce.rho, ce.rhop});
    return tri_price<WAVE, K>(te, edge[o], edges, p.base, lane, lane, u, z, p.left_u, p.left_v, ce.X, ce.Pe, ce.Pn, ce.type,
                              lds);
}

// Prices one tree wider than a group, alone in its wave.
__device__ __forceinline__ double price_tri_window(const OptConst *__restrict__ cst, const TriEdge *__restrict__ edge,
                                                   int o, int lane, lds_f64 *lds, double *park)
{
    const OptConst c = cst[o];
    const TreeShape t = uni(TreeShape{c.w, c.jmax, c.M, c.dr, c.dt, c.rho, c.rhop});
    const int n = uni(c.n), e = uni(c.e);
    const Reach reach = make_reach(c.sigmas, t.M, t.dr, t.dt, n, t.jmax);
    TriPhase p{};
    p.left_u = uni(sixfold_left(0, e));
    p.left_v = uni(sixfold_left(e, n));
    double price = 0.0;
    SixfoldScale scale;
    for (int back = 0; back < 2; ++back) {
        int at = back ? n : 0, l0 = 0, u0 = 0;
        if (back) {
            reach_at(reach, n, min(e, t.jmax) + (n - e), l0, u0);
            l0 = uni(l0);
            u0 = uni(u0);
        }
        p.back = back != 0;
        p.first = true;
        p.in_n = 0;
        do {
            const ReachPhase f = back ? reach_back<1>(t, reach, at, e, lane, l0, u0) : reach_ahead<1>(t, reach, at, e, lane);
            p.K = min(f.win.K, TRI_MAXK);
            p.base = f.win.base;
            p.steps = abs(f.end - at);
            p.last = f.end == e;
            switch (p.K) {
#define HWT_W(KK) case KK: price = tri_phase<KK>(cst, edge, o, p, lane, lds, park, scale); break;
                HWT_W(2) HWT_W(3) HWT_W(4) HWT_W(5) HWT_W(6) HWT_W(7) HWT_W(8) HWT_W(9) HWT_W(10)
            default: price = tri_phase<TRI_MAXK>(cst, edge, o, p, lane, lds, park, scale); break;
#undef HWT_W
            }
            p.in_base = p.base;
            p.in_n = WAVE * p.K;
            p.first = false;
            at = f.end;
        } while (!p.last);
        if (!back) {
            p.f_base = p.base;
            p.f_n = min(WAVE * p.K, t.w - p.base);
            __threadfence_block();
        }
    }
    return price;
}

} // namespace hwt
