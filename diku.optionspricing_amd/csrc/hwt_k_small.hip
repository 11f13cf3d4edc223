// hwt_k_small.hip -- FP64 batches of a few options: setup and pricing in one kernel.
#include "hwt_pricers.h"
#include "hwt_setup.h"

namespace hwt {

// The general routine, out of line: inside the kernel it took registers from the other
// two ways (114 spilled; 1,000 options 17.9 us a call instead of 17.4).
__device__ __noinline__ static double price_general(const OptConst *c, int lane, lds_f64 *lds, lds_f64 *etab, double *park)
{
    return price_option<double, MAXK>(*c, nullptr, lane, lds, etab, park);
}

// One wave per option, every wave resident at once (2 per SIMD): the option is set up
// by all lanes alike and priced as k_price_tri's spread batches are (16 lanes up to 64
// nodes, a wave above), so nothing is sorted, queued or counted, and prices are the
// same to the bit.  A batch this small waits for latencies, not for issue: the launches
// of the general pipeline (k_setup, k_order, the big trees' empty kernel, k_price_tri)
// took 34 us for 1,000 options, this one 17.4 (13.4 in the kernel).
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(2))) void k_price_small(
    DevOpts o, DevYield y, int32_t maxWidth, double unit_dmin, OptConst *__restrict__ cst,
    int32_t *__restrict__ tally, double *__restrict__ out, double *__restrict__ scratch)
{
    __shared__ double buf[WAVE * MAXK];  // the curve, then the tree
    __shared__ double etab[EDGE_TAB];
    __shared__ OptConst sc;
    __shared__ TriEdge se;
    static_assert(SMALL_YMAX * 12 <= (int)sizeof(buf), "the curve fits");
    const int lane = threadIdx.x, i = blockIdx.x;
    if (i == 0) {
        reinterpret_cast<unsigned long long *>(tally)[T_T0 / 2] = __builtin_amdgcn_s_memrealtime();
        tally[T_SMALL] = o.n;
    }
    OptFields f{};
    if (!o.consts) f = option_fields(o, i);
    // the curve as in k_setup
    double *yr = buf;
    int32_t *yd = reinterpret_cast<int32_t *>(buf + SMALL_YMAX);
    int unsorted = 0;
    for (int k = lane; k < y.n; k += WAVE) {
        yr[k] = y.rate[k];
        yd[k] = y.day[k];
        if (k + 1 < y.n && y.day[k] > y.day[k + 1]) unsorted = 1;
    }
    const bool sorted = __ballot(unsorted) == 0;
    __syncthreads();
    OptConst c{};
    TriEdge edges{};
    int64_t key = 0;
    double price = 0.0;
    option_record(o, i, f, maxWidth, c);
    const TriKind kind = tri_setup(c, f.term_unit, [&](double t, int tu) {
        return sorted ? yield_at_sorted(t, tu, yr, yd, y.n) : yield_at(t, tu, yr, yd, y.n);
    }, true, unit_dmin, edges, key, price);
    __syncthreads();  // the curve's last reads
    if (lane == 0) {
        cst[i] = c;  // for the counts at sync time
        sc = c;
        se = edges;
    }
    __syncthreads();
    const int way = uni((int)kind);
    lds_f64 *lds = (lds_f64 *)buf;
    double *park = scratch + (size_t)i * (WAVE * MAXK);
    if (way == TRI_GROUPED) {
        const int part = uni(tri_part(sc.w, true));
        price = part == 0   ? price_tri_group<16, tri_nodes(0)>(&sc, &se, 0, lane < 16, lds)
                : part == 1 ? price_tri_group<16, tri_nodes(1)>(&sc, &se, 0, lane < 16, lds)
                            : price_tri_group<16, tri_nodes(2)>(&sc, &se, 0, lane < 16, lds);
    } else if (way == TRI_WINDOWED) {
        price = price_tri_window(&sc, &se, 0, lane, lds, park);
    } else if (way == TRI_GENERAL) {
        price = price_general(&sc, lane, lds, (lds_f64 *)etab, park);
    }
    if (lane == 0) out[i] = price;
    stamp_wave_end(tally);
}

} // namespace hwt
