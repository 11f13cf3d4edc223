// hwt_k_tri.hip -- the FP64 pricing kernel: window tasks and groups (hwt_tri.h).
#include "hwt_pricers.h"
#include "hwt_tri.h"

namespace hwt {

// Persistent, one wave per workgroup: the window tasks from their queue, longest
// first, then the groups from theirs, so the short groups fill the time in
// which the last long trees finish.
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(3))) void k_price_tri(
    const OptConst *__restrict__ cst, const double *__restrict__ edge, const int32_t *__restrict__ order,
    int32_t *__restrict__ tally, double *__restrict__ out, double *__restrict__ scratch)
{
    clear_bucket_counts(tally);
    __shared__ double buf[TRI_MAX_NODES];
    lds_f64 *lds = (lds_f64 *)buf;
    const TriEdge *ed = reinterpret_cast<const TriEdge *>(edge);
    const int lane = threadIdx.x;
    const int first = uni(tally[T_TBIG]), last = uni(tally[T_TWIN]), ngroups = uni(tally[T_TNGROUP]);
    double *park = scratch + (size_t)blockIdx.x * TRI_MAX_NODES;
    // the wave's queue, and its place among the waves that share it
    const int queue = uni((int)blockIdx.x % TRI_QUEUES), rank = uni((int)blockIdx.x / TRI_QUEUES);
    const int sharing = uni(((int)gridDim.x - queue + TRI_QUEUES - 1) / TRI_QUEUES);
    int32_t *qwin = &tally[T_TQWIN + 32 * queue], *qgroup = &tally[T_TQGROUP + 32 * queue];
    // the first task by rank, then claimed; lane 0 stores a finished price and
    // claims the next task in one divergent region, every lane reads the claim
    // back together
    int t = first + queue + rank * TRI_QUEUES;
    while (t < last) {
        const int o = uni(order[t]);
        const double p = price_tri_window(cst, ed, o, lane, lds, park);
        int claim = 0;
        if (lane == 0) {
            out[o] = p;
            claim = atomicAdd(qwin, 1);
        }
        t = first + queue + (uni(__shfl(claim, 0, WAVE)) + sharing) * TRI_QUEUES;
    }
    // part starts, one per lane
    const int pstart = lane < TRI_PARTS ? tally[T_TSTART + lane] : 0;
    const int pgroup = lane < TRI_PARTS ? tally[T_TGROUP + lane] : INT_MAX;
    for (;;) {
        int claim = 0;
        if (lane == 0) claim = atomicAdd(qgroup, 1);
        const int g = queue + uni(__shfl(claim, 0, WAVE)) * TRI_QUEUES;
        if (g >= ngroups) break;
        const int j = __popcll(__ballot(pgroup <= g)) - 1;  // the last part that starts at or before g
        const int part = TRI_PARTS - 1 - j, L = tri_lanes(part);
        const int at = __builtin_amdgcn_readlane(pstart, j) + (g - __builtin_amdgcn_readlane(pgroup, j)) * (WAVE / L) + lane / L;
        const int mine = order[at];
        // a group's first slot is never idle; read in all lanes, outside the
        // choice below (inside it only the idle lanes would take part)
        const int head = uni(mine);
        const bool active = mine >= 0;
        const int o = active ? mine : head;
        double p = 0.0;
        switch (part) {
#define HWT_G(P) case P: p = price_tri_group<tri_lanes(P), tri_nodes(P)>(cst, ed, o, active, lds); break;
            HWT_G(0) HWT_G(1) HWT_G(2) HWT_G(3) HWT_G(4) HWT_G(5) HWT_G(6) HWT_G(7) HWT_G(8) HWT_G(9) HWT_G(10)
            HWT_G(11) HWT_G(12) HWT_G(13) HWT_G(14) HWT_G(15) HWT_G(16) HWT_G(17) HWT_G(18) HWT_G(19) HWT_G(20) HWT_G(21)
            HWT_G(22) HWT_G(23) HWT_G(24) HWT_G(25) HWT_G(26) HWT_G(27) HWT_G(28) HWT_G(29) HWT_G(30)
#undef HWT_G
        default: break;
        }
        if (active && lane % L == 0) out[o] = p;
    }
    stamp_wave_end(tally);
}

} // namespace hwt
