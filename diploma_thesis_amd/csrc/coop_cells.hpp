// coop_cells.hpp -- the 27-cell contact sum of one particle by a group of 16 lanes.
//
// One thread per particle walks its candidates one after another: a particle with hundreds of candidates
// (a range image puts about a hundred scene points into a cell) is then one long serial chain of loads,
// and a few thousand particles leave most of the chip idle.  Here 16 lanes share a particle: the
// lanes look up its 27 cells side by side, lay the cells' runs end to end, and test 16 candidates
// per step.  The forces of the hits are listed in LDS in candidate order, and three lanes (one per
// component) add them one by one, cell partial by cell partial, so every sum is formed in the same
// order as by one thread and has the same bits.
#pragma once

#include "kernels.hpp"

namespace arsim {

constexpr int kCoopLanes = 16;
constexpr int kCoopList = 64;   // listed hits per group before they are added up
struct CoopGroupLds {
    float4 list[kCoopList];     // force, cell
    unsigned off[28], beg[28];  // cell c holds the slots [off[c], off[c + 1]), its first candidate is beg[c]
};

// Adds the group's n listed forces: lane l adds component l (lanes 0..2; the others do no harm).
__device__ __forceinline__ void coop_drain(const CoopGroupLds &g, int n, int l, int &cur, float &F, float &csum) {
    const int comp = l < 3 ? l : 0;
    for (int k = 0; k < n; k += 4) {
        float v[4];
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {   // (entries past n hold stale values, which the guard below drops)
            const float *e = reinterpret_cast<const float *>(&g.list[(k + u) & (kCoopList - 1)]);
            v[u] = e[comp];
            c[u] = __float_as_int(e[3]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (k + u < n) {
                if (c[u] != cur) {
                    F = F + csum;
                    csum = 0.f;
                    cur = c[u];
                }
                csum = csum + v[u];
            }
        }
    }
}

// Σ over the 27 cells (cell c = 9 (dz + 1) + 3 (dy + 1) + dx + 1), per cell the partial sum of its hits in
// candidate order.  cell(c, begin, end) gives a cell's run of candidates, pair(j, f) candidate j's force
// (false: no contact).  Every lane of the wave calls it (valid: the group has a particle); lane l < 3
// of the group returns component l of the sum.
template <class CellFn, class PairFn>
__device__ __forceinline__ float coop_cells(CoopGroupLds &g, bool valid, CellFn cell, PairFn pair) {
    const int lane = (int)(threadIdx.x & 63u), l = lane & (kCoopLanes - 1), base = lane - l;
    unsigned b0 = 0u, e0 = 0u, b1 = 0u, e1 = 0u;
    if (valid) {
        cell(l, b0, e0);
        if (l + kCoopLanes < 27) cell(l + kCoopLanes, b1, e1);
    }
    // slots of the cells: exclusive sums over the cells 0..15, then 16..26
    const unsigned n0 = e0 - b0, n1 = e1 - b1;
    unsigned x0 = n0, x1 = n1;
#pragma unroll
    for (int d = 1; d < kCoopLanes; d <<= 1) {
        const unsigned y0 = __shfl_up(x0, d, kCoopLanes), y1 = __shfl_up(x1, d, kCoopLanes);
        if (l >= d) {
            x0 += y0;
            x1 += y1;
        }
    }
    const unsigned t0 = __shfl(x0, kCoopLanes - 1, kCoopLanes);
    const unsigned total = t0 + __shfl(x1, kCoopLanes - 1, kCoopLanes);
    float F = 0.f, csum = 0.f;
    if (!__any(total > 0u)) return F;
    g.off[l] = x0 - n0;
    g.beg[l] = b0;
    if (l + kCoopLanes < 28) {   // entry 27 closes the last cell: its lane holds no cell, x1 = the sum
        g.off[l + kCoopLanes] = t0 + x1 - n1;
        g.beg[l + kCoopLanes] = b1;
    }
    __builtin_amdgcn_wave_barrier();
    int n = 0, cur = -1, c = 0;
    for (unsigned s = 0u; __any(s < total); s += kCoopLanes) {
        const unsigned slot = s + (unsigned)l;
        bool hit = false;
        f3 f = mk3(0.f, 0.f, 0.f);
        if (slot < total) {
            while (slot >= g.off[c + 1]) ++c;
            hit = pair(g.beg[c] + (slot - g.off[c]), f);
        }
        const unsigned m = (unsigned)(__ballot(hit) >> base) & 0xffffu;
        if (hit) g.list[n + __popc(m & ((1u << l) - 1u))] = f4(f, __int_as_float(c));
        n += __popc(m);
        __builtin_amdgcn_wave_barrier();
        if (__any(n > kCoopList - kCoopLanes)) {
            coop_drain(g, n, l, cur, F, csum);
            n = 0;
            __builtin_amdgcn_wave_barrier();
        }
    }
    coop_drain(g, n, l, cur, F, csum);
    return F + csum;
}

}  // namespace arsim
