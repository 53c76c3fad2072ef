// grid.hip -- uniform-grid broadphase: cell bounds + reorder, and the 27-cell DEM kernel.
#include <type_traits>

#include "coop_cells.hpp"
#include "csr_fill.hpp"
#include "kernels.hpp"
#include "reduce_apply.hpp"

namespace arsim {

namespace {

// reorderDataAndFindCellStartD (Kernels/particleKernels.cu:193-258).  The previous key is read
// straight from global memory (it is in the same or the previous cache line).  The sorted copies
// carry the rbIndex in sortedPos.w and, when scene ids are given, the scene id in sortedVel.w.
__global__ void k_reorder(const unsigned *__restrict__ keys, const unsigned *__restrict__ idx,
                          const float4 *__restrict__ pos, const float4 *__restrict__ vel, const int *__restrict__ rb,
                          const uint16_t *__restrict__ scene, float4 *__restrict__ sPos, float4 *__restrict__ sVel,
                          unsigned *__restrict__ cs, unsigned *__restrict__ ce, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    unsigned h = keys[i];
    if (i == 0 || h != keys[i - 1]) {
        cs[h] = (unsigned)i;
        if (i > 0) ce[keys[i - 1]] = (unsigned)i;
    }
    if (i == n - 1) ce[h] = (unsigned)n;
    unsigned o = idx[i];
    float4 p = pos[o];
    p.w = __int_as_float(rb[o]);
    sPos[i] = p;
    float4 v = vel[o];
    if (scene) v.w = __int_as_float((int)scene[o]);
    sVel[i] = v;
}

// A particle's contact sum F, the walls added, to its body's force or to its velocity.
__device__ __forceinline__ void dem_write(f3 F, int ra, f3 pa, f3 va, unsigned orig, const DevPhys &ph,
                                          const SceneGeom &g, const DemOut &o) {
    if (!((ph.flags & kGrainClamp) && ra < 0)) F = add3(F, wall_force(pa, va, ph, g));
    if (ra >= 0) {
        o.pForce[orig] = f4(F, 0.0f);
        if (o.pTorque) o.pTorque[orig] = f4(cross3(xyz(o.relPos[orig]), F), 0.0f);
    } else {
        const float fs = (ph.flags & kRefUnits) ? 1.0f : ph.dt;
        o.vel[orig] = make_float4(va.x + F.x * fs, va.y + F.y * fs, va.z + F.z * fs, 0.0f);
    }
}

// Contacts found first and evaluated later.  A lane's candidate loop only tests distances and appends the sorted
// positions in reach to the lane's queue in LDS (kQueue entries, lane-interleaved); the pair forces are formed
// when a queue could overflow or the particle's cells are done, two at a time.  Formed in the candidate loop, a wave
// ran the pair force in every iteration in which any of its lanes had a contact; queued, it runs it about as often as
// its fullest lane has contacts.  Three candidates' loads together, 16 entries (12 drain too often: 922 us a step at
// the pile below, 16 874; two loads 900, four 878).  Settled pile of 2^22 particles: 634 -> 534 us.
// Where few candidates are contacts the positions read a second time cost more than that gives.
constexpr int kQueue = 16, kQueueAhead = 3;
constexpr int kQueueMax = (1 << 28) - 4;   // particles: an entry holds 16 times a sorted position, read up to kQueueAhead on
__device__ __forceinline__ float4 at16(const float4 *__restrict__ p, unsigned byteOffset) {
    return *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(p) + byteOffset);
}
struct ContactQueue {
    unsigned *first, *tail, *full;   // this lane's entries: first, first + stride, ..., tail; full: no room for kQueueAhead more
    unsigned stride;
    int cell;                        // code of the cell of the last entry appended
    f3 F, csum;
    __device__ __forceinline__ ContactQueue(unsigned *q, unsigned stride_)
        : first(q), tail(q), full(q + (kQueue - kQueueAhead) * stride_), stride(stride_), cell(-1),
          F(mk3(0.f, 0.f, 0.f)), csum(mk3(0.f, 0.f, 0.f)) {}
    // bit 0: the first contact of another cell, whose partial sum starts with it
    __device__ __forceinline__ void push(unsigned j16, int c) {
        *tail = j16 | (c != cell ? 1u : 0u);
        tail += stride;
        cell = c;
    }
    __device__ __forceinline__ void one(unsigned w, const float4 &Q, const float4 &V, f3 pa, f3 va, const DevPhys &ph) {
        if (w & 1u) {
            F = add3(F, csum);
            csum = mk3(0.f, 0.f, 0.f);
        }
        f3 fj;
        if (pair_force(pa, xyz(Q), va, xyz(V), ph, fj)) csum = add3(csum, fj);
    }
    __device__ __forceinline__ void drain(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel, f3 pa, f3 va,
                                          const DevPhys &ph) {
        for (unsigned *p = first; p < tail; p += 2 * stride) {
            const unsigned w0 = *p;
            const bool two = p + stride < tail;
            const unsigned w1 = two ? p[stride] : w0;
            const float4 Q0 = at16(sPos, w0 & ~15u), V0 = at16(sVel, w0 & ~15u);
            const float4 Q1 = at16(sPos, w1 & ~15u), V1 = at16(sVel, w1 & ~15u);
            __builtin_amdgcn_sched_barrier(0);
            one(w0, Q0, V0, pa, va, ph);
            if (two) one(w1, Q1, V1, pa, va, ph);
        }
        tail = first;
    }
    // Queues the contacts of a run [j, e) whose second and third cells (code + 1, + 2) start at b1 and b2.
    __device__ __forceinline__ void run(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel, unsigned j,
                                        unsigned b1, unsigned b2, unsigned e, int code, unsigned i16, int ra, f3 pa, f3 va,
                                        const DevPhys &ph) {
        const unsigned e16 = e << 4, b116 = b1 << 4, b216 = b2 << 4;
        for (unsigned j16 = j << 4; j16 < e16; j16 += 16u * kQueueAhead) {
            unsigned jj[kQueueAhead];
            float4 Q[kQueueAhead];
#pragma unroll
            for (int u = 0; u < kQueueAhead; ++u) {
                jj[u] = j16 + 16u * u;
                if (u && !(jj[u] < e16)) jj[u] = i16;   // the particle itself: never a contact
                Q[u] = at16(sPos, jj[u]);
            }
            __builtin_amdgcn_sched_barrier(0);   // every load issued before the first is waited for
#pragma unroll
            for (int u = 0; u < kQueueAhead; ++u) {
                const f3 rel = sub3(xyz(Q[u]), pa);
                const bool near = !(dot3(rel, rel) > ph.cd2Reject);
                if (near & (jj[u] != i16) & pair_allowed(ra, __float_as_int(Q[u].w)))
                    push(jj[u], code + (jj[u] >= b116 ? 1 : 0) + (jj[u] >= b216 ? 1 : 0));
            }
            if (tail > full) drain(sPos, sVel, pa, va, ph);
        }
    }
};

// FindAndHandleRigidBodyCollisionsUniformGridKernel (RigidBodies/UniformGridDEM.cu:133-204) and
// collideD (particleKernels.cu:302-406): 27 cells in z, y, x order, per-cell partial sums, the
// contact predicate j != i && (rbA != rbB || rbA == -1), then the wall term.  EMIT writes the
// contact list instead of forces.
template <bool EMIT>
__global__ void k_dem_grid(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                           const unsigned *__restrict__ sIdx, const unsigned *__restrict__ cs,
                           const unsigned *__restrict__ ce, int n, DevPhys ph, SceneView sv, int sceneInVelW,
                           DemOut o) {
    const int lb = xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int i = lb * (int)blockDim.x + (int)threadIdx.x;
    if (i >= n) return;
    const float4 P = sPos[i];
    const float4 Vq = sVel[i];
    const int ra = __float_as_int(P.w);
    const int s = sceneInVelW ? __float_as_int(Vq.w) : 0;
    SceneGeom g;
    load_geom(sv, s, g);
    const f3 pa = xyz(P), va = xyz(Vq);
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const unsigned orig = sIdx[i];
    f3 F = mk3(0.f, 0.f, 0.f);
    int cnt = 0;
    for (int z = -1; z <= 1; ++z)
        for (int y = -1; y <= 1; ++y)
            for (int x = -1; x <= 1; ++x) {
                unsigned h = g.cellBase + grid_hash(gx + x, gy + y, gz + z, g);
                unsigned st = cs[h];
                if (st == kEmpty) continue;
                unsigned en = ce[h];
                f3 csum = mk3(0.f, 0.f, 0.f);
                for (unsigned j = st; j < en; ++j) {
                    float4 Q = sPos[j];
                    if (!candidate(Q, pa, ra, (int)j == i, ph)) continue;
                    if (EMIT) {
                        if (in_contact(pa, xyz(Q), ph)) {
                            if (cnt < o.maxPer) o.pairs[(size_t)orig * o.maxPer + cnt] = (int)sIdx[j];
                            ++cnt;
                        }
                    } else {
                        f3 fj;
                        if (pair_force(pa, xyz(Q), va, xyz(sVel[j]), ph, fj)) csum = add3(csum, fj);
                    }
                }
                F = add3(F, csum);
            }
    if (EMIT) {
        o.counts[orig] = cnt;
        return;
    }
    if (!((ph.flags & kGrainClamp) && ra < 0)) F = add3(F, wall_force(pa, va, ph, g));
    if (ra >= 0) {
        o.pForce[orig] = f4(F, 0.0f);
        if (o.pTorque) o.pTorque[orig] = f4(cross3(xyz(o.relPos[orig]), F), 0.0f);
    } else {
        const float fs = (ph.flags & kRefUnits) ? 1.0f : ph.dt;
        o.vel[orig] = make_float4(va.x + F.x * fs, va.y + F.y * fs, va.z + F.z * fs, 0.0f);
    }
}

// The same sums over queued contacts, a row's three cells together: their starts in one round trip, then their ends,
// and where the cells' runs follow each other (unless x wraps they do in a sorted point set) one run of candidates.
// Bound by the table's lines: in a scattered scene with twice 64 MB of tables every row is a miss, and read cell by
// cell the eight waves a SIMD evicted each other's lines between a row's reads.  Cell by cell with one candidate at a
// time and no queue, cell by cell with the queue, and now: 2^20 scattered particles 157, 240 and 117 us, piles of
// 300,007 77, 57 and 49, of 2^22 848, 692 and 555, a mixed scene of 800,000 211, 192 and 163.
__global__ void k_dem_grid_ref_queue(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                     const unsigned *__restrict__ sIdx, const unsigned *__restrict__ cs,
                                     const unsigned *__restrict__ ce, int n, DevPhys ph, SceneGeom g, DemOut o) {
    extern __shared__ unsigned queueLds[];
    const int i = xcd_block((int)blockIdx.x, (int)gridDim.x) * (int)blockDim.x + (int)threadIdx.x;
    if (i >= n) return;
    const float4 P = sPos[i];
    const float4 Vq = sVel[i];
    const int ra = __float_as_int(P.w);
    const f3 pa = xyz(P), va = xyz(Vq);
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    ContactQueue cq(queueLds + threadIdx.x, blockDim.x);
    for (int r = 0; r < 9; ++r) {
        const int y = gy + r % 3 - 1, z = gz + r / 3 - 1;
        const unsigned h[3] = {g.cellBase + grid_hash(gx - 1, y, z, g), g.cellBase + grid_hash(gx, y, z, g),
                               g.cellBase + grid_hash(gx + 1, y, z, g)};
        unsigned b[3], e[3];
        bool some[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) b[k] = cs[h[k]];
#pragma unroll
        for (int k = 0; k < 3; ++k) e[k] = b[k] != kEmpty ? ce[h[k]] : 0u;
#pragma unroll
        for (int k = 0; k < 3; ++k) some[k] = b[k] < e[k];
        // the cells' runs lie one after another unless x wraps (or a caller's own table says otherwise)
        const unsigned last = some[2] ? e[2] : some[1] ? e[1] : e[0];
        const unsigned b2 = some[2] ? b[2] : last, b1 = some[1] ? b[1] : b2;
        const bool joined = (!some[0] || e[0] == b1) & (!some[1] || e[1] == b2);
        if (joined) {
            cq.run(sPos, sVel, some[0] ? b[0] : b1, b1, b2, last, 3 * r, (unsigned)i << 4, ra, pa, va, ph);
        } else {
#pragma unroll 1
            for (int k = 0; k < 3; ++k) {
                const unsigned st = k == 0 ? b[0] : k == 1 ? b[1] : b[2], en = k == 0 ? e[0] : k == 1 ? e[1] : e[2];
                if (st < en) cq.run(sPos, sVel, st, en, en, en, 3 * r + k, (unsigned)i << 4, ra, pa, va, ph);
            }
        }
    }
    cq.drain(sPos, sVel, pa, va, ph);
    dem_write(add3(cq.F, cq.csum), ra, pa, va, sIdx[i], ph, g, o);
}

// Engine form of the reorder: the same gather of the sorted copies, but instead of the two
// cell-sized tables it writes a dense CSR offset array over segments of 2^segBits cells:
// segStart[s] = first sorted index whose key >= s << segBits (segStart[numSegs] = n).  Every entry
// is rewritten each step, so nothing has to be cleared.  With segBits = 0 it is cellStart with
// cellEnd[c] = segStart[c + 1], one table instead of two.  numSegs < 2^32.
// The long runs handed over by wave_fill, one chunk of at most kLongChunk entries per workgroup
// (workgroup g takes chunks g, g + G, ...).  With nothing listed the kernel only reads the count.
constexpr unsigned kFillBlocks = 512u;
__global__ __launch_bounds__(256) void k_fill_long(unsigned *__restrict__ table, unsigned long long size, LongFill lf) {
    const unsigned cnt = min(*lf.count, lf.cap);
    for (unsigned r = blockIdx.x; r < cnt; r += gridDim.x) {
        const uint4 e = lf.list[r];
        // (the capacity bound means every listed entry was written; the clamp keeps stores in the table)
        const unsigned a = e.x, b = (unsigned long long)e.y < size ? e.y : (unsigned)size;
        if (a >= b) continue;
        // scalar head and tail, 16-byte stores for the aligned middle
        const unsigned a4 = (a + 3u) & ~3u, b4 = b & ~3u;
        if (a4 >= b4) {
            for (unsigned k = a + threadIdx.x; k < b; k += 256u) table[k] = e.z;
            continue;
        }
        if (threadIdx.x < a4 - a) table[a + threadIdx.x] = e.z;
        if (threadIdx.x < b - b4) table[b4 + threadIdx.x] = e.z;
        const uint4 v4 = make_uint4(e.z, e.z, e.z, e.z);
        for (unsigned k = a4 + 4u * threadIdx.x; k < b4; k += 1024u) *reinterpret_cast<uint4 *>(table + k) = v4;
    }
}

__global__ void k_reorder_seg(const unsigned *__restrict__ keys, const unsigned *__restrict__ idx,
                              const float4 *__restrict__ pos, const float4 *__restrict__ vel,
                              const int *__restrict__ rb, const uint16_t *__restrict__ scene,
                              const float4 *__restrict__ rec, float4 *__restrict__ sPos, float4 *__restrict__ sVel,
                              unsigned *__restrict__ segStart, int segBits, long long numSegs, int n,
                              LongFill lf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const unsigned k = valid ? keys[i] : 0u;
    const unsigned s = k >> segBits;
    const unsigned sp1 = (valid && i > 0) ? (keys[i - 1] >> segBits) + 1u : 0u;   // first segment not yet started
    wave_fill(segStart, valid && s + 1u > sp1, sp1, s + 1u, (unsigned)i, lf);
    wave_fill(segStart, i == n - 1, s + 1u, (unsigned)numSegs + 1u, (unsigned)n, lf);
    if (!valid) return;
    const unsigned o = idx[i];
    if (rec) {
        sPos[i] = rec[2 * (size_t)o];
        sVel[i] = rec[2 * (size_t)o + 1];
        return;
    }
    float4 p = pos[o];
    p.w = __int_as_float(rb[o]);
    sPos[i] = p;
    float4 v = vel[o];
    if (scene) v.w = __int_as_float((int)scene[o]);
    sVel[i] = v;
}

// Contacts of one sorted particle within the sorted-key run [j, ...) of cells h0..h1 (one row of
// up to three consecutive cells), cell by cell in ascending order, each cell's contacts summed
// into a partial that is added to F when the cell ends -- the same grouping and order as the
// 27-cell loop over cellStart / cellEnd.
// Forward scan of the sorted keys from j (a segment start at or before h0): skips keys below h0,
// stops past h1.  (Reading several candidates per round trip was measured slower: the extra
// registers cost more occupancy than the latency it hid.)
template <bool EMIT>
__device__ __forceinline__ void scan_cells(const unsigned *__restrict__ keys, const float4 *__restrict__ sPos,
                                           const float4 *__restrict__ sVel, const unsigned *__restrict__ sIdx,
                                           unsigned j, int n, unsigned h0, unsigned h1, int i, int ra, f3 pa, f3 va,
                                           const DevPhys &ph, f3 &F, int &cnt, unsigned orig, const DemOut &o) {
    unsigned cur = 0xffffffffu;
    f3 csum = mk3(0.f, 0.f, 0.f);
    for (; (int)j < n; ++j) {
        const unsigned kj = keys[j];
        if (kj > h1) break;
        if (kj < h0) continue;
        if (kj != cur) {
            if (cur != 0xffffffffu) F = add3(F, csum);
            csum = mk3(0.f, 0.f, 0.f);
            cur = kj;
        }
        const float4 Q = sPos[j];
        if (!candidate(Q, pa, ra, (int)j == i, ph)) continue;
        if (EMIT) {
            if (in_contact(pa, xyz(Q), ph)) {
                if (cnt < o.maxPer) o.pairs[(size_t)orig * o.maxPer + cnt] = (int)sIdx[j];
                ++cnt;
            }
        } else {
            f3 fj;
            if (pair_force(pa, xyz(Q), va, xyz(sVel[j]), ph, fj)) csum = add3(csum, fj);
        }
    }
    if (cur != 0xffffffffu) F = add3(F, csum);
}

// Contacts of one particle with the sorted run [j, e) that holds up to three consecutive cells, the
// second starting at b1 and the third at b2 (exact cell offsets: no key is read).  A cell's partial
// is added to F when a non-empty cell ends, as in the 27-cell loop.
// Candidates are loaded two at a time (the second index clamped into the run), so that a wave has
// two loads in flight per lane: the loop is bound by load latency, not by the force arithmetic.
// Three or more per round trip cost more occupancy (registers) than they hide.
// The particle itself is excluded by its sorted index i (SELF_BY_ORIG false), or, when the caller
// walks particles in their original order, by its original index: only a candidate at distance 0
// from a grain can be the grain itself, so only then is the candidate's original index read (a body
// particle's own copy is excluded by the same-body rule anyway).
template <bool EMIT, bool SELF_BY_ORIG = false>
__device__ __forceinline__ void scan_run(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                         const unsigned *__restrict__ sIdx, unsigned j, unsigned b1, unsigned b2,
                                         unsigned e, int i, int ra, f3 pa, f3 va, const DevPhys &ph, f3 &F, int &cnt,
                                         unsigned orig, const DemOut &o) {
    const unsigned j0 = j;
    f3 csum = mk3(0.f, 0.f, 0.f);
    auto visit = [&](unsigned jj, const float4 &Q) {
        if (jj != j0 && (jj == b1 || jj == b2)) {
            F = add3(F, csum);
            csum = mk3(0.f, 0.f, 0.f);
        }
        if (SELF_BY_ORIG) {
            const f3 rel = sub3(mk3(Q.x, Q.y, Q.z), pa);
            const float d2 = dot3(rel, rel);
            bool ok = !(d2 > ph.cd2Reject) & pair_allowed(ra, __float_as_int(Q.w));
            if (ok && ra < 0 && d2 == 0.0f) ok = sIdx[jj] != orig;
            if (!ok) return;
        } else {
            if (!candidate(Q, pa, ra, (int)jj == i, ph)) return;
        }
        if (EMIT) {
            if (in_contact(pa, xyz(Q), ph)) {
                if (cnt < o.maxPer) o.pairs[(size_t)orig * o.maxPer + cnt] = (int)sIdx[jj];
                ++cnt;
            }
        } else {
            f3 fj;
            if (pair_force(pa, xyz(Q), va, xyz(sVel[jj]), ph, fj)) csum = add3(csum, fj);
        }
    };
    for (; j < e; j += 2u) {
        const float4 Q0 = sPos[j];
        const float4 Q1 = sPos[j + 1u < e ? j + 1u : j];
        visit(j, Q0);
        if (j + 1u < e) visit(j + 1u, Q1);
    }
    if (e > j0) F = add3(F, csum);
}

// Σ of the pair forces on one particle over its 27 neighbour cells with the exact cell table
// (segStart = cellStart, numCells + 1 entries): for each of the 9 (dz, dy) rows in z, y order the
// three x-cells are one contiguous run [segStart[h0], segStart[h0 + 3]) unless x wraps, visited in
// the order x-1, x, x+1.  The walls are not included.
template <bool EMIT, bool SELF_BY_ORIG>
__device__ __forceinline__ f3 dem_rows_exact(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                             const unsigned *__restrict__ sIdx, const unsigned *__restrict__ segStart,
                                             const SceneGeom &g, int i, int ra, f3 pa, f3 va, const DevPhys &ph,
                                             int &cnt, unsigned orig, const DemOut &o) {
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const unsigned x0 = (unsigned)(gx - 1) & g.gridMask[0], x1 = (unsigned)gx & g.gridMask[0],
                   x2 = (unsigned)(gx + 1) & g.gridMask[0];
    const bool contiguous = (x0 + 1u == x1) && (x1 + 1u == x2);
    f3 F = mk3(0.f, 0.f, 0.f);
    auto row_of = [&](int r) {
        const unsigned uz = (unsigned)(gz + (r / 3) - 1) & g.gridMask[2];
        const unsigned uy = (unsigned)(gy + (r % 3) - 1) & g.gridMask[1];
        return g.cellBase + uz * g.gxy + uy * g.gx;
    };
    for (int r = 0; r < 9; ++r) {
        const unsigned row = row_of(r);
        if (contiguous) {
            // the row's four offsets in one 16-byte load (4-byte aligned): the kernel issues fewer
            // vector memory instructions, which bound it more than bytes do
            uint4 bnd;
            __builtin_memcpy(&bnd, segStart + row + x0, sizeof(bnd));
            scan_run<EMIT, SELF_BY_ORIG>(sPos, sVel, sIdx, bnd.x, bnd.y, bnd.z, bnd.w, i, ra, pa, va, ph, F, cnt,
                                         orig, o);
        } else {
            const unsigned xs[3] = {x0, x1, x2};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const unsigned h = row + xs[k];
                const unsigned e = segStart[h + 1];
                scan_run<EMIT, SELF_BY_ORIG>(sPos, sVel, sIdx, segStart[h], e, e, e, i, ra, pa, va, ph, F, cnt,
                                             orig, o);
            }
        }
    }
    return F;
}

// Engine DEM over the segment index: for each of the 9 (dz, dy) rows the three x-cells are
// consecutive keys unless x wraps, so one segment lookup and one forward scan of the sorted
// keys visit them in the order x-1, x, x+1.  EXACT (segments of one cell, segStart = cellStart
// with numCells + 1 entries): a row is the run [segStart[h0], segStart[h0 + 3]) with its cell
// boundaries read from the table, and the keys are not read at all.
// Where a block's scene geometry comes from: the one scene's, passed by value (kGeomSingle); for several
// scenes (scene id in sortedVel.w), the table entry of the block's scene when all of the block's
// particles belong to it (kGeomBlock: scalar loads), or each lane's own entry (kGeomLane).
enum { kGeomSingle = 0, kGeomBlock = 1, kGeomLane = 2 };
// The blocks of a batch's launch: first one workgroup per boundary between scenes k - 1 and k, which takes the
// block that holds the boundary with kGeomLane (if the boundary lies strictly inside a block and no
// earlier boundary lies strictly inside the same one), then every block, those of one scene being
// taken with kGeomBlock.  As a launch of their own after the others the boundary blocks were alone on the
// chip for 27 to 37 us: 128 scenes' step 314 -> 289 us, 24 larger scenes' 50 steps 14.7 -> 13.5 ms.  They are filled up
// to a multiple of the XCDs (sv.boundaryBlocks), so that the blocks after them run on the XCD whose L2 the bucket sort left
// them in, and the next step's bucket sort finds its own: 8 scenes of 16,000 particles step 68.8 -> 61.9 us.
__device__ __forceinline__ bool boundary_block(const SceneView &sv, int n, int &lb) {
    const int k = (int)blockIdx.x + 1, bs = (int)blockDim.x;
    const int b = sv.sceneStart[k], pb = sv.sceneStart[k - 1];
    lb = b / bs;
    if (b % bs == 0 || b >= n) return false;
    return !(k > 1 && pb / bs == lb && pb % bs != 0);
}
// Whether block lb lies in one scene.
__device__ __forceinline__ bool one_scene(const float4 *__restrict__ sVel, int lb, int n, int &scene) {
    const int first = lb * (int)blockDim.x, last = min(n, first + (int)blockDim.x) - 1;
    scene = __float_as_int(sVel[first].w);
    return scene == __float_as_int(sVel[last].w);
}
// Runs body(lb, g, lanes) for this workgroup's block: g its scene's geometry, or none (lanes true).
template <bool BATCH, class Body>
__device__ __forceinline__ void for_dem_block(const SceneView &sv, const float4 *__restrict__ sVel, int n, Body body) {
    if (!BATCH) {
        body(xcd_block((int)blockIdx.x, (int)gridDim.x), sv.single, std::integral_constant<int, kGeomSingle>{});
        return;
    }
    const int boundaries = sv.boundaryBlocks;
    int lb, scene;
    if ((int)blockIdx.x < boundaries) {
        if ((int)blockIdx.x >= sv.count - 1) return;   // (a block that only fills up)
        if (!boundary_block(sv, n, lb) || one_scene(sVel, lb, n, scene)) return;
        body(lb, SceneGeom{}, std::integral_constant<int, kGeomLane>{});
        return;
    }
    lb = xcd_block((int)blockIdx.x - boundaries, (int)gridDim.x - boundaries);
    if (!one_scene(sVel, lb, n, scene)) return;
    body(lb, sv.table[scene], std::integral_constant<int, kGeomBlock>{});
}
template <bool EMIT, bool EXACT, int GEOM>
__device__ __forceinline__ void dem_seg_block(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                              const unsigned *__restrict__ keys, const unsigned *__restrict__ sIdx,
                                              const unsigned *__restrict__ segStart, int segBits, int n,
                                              const DevPhys &ph, const SceneView &sv, const DemOut &o, int lb,
                                              SceneGeom g) {
    const int first = lb * (int)blockDim.x;
    const int i = first + (int)threadIdx.x;
    if (i >= n) return;
    const float4 P = sPos[i];
    const float4 Vq = sVel[i];
    const int ra = __float_as_int(P.w);
    if (GEOM == kGeomLane) g = sv.table[__float_as_int(Vq.w)];
    const f3 pa = xyz(P), va = xyz(Vq);
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const unsigned orig = sIdx[i];
    const unsigned x0 = (unsigned)(gx - 1) & g.gridMask[0], x1 = (unsigned)gx & g.gridMask[0],
                   x2 = (unsigned)(gx + 1) & g.gridMask[0];
    const bool contiguous = (x0 + 1u == x1) && (x1 + 1u == x2);
    f3 F = mk3(0.f, 0.f, 0.f);
    int cnt = 0;
    // the nine row starts are independent: issue all their loads before scanning any row
    auto row_of = [&](int r) {
        const unsigned uz = (unsigned)(gz + (r / 3) - 1) & g.gridMask[2];
        const unsigned uy = (unsigned)(gy + (r % 3) - 1) & g.gridMask[1];
        return g.cellBase + uz * g.gxy + uy * g.gx;
    };
    if (EXACT) {
        for (int r = 0; r < 9; ++r) {
            const unsigned row = row_of(r);
            if (contiguous) {
                const unsigned h0 = row + x0;
                // the row's four offsets in one 16-byte load (4-byte aligned): the kernel issues fewer
                // vector memory instructions, which bound it more than bytes do
                uint4 bnd;
                __builtin_memcpy(&bnd, segStart + h0, sizeof(bnd));
                scan_run<EMIT>(sPos, sVel, sIdx, bnd.x, bnd.y, bnd.z, bnd.w, i, ra, pa, va, ph, F, cnt, orig, o);
            } else {
                const unsigned xs[3] = {x0, x1, x2};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const unsigned h = row + xs[k];
                    const unsigned e = segStart[h + 1];
                    scan_run<EMIT>(sPos, sVel, sIdx, segStart[h], e, e, e, i, ra, pa, va, ph, F, cnt, orig, o);
                }
            }
        }
    } else {
        unsigned rowJ[9];
        if (contiguous) {
#pragma unroll
            for (int r = 0; r < 9; ++r) rowJ[r] = segStart[(row_of(r) + x0) >> segBits];
        }
        for (int r = 0; r < 9; ++r) {
            const unsigned row = row_of(r);
            if (contiguous) {
                const unsigned h0 = row + x0;
                scan_cells<EMIT>(keys, sPos, sVel, sIdx, rowJ[r], n, h0, h0 + 2u, i, ra, pa, va, ph, F, cnt, orig, o);
            } else {
                const unsigned xs[3] = {x0, x1, x2};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const unsigned h = row + xs[k];
                    scan_cells<EMIT>(keys, sPos, sVel, sIdx, segStart[h >> segBits], n, h, h, i, ra, pa, va, ph, F,
                                     cnt, orig, o);
                }
            }
        }
    }
    if (EMIT) {
        o.counts[orig] = cnt;
        return;
    }
    dem_write(F, ra, pa, va, orig, ph, g, o);
}
// Eight waves a SIMD, in 64 registers: with several scenes the kernels took 66 to 72, for seven (128 scenes' step 289 us,
// so 285; nothing is spilled).
template <bool EMIT, bool EXACT, bool BATCH>
__global__ __attribute__((amdgpu_waves_per_eu(8))) void k_dem_grid_seg(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                               const unsigned *__restrict__ keys, const unsigned *__restrict__ sIdx,
                               const unsigned *__restrict__ segStart, int segBits, int n, DevPhys ph, SceneView sv,
                               DemOut o) {
    for_dem_block<BATCH>(sv, sVel, n, [&](int lb, const SceneGeom &g, auto geom) {
        dem_seg_block<EMIT, EXACT, decltype(geom)::value>(sPos, sVel, keys, sIdx, segStart, segBits, n, ph, sv, o, lb, g);
    });
}

// The contact kernel over the exact cell table, contacts queued.
template <int GEOM>
__device__ __forceinline__ void dem_queue_block(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                                const unsigned *__restrict__ sIdx,
                                                const unsigned *__restrict__ segStart, int n, const DevPhys &ph,
                                                const SceneView &sv, const DemOut &o, int lb, SceneGeom g,
                                                unsigned *queue) {
    const int i = lb * (int)blockDim.x + (int)threadIdx.x;
    if (i >= n) return;
    const float4 P = sPos[i];
    const float4 Vq = sVel[i];
    const int ra = __float_as_int(P.w);
    if (GEOM == kGeomLane) g = sv.table[__float_as_int(Vq.w)];
    const f3 pa = xyz(P), va = xyz(Vq);
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const unsigned x0 = (unsigned)(gx - 1) & g.gridMask[0], x1 = (unsigned)gx & g.gridMask[0],
                   x2 = (unsigned)(gx + 1) & g.gridMask[0];
    const bool contiguous = (x0 + 1u == x1) && (x1 + 1u == x2);
    ContactQueue cq(queue, blockDim.x);
    for (int r = 0; r < 9; ++r) {
        const unsigned uz = (unsigned)(gz + (r / 3) - 1) & g.gridMask[2];
        const unsigned uy = (unsigned)(gy + (r % 3) - 1) & g.gridMask[1];
        const unsigned row = g.cellBase + uz * g.gxy + uy * g.gx;
        if (contiguous) {
            // the row's four offsets in one 16-byte load (4-byte aligned)
            uint4 bnd;
            __builtin_memcpy(&bnd, segStart + (row + x0), sizeof(bnd));
            cq.run(sPos, sVel, bnd.x, bnd.y, bnd.z, bnd.w, 3 * r, (unsigned)i << 4, ra, pa, va, ph);
        } else {
#pragma unroll 1
            for (int k = 0; k < 3; ++k) {
                const unsigned h = row + (k == 0 ? x0 : k == 1 ? x1 : x2);
                const unsigned e = segStart[h + 1u];
                cq.run(sPos, sVel, segStart[h], e, e, e, 3 * r + k, (unsigned)i << 4, ra, pa, va, ph);
            }
        }
    }
    cq.drain(sPos, sVel, pa, va, ph);
    dem_write(add3(cq.F, cq.csum), ra, pa, va, sIdx[i], ph, g, o);
}
template <bool BATCH>
__global__ __attribute__((amdgpu_waves_per_eu(8))) void k_dem_grid_queue(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                 const unsigned *__restrict__ sIdx, const unsigned *__restrict__ segStart, int n,
                                 DevPhys ph, SceneView sv, DemOut o) {
    extern __shared__ unsigned queueLds[];
    for_dem_block<BATCH>(sv, sVel, n, [&](int lb, const SceneGeom &g, auto geom) {
        dem_queue_block<decltype(geom)::value>(sPos, sVel, sIdx, segStart, n, ph, sv, o, lb, g, queueLds + threadIdx.x);
    });
}

// The contact kernel over the compact cell index: the occupied cells of all nine rows first (nine loads in
// flight, from an index of a quarter byte a cell where the table has four), then the rows that have any, each
// lane its own next one.  At the 2^20-particle scene it takes as long as with the table (68 us: what it saves in
// memory it spends in instructions), while the bucket sort, which wrote the table, goes from 45 to 31 us;
// at 128 mixed scenes 148 -> 144 and 117 -> 72 us.
template <int GEOM>
__device__ __forceinline__ void dem_index_block(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                                const unsigned *__restrict__ sIdx, const CellIndex &ix, int n,
                                                const DevPhys &ph, const SceneView &sv, const DemOut &o, int lb,
                                                SceneGeom g, unsigned *sRank) {
    const int first = lb * (int)blockDim.x;
    const int i = first + (int)threadIdx.x;
    if (i >= n) return;
    const float4 P = sPos[i];
    const float4 Vq = sVel[i];
    const int ra = __float_as_int(P.w);
    if (GEOM == kGeomLane) g = sv.table[__float_as_int(Vq.w)];
    const f3 pa = xyz(P), va = xyz(Vq);
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const unsigned orig = sIdx[i];
    const unsigned x0 = (unsigned)(gx - 1) & g.gridMask[0], x1 = (unsigned)gx & g.gridMask[0],
                   x2 = (unsigned)(gx + 1) & g.gridMask[0];
    const bool contiguous = (x0 + 1u == x1) && (x1 + 1u == x2);
    const int lgx = __ffs((int)g.gx) - 1, lgxy = __ffs((int)g.gxy) - 1;
    f3 F = mk3(0.f, 0.f, 0.f);
    int cnt = 0;
    auto row_of = [&](int r) {
        const unsigned uz = (unsigned)(gz + (r / 3) - 1) & g.gridMask[2];
        const unsigned uy = (unsigned)(gy + (r % 3) - 1) & g.gridMask[1];
        return g.cellBase + (uz << lgxy) + (uy << lgx);
    };
    if (contiguous) {
        unsigned rows = 0u;   // three bits a row: its occupied cells
#pragma unroll
        for (int z = 0; z < 3; ++z) {
            uint4 w[3];
#pragma unroll
            for (int y = 0; y < 3; ++y) __builtin_memcpy(&w[y], ix.words + ((row_of(3 * z + y) + x0) >> 5), sizeof(uint4));
#pragma unroll
            for (int y = 0; y < 3; ++y) {
                const int r = 3 * z + y;
                const unsigned sh = (row_of(r) + x0) & 31u;
                const unsigned lowBits = w[y].x >> sh;
                const unsigned bits = __builtin_amdgcn_alignbit(w[y].z, w[y].x, sh) & 7u;
                sRank[r * blockDim.x + threadIdx.x] =
                    lowBits ? w[y].y + __popc(w[y].x & ((1u << sh) - 1u)) : w[y].w;
                rows |= bits << (3 * r);
            }
        }
        while (rows) {
            const unsigned r = (unsigned)__builtin_ctz(rows) / 3u;
            const unsigned bits = (rows >> (3u * r)) & 7u;
            rows &= ~(7u << (3u * r));
            const unsigned slot = sRank[r * blockDim.x + threadIdx.x];
            uint4 s;
            __builtin_memcpy(&s, ix.starts + slot, sizeof(s));
            const unsigned n0 = bits & 1u, n01 = n0 + ((bits >> 1) & 1u), n012 = n01 + (bits >> 2);
            const unsigned b1 = n0 ? s.y : s.x;
            const unsigned b2 = n01 == 0u ? s.x : n01 == 1u ? s.y : s.z;
            const unsigned e = n012 == 1u ? s.y : n012 == 2u ? s.z : s.w;
            scan_run<false>(sPos, sVel, sIdx, s.x, b1, b2, e, i, ra, pa, va, ph, F, cnt, orig, o);
        }
    } else {
        for (int r = 0; r < 9; ++r) {
            const unsigned row = row_of(r);
#pragma unroll 1
            for (int k = 0; k < 3; ++k) {
                const unsigned h = row + (k == 0 ? x0 : k == 1 ? x1 : x2);
                const uint2 w = ix.words[h >> 5];
                if (!((w.x >> (h & 31u)) & 1u)) continue;
                const unsigned *st = ix.starts + w.y + __popc(w.x & ((1u << (h & 31u)) - 1u));
                const unsigned e = st[1];
                scan_run<false>(sPos, sVel, sIdx, st[0], e, e, e, i, ra, pa, va, ph, F, cnt, orig, o);
            }
        }
    }
    dem_write(F, ra, pa, va, orig, ph, g, o);
}
template <bool BATCH>
__global__ __attribute__((amdgpu_waves_per_eu(8))) void k_dem_grid_index(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                 const unsigned *__restrict__ sIdx, CellIndex ix, int n, DevPhys ph, SceneView sv,
                                 DemOut o) {
    extern __shared__ unsigned sRank[];   // per row and thread: slot of the row's first occupied cell
    for_dem_block<BATCH>(sv, sVel, n, [&](int lb, const SceneGeom &g, auto geom) {
        dem_index_block<decltype(geom)::value>(sPos, sVel, sIdx, ix, n, ph, sv, o, lb, g, sRank);
    });
}

// The contact kernel with 16 lanes per particle (coop_cells): cells of the reference's cellStart / cellEnd (REF)
// or of the exact table (cs = segStart); sceneTable: each particle's scene (its id in sortedVel.w), else the one
// scene g.  For the sizes at which there are too few waves to hide a thread's chain of lookups and candidate loads:
// 16,384 particles of c0's cubes 15.2 -> 9.6 us, 50,021 mixed ones 25 -> 17, a pile of 65,536 61 -> 28.  The lanes'
// shared steps (slots, ranks, the ordered adds) cost more than the chains from about (per thread and with 16 lanes, us)
//   one scene: 91,000 mixed 32 and 26.5, 98,000 25.7 and 27.1, 196,608 48 and 55; cubes 91,000 26 and 23, 196,608 30
//   and 43; piles 131,000 48.8 and 46.6 (the queue), 150,000 51.2 and 52.0, 196,608 54 and 64
//   several: 4 of 17,000 21.8 and 18.8, 24 of 3,000 21.4 and 20.2, 5 of 16,000 17.7 and 21.1,
//   12 of 16,000 21 and 40, 100 of 1,900 23 and 40
//   the reference's layout: 91,000 mixed 28 and 25, 98,000 20 and 26; piles 91,000 36 and 33, 115,000 36 and 40
constexpr int kCoopBlock = 128;
template <bool REF>
__global__ __launch_bounds__(kCoopBlock) void k_dem_grid_coop(const float4 *__restrict__ sPos,
                                                              const float4 *__restrict__ sVel,
                                                              const unsigned *__restrict__ sIdx,
                                                              const unsigned *__restrict__ cs,
                                                              const unsigned *__restrict__ ce, int n, DevPhys ph,
                                                              SceneGeom g, const SceneGeom *__restrict__ sceneTable,
                                                              DemOut o) {
    __shared__ CoopGroupLds sGroup[kCoopBlock / kCoopLanes];
    const int gl = (int)threadIdx.x / kCoopLanes, l = (int)threadIdx.x & (kCoopLanes - 1);
    const int i = xcd_block((int)blockIdx.x, (int)gridDim.x) * (kCoopBlock / kCoopLanes) + gl;
    const bool valid = i < n;
    const float4 P = sPos[valid ? i : n - 1], Vq = sVel[valid ? i : n - 1];
    const unsigned orig = sIdx[valid ? i : n - 1];
    const int ra = __float_as_int(P.w);
    const f3 pa = xyz(P), va = xyz(Vq);
    if (sceneTable) g = sceneTable[__float_as_int(Vq.w)];
    int gx, gy, gz;
    grid_pos(pa, g, gx, gy, gz);
    const float Fc = coop_cells(
        sGroup[gl], valid,
        [&](int c, unsigned &b, unsigned &e) {
            const unsigned h = g.cellBase + grid_hash(gx + c % 3 - 1, gy + (c / 3) % 3 - 1, gz + c / 9 - 1, g);
            b = cs[h];
            e = REF ? ce[h] : cs[h + 1];
            if (REF && (b == kEmpty || e < b)) b = e = 0u;   // an empty cell's end is not defined
        },
        [&](unsigned j, f3 &f) {
            const float4 Q = sPos[j];
            if (!candidate(Q, pa, ra, (int)j == i, ph)) return false;
            return pair_force(pa, xyz(Q), va, xyz(sVel[j]), ph, f);
        });
    f3 F = mk3(__shfl(Fc, 0, kCoopLanes), __shfl(Fc, 1, kCoopLanes), __shfl(Fc, 2, kCoopLanes));
    if (!valid || l > 3) return;
    if (!((ph.flags & kGrainClamp) && ra < 0)) F = add3(F, wall_force(pa, va, ph, g));
    auto pick = [l](f3 v) { return l == 0 ? v.x : l == 1 ? v.y : l == 2 ? v.z : 0.0f; };
    if (ra >= 0) {
        reinterpret_cast<float *>(o.pForce + orig)[l] = pick(F);
        if (o.pTorque) reinterpret_cast<float *>(o.pTorque + orig)[l] = pick(cross3(xyz(o.relPos[orig]), F));
    } else {
        const float fs = (ph.flags & kRefUnits) ? 1.0f : ph.dt;
        reinterpret_cast<float *>(o.vel + orig)[l] = pick(mk3(va.x + F.x * fs, va.y + F.y * fs, va.z + F.z * fs));
    }
}

// Grid DEM fused with the per-body reduction and apply (engine, exact cell table, no static set):
// one launch in place of k_dem_grid_seg + k_reduce_apply, with no per-particle force round trip
// through memory.  Waves [0, B) take one body each: lane l walks the body's particles l, l+64, ... in
// index order, computes each particle's force exactly as k_dem_grid_seg does (same cells, same order,
// same per-cell partials, walls last) and accumulates force and torque relPos × F in the order of
// k_reduce_apply; the butterfly and the apply follow.  The remaining waves take 64 grains each (grain
// indices in original order) and update their velocities.  A wave's lanes are then particles of one
// kind, close in space (one body, or grains in index order), so their candidate loops have similar
// lengths, where a wave of consecutive sorted particles mixes body particles and grains.
__global__ __launch_bounds__(256) void k_dem_fused(const float4 *__restrict__ sPos, const float4 *__restrict__ sVel,
                                                   const unsigned *__restrict__ sIdx,
                                                   const unsigned *__restrict__ segStart, FusedDemIn in, BodyBufs b,
                                                   int B, DevPhys ph, SceneView sv, int sceneInVelW) {
    const int lb = xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int wave = lb * 4 + (int)(threadIdx.x >> 6);
    const int lane = (int)(threadIdx.x & 63);
    const DemOut none{};
    int cnt = 0;
    if (wave < B) {
        const int body = wave;
        const int st = b.pstart[body], count = b.pcount[body];
        f3 aF = mk3(0.f, 0.f, 0.f), aT = mk3(0.f, 0.f, 0.f);
        for (int j = reduce_first(body, ph) + lane; j < count; j += 64) {
            const size_t o = (size_t)st + j;
            const float4 P = in.rec[2 * o], V = in.rec[2 * o + 1];
            const int ra = __float_as_int(P.w);
            SceneGeom g;
            load_geom(sv, sceneInVelW ? __float_as_int(V.w) : 0, g);
            const f3 pa = xyz(P), va = xyz(V);
            f3 F = dem_rows_exact<false, true>(sPos, sVel, sIdx, segStart, g, -1, ra, pa, va, ph, cnt, (unsigned)o,
                                               none);
            F = add3(F, wall_force(pa, va, ph, g));
            aF = add3(aF, F);
            aT = add3(aT, cross3(xyz(in.relPos[o]), F));
        }
        wave_reduce_apply(aF, aT, lane, body, b, ph);
        return;
    }
    const long long k = (long long)(wave - B) * 64 + lane;
    if (k >= in.numGrains) return;
    const unsigned o = (unsigned)in.grainIdx[k];
    const float4 P = in.rec[2 * (size_t)o], V = in.rec[2 * (size_t)o + 1];
    const int ra = __float_as_int(P.w);
    SceneGeom g;
    load_geom(sv, sceneInVelW ? __float_as_int(V.w) : 0, g);
    const f3 pa = xyz(P), va = xyz(V);
    f3 F = dem_rows_exact<false, true>(sPos, sVel, sIdx, segStart, g, -1, ra, pa, va, ph, cnt, o, none);
    if (!(ph.flags & kGrainClamp)) F = add3(F, wall_force(pa, va, ph, g));
    const float fs = (ph.flags & kRefUnits) ? 1.0f : ph.dt;
    in.vel[o] = make_float4(va.x + F.x * fs, va.y + F.y * fs, va.z + F.z * fs, 0.0f);
}

}  // namespace

void launch_reorder_seg(const unsigned *sortedKeys, const unsigned *sortedIdx, const float4 *pos, const float4 *vel,
                        const int *rb, const uint16_t *scene, const float4 *rec, float4 *sortedPos,
                        float4 *sortedVel, unsigned *segStart, int segBits, long long numSegs, int n,
                        const LongFill &lf, hipStream_t st) {
    if (n <= 0) return;
    const int block = 256;
    hipLaunchKernelGGL(k_reorder_seg, dim3((n + block - 1) / block), dim3(block), 0, st, sortedKeys, sortedIdx, pos,
                       vel, rb, scene, rec, sortedPos, sortedVel, segStart, segBits, numSegs, n, lf);
    if (lf.list) launch_fill_long(segStart, (unsigned long long)numSegs + 1ull, lf, st);
}

// Runs are disjoint and longer than kLongRange, so there are fewer than size / kLongRange of them, and
// each has at most len / kLongChunk + 1 chunks.
unsigned fill_long_capacity(unsigned long long tableSize) {
    return (unsigned)(tableSize / kLongRange + tableSize / kLongChunk + 4ull);
}

void launch_fill_long(unsigned *table, unsigned long long tableSize, const LongFill &lf, hipStream_t st) {
    unsigned long long blocks = (tableSize + kLongChunk - 1) / kLongChunk;
    if (blocks > kFillBlocks) blocks = kFillBlocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_fill_long, dim3((unsigned)blocks), dim3(256), 0, st, table, tableSize, lf);
}

void launch_dem_grid_seg(const float4 *sortedPos, const float4 *sortedVel, const unsigned *sortedKeys,
                         const unsigned *sortedIdx, const unsigned *segStart, int segBits, int n, const DevPhys &ph,
                         const SceneView &sv, bool sceneInVelW, const DemOut &o, bool coop, bool queue,
                         int block, hipStream_t st) {
    if (n <= 0) return;
    if (block <= 0) block = 128;
    if (coop && !o.pairs && segBits == 0) {
        const int per = kCoopBlock / kCoopLanes;
        hipLaunchKernelGGL(k_dem_grid_coop<false>, dim3((n + per - 1) / per), dim3(kCoopBlock), 0, st, sortedPos,
                           sortedVel, sortedIdx, segStart, nullptr, n, ph, sv.single, sceneInVelW ? sv.table : nullptr,
                           o);
        return;
    }
    dim3 grid((n + block - 1) / block);
    if (queue && !o.pairs && segBits == 0 && n < kQueueMax) {
        const size_t lds = (size_t)block * kQueue * sizeof(unsigned);
        if (sceneInVelW)
            hipLaunchKernelGGL(k_dem_grid_queue<true>, dim3(grid.x + (unsigned)sv.boundaryBlocks), dim3(block), lds, st,
                               sortedPos, sortedVel, sortedIdx, segStart, n, ph, sv, o);
        else
            hipLaunchKernelGGL(k_dem_grid_queue<false>, grid, dim3(block), lds, st, sortedPos, sortedVel, sortedIdx,
                               segStart, n, ph, sv, o);
        return;
    }
    auto run = [&](auto single, auto batch) {
        if (sceneInVelW)
            hipLaunchKernelGGL(batch, dim3(grid.x + (unsigned)sv.boundaryBlocks), dim3(block), 0, st, sortedPos, sortedVel,
                               sortedKeys, sortedIdx, segStart, segBits, n, ph, sv, o);
        else
            hipLaunchKernelGGL(single, grid, dim3(block), 0, st, sortedPos, sortedVel, sortedKeys, sortedIdx, segStart,
                               segBits, n, ph, sv, o);
    };
    if (o.pairs) {
        if (segBits == 0) run(k_dem_grid_seg<true, true, false>, k_dem_grid_seg<true, true, true>);
        else run(k_dem_grid_seg<true, false, false>, k_dem_grid_seg<true, false, true>);
    } else {
        if (segBits == 0) run(k_dem_grid_seg<false, true, false>, k_dem_grid_seg<false, true, true>);
        else run(k_dem_grid_seg<false, false, false>, k_dem_grid_seg<false, false, true>);
    }
}

void launch_dem_grid_index(const float4 *sortedPos, const float4 *sortedVel, const unsigned *sortedIdx,
                           const CellIndex &ix, int n, const DevPhys &ph, const SceneView &sv, bool sceneInVelW,
                           const DemOut &o, int block, hipStream_t st) {
    if (n <= 0) return;
    if (block <= 0) block = 128;
    const unsigned all = (unsigned)((n + block - 1) / block);
    const size_t lds = (size_t)9 * block * sizeof(unsigned);
    if (sceneInVelW)
        hipLaunchKernelGGL(k_dem_grid_index<true>, dim3(all + (unsigned)sv.boundaryBlocks), dim3(block), lds, st, sortedPos,
                           sortedVel, sortedIdx, ix, n, ph, sv, o);
    else
        hipLaunchKernelGGL(k_dem_grid_index<false>, dim3(all), dim3(block), lds, st, sortedPos, sortedVel, sortedIdx, ix,
                           n, ph, sv, o);
}

void launch_reorder(const unsigned *sortedKeys, const unsigned *sortedIdx, const float4 *pos, const float4 *vel,
                    const int *rb, const uint16_t *scene, float4 *sortedPos, float4 *sortedVel, unsigned *cellStart,
                    unsigned *cellEnd, int n, hipStream_t st) {
    if (n <= 0) return;
    const int block = 256;
    hipLaunchKernelGGL(k_reorder, dim3((n + block - 1) / block), dim3(block), 0, st, sortedKeys, sortedIdx, pos, vel,
                       rb, scene, sortedPos, sortedVel, cellStart, cellEnd, n);
}

void launch_dem_grid(const float4 *sortedPos, const float4 *sortedVel, const unsigned *sortedIdx,
                     const unsigned *cellStart, const unsigned *cellEnd, int n, const DevPhys &ph,
                     const SceneView &sv, bool sceneInVelW, const DemOut &o, int block, hipStream_t st) {
    if (n <= 0) return;
    if (block <= 0) block = 128;
    if (!o.pairs && !sceneInVelW && n <= kCoopMax) {
        const int per = kCoopBlock / kCoopLanes;
        hipLaunchKernelGGL(k_dem_grid_coop<true>, dim3((n + per - 1) / per), dim3(kCoopBlock), 0, st, sortedPos,
                           sortedVel, sortedIdx, cellStart, cellEnd, n, ph, sv.single, nullptr, o);
        return;
    }
    dim3 grid((n + block - 1) / block);
    if (!o.pairs && !sceneInVelW && n < kQueueMax)
        hipLaunchKernelGGL(k_dem_grid_ref_queue, grid, dim3(block), (size_t)block * kQueue * sizeof(unsigned), st,
                           sortedPos, sortedVel, sortedIdx, cellStart, cellEnd, n, ph, sv.single, o);
    else if (o.pairs)
        hipLaunchKernelGGL(k_dem_grid<true>, grid, dim3(block), 0, st, sortedPos, sortedVel, sortedIdx, cellStart,
                           cellEnd, n, ph, sv, sceneInVelW ? 1 : 0, o);
    else
        hipLaunchKernelGGL(k_dem_grid<false>, grid, dim3(block), 0, st, sortedPos, sortedVel, sortedIdx, cellStart,
                           cellEnd, n, ph, sv, sceneInVelW ? 1 : 0, o);
}

void launch_dem_fused(const float4 *sortedPos, const float4 *sortedVel, const unsigned *sortedIdx,
                      const unsigned *segStart, const FusedDemIn &in, const BodyBufs &b, int numBodies,
                      const DevPhys &ph, const SceneView &sv, bool sceneInVelW, hipStream_t st) {
    const long long waves = (long long)numBodies + (in.numGrains + 63) / 64;
    if (waves <= 0) return;
    const long long blocks = (waves + 3) / 4;
    hipLaunchKernelGGL(k_dem_fused, dim3((unsigned)blocks), dim3(256), 0, st, sortedPos, sortedVel, sortedIdx, segStart,
                       in, b, numBodies, ph, sv, sceneInVelW ? 1 : 0);
}

}  // namespace arsim
