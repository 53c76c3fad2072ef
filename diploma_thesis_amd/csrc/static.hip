// static.hip -- the static (augmented-reality) collider set: range image -> scene points and
// normals, the static points' grid index, and the DEM of the dynamic particles against them.
#include "coop_cells.hpp"
#include "csr_fill.hpp"
#include "kernels.hpp"

namespace arsim {

namespace {

// RGBDloader (Kernels/customRangeImageLoader.cu:14-109), one thread per pixel.  Intrinsics and the
// accelerometer rotation are the reference's constants; g is the normalised accelerometer vector.
// A 4x4 matrix-vector product is summed by columns as (c0 v0 + c1 v1) + (c2 v2 + c3 v3).
__global__ void k_range_image(const uint16_t *__restrict__ img, int W, int H, RangeCamera cam, float radius,
                              float4 *__restrict__ pos, float *__restrict__ radii, float *__restrict__ vao) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)W * H) return;
    if (idx > (long)(W - 1) * (long)(H - 1)) return;   // the reference's bound
    const int y = (int)(idx / W), x = (int)(idx - (long)y * W);
    float d = (float)img[idx];
    d = d / 5000.f;
    if (radii) radii[idx] = radius;
    if ((double)d < 0.01) d = -1000.f;
    const float X = d * ((float)x - 318.6f) / 517.3f;
    const float Y = d * ((float)y - 255.3f) / 516.5f;
    const float v0 = X, v1 = Y, v2 = d, v3 = 0.f;
    float t[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)   // transpose(cam): element (r, c) = cam[4 r + c]
        t[r] = (cam.m[4 * r + 0] * v0 + cam.m[4 * r + 1] * v1) + (cam.m[4 * r + 2] * v2 + cam.m[4 * r + 3] * v3);
    const float gx = cam.g[0], gy = cam.g[1], gz = cam.g[2];
    const float G[16] = {1.f, 0.f, 0.f, 0.f, -gx, -gy, -gz, 0.f, 0.f, gz, -gy, 0.f, 0.f, 0.f, 0.f, 1.f};
    float u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = (G[r] * t[0] + G[4 + r] * t[1]) + (G[8 + r] * t[2] + G[12 + r] * t[3]);
    const float px = u[0], py = -u[1], pz = -u[2];
    if (vao) {
        vao[5 * idx] = px;
        vao[5 * idx + 1] = py;
        vao[5 * idx + 2] = pz;
        vao[5 * idx + 3] = (float)x / (float)W;
        vao[5 * idx + 4] = (float)y / (float)H;
    }
    pos[idx] = make_float4(px, py, pz, 0.f);
}

// computeNormals (customRangeImageLoader.cu:118-162): interior pixels only,
// n = normalize(cross(P[y+1][x] - P[y-1][x], P[y][x+1] - P[y][x-1])), normalize = v * (1 / |v|).
__global__ void k_range_normals(const float4 *__restrict__ pos, int W, int H, float4 *__restrict__ norm) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)W * H) return;
    const int y = (int)(idx / W), x = (int)(idx - (long)y * W);
    if (x > W - 2 || x == 0 || y == 0 || y > H - 2) return;
    const float4 r = pos[idx + 1], l = pos[idx - 1], b = pos[idx + W], t = pos[idx - W];
    const float dx0 = r.x - l.x, dx1 = r.y - l.y, dx2 = r.z - l.z;
    const float dy0 = b.x - t.x, dy1 = b.y - t.y, dy2 = b.z - t.z;
    const float n0 = dy1 * dx2 - dy2 * dx1;
    const float n1 = dy2 * dx0 - dy0 * dx2;
    const float n2 = dy0 * dx1 - dy1 * dx0;
    const float inv = 1.0f / sqrtf(n0 * n0 + n1 * n1 + n2 * n2);
    norm[idx] = make_float4(n0 * inv, n1 * inv, n2 * inv, 0.f);
}

// Cell key of every static point (calcHashD for the static set) and the identity index.
__global__ void k_static_hash(const float4 *__restrict__ pos, int m, SceneGeom g, unsigned *__restrict__ keys) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    int gx, gy, gz;
    grid_pos(xyz(pos[j]), g, gx, gy, gz);
    keys[j] = grid_hash(gx, gy, gz, g);
}

// Sorted copies of the static points and normals plus the exact cell table:
// table[c] = first sorted index with key >= c, for c = 0 .. numCells.
__global__ void k_static_reorder(const unsigned *__restrict__ keys, const unsigned *__restrict__ idx,
                                 const float4 *__restrict__ pos, const float4 *__restrict__ norm, int m,
                                 unsigned numCells, float4 *__restrict__ sPos, float4 *__restrict__ sNorm,
                                 unsigned *__restrict__ table, LongFill lf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < m;
    const unsigned k = valid ? keys[i] : 0u;
    const unsigned kp1 = (valid && i > 0) ? keys[i - 1] + 1u : 0u;
    wave_fill(table, valid && k + 1u > kp1, kp1, k + 1u, (unsigned)i, lf);
    wave_fill(table, i == m - 1, k + 1u, numCells + 1u, (unsigned)m, lf);
    if (!valid) return;
    const unsigned o = idx[i];
    sPos[i] = pos[o];
    sNorm[i] = norm[o];
}

// FindAndHandleAugmentedRealityCollisionsUniformGridKernel (RigidBodies/UniformGridDEM.cu:306-378):
// per sorted dynamic particle, the 27 cells of the static grid in z, y, x order, each cell's
// contacts summed into a partial that is added to the total for every cell.
//  REF (reference layout): static cellStart / cellEnd with 0xffffffff for an empty cell, normals read
//    through the static sorted index, every particle: pForce += F, pTorque += relativePos x F.
//  engine: the exact static cell table and sorted normals, body particles only: pForce += F (the
//    torque is relativePos x pForce, formed by the reduction).
// A workgroup first tests its particles one per thread for any candidate (the 9 rows of cells, three
// consecutive cells each), then takes those that have some 16 lanes each (coop_cells) or, where that is the longer way,
// one thread each: the walk of a particle on a scanned surface, about a thousand candidates, is one serial chain per
// thread, bound by the latency of its loads.  16,384 particles on the points of a 640 x 480 depth image: 1,280 -> 97 us;
// a 2^20-particle scene over a floor of 2^20 points (few particles near it): step 286 -> 210 us.  Without
// the first test every particle takes 16 lanes, and that scene over 65,536 points costs 240 us a step
// instead of 187 (one thread per particle: 213).
constexpr int kStaticBlock = 128;
// Whether `count` particles of a workgroup with `candidates` of theirs in all take one thread each.  With 16 lanes eight at a
// time do, each in a time that grows with a 16th of the candidates; with one thread all of them at once.  (The numbers are
// a fit of both forms, 10^3 to 10^6 particles on points 1/50 of a cell to a cell apart.)  Every particle near the points, one
// thread each, 16 lanes each, and weighed (us): 10^6 and 9 points a particle 116, 260, 109; 36 points 201, 406, 183; 900
// points on a 16th of the scene 781, 1,482, 777; 200,000 and 9 points 37, 70, 37; 36 points 79, 104, 69; 900 points 773, 438, 504.
__device__ __forceinline__ bool one_thread_each(int count, unsigned candidates) {
    const long long rounds = (count + kStaticBlock / kCoopLanes - 1) / (kStaticBlock / kCoopLanes);
    return rounds * (47ll * count + candidates) > 75ll * count + 7ll * candidates;
}
// WEIGH: both forms are weighed (launch_dem_static), else 16 lanes each.
template <bool REF, bool WEIGH>
__global__ __launch_bounds__(kStaticBlock) void k_dem_static(
    const float4 *__restrict__ sPos, const float4 *__restrict__ sVel, const unsigned *__restrict__ sIdx, int n,
    int perBlock, int byXcd, const float4 *__restrict__ stPos, const float4 *__restrict__ stNorm,
    const unsigned *__restrict__ stIdx, const unsigned *__restrict__ cs, const unsigned *__restrict__ ce, DevPhys ph,
    SceneGeom g, float4 *__restrict__ pForce, float4 *__restrict__ pTorque, const float4 *__restrict__ relPos) {
    __shared__ CoopGroupLds sGroup[kStaticBlock / kCoopLanes];
    __shared__ int sList[kStaticBlock];
    __shared__ int sCount;
    __shared__ unsigned sCand;
    const int t = (int)threadIdx.x,
              first = (!WEIGH || byXcd ? xcd_block((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x) * perBlock;
    // cell h's run of candidates
    auto cell_run = [&](unsigned h, unsigned &b, unsigned &e) {
        b = cs[h];
        e = REF ? ce[h] : cs[h + 1];   // (both ends at once, the second not after the first)
        if (REF && (b == kEmpty || e < b)) b = e = 0u;   // an empty cell's end is not defined
    };
    if (t == 0) {
        sCount = 0;
        if (WEIGH) sCand = 0u;
    }
    __syncthreads();
    unsigned rows = 0u;   // of this thread's particle: those that have candidates
    if (t < perBlock && first + t < n) {
        const float4 P = sPos[first + t];
        unsigned cand = 0u;
        if (REF || __float_as_int(P.w) >= 0) {
            int gx, gy, gz;
            grid_pos(xyz(P), g, gx, gy, gz);
            constexpr unsigned kMost = 4096u;   // (counted of one row or cell, so that the sum fits)
            unsigned cells = 0u, at = 0u;
            for (int r = 0; r < 9; ++r) {
                const unsigned h0 = grid_hash(gx - 1, gy + r % 3 - 1, gz + r / 3 - 1, g);
                const unsigned h1 = grid_hash(gx, gy + r % 3 - 1, gz + r / 3 - 1, g);
                const unsigned h2 = grid_hash(gx + 1, gy + r % 3 - 1, gz + r / 3 - 1, g);
                if (!WEIGH) {   // (one bit for all rows: 16,384 particles on 640 x 480 points 117 us with the counts, 115 so)
                    bool any;
                    if (REF) any = (cs[h0] != kEmpty) | (cs[h1] != kEmpty) | (cs[h2] != kEmpty);
                    else if (h2 == h0 + 2u) any = cs[h0] != cs[h0 + 3u];
                    else any = (cs[h0] != cs[h0 + 1u]) | (cs[h1] != cs[h1 + 1u]) | (cs[h2] != cs[h2 + 1u]);
                    rows |= any ? 1u : 0u;
                    continue;
                }
                unsigned some;
                if (REF) {
                    const unsigned c0 = cs[h0], c1 = cs[h1], c2 = cs[h2];
                    some = (c0 != kEmpty ? 1u : 0u) + (c1 != kEmpty ? 1u : 0u) + (c2 != kEmpty ? 1u : 0u);
                    at = c0 != kEmpty ? h0 : c1 != kEmpty ? h1 : c2 != kEmpty ? h2 : at;
                    cells += some;
                } else {
                    if (h2 == h0 + 2u) some = min(cs[h0 + 3u] - cs[h0], kMost);
                    else
                        some = min(cs[h0 + 1u] - cs[h0], kMost) + min(cs[h1 + 1u] - cs[h1], kMost) +
                               min(cs[h2 + 1u] - cs[h2], kMost);
                    cand += some;
                }
                rows |= some ? 1u << r : 0u;
            }
            if (REF && WEIGH && cells) {   // estimated: every cell as full as one of them
                unsigned b, e;
                cell_run(at, b, e);
                cand = cells * max(min(e - b, kMost), 1u);
            }
        }
        if (rows) {   // (each particle is written by itself: any order)
            sList[atomicAdd(&sCount, 1)] = first + t;
            if (WEIGH) atomicAdd(&sCand, cand);
        } else if (REF) {   // nothing to add: a sum of no contacts is +0
            const unsigned o = sIdx[first + t];
            const float4 f = pForce[o], q = pTorque[o];
            const f3 tq = cross3(xyz(relPos[o]), mk3(0.f, 0.f, 0.f));
            pForce[o] = make_float4(f.x + 0.0f, f.y + 0.0f, f.z + 0.0f, f.w + 0.0f);
            pTorque[o] = make_float4(q.x + tq.x, q.y + tq.y, q.z + tq.z, q.w + 0.0f);
        }
    }
    __syncthreads();
    if (WEIGH && one_thread_each(sCount, sCand)) {
        if (!rows) return;
        const int i = first + t;
        const f3 pa = xyz(sPos[i]), va = xyz(sVel[i]);
        int gx, gy, gz;
        grid_pos(pa, g, gx, gy, gz);
        f3 F = mk3(0.f, 0.f, 0.f);
        for (; rows; rows &= rows - 1u) {   // (the others have no contact to add)
            const int r = __builtin_ctz(rows);
            for (int x = -1; x <= 1; ++x) {
                unsigned j, e;
                cell_run(grid_hash(gx + x, gy + r % 3 - 1, gz + r / 3 - 1, g), j, e);
                f3 csum = mk3(0.f, 0.f, 0.f);
                for (; j < e; ++j) {   // (a candidate's normal is read with its position, not after it)
                    const f3 ps = xyz(stPos[j]), ns = xyz(stNorm[REF ? stIdx[j] : j]);
                    f3 fj;
                    if (static_force(pa, ps, ns, va, ph, fj)) csum = add3(csum, fj);
                }
                F = add3(F, csum);
            }
        }
        const unsigned o = sIdx[i];
        const float4 old = pForce[o];
        pForce[o] = make_float4(old.x + F.x, old.y + F.y, old.z + F.z, old.w + 0.0f);
        if (REF) {
            const float4 q = pTorque[o];
            const f3 tq = cross3(xyz(relPos[o]), F);
            pTorque[o] = make_float4(q.x + tq.x, q.y + tq.y, q.z + tq.z, q.w + 0.0f);
        }
        return;
    }
    const int count = sCount, gl = t / kCoopLanes, l = t & (kCoopLanes - 1);
    // (a wave's four groups stay together: the bound is the wave's, not the group's)
    for (int k0 = (t >> 6) * (64 / kCoopLanes); k0 < count; k0 += kStaticBlock / kCoopLanes) {
        const int k = k0 + (gl & (64 / kCoopLanes - 1));
        const bool valid = k < count;
        const int i = sList[valid ? k : k0];
        const f3 pa = xyz(sPos[i]), va = xyz(sVel[i]);
        int gx, gy, gz;
        grid_pos(pa, g, gx, gy, gz);
        const float F = coop_cells(
            sGroup[gl], valid,
            [&](int c, unsigned &b, unsigned &e) {
                cell_run(grid_hash(gx + c % 3 - 1, gy + (c / 3) % 3 - 1, gz + c / 9 - 1, g), b, e);
            },
            [&](unsigned j, f3 &f) {
                const f3 ps = xyz(stPos[j]);
                if (!in_contact(pa, ps, ph)) return false;
                return static_force(pa, ps, xyz(stNorm[REF ? stIdx[j] : j]), va, ph, f);
            });
        const f3 F3 = mk3(__shfl(F, 0, kCoopLanes), __shfl(F, 1, kCoopLanes), __shfl(F, 2, kCoopLanes));
        if (!valid || l > 3) continue;
        const unsigned o = sIdx[i];
        auto pick = [l](f3 v) { return l == 0 ? v.x : l == 1 ? v.y : l == 2 ? v.z : 0.0f; };
        float *pf = reinterpret_cast<float *>(pForce + o) + l;
        *pf = *pf + pick(F3);
        if (REF) {
            float *pt = reinterpret_cast<float *>(pTorque + o) + l;
            *pt = *pt + pick(cross3(xyz(relPos[o]), F3));
        }
    }
}

}  // namespace

void launch_range_image(const uint16_t *img, int W, int H, const RangeCamera &cam, float radius, float4 *pos,
                        float4 *norm, float *radii, float *vao, hipStream_t st) {
    const long total = (long)W * H;
    if (total <= 0) return;
    const int block = 256;
    const dim3 grid((unsigned)((total + block - 1) / block));
    hipLaunchKernelGGL(k_range_image, grid, dim3(block), 0, st, img, W, H, cam, radius, pos, radii, vao);
    hipLaunchKernelGGL(k_range_normals, grid, dim3(block), 0, st, pos, W, H, norm);
}

void launch_static_hash(const float4 *pos, int m, const SceneGeom &g, unsigned *keys, hipStream_t st) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_static_hash, dim3((m + 255) / 256), dim3(256), 0, st, pos, m, g, keys);
}

void launch_static_reorder(const unsigned *keys, const unsigned *idx, const float4 *pos, const float4 *norm, int m,
                           unsigned numCells, float4 *sPos, float4 *sNorm, unsigned *table, const LongFill &lf,
                           hipStream_t st) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_static_reorder, dim3((m + 255) / 256), dim3(256), 0, st, keys, idx, pos, norm, m, numCells,
                       sPos, sNorm, table, lf);
    if (lf.list) launch_fill_long(table, (unsigned long long)numCells + 1ull, lf, st);
}

void launch_dem_static(const float4 *sPos, const float4 *sVel, const unsigned *sIdx, int n, const float4 *stPos,
                       const float4 *stNorm, const unsigned *stIdx, const unsigned *cs, const unsigned *ce,
                       const DevPhys &ph, const SceneGeom &g, float4 *pForce, float4 *pTorque,
                       const float4 *relPos, bool refLayout, hipStream_t st) {
    if (n <= 0) return;
    // Up to 65,536 particles a workgroup takes one per group of 16 lanes, so that the particles near a surface, few and
    // together, spread over the chip.  More of them load the chip either way, and then the two forms are weighed, in
    // workgroups of 32 as long as fuller ones would be too few, of 64, and of 128.  Consecutive workgroups run on one XCD
    // while the scene is small enough for its L2 to matter more than an even load (a scan that covers a 16th of 10^6
    // particles: 1,090 us by XCD, 778 in turn; one under all of 200,000 53 and 63).
    const bool weigh = n > 65536;
    const int perBlock = !weigh ? kStaticBlock / kCoopLanes : n <= (7 << 15) ? 32 : n <= 524288 ? 64 : kStaticBlock;
    const int byXcd = n <= 262144 ? 1 : 0;
    const dim3 grid((n + perBlock - 1) / perBlock);
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kStaticBlock), 0, st, sPos, sVel, sIdx, n, perBlock, byXcd, stPos, stNorm,
                           stIdx, cs, ce, ph, g, pForce, pTorque, relPos);
    };
    if (refLayout) weigh ? run(k_dem_static<true, true>) : run(k_dem_static<true, false>);
    else weigh ? run(k_dem_static<false, true>) : run(k_dem_static<false, false>);
}

}  // namespace arsim
