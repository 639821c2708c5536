// Triangle collision, CollisionTriangle::execute (Collision_triangle.cpp,
// collision_tri.cl:120-231 and 418-470; one particle and one triangle are
// tri_add in obstacles_device.h).
//
// Per triangle the host prepares, in the simulation scale, its vertices
// a, b, c (= v * scale), n = (b - a) x (c - a), the unit normal n / |n| and a
// bounding sphere.  A particle farther than radius + dist from the sphere's
// centre cannot get a hit closer than dist (tp lies in the triangle), so it
// skips the test; that changes no result.
//
// A system's triangles are loaded once and met in every step: a particle
// visits only those listed in its cell of a grid laid over them
// (bin_triangles), whose box, widened by dist, meets the cell, in triangle
// order.  Culling blocks of particles against the triangles instead leaves the
// blocks that span a change of row or plane with most of them: 97 us a step for
// 150,001 particles and 1,152 triangles, of which the sheet in the pool touches
// a fraction.
//
// The stage operator's triangles are met once, where making the lists costs
// the host more than they save: k_collision_tri culls by block.  Only for few
// particles, whose blocks leave most of the chip idle while each goes through
// all triangles, the lists are made there, too (kListParticles).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <limits>
#include <vector>

#include "obstacles_device.h"
#include "rtps_internal.h"

namespace rtps {

namespace {

constexpr int kBlockTri = 256;
constexpr int kWavesTri = kBlockTri / 64;
constexpr int kTriChunk = 256;   // triangles tested per chunk (one per thread); 20 KiB of TriPrep in LDS

__device__ __forceinline__ float wave_min(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Blocks of consecutive sorted particles are compact in space: per chunk of
// triangles, each thread tests one triangle's sphere (centre, reach squared)
// against the block's bounding box, and those that meet it are compacted into
// LDS in triangle order (ballot ranks, then per-wave offsets).
__global__ __launch_bounds__(kBlockTri) void k_collision_tri(int num, const float4* __restrict__ pos_s,
                                                             const float4* __restrict__ vel_s,
                                                             float4* __restrict__ force,
                                                             const TriPrep* __restrict__ tris,
                                                             const float4* __restrict__ sphere, int ntri,
                                                             rtps_sph_params sp) {
    __shared__ TriPrep lt[kTriChunk];
    __shared__ float box[kWavesTri][6];
    __shared__ int wave_n[kWavesTri];
    const int i = blockIdx.x * kBlockTri + threadIdx.x;
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const bool live = i < num;
    const float s = sp.simulation_scale;
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f), v = p;
    if (live) {
        p = pos_s[i];
        v = vel_s[i];
    }
    const float px = p.x * s, py = p.y * s, pz = p.z * s;
    // bounding box of the block's live particles
    {
        const float inf = __builtin_inff();
        const float lo[3] = {live ? px : inf, live ? py : inf, live ? pz : inf};
        const float hi[3] = {live ? px : -inf, live ? py : -inf, live ? pz : -inf};
        for (int c = 0; c < 3; ++c) {
            const float a = wave_min(lo[c]), b = wave_max(hi[c]);
            if (lane == 0) {
                box[wave][c] = a;
                box[wave][3 + c] = b;
            }
        }
    }
    __syncthreads();
    float bl[3], bh[3];
    for (int c = 0; c < 3; ++c) {
        bl[c] = box[0][c];
        bh[c] = box[0][3 + c];
        for (int w = 1; w < kWavesTri; ++w) {
            bl[c] = fminf(bl[c], box[w][c]);
            bh[c] = fmaxf(bh[c], box[w][3 + c]);
        }
    }
    float3 f = make_float3(0.f, 0.f, 0.f);
    for (int c0 = 0; c0 < ntri; c0 += kTriChunk) {
        const int t = c0 + (int)threadIdx.x;
        bool cand = false;
        if (t < ntri) {
            const float4 r = sphere[t];
            const float dx = fmaxf(fmaxf(bl[0] - r.x, r.x - bh[0]), 0.f);
            const float dy = fmaxf(fmaxf(bl[1] - r.y, r.y - bh[1]), 0.f);
            const float dz = fmaxf(fmaxf(bl[2] - r.z, r.z - bh[2]), 0.f);
            cand = dx * dx + dy * dy + dz * dz <= r.w;
        }
        const unsigned long long m = __ballot(cand);
        const int rank = __popcll(m & ((1ull << lane) - 1ull));
        __syncthreads();   // the previous chunk's triangles are no longer read
        if (lane == 0) wave_n[wave] = __popcll(m);
        __syncthreads();
        int base = 0, total = 0;
        for (int w = 0; w < kWavesTri; ++w) {
            if (w < wave) base += wave_n[w];
            total += wave_n[w];
        }
        if (cand) lt[base + rank] = tris[t];
        __syncthreads();
        if (!live) continue;
        for (int q = 0; q < total; ++q) {
            const TriPrep& T = lt[q];
            const float cx = px - T.cx, cy = py - T.cy, cz = pz - T.cz;
            if (!(cx * cx + cy * cy + cz * cz > T.reach2)) tri_add(f, px, py, pz, v, T, sp);
        }
    }
    if (!live) return;
    float4 F = force[i];
    F.x += f.x;
    F.y += f.y;
    F.z += f.z;
    force[i] = F;
}

// The spheres of the triangles in list order.
__global__ __launch_bounds__(kBlockTri) void k_list_spheres(uint32_t n, const uint32_t* __restrict__ list,
                                                            const TriPrep* __restrict__ tris,
                                                            float4* __restrict__ sphere) {
    const uint32_t q = blockIdx.x * kBlockTri + threadIdx.x;
    if (q >= n) return;
    const TriPrep& T = tris[list[q]];
    sphere[q] = make_float4(T.cx, T.cy, T.cz, T.reach2);
}

}  // namespace

// Where the lists pay for one call.  Measured for the operator (us, lists /
// blocks): 59 / 40 with 2 triangles and 86 / 74 with 128 (1,000 particles and
// more); with 1,152, 5,000 and 20,000 triangles 194 / 264, 422 / 845 and
// 1,475 / 2,380 at 1,000 particles, 147 / 172, 348 / 494 and 1,208 / 1,618 at
// 10,000, 134 / 125, 333 / 290 and 1,149 / 819 at 50,000, 137 / 154, 341 / 360
// and 1,165 / 1,014 at 600,000; with 180,000 14.9 / 22.0, 13.8 / 15.6,
// 13.0 / 6.2 and 9.8 / 7.9 ms.
constexpr int kListParticles = 1 << 14;
constexpr size_t kListTriangles = 1 << 10;

hipError_t collision_triangles(int num, const float4* pos_s, const float4* vel_s, float4* force,
                               const std::vector<TriPrep>& prep, const rtps_sph_params& sp, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num <= 0 || prep.empty()) return hipSuccess;
    if (num <= kListParticles && prep.size() >= kListTriangles) {
        TriDevice dev;
        hipError_t e = dev.load(prep, sp.boundary_distance, st);
        if (e == hipSuccess)
            e = launch_after_force(num, nullptr, nullptr, 0, pos_s, vel_s, nullptr, force, nullptr, nullptr, sp,
                                   AfterForce{}, GravitySources{}, Grid{}, &dev.set, nullptr, nullptr, nullptr,
                                   nullptr, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);   // the triangle memory goes with dev
        return e;
    }
    std::vector<float4> sphere(prep.size());
    for (size_t q = 0; q < prep.size(); ++q)
        sphere[q] = make_float4(prep[q].cx, prep[q].cy, prep[q].cz, prep[q].reach2);
    TriPrep* dev = nullptr;
    hipError_t e = hipMalloc((void**)&dev, prep.size() * (sizeof(TriPrep) + sizeof(float4)));
    if (e != hipSuccess) return e;
    float4* dev_sphere = reinterpret_cast<float4*>(dev + prep.size());
    e = hipMemcpyAsync(dev, prep.data(), prep.size() * sizeof(TriPrep), hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
        e = hipMemcpyAsync(dev_sphere, sphere.data(), sphere.size() * sizeof(float4), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        k_collision_tri<<<(num + kBlockTri - 1) / kBlockTri, kBlockTri, 0, st>>>(num, pos_s, vel_s, force, dev,
                                                                               dev_sphere, (int)prep.size(), sp);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);   // the triangles are freed below
    (void)hipFree(dev);
    return e;
}

std::vector<TriPrep> prepare_triangles(const rtps_triangle* tris, int n, float scale) {
#pragma clang fp contract(off)
    std::vector<TriPrep> out((size_t)n);
    for (int q = 0; q < n; ++q) {
        const rtps_triangle& T = tris[q];
        TriPrep& P = out[(size_t)q];
        const float ax = T.verts[0].x * scale, ay = T.verts[0].y * scale, az = T.verts[0].z * scale;
        const float bx = T.verts[1].x * scale, by = T.verts[1].y * scale, bz = T.verts[1].z * scale;
        const float cx = T.verts[2].x * scale, cy = T.verts[2].y * scale, cz = T.verts[2].z * scale;
        P.ax = ax; P.ay = ay; P.az = az;
        P.bx = bx; P.by = by; P.bz = bz;
        P.qx = cx; P.qy = cy; P.qz = cz;
        const float abx = bx - ax, aby = by - ay, abz = bz - az;
        const float acx = cx - ax, acy = cy - ay, acz = cz - az;
        P.nx = aby * acz - abz * acy;   // cross_product(ab, ac), collision_tri.cl:139
        P.ny = abz * acx - abx * acz;
        P.nz = abx * acy - aby * acx;
        const float nm = std::sqrt(P.nx * P.nx + P.ny * P.ny + P.nz * P.nz);
        P.ux = P.nx / nm; P.uy = P.ny / nm; P.uz = P.nz / nm;
        // bounding sphere: the centroid and the farthest vertex, widened by
        // the boundary distance later and by a margin for rounding
        const double mx = ((double)ax + bx + cx) / 3.0, my = ((double)ay + by + cy) / 3.0,
                     mz = ((double)az + bz + cz) / 3.0;
        double r2 = 0.0;
        const double vx[3] = {ax, bx, cx}, vy[3] = {ay, by, cy}, vz[3] = {az, bz, cz};
        for (int k = 0; k < 3; ++k)
            r2 = std::max(r2, (vx[k] - mx) * (vx[k] - mx) + (vy[k] - my) * (vy[k] - my) + (vz[k] - mz) * (vz[k] - mz));
        P.cx = (float)mx; P.cy = (float)my; P.cz = (float)mz;
        P.radius = (float)std::sqrt(r2);
        P.reach2 = 0.0f;   // set by set_triangle_reach once the boundary distance is known
    }
    return out;
}

void set_triangle_reach(std::vector<TriPrep>& t, float dist) {
    for (TriPrep& P : t) {
        const double r = ((double)P.radius + dist) * (1.0 + 1e-5) + 1e-6;
        P.reach2 = (float)(r * r);
    }
}

namespace {

// The grid over the triangles: cells of edge 1 / inv from min, the triangles
// of cell c in list[start[c]..start[c + 1]).
struct TriBins {
    float min[3] = {}, inv = 0.f;
    int n[3] = {};
    std::vector<uint32_t> start;
    struct Box {
        float lo[3], hi[3];   // around triangle id
        uint32_t id;
    };
    std::vector<Box> box;   // finite triangles
    double wide = 0.0;      // added to them on each side
    // cell(c) for every cell that box b may meet
    template <typename Cell>
    void each(const Box& b, Cell&& cell) const {
        int f[3], t[3];
        range(b, f, t);
        for (int z = f[2]; z <= t[2]; ++z)
            for (int y = f[1]; y <= t[1]; ++y)
                for (int x = f[0]; x <= t[0]; ++x) cell(((size_t)z * n[1] + y) * n[0] + x);
    }
    size_t range(const Box& b, int (&f)[3], int (&t)[3]) const {   // those cells, and their number
        size_t m = 1;
        for (int k = 0; k < 3; ++k) {   // no box begins below min
            f[k] = std::min((int)((b.lo[k] - (min[k] + wide)) * inv), n[k] - 1);
            t[k] = std::min((int)((b.hi[k] - (min[k] - wide)) * inv), n[k] - 1);
            m *= (size_t)(t[k] - f[k] + 1);
        }
        return m;
    }
};

// Cells about as large as the triangles: a triangle then lies in a few cells
// and a cell lists a few triangles.  Where that lists a triangle more than
// kTriLists times on average (few large ones among many small), or takes more
// than kTriCells cells, the cells are doubled until it does not; one cell lists
// every triangle once.
constexpr size_t kTriLists = 16, kTriCells = 1 << 18;

// The grid and its cells' starts in the lists (start[c + 1] holds the number
// before it, to be filled from there on).
TriBins bin_triangles(const std::vector<TriPrep>& prep, float dist) {
    TriBins B;
    constexpr double top = std::numeric_limits<float>::max();
    float first[3] = {(float)top, (float)top, (float)top}, last[3] = {(float)-top, (float)-top, (float)-top};
    double edge = 0.0;
    B.box.reserve(prep.size());
    for (size_t q = 0; q < prep.size(); ++q) {
        const TriPrep& P = prep[q];
        const float v[3][3] = {{P.ax, P.bx, P.qx}, {P.ay, P.by, P.qy}, {P.az, P.bz, P.qz}};
        TriBins::Box b;
        b.id = (uint32_t)q;
        float none = 0.f, side = 0.f;
        for (int k = 0; k < 3; ++k) {
            b.lo[k] = std::min(v[k][0], std::min(v[k][1], v[k][2]));
            b.hi[k] = std::max(v[k][0], std::max(v[k][1], v[k][2]));
            none += (v[k][0] - v[k][0]) + (v[k][1] - v[k][1]) + (v[k][2] - v[k][2]);
            side = std::max(side, b.hi[k] - b.lo[k]);
        }
        if (!(none == 0.f)) continue;   // infinite or not a number: no comparison of its test can hold
        for (int k = 0; k < 3; ++k) {
            first[k] = std::min(first[k], b.lo[k]);
            last[k] = std::max(last[k], b.hi[k]);
        }
        edge += side;
        B.box.push_back(b);
    }
    if (B.box.empty()) return B;
    double most = 0.0, extent = 0.0, size[3];   // the largest coordinate: the scale of the particle side's roundings
    for (int k = 0; k < 3; ++k) most = std::max({most, std::fabs((double)first[k]), std::fabs((double)last[k])});
    // wider than the roundings of the particle's side (its cell index, tp, the
    // distance), each below 1e-6 of the largest coordinate
    B.wide = dist * (1.0 + 1e-5) + 1e-6 + 1e-5 * most;
    for (int k = 0; k < 3; ++k) {
        B.min[k] = (float)std::max(first[k] - B.wide, -top);
        size[k] = last[k] + B.wide - B.min[k];
        extent = std::max(extent, size[k]);
    }
    edge = edge / (double)B.box.size() + 2.0 * B.wide;
    for (;; edge *= 2.0) {
        const bool one = !(edge < extent);
        B.inv = one ? 0.f : (float)(1.0 / edge);   // one cell: every index is 0
        size_t cells = 1;
        for (int k = 0; k < 3; ++k) {
            B.n[k] = one ? 1 : (int)std::min(1e6, std::floor(size[k] / edge) + 2.0);
            cells *= (size_t)B.n[k];
        }
        if (!one && cells > kTriCells) continue;
        int f[3], t[3];
        size_t total = 0;
        for (const TriBins::Box& b : B.box) total += B.range(b, f, t);
        if (!one && total > kTriLists * B.box.size()) continue;
        B.start.assign(cells + 2, 0);
        for (const TriBins::Box& b : B.box) B.each(b, [&](size_t c) { ++B.start[c + 2]; });
        for (size_t c = 0; c < cells; ++c) B.start[c + 2] += B.start[c + 1];
        return B;
    }
}

}  // namespace

hipError_t TriDevice::load(const std::vector<TriPrep>& prep, float dist, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    set = TriSet{};
    // a hit needs dist - |pos - tp| > 1e-6: none at a distance that is negative, zero, infinite or not a number
    if (prep.empty() || !(dist > 0.f) || !std::isfinite(dist)) return hipSuccess;
    TriBins B = bin_triangles(prep, dist);
    if (B.start.empty()) return hipSuccess;   // no finite triangle
    // one allocation: spheres in list order, records, cell starts, lists
    const size_t listed = B.start.back(), cells = B.start.size() - 2;
    std::vector<uint32_t> host(cells + 1 + listed);
    uint32_t* const list = host.data() + cells + 1;
    for (const TriBins::Box& b : B.box) B.each(b, [&](size_t c) { list[B.start[c + 1]++] = b.id; });
    std::copy_n(B.start.begin(), cells + 1, host.begin());
    const size_t o_tri = listed * sizeof(float4), o_start = o_tri + prep.size() * sizeof(TriPrep),
                 o_list = o_start + (cells + 1) * 4, bytes = o_list + listed * 4;
    hipError_t e = hipStreamSynchronize(st);   // launches that read the former triangles
    if (e == hipSuccess && bytes > cap) {
        if (mem) e = hipFree(mem);
        mem = nullptr;
        cap = 0;
        if (e == hipSuccess) e = hipMalloc((void**)&mem, bytes);
        if (e != hipSuccess) return e;
        cap = bytes;
    }
    if (e == hipSuccess) e = hipMemcpyAsync(mem + o_tri, prep.data(), o_start - o_tri, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipMemcpyAsync(mem + o_start, host.data(), bytes - o_start, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        k_list_spheres<<<(uint32_t)((listed + kBlockTri - 1) / kBlockTri), kBlockTri, 0, st>>>(
            (uint32_t)listed, (const uint32_t*)(mem + o_list), (const TriPrep*)(mem + o_tri), (float4*)mem);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);   // the host arrays are read
    if (e != hipSuccess) return e;
    set.n = (int)prep.size();
    set.sphere = (const float4*)mem;
    set.tris = (const TriPrep*)(mem + o_tri);
    set.start = (const uint32_t*)(mem + o_start);
    set.list = (const uint32_t*)(mem + o_list);
    set.min = make_float3(B.min[0], B.min[1], B.min[2]);
    set.inv = B.inv;
    set.nx = B.n[0];
    set.ny = B.n[1];
    set.nz = B.n[2];
    return hipSuccess;
}

}  // namespace rtps
