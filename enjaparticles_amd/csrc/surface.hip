// Colour field and iso-surface extraction (SPH::postProcess, SPH.cpp:338-386).
//
// Colour field (colorfield.cl:86-125, ColorField.cpp): node (s, t, r) of a
// res^3 lattice spanning the scaled boundary box takes
//     mass * sum_j Wspiky(max(|x - x_j|, eps), h) / rho_j,   |x - x_j| <= h,
// Wspiky(r, h) = 15 / (pi h^6) (h - r)^3 (cl_sph_kernels.h:71-78), over the
// 27 cells around the node, with the neighbour rows of the density kernel.
// Nodes are stored x fastest, then y, then z (a plain 3-D array instead of
// the reference's 2-D image of slices).
//
// Iso-surface (MarchingCubes.cpp with classifycubes.cl / constructhp.cl /
// traversehp.cl): the reference classifies cubes into a 2-D histogram
// pyramid and walks the pyramid once per output triangle.  Here the cubes
// are classified and their triangles counted in tiles, an exclusive scan gives
// each tile its first triangle, and the tiles write theirs, a vertex per thread:
// vertices interpolated linearly along the crossing edges, normals from the
// interpolated negative central differences of the field (pointing away from
// the fluid), as traversehp.cl:470-515 computes them.  The case table, the
// corner bits and the edge ends are the reference's (mc_table.h); a cube's
// triangles come out in the table's order, cubes in lattice order (x fastest).
// Vertices are in world coordinates of the boundary box, or in the
// reference's frame (lattice coordinates / (res - 1) * 10, traversehp.cl:512).

#include <hip/hip_runtime.h>

#include <mutex>

#include "mc_table.h"
#include "rtps_internal.h"
#include "sort_layout.h"
#include "sph_device.h"

namespace rtps {

namespace {

constexpr int kBlockSurf = 256;
constexpr int kTileCubes = kBlockSurf;                  // cubes per tile, one thread each
constexpr int kScanThreads = 1024, kScanItems = 8;       // of the scan of the tiles' counts, per thread

inline int blocks_of(long n, int bs) { return (int)((n + bs - 1) / bs); }

}  // namespace

// Corner offsets of the case bits and the edges' two ends (mc_table.h).
__constant__ int8_t c_mc_corner[8][3];
__constant__ int8_t c_mc_edge[12][6];

namespace {

// One wave per brick of 32 x 2 x 1 nodes.  The brick walks the rows of cells
// around it in ascending (z, y), which for every node is the order of its own
// nine rows; the union of its nodes' windows of a row is copied to LDS once
// (positions, with the density in w) and each node takes its window from there,
// 32 candidates at a time: the tests first, one bit each, then the terms of the
// accepted ones (an IEEE square root and division each, which in the test's
// branch would run for the whole wave when one lane accepts).  The next row's
// windows are looked up before the current row's walk.  A brick with no particle
// in the cells around it, most of a pool's box, ends after one look at them.
// Measured on a settled pool of 262,139 particles in a 128^3 lattice (14% of its
// nodes in the fluid): 81 us, with bricks of 16 x 2 x 2 and 16 x 4 x 1 nodes 86
// and 91, 8 x 4 x 2 97, 4 x 4 x 4 115; a thread per node that reads its windows
// from memory 150, in bricks of 4 x 4 x 4 166.  (Coarse lattices: bricks_pay.)
constexpr int kBrickX = 32, kBrickY = 2, kBrickZ = 1;   // 64 nodes
constexpr int kFieldCap = 256;   // candidates per LDS copy of a row (4 KB per wave)

template <bool SCALED>
__global__ __launch_bounds__(kBlockSurf) void k_color_field(int res, const float4* __restrict__ pos_s,
                                                            const float4* __restrict__ ve_s,
                                                            const uint32_t* __restrict__ start,
                                                            const uint32_t* __restrict__ end, rtps_sph_params sp,
                                                            Grid g, Win win, rtps_float4 bmin, rtps_float4 bmax,
                                                            float* __restrict__ field) {
    __shared__ float4 stage[kBlockSurf / 64][kFieldCap];
    float4* __restrict__ my = stage[threadIdx.x >> 6];
    const int bx = (res + kBrickX - 1) / kBrickX, by = (res + kBrickY - 1) / kBrickY,   // bricks per axis
              bz = (res + kBrickZ - 1) / kBrickZ;
    const long brick = (long)blockIdx.x * (kBlockSurf / 64) + (threadIdx.x >> 6);
    if (brick >= (long)bx * by * bz) return;
    const int lane = (int)threadIdx.x & 63;
    const int s0 = kBrickX * (int)(brick % bx) + lane % kBrickX;
    const int t0 = kBrickY * (int)((brick / bx) % by) + lane / kBrickX % kBrickY;
    const int r0 = kBrickZ * (int)(brick / ((long)bx * by)) + lane / (kBrickX * kBrickY);
    const bool inside = s0 < res && t0 < res && r0 < res;
    // lanes past the lattice repeat its last nodes: the copies take whole waves
    const int s = min(s0, res - 1), t = min(t0, res - 1), r = min(r0, res - 1);
    // texPos = (s, t, r) / (res - 1) * (bnd_max - bnd_min) + bnd_min (colorfield.cl:104-108)
    const float tmp = 1.0f / (float)(res - 1);
    const float px = (float)s * tmp * (bmax.x - bmin.x) + bmin.x;
    const float py = (float)t * tmp * (bmax.y - bmin.y) + bmin.y;
    const float pz = (float)r * tmp * (bmax.z - bmin.z) + bmin.z;
    const float scale = sp.simulation_scale;
    const float h = sp.smoothing_distance, h2 = h * h, eps = sp.EPSILON;
    const float h6 = h * h * h * h * h * h;
    const float alpha = 15.0f / 3.14159265f / h6;
    const int3 c = grid_cell(px, py, pz, g);
    float sum = 0.0f;
    // the cells of the brick (nodes ascend along every axis), one more on each side
    const int x_lo = __builtin_amdgcn_readlane(c.x, 0) - 1, x_hi = __builtin_amdgcn_readlane(c.x, 63) + 1;
    const int y_lo = __builtin_amdgcn_readlane(c.y, 0) - 1, y_hi = __builtin_amdgcn_readlane(c.y, 63) + 1;
    const int z_lo = __builtin_amdgcn_readlane(c.z, 0) - 1, z_hi = __builtin_amdgcn_readlane(c.z, 63) + 1;
    const int nx = x_hi - x_lo + 1, ny = y_hi - y_lo + 1, nz = z_hi - z_lo + 1, rows = ny * nz;
    bool wet = false;
    for (int k = lane; k < nx * rows; k += 64) {
        const uint32_t cell = (uint32_t)grid_hash(x_lo + k % nx, y_lo + (k / nx) % ny, z_lo + k / (nx * ny), g);
        wet = wet || (cell < (uint32_t)g.nb_cells && start[cell] != kEmpty);
    }
    if (__ballot(wet) != 0ull) {
        const WindowCtx wc = window_ctx(px, py, pz, g, c, h, win.keys, win.rx, win.ry, win.rz);
        auto dist2 = [&](float4 pj) {
            if (SCALED) { pj.x *= scale; pj.y *= scale; pj.z *= scale; }
            const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
            return rx * rx + ry * ry + rz * rz;
        };
        // the node's window of row k of the brick's rows, empty when the row is not one of its nine
        auto lookup = [&](int k, uint32_t& a, uint32_t& b) {
            const int dy = y_lo + k % ny - c.y, dz = z_lo + k / ny - c.z;
            a = b = 0u;
            if (dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1)
                row_window(wc, c, dy, dz, h2, g, start, end, win.keys, a, b, 0u, win.sub);
        };
        auto walk = [&](uint32_t a, uint32_t b, auto&& pos, auto&& rho) {
            for (uint32_t j0 = a; j0 < b; j0 += 32u) {
                const uint32_t n = min(b - j0, 32u);
                uint32_t m = 0u;   // accepted candidates, bit k = j0 + k
                uint32_t k = 0u;
                for (; k + kGroup <= n; k += kGroup) {
                    float4 q[kGroup];
#pragma unroll
                    for (int u = 0; u < kGroup; ++u) q[u] = pos(j0 + k + u);
#pragma unroll
                    for (int u = 0; u < kGroup; ++u) m |= dist2(q[u]) <= h2 ? 1u << (k + u) : 0u;
                }
                for (; k < n; ++k) m |= dist2(pos(j0 + k)) <= h2 ? 1u << k : 0u;
                while (m != 0u) {   // colorfield.cl:63-75
                    const uint32_t j = j0 + (uint32_t)__builtin_ctz(m);
                    m &= m - 1u;
                    const float4 pj = pos(j);
                    const float rlen = fmaxf(__builtin_sqrtf(dist2(pj)), eps);
                    const float hr = h - rlen;
                    sum += alpha * hr * hr * hr / rho(pj, j);
                }
            }
        };
        uint32_t a, b, a1 = 0u, b1 = 0u;
        lookup(0, a, b);
        for (int k = 0; k < rows; ++k, a = a1, b = b1) {
            const uint32_t A = __ockl_wfred_min_u32(a < b ? a : 0xFFFFFFFFu);
            const uint32_t B = __ockl_wfred_max_u32(a < b ? b : 0u);
            const bool staged = B > A && B - A <= (uint32_t)kFieldCap;
            if (staged)
                for (uint32_t q = lane; q < B - A; q += 64u) {
                    float4 p = pos_s[A + q];
                    p.w = ve_s[A + q].w;
                    my[q] = p;
                }
            if (k + 1 < rows) lookup(k + 1, a1, b1);
            __builtin_amdgcn_wave_barrier();   // the copies before any lane reads them
            if (staged) walk(a, b, [&](uint32_t j) { return my[j - A]; }, [](const float4& p, uint32_t) { return p.w; });
            else walk(a, b, [&](uint32_t j) { return pos_s[j]; }, [&](const float4&, uint32_t j) { return ve_s[j].w; });
            __builtin_amdgcn_wave_barrier();   // every read before the next row's copies
        }
    }
    if (inside) field[((long)r * res + t) * res + s] = sum * sp.mass;
}

// The same for coarse lattices, a thread per node that reads its nine windows
// from memory: the nodes of a wave are so far apart there that a brick's rows
// reach across the box, most of them not its nodes' own.
template <bool SCALED>
__global__ __launch_bounds__(kBlockSurf) void k_color_field_nodes(int res, const float4* __restrict__ pos_s,
                                                                  const float4* __restrict__ ve_s,
                                                                  const uint32_t* __restrict__ start,
                                                                  const uint32_t* __restrict__ end,
                                                                  rtps_sph_params sp, Grid g, Win win,
                                                                  rtps_float4 bmin, rtps_float4 bmax,
                                                                  float* __restrict__ field) {
    const long idx = (long)blockIdx.x * kBlockSurf + threadIdx.x;
    if (idx >= (long)res * res * res) return;
    const int s = (int)(idx % res), t = (int)((idx / res) % res), r = (int)(idx / ((long)res * res));
    const float tmp = 1.0f / (float)(res - 1);
    const float px = (float)s * tmp * (bmax.x - bmin.x) + bmin.x;
    const float py = (float)t * tmp * (bmax.y - bmin.y) + bmin.y;
    const float pz = (float)r * tmp * (bmax.z - bmin.z) + bmin.z;
    const float scale = sp.simulation_scale;
    const float h = sp.smoothing_distance, h2 = h * h, eps = sp.EPSILON;
    const float h6 = h * h * h * h * h * h;
    const float alpha = 15.0f / 3.14159265f / h6;
    const int3 c = grid_cell(px, py, pz, g);
    const WindowCtx wc = window_ctx(px, py, pz, g, c, h, win.keys, win.rx, win.ry, win.rz);
    float sum = 0.0f;
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy) {
            uint32_t a, b;
            row_window(wc, c, dy, dz, h2, g, start, end, win.keys, a, b, 0u, win.sub);
            auto term = [&](float4 pj, uint32_t j) {   // colorfield.cl:63-75
                if (SCALED) { pj.x *= scale; pj.y *= scale; pj.z *= scale; }
                const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
                const float r2 = rx * rx + ry * ry + rz * rz;
                if (r2 <= h2) {
                    const float rlen = fmaxf(__builtin_sqrtf(r2), eps);
                    const float hr = h - rlen;
                    sum += alpha * hr * hr * hr / ve_s[j].w;
                }
            };
            uint32_t j = a;
            for (; j + kGroup <= b; j += kGroup) {   // loads of a group issued together
                float4 q[kGroup];
#pragma unroll
                for (int k = 0; k < kGroup; ++k) q[k] = pos_s[j + k];
#pragma unroll
                for (int k = 0; k < kGroup; ++k) term(q[k], j + k);
            }
            for (; j < b; ++j) term(pos_s[j], j);
        }
    field[idx] = sum * sp.mass;
}

// Where the bricks pay: from kBrickRes nodes an axis, fewer being too few waves,
// at a node spacing of at most kBrickSpacing cells.  Measured (us, a thread per
// node / bricks; settled pools): 21 / 75 at 2 nodes an axis and 64 / 67 at 16 of
// 23 cells (20,011 particles); 31 / 75, 79 / 102, 139 / 103 and 158 / 96 at 3, 16,
// 31 and 104 of 52 cells (262,139); 44 / 96, 168 / 202, 204 / 191, 169 / 156 and
// 771 / 298 at 4, 40, 56, 80 and 159 of 79 cells (1,000,000).
constexpr int kBrickRes = 28;
constexpr float kBrickSpacing = 1.8f;
bool bricks_pay(int res, const Grid& g, const rtps_float4& bmin, const rtps_float4& bmax) {
    const float per = 1.0f / (float)(res - 1);   // along z a brick is one node
    return res >= kBrickRes && (bmax.x - bmin.x) * per * g.delta.x <= kBrickSpacing &&
           (bmax.y - bmin.y) * per * g.delta.y <= kBrickSpacing;
}

__device__ __forceinline__ float node(const float* __restrict__ f, int res, int x, int y, int z) {
    return f[((long)z * res + y) * res + x];
}

// Lattice position of cube k of a tile (cubes are numbered x fastest, m per
// axis): the tile's by one uniform 64-bit division, the cube's by 32-bit ones.
__device__ __forceinline__ int3 tile_cube(uint32_t tile, uint32_t k, int m) {
    const long base = (long)tile * kTileCubes;
    const uint32_t row0 = (uint32_t)(base / m), x0 = (uint32_t)(base % m) + k, n = (uint32_t)m;
    const uint32_t row = row0 + x0 / n;
    return make_int3((int)(x0 % n), (int)(row % n), (int)(row / n));
}

// Case of every cube (bit k set when the node at corner offset
// kMcCorner[k] exceeds the iso level, classifycubes.cl:44-55), and the
// triangles (nrOfTriangles, classifycubes.cl:37) of each tile of kTileCubes
// cubes.  The cubes' own counts are not stored: k_mc_emit has them again from
// the cases.
__global__ __launch_bounds__(kBlockSurf) void k_mc_classify(int res, float iso, const float* __restrict__ f,
                                                            const uint8_t* __restrict__ ntri,
                                                            uint8_t* __restrict__ cases, uint32_t* __restrict__ sums) {
    __shared__ uint32_t part[kBlockSurf / 64];
    const int m = res - 1;
    const long ncubes = (long)m * m * m;
    const long idx = (long)blockIdx.x * kTileCubes + threadIdx.x;
    uint32_t count = 0;
    if (idx < ncubes) {
        const int3 p = tile_cube(blockIdx.x, threadIdx.x, m);
        uint32_t cs = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c)
            cs |= (uint32_t)(node(f, res, p.x + c_mc_corner[c][0], p.y + c_mc_corner[c][1],
                                  p.z + c_mc_corner[c][2]) > iso) << c;
        cases[idx] = (uint8_t)cs;
        count = ntri[cs];
    }
    count = wave_incl_scan(count);
    if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = count;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Exclusive scan of the tiles' triangle counts in place, one block walking
// them in chunks; the grand total follows the last one.
__global__ __launch_bounds__(kScanThreads) void k_scan_sums(uint32_t* __restrict__ sums, int ntiles) {
    __shared__ uint32_t part[kScanThreads / 64];
    const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
    uint32_t carry = 0;
    for (int c0 = 0; c0 < ntiles; c0 += kScanThreads * kScanItems) {
        const int i = c0 + (int)threadIdx.x * kScanItems;
        uint32_t v[kScanItems], sum = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const uint32_t c = sums[min(i + k, ntiles - 1)];   // no branch: the loads are issued together
            v[k] = i + k < ntiles ? c : 0u;
            sum += v[k];
        }
        const uint32_t inc = wave_incl_scan(sum);
        if (lane == 63) part[w] = inc;
        __syncthreads();
        uint32_t run = carry + inc - sum;
#pragma unroll
        for (int q = 0; q < kScanThreads / 64; ++q) {
            if (q < w) run += part[q];
            carry += part[q];
        }
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (i + k < ntiles) sums[i + k] = run;
            run += v[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[ntiles] = carry;
}

__device__ __forceinline__ float3 neg_gradient(const float* __restrict__ f, int res, int x, int y, int z) {
    // traversehp.cl:470-502: -(f(p + e) - f(p - e)) per axis, indices clamped to the lattice
    const int xp = min(x + 1, res - 1), xm = max(x - 1, 0);
    const int yp = min(y + 1, res - 1), ym = max(y - 1, 0);
    const int zp = min(z + 1, res - 1), zm = max(z - 1, 0);
    return make_float3(node(f, res, xm, y, z) - node(f, res, xp, y, z), node(f, res, x, ym, z) - node(f, res, x, yp, z),
                       node(f, res, x, y, zm) - node(f, res, x, y, zp));
}

// Triangles of every cube at its scanned offset (at most `capacity` in all):
// 9 floats per triangle in `verts` and `normals`; frame 0 = world
// coordinates of [wmin, wmax], 1 = the reference's lattice / (res - 1) * 10.
// One block per tile of cubes; most have none and end at once.  The others list
// their triangles (cube and number) in LDS and then take one vertex per thread,
// in the order of the output.  With the counting that it repeats in place of
// stored counts and offsets (8 bytes a cube), classifying, scanning and
// emitting a 128^3 lattice takes 39 us instead of 46; tiles of 2,048 cubes take
// 70 us here, as a flat surface lies in a few of them.
__global__ __launch_bounds__(kBlockSurf) void k_mc_emit(int res, float iso, const float* __restrict__ f,
                                                        const uint8_t* __restrict__ cases,
                                                        const uint8_t* __restrict__ ntri,
                                                        const uint32_t* __restrict__ tile_offs,
                                                        const uint64_t* __restrict__ words, rtps_float4 wmin,
                                                        rtps_float4 wmax, int frame, long capacity,
                                                        float* __restrict__ verts, float* __restrict__ normals) {
    __shared__ uint16_t list[kTileCubes * 5];   // cube << 3 | triangle; a case has at most five
    __shared__ uint8_t tile_cases[kTileCubes];
    __shared__ uint32_t part[kBlockSurf / 64];
    const uint32_t first = tile_offs[blockIdx.x], count = tile_offs[blockIdx.x + 1] - first;
    if (count == 0) return;
    const int m = res - 1, tid = (int)threadIdx.x;
    const long ncubes = (long)m * m * m, base = (long)blockIdx.x * kTileCubes;
    const uint8_t cs = base + tid < ncubes ? cases[base + tid] : (uint8_t)0;   // case 0: no triangle
    tile_cases[tid] = cs;
    const uint32_t n = ntri[cs], inc = wave_incl_scan(n);
    if ((tid & 63) == 63) part[tid >> 6] = inc;
    __syncthreads();
    uint32_t at = inc - n;
    for (int q = 0; q < tid >> 6; ++q) at += part[q];
    for (uint32_t q = 0; q < n; ++q) list[at + q] = (uint16_t)(tid << 3 | q);
    __syncthreads();
    const float inv = 1.0f / (float)(res - 1);
    for (uint32_t u = tid; u < 3 * count; u += kBlockSurf) {
        const uint32_t tri = u / 3, v = u - 3 * tri, entry = list[tri];
        const long o = (long)first + tri;
        if (o >= capacity) return;
        const uint32_t cube = entry >> 3, q = entry & 7u;
        const int3 p = tile_cube(blockIdx.x, cube, m);
        const uint64_t w = words[tile_cases[cube]];
        const int e = (int)((w >> (4 * (3 * q + v))) & 0xFu);
        const int8_t* ee = c_mc_edge[e];
        const int ax = p.x + ee[0], ay = p.y + ee[1], az = p.z + ee[2];
        const int bx = p.x + ee[3], by = p.y + ee[4], bz = p.z + ee[5];
        const float v0 = node(f, res, ax, ay, az), v1 = node(f, res, bx, by, bz);
        const float d = (iso - v0) / (v1 - v0);   // traversehp.cl:506-511
        const float gx = (float)ax + d * (float)(bx - ax);
        const float gy = (float)ay + d * (float)(by - ay);
        const float gz = (float)az + d * (float)(bz - az);
        const float3 n0 = neg_gradient(f, res, ax, ay, az), n1 = neg_gradient(f, res, bx, by, bz);
        const float nx = n0.x + d * (n1.x - n0.x), ny = n0.y + d * (n1.y - n0.y), nz = n0.z + d * (n1.z - n0.z);
        const float len2 = nx * nx + ny * ny + nz * nz;
        const float il = len2 > 0.0f ? __builtin_amdgcn_rsqf(len2) : 0.0f;
        float* pv = verts + (o * 3 + v) * 3;
        float* pn = normals + (o * 3 + v) * 3;
        if (frame == 1) {   // mix(p0, p1, d) / (res - 1) * 10 (traversehp.cl:512)
            const float rm = (float)(res - 1);
            pv[0] = gx / rm * 10.0f;
            pv[1] = gy / rm * 10.0f;
            pv[2] = gz / rm * 10.0f;
        } else {
            pv[0] = wmin.x + gx * inv * (wmax.x - wmin.x);
            pv[1] = wmin.y + gy * inv * (wmax.y - wmin.y);
            pv[2] = wmin.z + gz * inv * (wmax.z - wmin.z);
        }
        pn[0] = nx * il;
        pn[1] = ny * il;
        pn[2] = nz * il;
    }
}

}  // namespace

size_t surface_scan_tiles(long ncubes) { return (size_t)((ncubes + kTileCubes - 1) / kTileCubes); }

hipError_t launch_color_field(int res, const float4* pos_s, const float4* ve_s, const uint32_t* start,
                              const uint32_t* end, const rtps_sph_params& sp, const Grid& g, const Win& win,
                              const rtps_float4& bmin_scaled, const rtps_float4& bmax_scaled, float* field,
                              hipStream_t st) {
    (void)hipGetLastError();
    if (res < 2) return hipErrorInvalidValue;
    const bool scaled = sp.simulation_scale != 1.0f, bricks = bricks_pay(res, g, bmin_scaled, bmax_scaled);
    const long bx = (res + kBrickX - 1) / kBrickX, by = (res + kBrickY - 1) / kBrickY, bz = (res + kBrickZ - 1) / kBrickZ;
    const long n = bricks ? bx * by * bz * 64 : (long)res * res * res;   // one wave per brick, or a thread per node
    auto* kernel = bricks ? (scaled ? k_color_field<true> : k_color_field<false>)
                          : (scaled ? k_color_field_nodes<true> : k_color_field_nodes<false>);
    kernel<<<blocks_of(n, kBlockSurf), kBlockSurf, 0, st>>>(res, pos_s, ve_s, start, end, sp, g, win, bmin_scaled,
                                                            bmax_scaled, field);
    return hipGetLastError();
}

hipError_t launch_mc_count(int res, float iso, const float* field, const uint8_t* ntri, uint8_t* cases,
                           uint32_t* tile_sums, hipStream_t st) {
    (void)hipGetLastError();
    if (res < 2) return hipErrorInvalidValue;
    const long m = res - 1, ncubes = m * m * m;
    const int ntiles = (int)surface_scan_tiles(ncubes);
    k_mc_classify<<<ntiles, kBlockSurf, 0, st>>>(res, iso, field, ntri, cases, tile_sums);
    k_scan_sums<<<1, kScanThreads, 0, st>>>(tile_sums, ntiles);
    return hipGetLastError();
}

hipError_t mc_upload_geometry() {
    static std::mutex mu;
    static bool done[64] = {};
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (done[dev]) return hipSuccess;   // each device holds its own constant memory
    err = hipMemcpyToSymbol(HIP_SYMBOL(c_mc_corner), kMcCorner, sizeof(kMcCorner));
    if (err == hipSuccess) err = hipMemcpyToSymbol(HIP_SYMBOL(c_mc_edge), kMcEdgeEnds, sizeof(kMcEdgeEnds));
    if (err == hipSuccess) done[dev] = true;
    return err;
}

hipError_t launch_mc_emit(int res, float iso, const float* field, const uint8_t* cases, const uint8_t* ntri,
                          const uint32_t* tile_offs, const uint64_t* words,
                          const rtps_float4& wmin, const rtps_float4& wmax, int frame, long capacity, float* verts,
                          float* normals, hipStream_t st) {
    (void)hipGetLastError();
    if (res < 2) return hipErrorInvalidValue;
    const long m = res - 1;
    k_mc_emit<<<(int)surface_scan_tiles(m * m * m), kBlockSurf, 0, st>>>(
        res, iso, field, cases, ntri, tile_offs, words, wmin, wmax, frame, capacity, verts, normals);
    return hipGetLastError();
}

}  // namespace rtps
