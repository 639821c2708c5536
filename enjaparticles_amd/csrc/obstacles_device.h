// Forces of the obstacles on one fluid particle: loaded triangles and the
// particles of rigid bodies.
#pragma once

#include <hip/hip_runtime.h>

#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

// Triangle collision of collision_tri.cl:120-231, 418-470 for one particle at
// px, py, pz (scaled) with velocity v and one triangle: the segment
// pos +- dist * v/|v| (dist = boundary_distance) is intersected with it
// (Ericson, Real-Time Collision Detection, pp. 191-192); on a hit at tp,
// penetration = dist - |pos - tp| and, when it exceeds 1e-6, the repulsion
// and friction of cl_sph_collision.h:31-73 along the triangle's unit normal
// are added to f.
__device__ __forceinline__ void tri_add(float3& f, float px, float py, float pz, float4 v, const TriPrep& T,
                                        const rtps_sph_params& sp) {
    const float dist = sp.boundary_distance, k = sp.boundary_stiffness, damp = sp.boundary_dampening;
    // v3normalize (collision_tri.cl:46-50): NaN for v = 0, and then no hit
    const float mag = __builtin_sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
    const float vnx = v.x / mag, vny = v.y / mag, vnz = v.z / mag;
    // segment ends p = pos - vn dist, q = pos + vn dist (collision_tri.cl:135-137)
    const float sx = px - vnx * dist, sy = py - vny * dist, sz = pz - vnz * dist;
    const float qx = px + vnx * dist, qy = py + vny * dist, qz = pz + vnz * dist;
    const float qpx = sx - qx, qpy = sy - qy, qpz = sz - qz;
    // Ericson segment-triangle test (collision_tri.cl:120-170)
    const float d = qpx * T.nx + qpy * T.ny + qpz * T.nz;
    if (d <= 0.0f) return;
    const float apx = sx - T.ax, apy = sy - T.ay, apz = sz - T.az;
    float tt = apx * T.nx + apy * T.ny + apz * T.nz;
    if (tt < 0.0f || tt > d) return;
    const float ex = qpy * apz - qpz * apy, ey = qpz * apx - qpx * apz, ez = qpx * apy - qpy * apx;
    const float abx = T.bx - T.ax, aby = T.by - T.ay, abz = T.bz - T.az;
    const float acx = T.qx - T.ax, acy = T.qy - T.ay, acz = T.qz - T.az;
    float vv = acx * ex + acy * ey + acz * ez;
    if (vv < 0.0f || vv > d) return;
    float ww = -(abx * ex + aby * ey + abz * ez);
    if (ww < 0.0f || vv + ww > d) return;
    const float ood = 1.0f / d;
    vv *= ood;
    ww *= ood;
    const float uu = 1.0f - vv - ww;
    const float tx = uu * T.ax + vv * T.bx + ww * T.qx;   // tp = u a + v b + w c
    const float ty = uu * T.ay + vv * T.by + ww * T.qy;
    const float tz = uu * T.az + vv * T.bz + ww * T.qz;
    const float ddx = px - tx, ddy = py - ty, ddz = pz - tz;
    const float pen = dist - __builtin_sqrtf(ddx * ddx + ddy * ddy + ddz * ddz);
    if (!(pen > 1e-6f)) return;   // collision_tri.cl:196
    // calculateRepulsionForce + calculateFrictionForce (zero coefficients)
    const float ndv = T.ux * v.x + T.uy * v.y + T.uz * v.z;
    const float m2 = k * pen - damp * ndv;
    f.x += m2 * T.ux;
    f.y += m2 * T.uy;
    f.z += m2 * T.uz;
    const float vtx = v.x - v.x * ndv, vty = v.y - v.y * ndv, vtz = v.z - v.z * ndv;
    if ((vtx + vty + vtz) / 3.0f > 0.0f) {
        f.x -= vtx;
        f.y -= vty;
        f.z -= vtz;
    }
}

// The forces of the triangles listed in the particle's cell (p, v unscaled),
// in triangle order.
__device__ __forceinline__ float3 tri_forces(float4 p, float4 v, const TriSet& S, const rtps_sph_params& sp) {
    const float s = sp.simulation_scale;
    const float px = p.x * s, py = p.y * s, pz = p.z * s;
    float3 f = make_float3(0.f, 0.f, 0.f);
    const float ux = (px - S.min.x) * S.inv, uy = (py - S.min.y) * S.inv, uz = (pz - S.min.z) * S.inv;
    if (!(ux >= 0.f && ux < (float)S.nx && uy >= 0.f && uy < (float)S.ny && uz >= 0.f && uz < (float)S.nz)) return f;
    const int c = ((int)uz * S.ny + (int)uy) * S.nx + (int)ux;
    const uint32_t q1 = S.start[c + 1];
    constexpr int kGroupTri = 4;   // spheres loaded together
    for (uint32_t q0 = S.start[c]; q0 < q1; q0 += kGroupTri) {
        float4 sphere[kGroupTri];   // centre, reach squared
#pragma unroll
        for (int g = 0; g < kGroupTri; ++g) sphere[g] = S.sphere[min(q0 + g, q1 - 1u)];
        uint32_t meet = 0u;
#pragma unroll
        for (int g = 0; g < kGroupTri; ++g) {
            const float4 r = sphere[g];
            const float cx = px - r.x, cy = py - r.y, cz = pz - r.z;
            const bool outside = cx * cx + cy * cy + cz * cz > r.w;   // no hit within dist
            meet |= !outside && q0 + g < q1 ? 1u << g : 0u;
        }
        for (; meet != 0u; meet &= meet - 1u)
            tri_add(f, px, py, pz, v, S.tris[S.list[q0 + (uint32_t)__builtin_ctz(meet)]], sp);
    }
    return f;
}

// Rigid-body particles around one fluid particle (SPH::interact;
// rigidbody_force.cl:118-193 for a moving body, staticrigidbody_force.cl:45-146
// for the static boundary): the 27 cells around it, cut-off 2 h.  p unscaled,
// e = veleval.xyz | density.  Adds to f.  Particles none of whose 27 cells
// holds one (RigidDev::near) are done after one load.
template <bool MOVING>
__device__ __forceinline__ void rigid_force(float4& f, float4 p, float4 e, const RigidDev& r, int nb_cells,
                                            const rtps_sph_params& sp, const Grid& gs) {
    const float scale = sp.simulation_scale, h = sp.smoothing_distance, eps = sp.EPSILON, m = sp.mass;
    const float h2x = 2.0f * h;
    const float px = p.x * scale, py = p.y * scale, pz = p.z * scale;
    const float stiff = r.s0 * m;
    float fx = 0.f, fy = 0.f, fz = 0.f, vx = 0.f, vy = 0.f, vz = 0.f;
    const int3 c = grid_cell(px, py, pz, gs);
    if (r.near && (uint32_t)c.x < (uint32_t)gs.irx && (uint32_t)c.y < (uint32_t)gs.iry && c.z >= 0) {
        const uint32_t own = (uint32_t)grid_hash(c.x, c.y, c.z, gs);
        if (own < (uint32_t)nb_cells && !r.near[own]) return;   // no pair: nothing to add
    }
    for (int z = c.z - 1; z <= c.z + 1; ++z) {
        // The plane's nine cells are looked up together (one by one, each
        // waited for the loads of the one before): a row's three cells are one
        // run of the sorted particles.  Only on the largest grids, whose float
        // hashes are no longer exact, the cells are taken one at a time.
        const bool rows = nb_cells < (1 << 23);
        uint32_t lo[3], hi[3];
        auto run = [&](int x0, int n, int y, uint32_t& a, uint32_t& b) {
            uint32_t first[3], last[3];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                const uint32_t ch = x < n ? min((uint32_t)grid_hash(x0 + x, y, z, gs), (uint32_t)nb_cells) : (uint32_t)nb_cells;
                first[x] = r.start[ch];
                last[x] = r.end[ch];   // of an empty cell: not used
                if (ch >= (uint32_t)nb_cells) first[x] = kEmpty;
            }
            a = min(first[0], min(first[1], first[2]));
            b = 0u;
#pragma unroll
            for (int x = 0; x < 3; ++x) b = first[x] != kEmpty ? max(b, last[x]) : b;
        };
        if (rows) {
#pragma unroll
            for (int k = 0; k < 3; ++k) run(c.x - 1, 3, c.y - 1 + k, lo[k], hi[k]);
        }
#pragma unroll 1
        for (int k = 0; k < (rows ? 3 : 9); ++k) {
            uint32_t a = k == 0 ? lo[0] : (k == 1 ? lo[1] : lo[2]), b = k == 0 ? hi[0] : (k == 1 ? hi[1] : hi[2]);
            if (!rows) run(c.x - 1 + k % 3, 1, c.y - 1 + k / 3, a, b);
            for (uint32_t j = a; j < b; ++j) {
                const float4 q = r.pos[j];
                const float rx = q.x * scale - px, ry = q.y * scale - py, rz = q.z * scale - pz;
                float rl = __builtin_sqrtf(rx * rx + ry * ry + rz * rz);
                if (!(rl <= h2x)) continue;
                rl = fmaxf(rl, eps);
                const float inv = 1.0f / rl;
                const float nx = rx * inv, ny = ry * inv, nz = rz * inv;
                float ux = -e.x, uy = -e.y, uz = -e.z, mn;
                if (MOVING) {
                    const float4 v = r.vel[j];
                    ux += v.x;
                    uy += v.y;
                    uz += v.z;
                    const float mj = r.mass[j];
                    mn = (m * mj) / (m + mj);
                } else {
                    mn = (m * m) / (m + m);
                }
                const float un = ux * nx + uy * ny + uz * nz;
                const float spr = -stiff * (h2x - rl);
                const float dmp = r.s1 * __builtin_sqrtf(stiff * mn);
                fx += spr * nx + dmp * (un * nx);
                fy += spr * ny + dmp * (un * ny);
                fz += spr * nz + dmp * (un * nz);
                const float lap = h - rl;
                if (MOVING) {
                    ux -= un * nx;
                    uy -= un * ny;
                    uz -= un * nz;
                }
                vx += ux * lap;
                vy += uy * lap;
                vz += uz * lap;
            }
        }
    }
    const float cv = m * (1.0f / (e.w * e.w)) * (sp.viscosity * sp.wvisc_dd_coef);
    const float sg = MOVING ? cv : -cv;
    f.x += fx / m + sg * vx;
    f.y += fy / m + sg * vy;
    f.z += fz / m + sg * vz;
}

}  // namespace rtps
