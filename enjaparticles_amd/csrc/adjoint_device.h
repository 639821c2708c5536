// Per-particle bodies of the adjoint kernels, shared by the single-system
// launches (adjoint.hip) and the batched ones (batch_adjoint.hip).  No
// reference counterpart; the forward step they differentiate is
// density.cl, force.cl, collision_wall.cl and leapfrog.cl (simulation_scale
// 1, no point sources, neighbour pairs held fixed):
//   rho_i = c_rho sum_j (h^2 - q^2)^3
//   a_i   = sum_j [ c_ij phi(q) r_ij + beta_ij psi(q) (e_j - e_i) ]
//           c_ij = m cp K (rho_i + rho_j - 2 rho0) / (rho_i rho_j), phi = (h-q)^2/q
//           beta_ij = m mu cv / (rho_i rho_j),                 psi = h - q
//   X_i   = cx sum_j (h^2 - q^2)^3 (e_j - e_i) / (rho_i + rho_j)
//   f_i   = clamp(a_i + walls(x_i, v_i) + g)
//   v' = v + dt f + xi X,  e' = (v + v')/2,  x' = x + dt v'
// c_ij, beta_ij and the XSPH weight are symmetric in (i, j), so every pair
// term of the backward pass is a gather over the same neighbour rows:
//   B1  per particle: leapfrog, velocity clamp and walls backwards -> adjoints
//       of a (ga) and X (gX), lambda_v of step n, the direct part of lambda_x
//   B2  pair loop: d/dx, d/de and d/drho of the pressure, viscosity and XSPH
//       terms, plus this particle's share of dL/dmu and dL/dK
//   B3  pair loop: density backwards, d rho / dx with the grho of both ends,
//       then lambda_x, lambda_e of step n scattered to the original order.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sph_device.h"

namespace rtps {

__device__ __forceinline__ float3 f3(float4 v) { return make_float3(v.x, v.y, v.z); }
__device__ __forceinline__ float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// The neighbour rows of a recorded step (Win::rows: the forward step's density
// kernel wrote them): for sorted particle i and row r = 3 (dz + 1) + (dy + 1)
// the three words at rows + 3 (r * stride + i) hold its window [a, b) and the
// rejection bits of the window's last min(b - a, 32) candidates.
struct AdjRows {
    const uint32_t* rows;
    uint32_t stride;
};

// B2 and B3 run blocks of kAdjThreads = three waves over a tile of 64
// particles, one plane (dz) of the neighbourhood each (the split tiles of
// sph_kernels.hip, here at every size: a tile's sums must not depend on how
// many tiles a launch holds).
constexpr int kAdjThreads = 192;

// Candidates per LDS copy of a row in B2 (4 records each) and B3 (a position
// and a float each): 6 KB and 5 KB per wave.
constexpr int kAdjStageCap = 96;
constexpr int kAdjB3StageCap = 256;
// LDS slice of a wave in B2 and B3 (float4 units).
constexpr int kAdjB2Slice = 4 * kAdjStageCap;
constexpr int kAdjB3Slice = kAdjB3StageCap + kAdjB3StageCap / 4;

// The wave's live lanes and this lane's rank among them; the union [A, B) of
// the live lanes' row windows (A >= B: no lane has candidates).
struct WaveLanes {
    uint32_t n, rank;
};
__device__ __forceinline__ WaveLanes wave_lanes() {
    const uint64_t live = __ballot(true);
    return WaveLanes{(uint32_t)__popcll(live),
                     (uint32_t)__popcll(live & ((1ull << (threadIdx.x & 63)) - 1ull))};
}
__device__ __forceinline__ void wave_range(uint32_t a, uint32_t b, uint32_t& A, uint32_t& B) {
    A = __ockl_wfred_min_u32(a < b ? a : 0xFFFFFFFFu);
    B = __ockl_wfred_max_u32(a < b ? b : 0u);
}

// B1 for sorted particle i.  lam_x/v/e: adjoints of step n+1 (original
// order; lam_v and lam_e may be null: zero).  Writes ga/gX (sorted), lam_v of
// step n (original order) and the direct part of lam_x (sorted).
__device__ __forceinline__ void adj_b1_body(int i, const uint32_t* __restrict__ idx, const float4* __restrict__ pos_s,
                                            const float4* __restrict__ vel_s, const float4* __restrict__ force_s,
                                            const rtps_sph_params& sp, const rtps_float4& bmin,
                                            const rtps_float4& bmax, int collision, float dt,
                                            const float4* __restrict__ lam_x, const float4* __restrict__ lam_v,
                                            const float4* __restrict__ lam_e, float4* __restrict__ ga_s,
                                            float4* __restrict__ gX_s, float4* __restrict__ lam_v_out,
                                            float4* __restrict__ lxp_s) {
    const uint32_t o = idx[i];
    const float3 none = make_float3(0.f, 0.f, 0.f);
    const float3 lx = f3(lam_x[o]), lv = lam_v ? f3(lam_v[o]) : none, le = lam_e ? f3(lam_e[o]) : none;
    // adjoint of v' (x' = x + dt v', e' = (v + v')/2)
    const float3 lvb = make_float3(lv.x + dt * lx.x + 0.5f * le.x, lv.y + dt * lx.y + 0.5f * le.y,
                                   lv.z + dt * lx.z + 0.5f * le.z);
    const float4 p = pos_s[i], v4 = vel_s[i];
    const float3 v = f3(v4);
    // f = force + walls + g, then the velocity clamp
    float4 F = force_s[i];
    if (collision) collision_wall(F, p, v4, sp, bmin, bmax);
    const float3 f = make_float3(F.x + sp.gravity.x, F.y + sp.gravity.y, F.z + sp.gravity.z);
    float3 gfc = make_float3(dt * lvb.x, dt * lvb.y, dt * lvb.z);   // adjoint of the clamped force
    float3 gf = gfc;
    const float speed = sqrtf(dot3(f, f));
    if (speed > sp.velocity_limit) {
        const float k = sp.velocity_limit / speed;
        const float3 u = make_float3(f.x / speed, f.y / speed, f.z / speed);
        const float ug = dot3(u, gfc);
        gf = make_float3(k * (gfc.x - u.x * ug), k * (gfc.y - u.y * ug), k * (gfc.z - u.z * ug));
    }
    const float xi = sp.xsph_factor;
    ga_s[i] = make_float4(gf.x, gf.y, gf.z, 0.f);
    gX_s[i] = make_float4(xi * lvb.x, xi * lvb.y, xi * lvb.z, 0.f);
    float3 gv = make_float3(lvb.x + 0.5f * le.x, lvb.y + 0.5f * le.y, lvb.z + 0.5f * le.z);
    float3 gx = lx;
    if (collision) {
        // active walls: d w / d x = -k s n n^T, d w / d v = -d n n^T, friction -v_t (v_t = v (1 - n.v))
        const float s = sp.simulation_scale, bd = sp.rest_distance * 0.5f;
        const float px = p.x * s, py = p.y * s, pz = p.z * s;
        const float diffs[6] = {bd - (pz - bmin.z), bd - (bmax.z - pz), bd - (py - bmin.y),
                                bd - (bmax.y - py), bd - (px - bmin.x), bd - (bmax.x - px)};
        const float3 ns[6] = {make_float3(0, 0, 1), make_float3(0, 0, -1), make_float3(0, 1, 0),
                              make_float3(0, -1, 0), make_float3(1, 0, 0), make_float3(-1, 0, 0)};
#pragma unroll
        for (int w = 0; w < 6; ++w) {
            if (!(diffs[w] > sp.EPSILON)) continue;
            const float3 n = ns[w];
            const float ng = dot3(n, gf);
            const float kx = -sp.boundary_stiffness * s * ng, kv = -sp.boundary_dampening * ng;
            gx.x += kx * n.x; gx.y += kx * n.y; gx.z += kx * n.z;
            gv.x += kv * n.x; gv.y += kv * n.y; gv.z += kv * n.z;
            const float ndv = dot3(n, v);
            const float3 vt = make_float3(v.x - v.x * ndv, v.y - v.y * ndv, v.z - v.z * ndv);
            if ((vt.x + vt.y + vt.z) / 3.0f > 0.0f) {
                // friction f = -v_t:  (d f / d v)^T g = -(1 - n.v) g + n (v . g)
                const float vg = dot3(v, gf);
                gv.x += -(1.f - ndv) * gf.x + n.x * vg;
                gv.y += -(1.f - ndv) * gf.y + n.y * vg;
                gv.z += -(1.f - ndv) * gf.z + n.z * vg;
            }
        }
    }
    lam_v_out[o] = make_float4(gv.x, gv.y, gv.z, 0.f);
    lxp_s[i] = make_float4(gx.x, gx.y, gx.z, 0.f);
}

// The accepted candidates of particle i in plane dz of its recorded rows, in
// ascending order.  Per row the wave's live lanes copy the union of their
// windows (when it holds at most CAP candidates) into the wave's LDS slice:
// `copy(t, j)` stores what candidate j needs besides its position at slot t,
// the position goes to st[t].  Wider unions are read from global memory.
// A lane's window is taken in chunks, the first ragged (1-32 candidates), the
// rest 32 long, so that the last chunk is what the record's bits cover; only
// earlier chunks are tested again.  pair(staged, o, r, r2): slot or index o of
// a candidate within h (not i itself), r = p_i - p_j.
template <int CAP, typename Copy, typename Pair>
__device__ __forceinline__ void adj_plane(int i, int dz, const AdjRows& rows, const float4& pi, float h2,
                                          const float4* __restrict__ pos_s, float4* __restrict__ st, Copy&& copy,
                                          Pair&& pair) {
    const WaveLanes wl = wave_lanes();
    uint32_t a[3], b[3], rej_last[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {   // the plane's records are loaded together
        const uint32_t* __restrict__ o = rows.rows + 3 * ((size_t)(3 * (dz + 1) + k) * rows.stride + (size_t)i);
        a[k] = o[0];
        b[k] = o[1];
        rej_last[k] = o[2];
    }
    auto walk = [&](auto staged, uint32_t a, uint32_t b, uint32_t off, uint32_t last) {
        const float4* __restrict__ P = decltype(staged)::value ? st : pos_s;
        uint32_t n = ((b - a - 1u) & 31u) + 1u;
        for (uint32_t j0 = a; j0 < b; j0 += n, n = 32u) {
            const uint32_t o0 = j0 - off;
            uint32_t rej = last;
            if (j0 + n != b) {
                rej = 0u;
                for (uint32_t k = 0; k < n; ++k) {
                    const float4 p = P[o0 + k];
                    rej = rej_bit(rej, h2_minus_r2(pi.x - p.x, pi.y - p.y, pi.z - p.z, h2));
                }
            }
            uint32_t m = __builtin_bitreverse32(~rej) >> (32u - n);   // bit t = candidate t
            const uint32_t self = (uint32_t)i - j0;   // the particle itself passes (r = 0): drop it
            if (self < n) m &= ~(1u << self);
            while (m != 0u) {
                const uint32_t o = o0 + (uint32_t)__builtin_ctz(m);
                m &= m - 1u;
                const float4 p = P[o];
                const float3 r = make_float3(pi.x - p.x, pi.y - p.y, pi.z - p.z);
                pair(staged, o, r, dot3(r, r));
            }
        }
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t A, B;
        wave_range(a[k], b[k], A, B);
        if (B <= A) continue;
        if (B - A <= (uint32_t)CAP) {
            for (uint32_t t = wl.rank; t < B - A; t += wl.n) {
                st[t] = pos_s[A + t];
                copy(t, A + t);
            }
            __builtin_amdgcn_wave_barrier();   // the copies before any lane reads them
            walk(std::true_type{}, a[k], b[k], A, rej_last[k]);
            __builtin_amdgcn_wave_barrier();   // every read before the next row's copies
        } else {
            walk(std::false_type{}, a[k], b[k], 0u, rej_last[k]);
        }
    }
}

// What B2 sums for a particle.
struct B2Acc {
    float3 gx, ge;
    float grho, gmu, gK;
};

// B2's pair terms of sorted particle i over plane dz.  ve_s = veleval.xyz |
// density (sorted).  Hardware rsq / rcp (~1 ulp) replace the square root and
// the divisions.  stage: kAdjB2Slice of the wave.
__device__ __forceinline__ B2Acc adj_b2_plane(int i, int dz, const float4* __restrict__ pos_s,
                                              const float4* __restrict__ ve_s, const float4* __restrict__ ga_s,
                                              const float4* __restrict__ gX_s, const AdjRows& rows,
                                              const rtps_sph_params& sp, float4* __restrict__ stage) {
    const float h = sp.smoothing_distance, h2 = h * h, eps = sp.EPSILON, eps2 = eps * eps;
    const float m = sp.mass, rho0 = sp.rest_density, K = sp.K, mu = sp.viscosity;
    const float cp = -0.5f * sp.wspiky_d_coef, cv = sp.wvisc_dd_coef;
    const float cx = 2.0f * sp.mass * sp.wpoly6_coef;
    const float4 pi = pos_s[i], vei = ve_s[i];
    const float3 ei = f3(vei), gai = f3(ga_s[i]), gXi = f3(gX_s[i]);
    const float ri = vei.w;
    const float inv_ri = __builtin_amdgcn_rcpf(ri);
    float3 gx = make_float3(0, 0, 0), ge = make_float3(0, 0, 0);
    float grho = 0.f, gmu = 0.f, gK = 0.f;
    // one accepted pair (within_h, j != i)
    auto pair = [&](const float3 r, const float q2, const float4 vej, const float4 gaj4, const float4 gXj4) {
        const float3 ej = f3(vej), gaj = f3(gaj4), gXj = f3(gXj4);
        const float rj = vej.w;
        const float q2c = fmaxf(q2, eps2);
        const float rinv = __builtin_amdgcn_rsqf(q2c);   // 1 / max(|r|, eps)
        const float q = q2c * rinv;                        // max(|r|, eps)
        const float dq = q2 > eps2 ? 1.f : 0.f;            // d q / d |r|
        const float inv_rr = __builtin_amdgcn_rcpf(ri * rj);
        const float3 dga = make_float3(gai.x - gaj.x, gai.y - gaj.y, gai.z - gaj.z);
        const float3 de = make_float3(ej.x - ei.x, ej.y - ei.y, ej.z - ei.z);
        const float3 rh = make_float3(r.x * rinv, r.y * rinv, r.z * rinv);   // used only where dq = 1
        // pressure: T_ij = c phi r
        const float hq = h - q;
        const float phi = hq * hq * rinv;
        const float dphi = -hq * (h + q) * rinv * rinv * dq;   // d phi / d |r|
        const float cK = m * cp * (ri + rj - 2.f * rho0) * inv_rr;   // c / K
        const float cc = K * cK;
        const float rdga = dot3(r, dga);
        const float sig = phi * rdga;
        gx.x += cc * (phi * dga.x + dphi * rdga * rh.x);
        gx.y += cc * (phi * dga.y + dphi * rdga * rh.y);
        gx.z += cc * (phi * dga.z + dphi * rdga * rh.z);
        grho += sig * m * cp * K * (2.f * rho0 - rj) * inv_rr * inv_ri;
        gK += cK * phi * dot3(r, gai);
        // viscosity: V_ij = beta psi (e_j - e_i), psi = h - q
        const float bmu = m * cv * inv_rr;           // beta / mu
        const float beta = mu * bmu;
        const float psi = hq;
        const float3 nga = make_float3(-dga.x, -dga.y, -dga.z);   // ga_j - ga_i
        ge.x += beta * psi * nga.x;
        ge.y += beta * psi * nga.y;
        ge.z += beta * psi * nga.z;
        const float deg = dot3(de, nga);
        gx.x += beta * deg * dq * rh.x;
        gx.y += beta * deg * dq * rh.y;
        gx.z += beta * deg * dq * rh.z;
        grho += -(beta * inv_ri) * psi * dot3(de, dga);
        gmu += bmu * psi * dot3(de, gai);
        // XSPH: Y_ij = cx w6 (e_j - e_i) / D
        const float t = h2 - q2;
        const float w6 = t * t * t;
        const float inv_D = __builtin_amdgcn_rcpf(ri + rj);
        const float3 dgX = make_float3(gXi.x - gXj.x, gXi.y - gXj.y, gXi.z - gXj.z);
        const float yk = cx * w6 * inv_D;
        ge.x -= yk * dgX.x;
        ge.y -= yk * dgX.y;
        ge.z -= yk * dgX.z;
        const float dedgX = dot3(de, dgX);
        const float yr = cx * inv_D * (-6.f) * t * t * dedgX;
        gx.x += yr * r.x;
        gx.y += yr * r.y;
        gx.z += yr * r.z;
        grho += -yk * inv_D * dedgX;
    };
    float4* __restrict__ sv = stage + kAdjStageCap;
    float4* __restrict__ sga = stage + 2 * kAdjStageCap;
    float4* __restrict__ sgx = stage + 3 * kAdjStageCap;
    adj_plane<kAdjStageCap>(
        i, dz, rows, pi, h2, pos_s, stage,
        [&](uint32_t t, uint32_t j) {
            sv[t] = ve_s[j];
            sga[t] = ga_s[j];
            sgx[t] = gX_s[j];
        },
        [&](auto staged, uint32_t o, const float3 r, float r2) {
            if constexpr (decltype(staged)::value) pair(r, r2, sv[o], sga[o], sgx[o]);
            else pair(r, r2, ve_s[o], ga_s[o], gX_s[o]);
        });
    return B2Acc{gx, ge, grho, gmu, gK};
}

// B2 for the block's tile: wave w takes plane w - 1 of particle i (the same 64
// particles in each wave; valid: i is one of them); wave 0 adds the planes in
// ascending order and writes gx2 (d/dx of the pair terms), ge (d/de) and grho
// (sorted), and the tile's share of dL/dmu and dL/dK goes to *partial.
__device__ __forceinline__ void adj_b2_tile(int i, bool valid, const float4* __restrict__ pos_s,
                                            const float4* __restrict__ ve_s, const float4* __restrict__ ga_s,
                                            const float4* __restrict__ gX_s, const AdjRows& rows,
                                            const rtps_sph_params& sp, float4* __restrict__ gx2_s,
                                            float4* __restrict__ ge_s, float* __restrict__ grho_s,
                                            float2* __restrict__ partial) {
    __shared__ float4 stage[3][kAdjB2Slice];
    __shared__ float2 share[3];
    const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
    B2Acc s = {make_float3(0, 0, 0), make_float3(0, 0, 0), 0.f, 0.f, 0.f};
    if (valid) s = adj_b2_plane(i, w - 1, pos_s, ve_s, ga_s, gX_s, rows, sp, stage[w]);
    for (int off = 32; off > 0; off >>= 1) {   // idle lanes add zero
        s.gmu += __shfl_down(s.gmu, off, 64);
        s.gK += __shfl_down(s.gK, off, 64);
    }
    if (lane == 0) share[w] = make_float2(s.gmu, s.gK);
    __builtin_amdgcn_wave_barrier();   // the last row's reads before the slice's reuse
    if (w > 0) {
        float* __restrict__ p = (float*)stage[w] + lane;
        p[0] = s.gx.x; p[64] = s.gx.y; p[128] = s.gx.z;
        p[192] = s.ge.x; p[256] = s.ge.y; p[320] = s.ge.z;
        p[384] = s.grho;
    }
    __syncthreads();
    if (w > 0) return;
    if (lane == 0)
        *partial = make_float2((share[0].x + share[1].x) + share[2].x, (share[0].y + share[1].y) + share[2].y);
    if (!valid) return;
    for (int q = 1; q <= 2; ++q) {
        const float* __restrict__ p = (const float*)stage[q] + lane;
        s.gx.x += p[0]; s.gx.y += p[64]; s.gx.z += p[128];
        s.ge.x += p[192]; s.ge.y += p[256]; s.ge.z += p[320];
        s.grho += p[384];
    }
    gx2_s[i] = make_float4(s.gx.x, s.gx.y, s.gx.z, 0.f);
    ge_s[i] = make_float4(s.ge.x, s.ge.y, s.ge.z, 0.f);
    grho_s[i] = s.grho;
}

// B3 for the block's tile (as adj_b2_tile): density backwards and the scatter
// of lambda_x, lambda_e of step n (lam_e_out may be null).
__device__ __forceinline__ void adj_b3_tile(int i, bool valid, const uint32_t* __restrict__ idx,
                                            const float4* __restrict__ pos_s, const float* __restrict__ grho_s,
                                            const float4* __restrict__ lxp_s, const float4* __restrict__ gx2_s,
                                            const float4* __restrict__ ge_s, const AdjRows& rows,
                                            const rtps_sph_params& sp, float4* __restrict__ lam_x_out,
                                            float4* __restrict__ lam_e_out) {
    __shared__ float4 stage[3][kAdjB3Slice];
    const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
    float3 gx = make_float3(0, 0, 0);
    if (valid) {
        const float h = sp.smoothing_distance, h2 = h * h;
        const float c6 = sp.wpoly6_coef * sp.mass * -6.f;
        const float gri = grho_s[i];
        float* __restrict__ sgr = (float*)(stage[w] + kAdjB3StageCap);
        adj_plane<kAdjB3StageCap>(
            i, w - 1, rows, pos_s[i], h2, pos_s, stage[w], [&](uint32_t t, uint32_t j) { sgr[t] = grho_s[j]; },
            [&](auto staged, uint32_t o, const float3 r, float r2) {
                float grj;
                if constexpr (decltype(staged)::value) grj = sgr[o];
                else grj = grho_s[o];
                const float t = h2 - r2;
                const float k = c6 * t * t * (gri + grj);
                gx.x += k * r.x;
                gx.y += k * r.y;
                gx.z += k * r.z;
            });
    }
    __builtin_amdgcn_wave_barrier();   // the last row's reads before the slice's reuse
    if (w > 0) {
        float* __restrict__ p = (float*)stage[w] + lane;
        p[0] = gx.x; p[64] = gx.y; p[128] = gx.z;
    }
    __syncthreads();
    if (w > 0 || !valid) return;
    for (int q = 1; q <= 2; ++q) {
        const float* __restrict__ p = (const float*)stage[q] + lane;
        gx.x += p[0]; gx.y += p[64]; gx.z += p[128];
    }
    const float4 lp = lxp_s[i], g2 = gx2_s[i];
    const uint32_t o = idx[i];
    lam_x_out[o] = make_float4(lp.x + g2.x + gx.x, lp.y + g2.y + gx.y, lp.z + g2.z + gx.z, 0.f);
    if (lam_e_out) lam_e_out[o] = ge_s[i];
}

// Sum of the n tile shares at partial in FP64, fixed order, by one block of
// 256 threads, into out[0], out[1].
__device__ __forceinline__ void adj_reduce_body(const float2* __restrict__ partial, int n,
                                                double* __restrict__ out) {
    __shared__ double s0[256], s1[256];
    double a = 0.0, b = 0.0;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        a += (double)partial[k].x;
        b += (double)partial[k].y;
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = b;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s0[threadIdx.x] += s0[threadIdx.x + w];
            s1[threadIdx.x] += s1[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s0[0];
        out[1] = s1[0];
    }
}

}  // namespace rtps
