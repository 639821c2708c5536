// What follows the pair sums of a step, per sorted particle, in one kernel:
// point sources (gravity.cl), walls (collision_wall.cl), triangles
// (collision_tri.cl), rigid-body particles (SPH::interact) and the integration
// (leapfrog.cl or euler.cl) with the count commit of a deletion step.  The
// step with obstacles, update() / interact() / integrate() and the stage
// operators launch it with the parts they want; the plain step's force kernel
// does its own parts itself.
//
// As kernels of their own these were five passes over the particles, and the
// triangles and boundary particles were searched by every particle: 154 us a
// step for 150,001 particles, 1,152 triangles and a boundary of 1,105
// particles, of which 97 culled triangles and 40 looked boundary particles
// up.  With the triangles listed per cell and the cells near boundary
// particles marked, one kernel takes 30 us.

#include <hip/hip_runtime.h>

#include "obstacles_device.h"
#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

constexpr int kAfBlock = 256;

// OBSTACLES: triangles or rigid-body particles are loaded (their code takes
// registers that the memory-bound rest does not need).
// d_num is not __restrict__: it is read and, by a deletion step's commit,
// written here (as in the force kernel, either count gives the same result).
template <bool OBSTACLES>
__global__ __launch_bounds__(kAfBlock) void k_after_force(int num_host, int* d_num,
                                                          const uint32_t* __restrict__ start, int nb_cells,
                                                          const float4* __restrict__ pos_s,
                                                          const float4* __restrict__ vel_s,
                                                          const float4* __restrict__ ve_s, float4* __restrict__ force,
                                                          const float4* __restrict__ xsph,
                                                          const uint32_t* __restrict__ idx, rtps_sph_params sp,
                                                          AfterForce a, GravitySources gsrc, Grid gs, TriSet tri,
                                                          RigidDev moving, RigidDev fixed, float4* __restrict__ pos_u,
                                                          float4* __restrict__ vel_u, float4* __restrict__ veleval_u,
                                                          const float4* __restrict__ color_s,
                                                          float4* __restrict__ color_u) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int num = d_num ? *d_num : num_host;
    bool deleted = false;
    if (d_num) deleted = effective_num(num, start, nb_cells, num);
    if (a.integrate && deleted && i == 0) *d_num = num;
    if (i >= num) return;
    const float4 p = pos_s[i];
    float4 f = force[i];
    if (a.gravity) gravity_sources(f, p, gsrc, sp.simulation_scale);
    if (a.walls) collision_wall(f, p, vel_s[i], sp, a.bmin, a.bmax);
    if constexpr (OBSTACLES) {
        if (tri.n > 0) {
            const float3 t = tri_forces(p, vel_s[i], tri, sp);
            f.x += t.x;
            f.y += t.y;
            f.z += t.z;
        }
        if (moving.n > 0) rigid_force<true>(f, p, ve_s[i], moving, nb_cells, sp, gs);
        if (fixed.n > 0) rigid_force<false>(f, p, ve_s[i], fixed, nb_cells, sp, gs);
    }
    if (a.store) force[i] = f;
    if (!a.integrate) return;
    const uint32_t o = deleted ? (uint32_t)i : idx[i];
    float4 po, vo;
    if (a.integrate == AfterForce::kEuler) {
        // euler.cl:33-78 leaves veleval alone; on a deletion step the
        // survivors' sorted records become the unsorted ones (call_prep,
        // SPH.cpp:445-457), so veleval and the colours are copied from the
        // sorted arrays there.  The sorted veleval array holds veleval.xyz |
        // density; its copy gets w = 0 (no kernel reads veleval.w).
        euler(p, vel_s[i], f, sp, a.dt, po, vo);
        if (deleted) {
            const float4 e = ve_s[i];
            veleval_u[i] = make_float4(e.x, e.y, e.z, 0.0f);
        }
    } else {   // leapfrog.cl:30-121
        float4 eo;
        leapfrog(p, vel_s[i], f, xsph[i], sp, a.dt, po, vo, eo);
        veleval_u[o] = eo;
    }
    pos_u[o] = po;
    vel_u[o] = vo;
    if (deleted && color_u) color_u[i] = color_s[i];   // leapfrog.cl:107
}

hipError_t launch_after_force(int num, int* d_num, const uint32_t* start, int nb_cells, const float4* pos_s,
                              const float4* vel_s, const float4* ve_s, float4* force, const float4* xsph,
                              const uint32_t* idx, const rtps_sph_params& sp, const AfterForce& a,
                              const GravitySources& gsrc, const Grid& gs, const TriSet* tri, const RigidDev* rigid,
                              float4* pos_u, float4* vel_u, float4* veleval_u, hipStream_t st, const float4* color_s,
                              float4* color_u) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    const TriSet t = tri ? *tri : TriSet{};
    const RigidDev none{}, &moving = rigid ? rigid[0] : none, &fixed = rigid ? rigid[1] : none;
    const bool obstacles = t.n > 0 || moving.n > 0 || fixed.n > 0;
    if (num <= 0 || (!a.gravity && !a.walls && !obstacles && !a.integrate)) return hipSuccess;
    const int blocks = (num + kAfBlock - 1) / kAfBlock;
    if (obstacles)
        k_after_force<true><<<blocks, kAfBlock, 0, st>>>(num, d_num, start, nb_cells, pos_s, vel_s, ve_s, force, xsph,
                                                         idx, sp, a, gsrc, gs, t, moving, fixed, pos_u, vel_u,
                                                         veleval_u, color_s, color_u);
    else
        k_after_force<false><<<blocks, kAfBlock, 0, st>>>(num, d_num, start, nb_cells, pos_s, vel_s, ve_s, force,
                                                          xsph, idx, sp, a, gsrc, gs, t, moving, fixed, pos_u, vel_u,
                                                          veleval_u, color_s, color_u);
    return hipGetLastError();
}

}  // namespace rtps
