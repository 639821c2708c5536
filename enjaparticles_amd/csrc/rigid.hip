// Rigid-body coupling of SPH::interact (rtpslib/system/SPH.cpp:610-663): the
// fluid against the particles of a rigid-body system, found through that
// system's own cell tables on the fluid's grid.
//
// A set of rigid-body particles (positions, and for a moving body velocities
// and masses) is hashed into the fluid's cell grid, sorted and given cell
// start/end tables with the same kernels as the fluid (System::hash_and_sort,
// System.cpp:145-170, on the rigid system).  rigid_force (obstacles_device.h)
// then adds, for each sorted fluid particle i and every set particle j in the 27 cells around i's
// cell with |r| <= 2h (cl_sph_neighbors.h:99-140 iteration, 2h cut-off):
//   norm = (x_j - x_i) / max(|r|, eps), stiff = s0 m
//   F += -stiff (2h - |r|) norm + s1 sqrt(stiff mn) ((vrel . norm) norm)
//   V += w (h - |r|)          (Wvisc_lapl, negative between h and 2h)
// static set  (staticrigidbody_force.cl:45-146): vrel = -e_i, mn = m / 2,
//             w = vrel, force_i += F / m - m mu c V / rho_i^2
// moving set  (rigidbody_force.cl:118-193): vrel = v_j - e_i,
//             mn = m m_j / (m + m_j), w = tangential part of vrel,
//             force_i += F / m + m mu c V / rho_i^2
// with e_i the fluid particle's veleval and c = wvisc_dd_coef.

#include <hip/hip_runtime.h>

#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

namespace {
constexpr int kRBlock = 256;
inline int rblocks(long n) { return (int)((n + kRBlock - 1) / kRBlock); }
}  // namespace

__global__ __launch_bounds__(kRBlock) void k_rigid_gather(int n, const uint32_t* __restrict__ idx,
                                                          const float4* __restrict__ pu,
                                                          const float4* __restrict__ vu,
                                                          const float* __restrict__ mu, float4* __restrict__ ps,
                                                          float4* __restrict__ vs, float* __restrict__ ms) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t s = idx[i];
    ps[i] = pu[s];
    if (vs) vs[i] = vu[s];
    if (ms) ms[i] = mu[s];
}

// Marks every cell one of whose 27 cells (linear hashes, as the force's own
// loop forms them) holds one of the n sorted particles.
__global__ __launch_bounds__(kRBlock) void k_rigid_near(int n, const uint32_t* __restrict__ keys, int nb_cells, int rx,
                                                        int ry, uint8_t* __restrict__ near) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || (i > 0 && keys[i - 1] == keys[i])) return;
    const int h = (int)keys[i];
    if (h >= nb_cells) return;
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                const long t = (long)h - (((long)dz * ry + dy) * rx + dx);
                if (t >= 0 && t < nb_cells) near[t] = 1;
            }
}

hipError_t rigid_prepare(int n, const float4* pos_u, const float4* vel_u, const float* mass_u, RigidDev& r,
                         const Grid& g, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    const int bits = sort_key_bits(g.nb_cells);
    const uint32_t pad = bits >= 32 ? 0xFFFFFFFFu : ((1u << bits) - 1u);
    hipError_t e = launch_hash(n, nullptr, n, pad, pos_u, r.keys, r.idx, g, r.start, g.nb_cells + 1, 0, st);
    if (e != hipSuccess) return e;
    uint32_t *ks = r.keys, *is = r.idx;
    e = sort_pairs_pingpong(n, bits, r.keys, r.idx, r.sort_tmp, st, &ks, &is);
    if (e != hipSuccess) return e;
    e = launch_cellindices(n, nullptr, ks, g.nb_cells, r.start, r.end, 0, st);
    if (e != hipSuccess) return e;
    if (n > 0)
        k_rigid_gather<<<rblocks(n), kRBlock, 0, st>>>(n, is, pos_u, vel_u, mass_u, r.pos, vel_u ? r.vel : nullptr,
                                                       mass_u ? r.mass : nullptr);
    if (r.near) {
        e = launch_fill_u32((uint32_t*)r.near, 0u, ((long)g.nb_cells + 3) / 4, st);
        if (e != hipSuccess) return e;
        if (n > 0) k_rigid_near<<<rblocks(n), kRBlock, 0, st>>>(n, ks, g.nb_cells, g.irx, g.iry, r.near);
    }
    return hipGetLastError();
}

}  // namespace rtps
