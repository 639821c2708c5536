// Launchers of the adjoint kernels (adjoint.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "sph_device.h"

namespace rtps {

// Tile order (remap_tile) of the recorded steps and of B2 and B3: one contiguous
// eighth of the particles per XCD, whose L2 then serves its tiles' rows; for larger
// runs chunks of 16 tiles in turn, as a pool's dense bottom would make one XCD's
// eighth the slowest (force at 150,001 settled particles: 52 us in plain order and in chunks, 66 in
// eighths; 43 and 42 at 65,536).  A gradient over 20 steps of 65,536 particles
// takes 2.41 ms in plain order, 2.31 in eighths.
__host__ __device__ inline int adj_remap(int num) { return num <= 1 << 16 ? 1 : 16; }
// How many of the `want` step records of a segment, `bytes` each, a handle keeps:
// what half of the device's free memory holds.  The rest is the caller's (a
// segment is then replayed once per part, and a record of 177 bytes a particle
// would otherwise leave 4 of 286 GiB: 4,194,304 particles, segments of 400 steps).
int adjoint_records(int want, size_t bytes);
// The parts of a record of n particles in one allocation (the device gives out
// whole 2 MiB: six of their own took 34 MiB instead of 24 at 131,072 particles).
struct RecordLayout {
    size_t idx, rows, pos, vel, ve, force, bytes;
    RecordLayout(size_t n, size_t row_words) {
        size_t at = 0;
        auto part = [&at](size_t size) {
            const size_t o = at;
            at += (size + 255) & ~(size_t)255;
            return o;
        };
        idx = part(4 * n);
        rows = part(4 * row_words);
        pos = part(16 * n);
        vel = part(16 * n);
        ve = part(16 * n);
        force = part(16 * n);
        bytes = at;
    }
};
int adjoint_tiles(int num);   // tiles of B2 (shares of dL/dmu, dL/dK it writes)
// A state's copy at the start of a run: pos and vel copied, veleval zero.
hipError_t launch_adj_start(int num, const float4* pos, const float4* vel, float4* pos_out, float4* vel_out,
                            float4* ve_out, hipStream_t st);
// lam_v and lam_e may be null (zero)
hipError_t launch_adj_b1(int num, const uint32_t* idx, const float4* pos_s, const float4* vel_s,
                         const float4* force_s, const rtps_sph_params& sp, const rtps_grid_params& gps, int collision,
                         float dt, const float4* lam_x, const float4* lam_v, const float4* lam_e, float4* ga_s,
                         float4* gX_s, float4* lam_v_out, float4* lxp_s, hipStream_t st);
// rows, stride: the step's recorded neighbour rows (Win::rows)
hipError_t launch_adj_b2(int num, const float4* pos_s, const float4* ve_s, const float4* ga_s, const float4* gX_s,
                         const uint32_t* rows, uint32_t stride, const rtps_sph_params& sp, float4* gx2_s,
                         float4* ge_s, float* grho_s, float2* partial, hipStream_t st);
// lam_e_out may be null
hipError_t launch_adj_b3(int num, const uint32_t* idx, const float4* pos_s, const float* grho_s, const float4* lxp_s,
                         const float4* gx2_s, const float4* ge_s, const uint32_t* rows, uint32_t stride,
                         const rtps_sph_params& sp, float4* lam_x_out, float4* lam_e_out, hipStream_t st);
// out[2 k], out[2 k + 1] = the sums of the n shares of step k < steps
hipError_t launch_adj_reduce(int steps, const float2* partial, int n, double* out, hipStream_t st);

}  // namespace rtps
