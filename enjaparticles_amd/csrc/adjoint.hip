// Single-system launches of the hand-written adjoint of the SPH step (no
// reference counterpart).  The per-particle bodies and the derivation live in
// adjoint_device.h; here each kernel maps thread i to sorted particle i (B1),
// or a block of three waves to 64 sorted particles (B2, B3).
//
// B2 and B3 were bound by latency and by work on rejected candidates: 56 and
// 41 us for 65,536 particles (one wave per SIMD, nine rows each looked up by
// binary search, then tested).  On the rows that the forward step's density
// kernel recorded, a plane per wave, they take 20 and 9 us.

#include <hip/hip_runtime.h>

#include "adjoint.h"
#include "adjoint_device.h"
#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

constexpr int kABlock = 256;

static inline int ablocks(long n) { return (int)((n + kABlock - 1) / kABlock); }

__global__ __launch_bounds__(kABlock) void k_adj_start(int num, const float4* __restrict__ pos,
                                                       const float4* __restrict__ vel, float4* __restrict__ pos_out,
                                                       float4* __restrict__ vel_out, float4* __restrict__ ve_out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    pos_out[i] = pos[i];
    vel_out[i] = vel[i];
    ve_out[i] = make_float4(0.f, 0.f, 0.f, 0.f);   // veleval starts at zero
}

__global__ __launch_bounds__(kABlock) void k_adj_b1(int num, const uint32_t* __restrict__ idx,
                                                    const float4* __restrict__ pos_s,
                                                    const float4* __restrict__ vel_s,
                                                    const float4* __restrict__ force_s, rtps_sph_params sp,
                                                    rtps_float4 bmin, rtps_float4 bmax, int collision, float dt,
                                                    const float4* __restrict__ lam_x, const float4* __restrict__ lam_v,
                                                    const float4* __restrict__ lam_e, float4* __restrict__ ga_s,
                                                    float4* __restrict__ gX_s, float4* __restrict__ lam_v_out,
                                                    float4* __restrict__ lxp_s) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    adj_b1_body(i, idx, pos_s, vel_s, force_s, sp, bmin, bmax, collision, dt, lam_x, lam_v, lam_e, ga_s, gX_s,
                lam_v_out, lxp_s);
}

__global__ __launch_bounds__(kAdjThreads) void k_adj_b2(int num, const float4* __restrict__ pos_s,
                                                        const float4* __restrict__ ve_s,
                                                        const float4* __restrict__ ga_s,
                                                        const float4* __restrict__ gX_s, AdjRows rows,
                                                        rtps_sph_params sp, float4* __restrict__ gx2_s,
                                                        float4* __restrict__ ge_s, float* __restrict__ grho_s,
                                                        float2* __restrict__ partial) {
    const int tile = remap_tile(adj_remap(num), blockIdx.x, gridDim.x), i = tile * 64 + ((int)threadIdx.x & 63);
    adj_b2_tile(i, i < num, pos_s, ve_s, ga_s, gX_s, rows, sp, gx2_s, ge_s, grho_s, partial + tile);
}

__global__ __launch_bounds__(kAdjThreads) void k_adj_b3(int num, const uint32_t* __restrict__ idx,
                                                        const float4* __restrict__ pos_s,
                                                        const float* __restrict__ grho_s,
                                                        const float4* __restrict__ lxp_s,
                                                        const float4* __restrict__ gx2_s,
                                                        const float4* __restrict__ ge_s, AdjRows rows,
                                                        rtps_sph_params sp, float4* __restrict__ lam_x_out,
                                                        float4* __restrict__ lam_e_out) {
    const int i = remap_tile(adj_remap(num), blockIdx.x, gridDim.x) * 64 + ((int)threadIdx.x & 63);
    adj_b3_tile(i, i < num, idx, pos_s, grho_s, lxp_s, gx2_s, ge_s, rows, sp, lam_x_out, lam_e_out);
}

// Block k adds the shares of step k (fixed order).
__global__ void k_adj_reduce(const float2* __restrict__ partial, int n, double* __restrict__ out) {
    adj_reduce_body(partial + (size_t)blockIdx.x * n, n, out + 2 * blockIdx.x);
}

int adjoint_tiles(int num) { return (int)(((long)num + 63) / 64); }

hipError_t launch_adj_start(int num, const float4* pos, const float4* vel, float4* pos_out, float4* vel_out,
                            float4* ve_out, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num <= 0) return hipSuccess;
    k_adj_start<<<ablocks(num), kABlock, 0, st>>>(num, pos, vel, pos_out, vel_out, ve_out);
    return hipGetLastError();
}

hipError_t launch_adj_b1(int num, const uint32_t* idx, const float4* pos_s, const float4* vel_s,
                         const float4* force_s, const rtps_sph_params& sp, const rtps_grid_params& gps, int collision,
                         float dt, const float4* lam_x, const float4* lam_v, const float4* lam_e, float4* ga_s,
                         float4* gX_s, float4* lam_v_out, float4* lxp_s, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num <= 0) return hipSuccess;
    k_adj_b1<<<ablocks(num), kABlock, 0, st>>>(num, idx, pos_s, vel_s, force_s, sp, gps.bnd_min, gps.bnd_max,
                                               collision, dt, lam_x, lam_v, lam_e, ga_s, gX_s, lam_v_out, lxp_s);
    return hipGetLastError();
}

hipError_t launch_adj_b2(int num, const float4* pos_s, const float4* ve_s, const float4* ga_s, const float4* gX_s,
                         const uint32_t* rows, uint32_t stride, const rtps_sph_params& sp, float4* gx2_s,
                         float4* ge_s, float* grho_s, float2* partial, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num <= 0) return hipSuccess;
    if (!rows || stride < (uint32_t)num) return hipErrorInvalidValue;
    k_adj_b2<<<adjoint_tiles(num), kAdjThreads, 0, st>>>(num, pos_s, ve_s, ga_s, gX_s, AdjRows{rows, stride}, sp,
                                                         gx2_s, ge_s, grho_s, partial);
    return hipGetLastError();
}

hipError_t launch_adj_b3(int num, const uint32_t* idx, const float4* pos_s, const float* grho_s, const float4* lxp_s,
                         const float4* gx2_s, const float4* ge_s, const uint32_t* rows, uint32_t stride,
                         const rtps_sph_params& sp, float4* lam_x_out, float4* lam_e_out, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num <= 0) return hipSuccess;
    if (!rows || stride < (uint32_t)num) return hipErrorInvalidValue;
    k_adj_b3<<<adjoint_tiles(num), kAdjThreads, 0, st>>>(num, idx, pos_s, grho_s, lxp_s, gx2_s, ge_s,
                                                         AdjRows{rows, stride}, sp, lam_x_out, lam_e_out);
    return hipGetLastError();
}

hipError_t launch_adj_reduce(int steps, const float2* partial, int n, double* out, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (steps <= 0) return hipSuccess;
    k_adj_reduce<<<steps, 256, 0, st>>>(partial, n, out);
    return hipGetLastError();
}

}  // namespace rtps
