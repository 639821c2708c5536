// Batched adjoint launches (no reference counterpart): the adjoint bodies of
// adjoint_device.h run over every scene of a batch at once.  One block per
// work item (a 256-slot tile of one scene; in B2 and B3 a 64-slot tile, one
// plane of the neighbourhood per wave), so the scene's parameters are uniform
// per block, and the dL/dmu, dL/dK share of B2's block b belongs to the scene
// of item b; k_badj_reduce then adds each scene's items in a fixed order
// (FP64), one block per scene and step.  Items tile each scene from its first
// slot, exactly as the single-system launches tile a system from sorted
// index 0, so every scene gets the single system's block partition.

#include <hip/hip_runtime.h>

#include "adjoint_device.h"
#include "batch_adjoint.h"
#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

constexpr int kBABlock = 256;

struct ItemCtx {
    int s, i;
    bool valid;
};

__device__ __forceinline__ ItemCtx item_ctx(const BatchItem* __restrict__ items) {
    const BatchItem it = items[xcd_tile(blockIdx.x, gridDim.x)];
    ItemCtx c;
    c.s = __builtin_amdgcn_readfirstlane(it.scene);
    c.i = it.first + (int)threadIdx.x;
    c.valid = (int)threadIdx.x < it.count;
    return c;
}

__global__ __launch_bounds__(kBABlock) void k_badj_b1(const BatchItem* __restrict__ items,
                                                      const SceneDev* __restrict__ scenes,
                                                      const uint32_t* __restrict__ idx,
                                                      const float4* __restrict__ pos_s,
                                                      const float4* __restrict__ vel_s,
                                                      const float4* __restrict__ force_s,
                                                      const float4* __restrict__ lam_x,
                                                      const float4* __restrict__ lam_v,
                                                      const float4* __restrict__ lam_e, float4* __restrict__ ga_s,
                                                      float4* __restrict__ gX_s, float4* __restrict__ lam_v_out,
                                                      float4* __restrict__ lxp_s) {
    const ItemCtx c = item_ctx(items);
    if (!c.valid) return;
    const SceneDev& S = scenes[c.s];
    adj_b1_body(c.i, idx, pos_s, vel_s, force_s, S.sp, S.bmin, S.bmax, S.collision, S.dt, lam_x, lam_v, lam_e, ga_s,
                gX_s, lam_v_out, lxp_s);
}

// The 64-slot item of a block of B2 or B3: slot of the calling lane.
__device__ __forceinline__ ItemCtx item64_ctx(const BatchItem* __restrict__ items) {
    const BatchItem it = items[xcd_tile(blockIdx.x, gridDim.x)];
    const int lane = (int)threadIdx.x & 63;
    return ItemCtx{__builtin_amdgcn_readfirstlane(it.scene), it.first + lane, lane < it.count};
}

__global__ __launch_bounds__(kAdjThreads) void k_badj_b2(const BatchItem* __restrict__ items,
                                                         const SceneDev* __restrict__ scenes,
                                                         const float4* __restrict__ pos_s,
                                                         const float4* __restrict__ ve_s,
                                                         const float4* __restrict__ ga_s,
                                                         const float4* __restrict__ gX_s, AdjRows rows,
                                                         float4* __restrict__ gx2_s, float4* __restrict__ ge_s,
                                                         float* __restrict__ grho_s, float2* __restrict__ partial) {
    const ItemCtx c = item64_ctx(items);
    adj_b2_tile(c.i, c.valid, pos_s, ve_s, ga_s, gX_s, rows, scenes[c.s].sp, gx2_s, ge_s, grho_s,
                partial + xcd_tile(blockIdx.x, gridDim.x));
}

__global__ __launch_bounds__(kAdjThreads) void k_badj_b3(const BatchItem* __restrict__ items,
                                                         const SceneDev* __restrict__ scenes,
                                                         const uint32_t* __restrict__ idx,
                                                         const float4* __restrict__ pos_s,
                                                         const float* __restrict__ grho_s,
                                                         const float4* __restrict__ lxp_s,
                                                         const float4* __restrict__ gx2_s,
                                                         const float4* __restrict__ ge_s, AdjRows rows,
                                                         float4* __restrict__ lam_x_out,
                                                         float4* __restrict__ lam_e_out) {
    const ItemCtx c = item64_ctx(items);
    adj_b3_tile(c.i, c.valid, idx, pos_s, grho_s, lxp_s, gx2_s, ge_s, rows, scenes[c.s].sp, lam_x_out, lam_e_out);
}

// Block (s, k) adds the shares of scene s's items in step k.
__global__ void k_badj_reduce(const int* __restrict__ item_first, int n_items64, const float2* __restrict__ partial,
                              double* __restrict__ out) {
    const int s = blockIdx.x, f = item_first[s];
    adj_reduce_body(partial + (size_t)blockIdx.y * n_items64 + f, item_first[s + 1] - f,
                    out + 2 * ((size_t)blockIdx.y * gridDim.x + s));
}

hipError_t launch_badj_b1(int n_items, const BatchItem* items, const SceneDev* scenes, const uint32_t* idx,
                          const float4* pos_s, const float4* vel_s, const float4* force_s, const float4* lam_x,
                          const float4* lam_v, const float4* lam_e, float4* ga_s, float4* gX_s, float4* lam_v_out,
                          float4* lxp_s, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (n_items <= 0) return hipSuccess;
    k_badj_b1<<<n_items, kBABlock, 0, st>>>(items, scenes, idx, pos_s, vel_s, force_s, lam_x, lam_v, lam_e, ga_s,
                                            gX_s, lam_v_out, lxp_s);
    return hipGetLastError();
}

hipError_t launch_badj_b2(int n_items64, const BatchItem* items64, const SceneDev* scenes, const float4* pos_s,
                          const float4* ve_s, const float4* ga_s, const float4* gX_s, const uint32_t* rows,
                          uint32_t stride, float4* gx2_s, float4* ge_s, float* grho_s, float2* partial,
                          hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (n_items64 <= 0) return hipSuccess;
    if (!rows || stride == 0) return hipErrorInvalidValue;
    k_badj_b2<<<n_items64, kAdjThreads, 0, st>>>(items64, scenes, pos_s, ve_s, ga_s, gX_s, AdjRows{rows, stride},
                                                 gx2_s, ge_s, grho_s, partial);
    return hipGetLastError();
}

hipError_t launch_badj_b3(int n_items64, const BatchItem* items64, const SceneDev* scenes, const uint32_t* idx,
                          const float4* pos_s, const float* grho_s, const float4* lxp_s, const float4* gx2_s,
                          const float4* ge_s, const uint32_t* rows, uint32_t stride, float4* lam_x_out,
                          float4* lam_e_out, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (n_items64 <= 0) return hipSuccess;
    if (!rows || stride == 0) return hipErrorInvalidValue;
    k_badj_b3<<<n_items64, kAdjThreads, 0, st>>>(items64, scenes, idx, pos_s, grho_s, lxp_s, gx2_s, ge_s,
                                                 AdjRows{rows, stride}, lam_x_out, lam_e_out);
    return hipGetLastError();
}

hipError_t launch_badj_reduce(int steps, int num_scenes, const int* item_first, int n_items64, const float2* partial,
                              double* out, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (num_scenes <= 0 || steps <= 0) return hipSuccess;
    k_badj_reduce<<<dim3(num_scenes, steps), 256, 0, st>>>(item_first, n_items64, partial, out);
    return hipGetLastError();
}

}  // namespace rtps
