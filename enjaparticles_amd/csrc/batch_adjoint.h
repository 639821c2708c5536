// Launchers of the batched adjoint kernels (batch_adjoint.hip): one block per
// 256-slot work item of the batch layout, or per 64-slot item in B2 and B3.
#pragma once

#include <hip/hip_runtime.h>

#include "batch_types.h"

namespace rtps {

// lam_v and lam_e may be null (zero)
hipError_t launch_badj_b1(int n_items, const BatchItem* items, const SceneDev* scenes, const uint32_t* idx,
                          const float4* pos_s, const float4* vel_s, const float4* force_s, const float4* lam_x,
                          const float4* lam_v, const float4* lam_e, float4* ga_s, float4* gX_s, float4* lam_v_out,
                          float4* lxp_s, hipStream_t st);
// B2 and B3: one block per 64-slot item; rows, stride: the step's recorded
// neighbour rows (T slots per plane); partial: one share per item
hipError_t launch_badj_b2(int n_items64, const BatchItem* items64, const SceneDev* scenes, const float4* pos_s,
                          const float4* ve_s, const float4* ga_s, const float4* gX_s, const uint32_t* rows,
                          uint32_t stride, float4* gx2_s, float4* ge_s, float* grho_s, float2* partial,
                          hipStream_t st);
hipError_t launch_badj_b3(int n_items64, const BatchItem* items64, const SceneDev* scenes, const uint32_t* idx,
                          const float4* pos_s, const float* grho_s, const float4* lxp_s, const float4* gx2_s,
                          const float4* ge_s, const uint32_t* rows, uint32_t stride, float4* lam_x_out,
                          float4* lam_e_out, hipStream_t st);
// out[2 (k num_scenes + s)], [.. + 1] = the sums of scene s's shares of step
// k < steps; item_first: first 64-slot item of every scene, then their number
hipError_t launch_badj_reduce(int steps, int num_scenes, const int* item_first, int n_items64, const float2* partial,
                              double* out, hipStream_t st);

}  // namespace rtps
