// rtps_badj: forward and adjoint of many independent scenes at once (no
// reference counterpart).  Every scene runs the step of the single-system
// adjoint handle (adjoint_system.cpp) with its own settings, viscosity and
// gas constant; each stage is one launch for the whole batch (segmented keys
// (scene << 24) | (cell << 4) | xq as in the batched system), and the
// backward pass gives dL/dv0, dL/dx0 per particle and dL/dmu_s, dL/dK_s per
// scene.  Scene s holds exactly the max_num_particles of its settings, in
// slots [off_s, off_s + n_s) of the concatenated arrays.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "adjoint.h"
#include "batch_adjoint.h"
#include "batch_layout.h"
#include "batch_types.h"
#include "rtps_internal.h"
#include "sph_device.h"

using namespace rtps;

namespace {

struct BRecord {   // one forward step's sorted state of the whole batch
    uint32_t *idx = nullptr, *rows = nullptr;   // rows: the neighbour rows its density kernel recorded
    float4 *pos_s = nullptr, *vel_s = nullptr, *ve_s = nullptr, *force_s = nullptr;
};

struct BState {   // in original order
    float4 *pos = nullptr, *vel = nullptr, *ve = nullptr;
};

// Whether float4 kernels may use a caller's array (else it is copied).
bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

struct rtps_badj {
    BatchLayout L;
    int S = 0, T = 0, C = 0, ck = 20, steps = 0, n_items = 0, n_items64 = 0;
    std::vector<void*> allocs;
    SceneDev* scenes = nullptr;
    int *d_num = nullptr, *item_first = nullptr, *left_grid = nullptr;
    uint16_t* sid = nullptr;
    BatchItem *items = nullptr, *items64 = nullptr;
    BState slot[2];                    // states between checkpoints
    std::vector<BState> ck_state;      // checkpoints
    std::vector<BRecord> rec;          // records of one segment's steps (or of as many as fit)
    uint32_t *keys = nullptr, *start = nullptr, *end = nullptr, *sub = nullptr;   // of the step at hand
    bool by_cell = false;   // sorted by cell_sort.hip's counting sort
    void* sort_tmp = nullptr;
    float4 *lam_x[2] = {}, *lam_v[2] = {}, *lam_e[2] = {};
    float4 *ga = nullptr, *gX = nullptr, *lxp = nullptr, *gx2 = nullptr, *ge = nullptr;
    float* grho = nullptr;
    float2* partial = nullptr;         // B2's shares of dL/dmu, dL/dK: [record][64-slot item]
    double* sums = nullptr;            // and their sums: [step][scene]
    std::vector<double> sums_h;
    bool have_forward = false;
    int rec_lo = 0, rec_hi = 0;   // rec[0..] hold the steps rec_lo..rec_hi-1 of the last forward run

    ~rtps_badj() {
        (void)hipDeviceSynchronize();
        for (void* p : allocs) (void)hipFree(p);
    }
    template <typename T>
    hipError_t alloc(T** p, size_t count) {
        hipError_t e = hipMalloc((void**)p, count * sizeof(T) + 16);
        if (e == hipSuccess) allocs.push_back(*p);
        return e;
    }
};

namespace {

#define RTPS_TRY_HIP(expr)                                 \
    do {                                                   \
        hipError_t e_ = (expr);                            \
        if (e_ != hipSuccess) return hip_error(e_, #expr); \
    } while (0)

// Records for `want` steps or as many as adjoint_records allows, and half as many
// while the device has no room.
hipError_t alloc_records(rtps_badj* a, int want) {
    const size_t N = (size_t)a->T;
    const RecordLayout L(N, 27 * N);
    want = adjoint_records(want, L.bytes);
    for (;; want = (want + 1) / 2) {
        const size_t before = a->allocs.size();
        a->rec.assign((size_t)want, BRecord());
        hipError_t e = hipSuccess;
        for (BRecord& r : a->rec) {
            char* p = nullptr;
            e = a->alloc(&p, L.bytes);
            if (e != hipSuccess) break;
            r.idx = (uint32_t*)(p + L.idx);
            r.rows = (uint32_t*)(p + L.rows);
            r.pos_s = (float4*)(p + L.pos);
            r.vel_s = (float4*)(p + L.vel);
            r.ve_s = (float4*)(p + L.ve);
            r.force_s = (float4*)(p + L.force);
        }
        if (e == hipSuccess || e != hipErrorOutOfMemory || want == 1) return e;
        (void)hipGetLastError();
        for (size_t k = before; k < a->allocs.size(); ++k) (void)hipFree(a->allocs[k]);
        a->allocs.resize(before);
    }
}

// One forward step of every scene from state `in` to `out`, its sorted state
// left in r; force: also the SPH force, which only the adjoint reads.
int forward_step(rtps_badj* a, const BState& in, const BState& out, BRecord& r, bool force, hipStream_t st) {
    const int T = a->T;
    uint32_t* ks = a->keys;
    if (a->by_cell) {
        RTPS_TRY_HIP(cell_sort_place_b(T, a->sid, a->scenes, a->d_num, in.pos, a->C, a->keys, r.idx, a->start, a->end,
                                       a->sort_tmp, st));
        RTPS_TRY_HIP(cell_sort_finish_b(T, a->sid, a->scenes, a->d_num, a->C, a->start, a->end, a->sub, a->keys,
                                        r.idx, in.pos, in.vel, in.ve, r.pos_s, r.vel_s, r.ve_s, a->sort_tmp, st));
    } else {
        RTPS_TRY_HIP(launch_hash_b(T, a->sid, a->scenes, a->d_num, in.pos, a->keys, r.idx, a->start, a->C, st));
        uint32_t* is;
        RTPS_TRY_HIP(sort_pairs_passes(T, a->L.shifts, a->L.widths, a->L.npasses, a->keys, r.idx, a->sort_tmp, st, &ks,
                                       &is));
        if (is != r.idx) RTPS_TRY_HIP(hipMemcpyAsync(r.idx, is, (size_t)T * 4, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(launch_cellindices_b(T, ks, a->scenes, a->start, a->end, st, a->sub));
        RTPS_TRY_HIP(launch_permute(T, nullptr, r.idx, in.pos, in.vel, in.ve, r.pos_s, r.vel_s, r.ve_s, st));
    }
    for (int mode : {kPairsDensity, kPairsForceStep})
        RTPS_TRY_HIP(launch_pairs_split_b(mode, a->n_items64, a->items64, a->scenes, r.pos_s, a->start, a->end, ks,
                                          r.ve_s, r.vel_s, r.idx, out.pos, out.vel, out.ve,
                                          force ? r.force_s : nullptr, a->left_grid, a->sub, r.rows, (uint32_t)T,
                                          st));
    return RTPS_OK;
}

}  // namespace

extern "C" {

int rtps_badj_create(int num_scenes, const int* n_settings, const char* const* keys, const char* const* vals,
                     int checkpoint_every, int max_steps, rtps_badj** out) {
    try {
        if (!out || checkpoint_every <= 0 || max_steps <= 0)
            return set_error(RTPS_ERR_ARG, "rtps_badj_create: bad arguments");
        *out = nullptr;
        std::unique_ptr<rtps_badj> a(new rtps_badj());
        int rc = build_batch_layout(num_scenes, n_settings, keys, vals, a->L);
        if (rc) return rc;
        for (int s = 0; s < num_scenes; ++s) {
            const SceneDev& d = a->L.scenes[s];
            if (d.sp.simulation_scale != 1.0f)
                return set_error(RTPS_ERR_ARG, "scene " + std::to_string(s) + ": the adjoint supports "
                                                                               "simulation_scale = 1 only");
            for (float x : a->L.settings[s].GetSettingAs<std::vector<float>>("gravity_alphas"))
                if (x != 0.f)
                    return set_error(RTPS_ERR_ARG, "scene " + std::to_string(s) +
                                                       ": the adjoint does not support point gravity sources");
        }
        a->S = num_scenes;
        a->T = (int)a->L.T;
        a->C = (int)a->L.total_cells;
        a->ck = checkpoint_every;
        a->n_items = (int)a->L.items.size();
        a->n_items64 = (int)a->L.items64.size();
        const size_t N = (size_t)a->T, C = (size_t)a->C;
        RTPS_TRY_HIP(a->alloc(&a->scenes, (size_t)num_scenes));
        RTPS_TRY_HIP(a->alloc(&a->d_num, (size_t)num_scenes));
        RTPS_TRY_HIP(a->alloc(&a->item_first, (size_t)num_scenes + 1));
        RTPS_TRY_HIP(a->alloc(&a->left_grid, 1));
        RTPS_TRY_HIP(a->alloc(&a->sid, N));
        RTPS_TRY_HIP(a->alloc(&a->items, (size_t)a->n_items));
        RTPS_TRY_HIP(a->alloc(&a->items64, (size_t)a->n_items64));
        const int nck = (max_steps + checkpoint_every - 1) / checkpoint_every;
        a->ck_state.resize(nck);
        auto alloc_state = [&](BState& s) {
            hipError_t e = a->alloc(&s.pos, N);
            if (e == hipSuccess) e = a->alloc(&s.vel, N);
            return e == hipSuccess ? a->alloc(&s.ve, N) : e;
        };
        for (int s = 0; s < 2; ++s) {
            RTPS_TRY_HIP(alloc_state(a->slot[s]));
            RTPS_TRY_HIP(a->alloc(&a->lam_x[s], N));
            RTPS_TRY_HIP(a->alloc(&a->lam_v[s], N));
            RTPS_TRY_HIP(a->alloc(&a->lam_e[s], N));
        }
        for (BState& s : a->ck_state) RTPS_TRY_HIP(alloc_state(s));
        RTPS_TRY_HIP(a->alloc(&a->keys, N));
        RTPS_TRY_HIP(a->alloc(&a->start, C));
        RTPS_TRY_HIP(a->alloc(&a->end, C));
        if (C * kSubCells * sizeof(uint32_t) <= ((size_t)2 << 30))   // as the batched system's
            RTPS_TRY_HIP(a->alloc(&a->sub, C * kSubCells));
        a->by_cell = cell_sort_fits_b((long)N, (long)C);
        RTPS_TRY_HIP(a->alloc((char**)&a->sort_tmp, a->by_cell ? cell_sort_temp_bytes((int)N, (int)C - 1)
                                                               : sort_temp_bytes((int)N, 32)));
        RTPS_TRY_HIP(a->alloc(&a->ga, N));
        RTPS_TRY_HIP(a->alloc(&a->gX, N));
        RTPS_TRY_HIP(a->alloc(&a->lxp, N));
        RTPS_TRY_HIP(a->alloc(&a->gx2, N));
        RTPS_TRY_HIP(a->alloc(&a->ge, N));
        RTPS_TRY_HIP(a->alloc(&a->grho, N));
        const size_t nsums = 2 * (size_t)num_scenes * nck * checkpoint_every;
        RTPS_TRY_HIP(a->alloc(&a->sums, nsums));
        a->sums_h.resize(nsums);
        RTPS_TRY_HIP(alloc_records(a.get(), std::min(checkpoint_every, max_steps)));
        RTPS_TRY_HIP(a->alloc(&a->partial, a->rec.size() * (size_t)a->n_items64));
        std::vector<uint16_t> sid(N);
        std::vector<int> counts(num_scenes);
        for (int s = 0; s < num_scenes; ++s) {
            const SceneDev& d = a->L.scenes[s];
            std::fill(sid.begin() + d.off, sid.begin() + d.off + d.cap, (uint16_t)s);
            counts[s] = d.cap;   // every slot holds a particle
        }
        RTPS_TRY_HIP(hipMemcpy(a->sid, sid.data(), N * sizeof(uint16_t), hipMemcpyHostToDevice));
        RTPS_TRY_HIP(hipMemcpy(a->d_num, counts.data(), sizeof(int) * num_scenes, hipMemcpyHostToDevice));
        RTPS_TRY_HIP(hipMemcpy(a->items, a->L.items.data(), sizeof(BatchItem) * a->L.items.size(),
                               hipMemcpyHostToDevice));
        RTPS_TRY_HIP(hipMemcpy(a->items64, a->L.items64.data(), sizeof(BatchItem) * a->L.items64.size(),
                               hipMemcpyHostToDevice));
        RTPS_TRY_HIP(hipMemcpy(a->item_first, a->L.item_first.data(), sizeof(int) * (num_scenes + 1),
                               hipMemcpyHostToDevice));
        RTPS_TRY_HIP(hipMemcpy(a->scenes, a->L.scenes.data(), sizeof(SceneDev) * num_scenes, hipMemcpyHostToDevice));
        RTPS_TRY_HIP(a->by_cell ? cell_sort_clear_temp(a->sort_tmp, (int)C - 1, nullptr)
                                : sort_clear_temp(a->sort_tmp, (int)N, nullptr));
        RTPS_TRY_HIP(launch_fill_u32(a->end, 0u, (long)C, nullptr));
        RTPS_TRY_HIP(hipDeviceSynchronize());
        *out = a.release();
        return RTPS_OK;
    } catch (const std::exception& e) {
        return set_error(RTPS_ERR_ARG, std::string("rtps_badj_create: ") + e.what());
    }
}

int rtps_badj_destroy(rtps_badj* a) {
    delete a;
    return RTPS_OK;
}

int rtps_badj_layout(rtps_badj* a, int* num_scenes, int* total, int* offsets) {
    if (!a) return set_error(RTPS_ERR_ARG, "null handle");
    if (num_scenes) *num_scenes = a->S;
    if (total) *total = a->T;
    if (offsets) {
        for (int s = 0; s < a->S; ++s) offsets[s] = a->L.scenes[s].off;
        offsets[a->S] = a->T;
    }
    return RTPS_OK;
}

int rtps_badj_forward(rtps_badj* a, const rtps_float4* pos0, const rtps_float4* vel0, int nsteps,
                      const float* viscosity, const float* gas_constant, int collision, rtps_float4* pos_T,
                      rtps_float4* vel_T, void* stream) {
    if (!a || !pos0 || !vel0 || !pos_T || !viscosity || !gas_constant || nsteps <= 0 ||
        (size_t)((nsteps + a->ck - 1) / a->ck) > a->ck_state.size())
        return set_error(RTPS_ERR_ARG, "rtps_badj_forward: bad arguments or more steps than the handle holds");
    hipStream_t st = (hipStream_t)stream;
    for (int s = 0; s < a->S; ++s) {
        SceneDev& d = a->L.scenes[s];
        d.sp.viscosity = viscosity[s];
        d.sp.K = gas_constant[s];
        d.collision = collision ? 1 : 0;
    }
    RTPS_TRY_HIP(hipMemcpyAsync(a->scenes, a->L.scenes.data(), sizeof(SceneDev) * a->S, hipMemcpyHostToDevice, st));
    a->steps = nsteps;
    const size_t nb = (size_t)a->T * 16;
    const BState& s0 = a->ck_state[0];
    if (aligned16(pos0) && aligned16(vel0)) {
        RTPS_TRY_HIP(launch_adj_start(a->T, (const float4*)pos0, (const float4*)vel0, s0.pos, s0.vel, s0.ve, st));
    } else {
        RTPS_TRY_HIP(hipMemcpyAsync(s0.pos, pos0, nb, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(hipMemcpyAsync(s0.vel, vel0, nb, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(launch_fill_u32((uint32_t*)s0.ve, 0u, (long)a->T * 4, st));   // veleval starts at zero
    }
    RTPS_TRY_HIP(launch_fill_u32((uint32_t*)a->left_grid, 0u, 1, st));
    // The last segment's steps are recorded on the way: the adjoint starts
    // there, and its replay begins with the segment before.
    const int last_first = (nsteps - 1) / a->ck * a->ck, rec_lo = std::max(last_first, nsteps - (int)a->rec.size());
    a->rec_lo = a->rec_hi = 0;
    for (int n = 0; n < nsteps; ++n) {
        const BState& in = n % a->ck == 0 ? a->ck_state[n / a->ck] : a->slot[n & 1];
        BState out = (n + 1) % a->ck == 0 && n + 1 < nsteps ? a->ck_state[(n + 1) / a->ck] : a->slot[(n + 1) & 1];
        if (n + 1 == nsteps) {   // the last state goes to the caller
            if (aligned16(pos_T)) out.pos = (float4*)pos_T;
            if (vel_T && aligned16(vel_T)) out.vel = (float4*)vel_T;
        }
        int rc = forward_step(a, in, out, a->rec[std::max(n - rec_lo, 0)], n >= rec_lo, st);
        if (rc) return rc;
        if (n + 1 < nsteps) continue;
        if (!aligned16(pos_T)) RTPS_TRY_HIP(hipMemcpyAsync(pos_T, out.pos, nb, hipMemcpyDeviceToDevice, st));
        if (vel_T && !aligned16(vel_T)) RTPS_TRY_HIP(hipMemcpyAsync(vel_T, out.vel, nb, hipMemcpyDeviceToDevice, st));
    }
    int left = 0;
    RTPS_TRY_HIP(hipMemcpyAsync(&left, a->left_grid, sizeof(int), hipMemcpyDeviceToHost, st));
    RTPS_TRY_HIP(hipStreamSynchronize(st));
    a->have_forward = true;
    a->rec_lo = rec_lo;
    a->rec_hi = nsteps;
    if (left) return set_error(RTPS_ERR_STATE, "particles left the grid during the forward run (no deletion path in "
                                               "the adjoint)");
    return RTPS_OK;
}

int rtps_badj_backward(rtps_badj* a, const rtps_float4* dL_dpos_T, const rtps_float4* dL_dvel_T,
                       rtps_float4* dL_dvel0, rtps_float4* dL_dpos0, double* dL_dvisc, double* dL_dgas,
                       void* stream) {
    if (!a || !dL_dpos_T || !dL_dvel0) return set_error(RTPS_ERR_ARG, "rtps_badj_backward: bad arguments");
    if (!a->have_forward) return set_error(RTPS_ERR_STATE, "rtps_badj_backward needs a forward run");
    hipStream_t st = (hipStream_t)stream;
    const size_t nb = (size_t)a->T * 16;
    // the adjoints of the state at hand (original order); lam_e is zero at the end of the run
    const float4 *lx = (const float4*)dL_dpos_T, *lv = (const float4*)dL_dvel_T, *le = nullptr;
    if (!aligned16(lx)) {
        RTPS_TRY_HIP(hipMemcpyAsync(a->lam_x[0], lx, nb, hipMemcpyDeviceToDevice, st));
        lx = a->lam_x[0];
    }
    if (lv && !aligned16(lv)) {
        RTPS_TRY_HIP(hipMemcpyAsync(a->lam_v[0], lv, nb, hipMemcpyDeviceToDevice, st));
        lv = a->lam_v[0];
    }
    const int nck = (a->steps + a->ck - 1) / a->ck, R = (int)a->rec.size();
    const uint32_t T = (uint32_t)a->T;
    int L = 0;   // the adjoints at hand are in the buffers L (or still the caller's)
    for (int c = nck - 1; c >= 0; --c) {
        const int first = c * a->ck, last = std::min(a->steps, first + a->ck);
        for (int hi = last, lo; hi > first; hi = lo) {
            lo = std::max(first, hi - R);
            // replay the segment from its checkpoint, recording the steps lo..hi-1
            // (unless they are the ones recorded last)
            const bool recorded = a->rec_lo == lo && a->rec_hi == hi;
            if (!recorded) a->rec_lo = a->rec_hi = 0;
            for (int s = recorded ? hi : first; s < hi; ++s) {
                const BState& in = s == first ? a->ck_state[c] : a->slot[s & 1];
                int rc = forward_step(a, in, a->slot[(s + 1) & 1], a->rec[s < lo ? 0 : s - lo], s >= lo, st);
                if (rc) return rc;
            }
            a->rec_lo = lo;
            a->rec_hi = hi;
            for (int s = hi - 1; s >= lo; --s) {
                const BRecord& r = a->rec[s - lo];
                float4 *lv_out = a->lam_v[1 - L], *lx_out = a->lam_x[1 - L], *le_out = a->lam_e[1 - L];
                if (s == 0) {   // the initial state's adjoints go to the caller
                    if (aligned16(dL_dvel0)) lv_out = (float4*)dL_dvel0;
                    if (dL_dpos0 && aligned16(dL_dpos0)) lx_out = (float4*)dL_dpos0;
                    le_out = nullptr;
                }
                RTPS_TRY_HIP(launch_badj_b1(a->n_items, a->items, a->scenes, r.idx, r.pos_s, r.vel_s, r.force_s, lx,
                                            lv, le, a->ga, a->gX, lv_out, a->lxp, st));
                RTPS_TRY_HIP(launch_badj_b2(a->n_items64, a->items64, a->scenes, r.pos_s, r.ve_s, a->ga, a->gX,
                                            r.rows, T, a->gx2, a->ge, a->grho,
                                            a->partial + (size_t)(s - lo) * a->n_items64, st));
                RTPS_TRY_HIP(launch_badj_b3(a->n_items64, a->items64, a->scenes, r.idx, r.pos_s, a->grho, a->lxp,
                                            a->gx2, a->ge, r.rows, T, lx_out, le_out, st));
                lx = lx_out;
                lv = lv_out;
                le = le_out;
                L = 1 - L;
            }
            RTPS_TRY_HIP(launch_badj_reduce(hi - lo, a->S, a->item_first, a->n_items64, a->partial,
                                            a->sums + 2 * (size_t)a->S * lo, st));
        }
    }
    if (lv != (const float4*)dL_dvel0) RTPS_TRY_HIP(hipMemcpyAsync(dL_dvel0, lv, nb, hipMemcpyDeviceToDevice, st));
    if (dL_dpos0 && lx != (const float4*)dL_dpos0)
        RTPS_TRY_HIP(hipMemcpyAsync(dL_dpos0, lx, nb, hipMemcpyDeviceToDevice, st));
    RTPS_TRY_HIP(hipMemcpyAsync(a->sums_h.data(), a->sums, 2 * sizeof(double) * (size_t)a->S * a->steps,
                                hipMemcpyDeviceToHost, st));
    RTPS_TRY_HIP(hipStreamSynchronize(st));
    for (int s = 0; s < a->S; ++s) {   // steps from the last, in FP64
        double acc[2] = {0, 0};
        for (int n = a->steps - 1; n >= 0; --n)
            for (int k = 0; k < 2; ++k) acc[k] += a->sums_h[2 * ((size_t)n * a->S + s) + k];
        if (dL_dvisc) dL_dvisc[s] = acc[0];
        if (dL_dgas) dL_dgas[s] = acc[1];
    }
    return RTPS_OK;
}

}  // extern "C"
