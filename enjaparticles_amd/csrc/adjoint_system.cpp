// rtps_adj: forward SPH simulation with checkpoints and its hand-written
// adjoint (no reference counterpart).
//
// forward(pos0, vel0, T steps, mu, K) runs the plain system's step kernels
// (sort, cells + permute, density, force + walls + leapfrog) from the
// given state (veleval starts at zero, SPH.cpp:491-492) and keeps the state
// every `checkpoint_every` steps.  backward(dL/dx_T, dL/dv_T) walks the
// segments from the last: it replays a segment from its checkpoint, keeping
// every step's sorted records (idx, sorted pos/vel/veleval + density, SPH
// force and the neighbour rows the density kernel recorded), then runs the
// adjoint kernels B1-B3 (adjoint.hip) backwards through the segment.  The
// neighbour structure of each step is the one of the forward step (held
// fixed).  Gradients: dL/dv0, dL/dx0 and dL/dmu, dL/dK (accumulated in FP64).
// States are written where they are needed next (a checkpoint, the caller's
// result), so no step copies them.
//
// Where a segment's records would take more than half of the device's free
// memory, fewer are kept (`rec`) and a segment is replayed once per part of it.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "adjoint.h"
#include "rtps_internal.h"
#include "sph_device.h"

using namespace rtps;

namespace {

struct Record {   // one forward step's sorted state
    uint32_t *idx = nullptr, *rows = nullptr;
    float4 *pos_s = nullptr, *vel_s = nullptr, *ve_s = nullptr, *force_s = nullptr;
};

struct State {   // in original order
    float4 *pos = nullptr, *vel = nullptr, *ve = nullptr;
};

// Whether float4 kernels may use a caller's array (else it is copied).
bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

namespace rtps {

int adjoint_records(int want, size_t bytes) {
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) {
        (void)hipGetLastError();
        return want;
    }
    bytes = (bytes + (2 << 20) - 1) >> 21 << 21;
    return std::max(1, (int)std::min((size_t)want, free / 2 / bytes));
}

}  // namespace rtps

struct rtps_adj {
    RTPSSettings settings;
    rtps_sph_params sp{};
    rtps_grid_params gp{}, gps{};
    Grid g{}, gs{};
    float dt = 0.f;
    int N = 0, nb_cells = 0, key_bits = 0, ck = 20, T = 0, collision = 1;
    uint32_t pad_key = 0;
    std::vector<void*> allocs;
    State slot[2];                    // states between checkpoints
    std::vector<State> ck_state;      // checkpoints
    std::vector<Record> rec;          // per-step records of one segment (or of as many steps as fit)
    uint32_t *keys = nullptr, *start = nullptr, *end = nullptr, *sub = nullptr;   // of the step at hand
    void* sort_tmp = nullptr;
    // adjoint temporaries
    float4 *lam_x[2] = {}, *lam_v[2] = {}, *lam_e[2] = {};
    float4 *ga = nullptr, *gX = nullptr, *lxp = nullptr, *gx2 = nullptr, *ge = nullptr;
    float* grho = nullptr;
    float2* partial = nullptr;        // B2's shares of dL/dmu, dL/dK: [record][tile]
    double* sums = nullptr;           // and their sums per step
    std::vector<double> sums_h;
    int* left_grid = nullptr;
    bool have_forward = false;
    int rec_lo = 0, rec_hi = 0;   // rec[0..] hold the steps rec_lo..rec_hi-1 of the last forward run

    ~rtps_adj() {
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
hipError_t alloc_records(rtps_adj* a, int want) {
    const size_t N = (size_t)a->N;
    const RecordLayout L(N, 27 * N + 18 * ((N + 63) / 64));
    want = adjoint_records(want, L.bytes);
    for (;; want = (want + 1) / 2) {
        const size_t before = a->allocs.size();
        a->rec.assign((size_t)want, Record());
        hipError_t e = hipSuccess;
        for (Record& r : a->rec) {
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

// One forward step from state `in` to state `out`, its sorted state left in r;
// force: also the SPH force, which only the adjoint reads.
int forward_step(rtps_adj* a, const State& in, const State& out, Record& r, bool force, hipStream_t st) {
    const int n = a->N;
    const uint32_t* keys = a->keys;
    if (cell_sort_fits(n, a->nb_cells)) {
        RTPS_TRY_HIP(cell_sort_place(n, n, nullptr, in.pos, a->g, a->pad_key, a->keys, r.idx, a->start, a->end, a->sort_tmp, st));
        RTPS_TRY_HIP(cell_sort_finish(n, n, nullptr, a->pad_key, a->g, a->start, a->end, a->sub, a->keys, r.idx,
                                      in.pos, in.vel, in.ve, r.pos_s, r.vel_s, r.ve_s, a->sort_tmp, st, nullptr,
                                      nullptr, a->left_grid));
    } else {
        uint32_t *ks = a->keys, *is = r.idx;
        if (bucket_sort_fits(n, a->key_bits))
            RTPS_TRY_HIP(hash_bucket_sort(n, a->key_bits, in.pos, n, nullptr, a->pad_key, a->g, kSubBits, a->start,
                                          a->nb_cells + 1, a->keys, r.idx, a->sort_tmp, st));
        else
            RTPS_TRY_HIP(hash_sort_pairs(n, a->key_bits, in.pos, n, nullptr, a->pad_key, a->g, kSubBits, a->start,
                                         a->nb_cells + 1, a->keys, r.idx, a->sort_tmp, st, &ks, &is));
        if (is != r.idx) RTPS_TRY_HIP(hipMemcpyAsync(r.idx, is, (size_t)n * 4, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(launch_cells_permute(n, nullptr, ks, a->nb_cells, a->start, a->end, kSubBits, a->sub, r.idx,
                                          in.pos, in.vel, in.ve, r.pos_s, r.vel_s, r.ve_s, st, nullptr, nullptr,
                                          a->left_grid));
        keys = ks;
    }
    // force loop 5 on recorded rows, which the adjoint reads as well
    Win w{keys, a->gps.grid_res.x, a->gps.grid_res.y, a->gps.grid_res.z, adj_remap(n), 0, 5};
    w.sub = a->sub;
    w.rows = r.rows;
    w.rows_stride = (uint32_t)n;
    w.rows_share = rows_share_of(a->sp);
    w.split = Win::kAlways;
    RTPS_TRY_HIP(launch_density(n, nullptr, r.pos_s, a->start, a->end, a->sp, a->gs, w, nullptr, r.ve_s, st));
    const GravitySources none{};
    RTPS_TRY_HIP(launch_force_fused(n, nullptr, r.pos_s, r.ve_s, a->start, a->end, a->sp, a->gs, w,
                                    force ? r.force_s : nullptr, nullptr, r.vel_s, r.idx, none, a->collision, a->gps,
                                    a->dt, out.pos, out.vel, out.ve, st));
    return RTPS_OK;
}

}  // namespace

extern "C" {

int rtps_adj_create(const char* const* keys, const char* const* vals, int n, int max_particles,
                    int checkpoint_every, int max_steps, rtps_adj** out) {
    try {
        if (!out || n < 0 || max_particles <= 0 || checkpoint_every <= 0 || max_steps <= 0)
            return set_error(RTPS_ERR_ARG, "rtps_adj_create: bad arguments");
        *out = nullptr;
        std::unique_ptr<rtps_adj> a(new rtps_adj());
        for (int i = 0; i < n; ++i) {
            if (!keys[i] || !vals[i]) return set_error(RTPS_ERR_ARG, "null key or value");
            a->settings.SetSetting<std::string>(keys[i], vals[i]);
        }
        derive_params(a->settings, a->sp, a->gp, a->gps);
        if (a->sp.simulation_scale != 1.0f)
            return set_error(RTPS_ERR_ARG, "the adjoint supports simulation_scale = 1 only");
        if (a->settings.GetSettingAs<std::vector<float>>("gravity_alphas").size() &&
            [&] {
                for (float x : a->settings.GetSettingAs<std::vector<float>>("gravity_alphas"))
                    if (x != 0.f) return true;
                return false;
            }())
            return set_error(RTPS_ERR_ARG, "the adjoint does not support point gravity sources");
        if (integrator_of(a->settings) != 0)
            return set_error(RTPS_ERR_ARG, "the adjoint differentiates the leapfrog step only (integrator " +
                                               a->settings.GetSettingAs<std::string>("integrator") + ")");
        a->dt = a->settings.GetSettingAs<float>("time_step");
        a->g = make_grid(a->gp);
        a->gs = make_grid(a->gps);
        a->nb_cells = a->gp.nb_cells;
        if (a->nb_cells <= 0 || a->nb_cells > (1 << 28) - 2)
            return set_error(RTPS_ERR_ARG, "grid has no cells or more than 2^28 - 2 cells (" +
                                               std::to_string(a->nb_cells) + ")");
        a->key_bits = sort_key_bits(a->nb_cells) + kSubBits;
        a->pad_key = a->key_bits >= 32 ? 0xFFFFFFFFu : (1u << a->key_bits) - 1u;
        a->N = max_particles;
        a->ck = checkpoint_every;
        const size_t N = (size_t)max_particles, C = (size_t)a->nb_cells + 1;
        const int nck = (max_steps + checkpoint_every - 1) / checkpoint_every;
        a->ck_state.resize(nck);
        auto alloc_state = [&](State& s) {
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
        for (State& s : a->ck_state) RTPS_TRY_HIP(alloc_state(s));
        RTPS_TRY_HIP(a->alloc(&a->keys, N));
        RTPS_TRY_HIP(a->alloc(&a->start, C));
        RTPS_TRY_HIP(a->alloc(&a->end, C));
        if ((size_t)a->nb_cells * kSubCells * sizeof(uint32_t) <= ((size_t)2 << 30))   // as the system's
            RTPS_TRY_HIP(a->alloc(&a->sub, (size_t)a->nb_cells * kSubCells));
        const bool by_cell = cell_sort_fits((int)N, a->nb_cells);
        RTPS_TRY_HIP(a->alloc((char**)&a->sort_tmp, by_cell ? cell_sort_temp_bytes((int)N, a->nb_cells)
                                                            : bucket_temp_bytes((int)N, a->key_bits)));
        RTPS_TRY_HIP(a->alloc(&a->ga, N));
        RTPS_TRY_HIP(a->alloc(&a->gX, N));
        RTPS_TRY_HIP(a->alloc(&a->lxp, N));
        RTPS_TRY_HIP(a->alloc(&a->gx2, N));
        RTPS_TRY_HIP(a->alloc(&a->ge, N));
        RTPS_TRY_HIP(a->alloc(&a->grho, N));
        RTPS_TRY_HIP(a->alloc(&a->sums, 2 * (size_t)nck * checkpoint_every));
        a->sums_h.resize(2 * (size_t)nck * checkpoint_every);
        RTPS_TRY_HIP(a->alloc(&a->left_grid, 1));
        RTPS_TRY_HIP(alloc_records(a.get(), std::min(checkpoint_every, max_steps)));
        RTPS_TRY_HIP(a->alloc(&a->partial, a->rec.size() * (size_t)adjoint_tiles((int)N)));
        RTPS_TRY_HIP(by_cell ? cell_sort_clear_temp(a->sort_tmp, a->nb_cells, nullptr)
                             : sort_clear_temp(a->sort_tmp, (int)N, nullptr));
        RTPS_TRY_HIP(launch_fill_u32(a->end, 0u, (long)C, nullptr));
        RTPS_TRY_HIP(hipDeviceSynchronize());
        *out = a.release();
        return RTPS_OK;
    } catch (const std::exception& e) {
        return set_error(RTPS_ERR_ARG, std::string("rtps_adj_create: ") + e.what());
    }
}

int rtps_adj_destroy(rtps_adj* a) {
    delete a;
    return RTPS_OK;
}

int rtps_adj_forward(rtps_adj* a, const rtps_float4* pos0, const rtps_float4* vel0, int nsteps, float viscosity,
                     float gas_constant, int collision, rtps_float4* pos_T, rtps_float4* vel_T, void* stream) {
    if (!a || !pos0 || !vel0 || !pos_T || nsteps <= 0 ||
        (size_t)((nsteps + a->ck - 1) / a->ck) > a->ck_state.size())
        return set_error(RTPS_ERR_ARG, "rtps_adj_forward: bad arguments or more steps than the handle holds");
    hipStream_t st = (hipStream_t)stream;
    a->sp.viscosity = viscosity;
    a->sp.K = gas_constant;
    a->collision = collision ? 1 : 0;
    a->T = nsteps;
    const size_t nb = (size_t)a->N * 16;
    const State& s0 = a->ck_state[0];
    if (aligned16(pos0) && aligned16(vel0)) {
        RTPS_TRY_HIP(launch_adj_start(a->N, (const float4*)pos0, (const float4*)vel0, s0.pos, s0.vel, s0.ve, st));
    } else {
        RTPS_TRY_HIP(hipMemcpyAsync(s0.pos, pos0, nb, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(hipMemcpyAsync(s0.vel, vel0, nb, hipMemcpyDeviceToDevice, st));
        RTPS_TRY_HIP(launch_fill_u32((uint32_t*)s0.ve, 0u, (long)a->N * 4, st));   // veleval starts at zero
    }
    RTPS_TRY_HIP(launch_fill_u32((uint32_t*)a->left_grid, 0u, 1, st));
    // The last segment's steps are recorded on the way: the adjoint starts
    // there, and its replay begins with the segment before.
    const int last_first = (nsteps - 1) / a->ck * a->ck, rec_lo = std::max(last_first, nsteps - (int)a->rec.size());
    a->rec_lo = a->rec_hi = 0;
    for (int n = 0; n < nsteps; ++n) {
        const State& in = n % a->ck == 0 ? a->ck_state[n / a->ck] : a->slot[n & 1];
        State out = (n + 1) % a->ck == 0 && n + 1 < nsteps ? a->ck_state[(n + 1) / a->ck] : a->slot[(n + 1) & 1];
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

int rtps_adj_backward(rtps_adj* a, const rtps_float4* dL_dpos_T, const rtps_float4* dL_dvel_T, rtps_float4* dL_dvel0,
                      rtps_float4* dL_dpos0, double* dL_dvisc, double* dL_dgas, void* stream) {
    if (!a || !dL_dpos_T || !dL_dvel0) return set_error(RTPS_ERR_ARG, "rtps_adj_backward: bad arguments");
    if (!a->have_forward) return set_error(RTPS_ERR_STATE, "rtps_adj_backward needs a forward run");
    hipStream_t st = (hipStream_t)stream;
    const int n = a->N;
    const size_t nb = (size_t)n * 16;
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
    const int nck = (a->T + a->ck - 1) / a->ck, R = (int)a->rec.size();
    const int ntiles = adjoint_tiles(n);
    int L = 0;   // the adjoints at hand are in the buffers L (or still the caller's)
    for (int c = nck - 1; c >= 0; --c) {
        const int first = c * a->ck, last = std::min(a->T, first + a->ck);
        for (int hi = last, lo; hi > first; hi = lo) {
            lo = std::max(first, hi - R);
            // replay the segment from its checkpoint, recording the steps lo..hi-1
            // (unless they are the ones recorded last)
            const bool recorded = a->rec_lo == lo && a->rec_hi == hi;
            if (!recorded) a->rec_lo = a->rec_hi = 0;
            for (int s = recorded ? hi : first; s < hi; ++s) {
                const State& in = s == first ? a->ck_state[c] : a->slot[s & 1];
                int rc = forward_step(a, in, a->slot[(s + 1) & 1], a->rec[s < lo ? 0 : s - lo], s >= lo, st);
                if (rc) return rc;
            }
            a->rec_lo = lo;
            a->rec_hi = hi;
            // adjoint through them, last step first
            for (int s = hi - 1; s >= lo; --s) {
                const Record& r = a->rec[s - lo];
                float4 *lv_out = a->lam_v[1 - L], *lx_out = a->lam_x[1 - L], *le_out = a->lam_e[1 - L];
                if (s == 0) {   // the initial state's adjoints go to the caller
                    if (aligned16(dL_dvel0)) lv_out = (float4*)dL_dvel0;
                    if (dL_dpos0 && aligned16(dL_dpos0)) lx_out = (float4*)dL_dpos0;
                    le_out = nullptr;
                }
                RTPS_TRY_HIP(launch_adj_b1(n, r.idx, r.pos_s, r.vel_s, r.force_s, a->sp, a->gps, a->collision, a->dt,
                                           lx, lv, le, a->ga, a->gX, lv_out, a->lxp, st));
                RTPS_TRY_HIP(launch_adj_b2(n, r.pos_s, r.ve_s, a->ga, a->gX, r.rows, (uint32_t)n, a->sp, a->gx2,
                                           a->ge, a->grho, a->partial + (size_t)(s - lo) * ntiles, st));
                RTPS_TRY_HIP(launch_adj_b3(n, r.idx, r.pos_s, a->grho, a->lxp, a->gx2, a->ge, r.rows, (uint32_t)n,
                                           a->sp, lx_out, le_out, st));
                lx = lx_out;
                lv = lv_out;
                le = le_out;
                L = 1 - L;
            }
            RTPS_TRY_HIP(launch_adj_reduce(hi - lo, a->partial, ntiles, a->sums + 2 * (size_t)lo, st));
        }
    }
    if (lv != (const float4*)dL_dvel0) RTPS_TRY_HIP(hipMemcpyAsync(dL_dvel0, lv, nb, hipMemcpyDeviceToDevice, st));
    if (dL_dpos0 && lx != (const float4*)dL_dpos0)
        RTPS_TRY_HIP(hipMemcpyAsync(dL_dpos0, lx, nb, hipMemcpyDeviceToDevice, st));
    RTPS_TRY_HIP(hipMemcpyAsync(a->sums_h.data(), a->sums, 2 * sizeof(double) * (size_t)a->T, hipMemcpyDeviceToHost,
                                st));
    RTPS_TRY_HIP(hipStreamSynchronize(st));
    double acc[2] = {0, 0};
    for (int s = a->T - 1; s >= 0; --s)
        for (int k = 0; k < 2; ++k) acc[k] += a->sums_h[2 * (size_t)s + k];
    if (dL_dvisc) *dL_dvisc = acc[0];
    if (dL_dgas) *dL_dgas = acc[1];
    return RTPS_OK;
}

}  // extern "C"
