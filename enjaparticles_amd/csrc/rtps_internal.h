// Internal declarations shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "rtps_c.h"
#include "rtps/RTPSSettings.h"

namespace rtps {

// Flags of the library's timing events (stage timers, autotuners): they only
// time work on their stream and are never used to make device memory visible
// to the host, so their records skip the system-scope fence (a cache
// write-back and invalidate per record, which also leaves the next kernel's
// caches cold).
constexpr unsigned kTimingEvent = hipEventDisableSystemFence;

struct Grid;
struct GravitySources;
struct Win;

// ---- error reporting (capi.cpp) ----
int set_error(int code, const std::string& msg);
int hip_error(hipError_t e, const char* where);

// ---- runs of steps (sph_system.cpp, batch_system.cpp) ----
// Between two graph launches the device is idle for 8 to 10 us, a fifth of a step
// of 2,048 particles; so runs of four and of two steps are graphs, too, next to a
// handle's graph of one.  Each is captured by a call that could use it and finds
// the one-step graph of an earlier call still valid (not where options change
// from call to call), once that call's own steps are under way.
class StepRuns {
public:
    StepRuns() = default;
    StepRuns(const StepRuns&) = delete;
    StepRuns& operator=(const StepRuns&) = delete;
    ~StepRuns() { drop(); }
    void drop() {   // the one-step graph has changed
        for (hipGraphExec_t& e : run_) {
            if (e) (void)hipGraphExecDestroy(e);
            e = nullptr;
        }
        failed_ = false;
    }
    // nsteps steps: runs where they are there, the rest by `one`; kept: it is an
    // earlier call's.  capture(steps, &exec) captures that many steps (RTPS_OK).
    template <class Capture>
    hipError_t replay(hipGraphExec_t one, bool kept, int nsteps, hipStream_t st, Capture&& capture) {
        int left = nsteps;
        for (int r = 0; r < 2; ++r)
            for (; run_[r] && left >= kSteps[r]; left -= kSteps[r]) {
                const hipError_t e = hipGraphLaunch(run_[r], st);
                if (e != hipSuccess) return e;
            }
        for (; left > 0; --left) {
            const hipError_t e = hipGraphLaunch(one, st);
            if (e != hipSuccess) return e;
        }
        for (int r = 0, n = nsteps; r < 2 && kept && !failed_; n %= kSteps[r], ++r)
            if (!run_[r] && n >= kSteps[r]) failed_ = capture(kSteps[r], &run_[r]) != 0;   // then by the others
        return hipSuccess;
    }

private:
    static constexpr int kSteps[2] = {4, 2};
    hipGraphExec_t run_[2] = {};
    bool failed_ = false;
};

// ---- parameter derivation (params.cpp) ----
// SPH::calculate (SPHSettings.cpp:30-144) on `s` (writes the derived keys),
// then SPH::updateParams (:149-201) and System::setupDomain (System.cpp:294-329).
void derive_params(RTPSSettings& s, rtps_sph_params& sp, rtps_grid_params& gp, rtps_grid_params& gps);
// SPH::updateParams only (re-read of the settings after a change).
void read_sph_params(const RTPSSettings& s, rtps_sph_params& sp);
int sort_key_bits(int nb_cells);
void gravity_sources_of(const RTPSSettings& st, GravitySources& g);
int integrator_of(const RTPSSettings& st);

// ---- kernels (sph_kernels.hip) ----
extern int g_density_stage;   // 1 = density rows staged through LDS (default), 0 = read from global memory
extern int g_force_variant;   // force loop: 0 = direct, 4 = rows staged in LDS, 5 = staged with accepted bits
hipError_t launch_hash(int num, const int* d_num, int n_pad, uint32_t pad_key, const float4* pos_u, uint32_t* keys,
                       uint32_t* idx, const Grid& g, uint32_t* start_clear, int n_clear, int sub_bits,
                       hipStream_t st);
// sub (optional, sub_bits = 4 only): the sub-cell start table of the
// windowed neighbour rows, 16 entries per cell
hipError_t launch_cellindices(int num, const int* d_num, const uint32_t* keys, int nb_cells, uint32_t* start,
                              uint32_t* end, int sub_bits, hipStream_t st, uint32_t* sub = nullptr);
hipError_t launch_read_nc(const uint32_t* start, int nb_cells, int* nc, hipStream_t st);
// cu/cs (optional): particle colours, permuted like the positions
hipError_t launch_permute(int num, const int* d_num, const uint32_t* idx, const float4* pu, const float4* vu,
                          const float4* eu, float4* ps, float4* vs, float4* es, hipStream_t st,
                          const float4* cu = nullptr, float4* cs = nullptr);
// launch_cellindices and launch_permute in one kernel (the system's step);
// left (optional) is set to 1 when a particle lies outside the grid
hipError_t launch_cells_permute(int num, const int* d_num, const uint32_t* keys, int nb_cells, uint32_t* start,
                                uint32_t* end, int sub_bits, uint32_t* sub, const uint32_t* idx, const float4* pu,
                                const float4* vu, const float4* eu, float4* ps, float4* vs, float4* es,
                                hipStream_t st, const float4* cu = nullptr, float4* cs = nullptr,
                                int* left = nullptr);
hipError_t launch_density(int num, const int* d_num, const float4* pos_s, const uint32_t* start, const uint32_t* end,
                          const rtps_sph_params& sp, const Grid& g, const Win& win, float* dens, float4* packed,
                          hipStream_t st);
hipError_t launch_force(int num, int* d_num, const float4* pos_s, const float* dens, const float4* ve,
                        bool packed, const uint32_t* start, const uint32_t* end, const rtps_sph_params& sp,
                        const Grid& g, const Win& win, float4* force, float4* xsph, hipStream_t st);
// force, xsph (optional): stored as well
hipError_t launch_force_fused(int num, int* d_num, const float4* pos_s, const float4* ve_packed,
                              const uint32_t* start, const uint32_t* end, const rtps_sph_params& sp, const Grid& g,
                              const Win& win, float4* force, float4* xsph, const float4* vel_s, const uint32_t* idx,
                              const GravitySources& gsrc, int collision, const rtps_grid_params& gps, float dt,
                              float4* pos_u, float4* vel_u, float4* veleval_u, hipStream_t st,
                              const float4* color_s = nullptr, float4* color_u = nullptr);
// The same for small launches on recorded rows, nine waves per 64 particles
// (row_tiles.hip); the split order (Win::split) where the caller asks for it.
hipError_t launch_density_rows(int num, const int* d_num, const float4* pos_s, const uint32_t* start,
                               const uint32_t* end, const rtps_sph_params& sp, const Grid& g, const Win& win,
                               float4* packed, hipStream_t st);
hipError_t launch_force_rows(int num, int* d_num, const float4* pos_s, const float4* ve, const uint32_t* start,
                             const rtps_sph_params& sp, const Grid& g, const Win& win, float4* force, float4* xsph,
                             bool fused, const float4* vel_s, const uint32_t* idx, const GravitySources& gsrc,
                             int collision, const rtps_float4& bmin, const rtps_float4& bmax, float dt, float4* pos_u,
                             float4* vel_u, float4* veleval_u, const float4* color_s, float4* color_u,
                             hipStream_t st);
// Whether launch_density / launch_force (packed) take these (Win::block is then
// without effect), and how many of the two may at this count.
bool density_by_rows(int num, const Win& win);
bool force_by_rows(int num, const Win& win);
int kernels_by_rows(int num, float share);
float rows_share_of(const rtps_sph_params& sp);   // Win::rows_share
hipError_t launch_count_pairs(int num, const int* d_num, const float4* pos_s, const uint32_t* start,
                              const uint32_t* end, const rtps_sph_params& sp, const Grid& g, const Win& win,
                              unsigned long long* out, hipStream_t st);
// the maxima of parts of v[0, n) to out[0, *blocks), at most kMaxBlocks of them
constexpr int kMaxBlocks = 256;
hipError_t launch_max_i32(int n, const int32_t* v, int32_t* out, int* blocks, hipStream_t st);
hipError_t launch_fill_u32(uint32_t* p, uint32_t v, long n, hipStream_t st);

// Default particle colour of System::pushParticles (System.h:160).
constexpr rtps_float4 kDefaultColor{1.0f, 0.0f, 0.0f, 1.0f};

// ---- triangle collision (collision_tri.hip) ----
// One triangle in the simulation scale: vertices a, b, c (q* = c), the
// unnormalised normal n = (b - a) x (c - a), the unit normal u, and the
// bounding sphere (centre c*, radius) with reach2 = (radius + dist)^2 widened.
struct TriPrep {
    float ax, ay, az, bx, by, bz, qx, qy, qz;
    float nx, ny, nz, ux, uy, uz;
    float cx, cy, cz, radius, reach2;
};
std::vector<TriPrep> prepare_triangles(const rtps_triangle* tris, int n, float scale);
void set_triangle_reach(std::vector<TriPrep>& t, float dist);
// Adds the triangles' forces to force, once (waits for the stream).
hipError_t collision_triangles(int num, const float4* pos_s, const float4* vel_s, float4* force,
                               const std::vector<TriPrep>& prep, const rtps_sph_params& sp, hipStream_t st);
// The triangles on the device, and a grid over them: a particle in cell c can
// touch the triangles list[q], q in start[c]..start[c + 1] - 1, whose bounding
// spheres (centre, reach squared) are sphere[q].
struct TriSet {
    int n = 0;   // 0 = none
    const TriPrep* tris = nullptr;
    const float4* sphere = nullptr;
    const uint32_t *start = nullptr, *list = nullptr;
    float3 min{};
    float inv = 0.f;   // cells per unit of length
    int nx = 0, ny = 0, nz = 0;
};
// Owner of a TriSet's device memory.
struct TriDevice {
    TriSet set;
    char* mem = nullptr;
    size_t cap = 0;
    TriDevice() = default;
    TriDevice(const TriDevice&) = delete;
    TriDevice& operator=(const TriDevice&) = delete;
    ~TriDevice() {
        if (mem) (void)hipFree(mem);
    }
    // Replaces the set (waits for the work on st).
    hipError_t load(const std::vector<TriPrep>& prep, float dist, hipStream_t st);
};

// ---- colour field and iso-surface (surface.hip) ----
size_t surface_scan_tiles(long ncubes);
hipError_t launch_color_field(int res, const float4* pos_s, const float4* ve_s, const uint32_t* start,
                              const uint32_t* end, const rtps_sph_params& sp, const Grid& g, const Win& win,
                              const rtps_float4& bmin_scaled, const rtps_float4& bmax_scaled, float* field,
                              hipStream_t st);
// tile_sums: surface_scan_tiles() + 1 words, afterwards each tile's first triangle and the total
hipError_t launch_mc_count(int res, float iso, const float* field, const uint8_t* ntri, uint8_t* cases,
                           uint32_t* tile_sums, hipStream_t st);
// the corner and edge tables into the emit kernel's constant memory (once per process)
hipError_t mc_upload_geometry();
// The surface's triangles at their scanned offsets.
hipError_t launch_mc_emit(int res, float iso, const float* field, const uint8_t* cases, const uint8_t* ntri,
                          const uint32_t* tile_offs, const uint64_t* words, const rtps_float4& wmin,
                          const rtps_float4& wmax, int frame, long capacity, float* verts, float* normals,
                          hipStream_t st);

// ---- rigid-body coupling (rigid.hip) ----
// One set of rigid-body particles in the fluid's grid: sorted positions (and,
// for a moving body, velocities and masses), its cell start/end tables, and
// the staging arrays of the host upload.  s0 / s1: the rigid system's
// "spring" and "dampening" settings.
struct RigidDev {
    int n = 0, cap = 0;
    bool moving = false;
    float s0 = 0.f, s1 = 0.f;
    float4 *pos = nullptr, *vel = nullptr, *in_pos = nullptr, *in_vel = nullptr;
    float *mass = nullptr, *in_mass = nullptr;
    uint32_t *keys = nullptr, *idx = nullptr, *start = nullptr, *end = nullptr;
    void* sort_tmp = nullptr;
    uint8_t* near = nullptr;   // per cell: 1 where one of its 27 cells holds a particle (nullptr: not kept)
};
// Hashes, sorts and tables n particles of pos_u (vel_u / mass_u may be null)
// into r on the unscaled grid g.
hipError_t rigid_prepare(int n, const float4* pos_u, const float4* vel_u, const float* mass_u, RigidDev& r,
                         const Grid& g, hipStream_t st);

// ---- after the pair sums (after_force.hip) ----
struct AfterForce {
    enum { kNone = 0, kLeapfrog = 1, kEuler = 2 };
    bool gravity = false;          // point sources
    bool walls = false;            // of the domain bmin..bmax (scaled)
    bool store = true;             // the force with what was added
    int integrate = kNone;         // with the count commit of a deletion step
    float dt = 0.f;
    rtps_float4 bmin{}, bmax{};
};
// tri, rigid[2] (moving body, static boundary): optional.  idx, xsph and the
// unsorted arrays are used by the integration, ve_s by rigid bodies and euler.
hipError_t launch_after_force(int num, int* d_num, const uint32_t* start, int nb_cells, const float4* pos_s,
                              const float4* vel_s, const float4* ve_s, float4* force, const float4* xsph,
                              const uint32_t* idx, const rtps_sph_params& sp, const AfterForce& a,
                              const GravitySources& gsrc, const Grid& gs, const TriSet* tri, const RigidDev* rigid,
                              float4* pos_u, float4* vel_u, float4* veleval_u, hipStream_t st,
                              const float4* color_s = nullptr, float4* color_u = nullptr);

// ---- hoses (hose.cpp) ----
std::vector<rtps_float4> hose_spray(rtps_hose* h);

// ---- radix sort (radix_sort.hip) ----
extern int g_sort_items;   // one-sweep tile: threads * 100 + keys per thread, 0 = by size (process-wide)
bool sort_config_valid(int block, int keys_per_thread);
int sort_passes(int key_bits);
size_t sort_temp_bytes(int n, int key_bits);
hipError_t sort_clear_temp(void* temp, int n, hipStream_t st);
hipError_t sort_pairs_pingpong(int n, int key_bits, uint32_t* keys, uint32_t* vals, void* temp, hipStream_t st,
                               uint32_t** out_keys, uint32_t** out_vals);
hipError_t sort_pairs_inplace(int n, int key_bits, uint32_t* keys, uint32_t* vals, void* temp, hipStream_t st);
hipError_t sort_pairs_passes(int n, const int* shifts, const int* widths, int npasses, uint32_t* keys,
                             uint32_t* vals, void* temp, hipStream_t st, uint32_t** out_keys, uint32_t** out_vals);
int sort_plan(int key_bits, int* shifts, int* widths);
// launch_hash (keys of pos_u, pad_key past num, start[0..n_clear) cleared)
// and sort_pairs_pingpong of its (keys, idx) with the hash fused into the
// sort's histogram kernel: one kernel fewer per step.
hipError_t hash_sort_pairs(int n, int key_bits, const float4* pos_u, int num_host, const int* d_num, uint32_t pad_key,
                           const Grid& g, int sub_bits, uint32_t* start_clear, int n_clear, uint32_t* keys,
                           uint32_t* vals, void* temp, hipStream_t st, uint32_t** out_keys, uint32_t** out_vals);
hipError_t sort_segments(int batch, int length, int dir, uint32_t* dkeys, uint32_t* dvals, const uint32_t* skeys,
                         const uint32_t* svals, void* temp, hipStream_t st);

// ---- counting sort of the step's particles by cell (cell_sort.hip) ----
constexpr int kCellSortMax = 5 << 16;      // particles
constexpr int kCellSortOneMax = 1 << 12;   // particles that one block sorts
// True when cell_sort_place takes n particles on a grid of nb_cells cells.
bool cell_sort_fits(int n, int nb_cells);
size_t cell_sort_temp_bytes(int n, int nb_cells);   // for every count up to n
hipError_t cell_sort_clear_temp(void* temp, int nb_cells, hipStream_t st);   // before the first sort
// hash, sort and cellindices up to the order inside the cells; then that order
// (keys, idx: hash_sort_pairs's result), the sub-cell table (may be null) and the
// permute, as launch_cells_permute.  start and end are valid after both (small
// launches write them in the second).
hipError_t cell_sort_place(int n, int num_host, const int* d_num, const float4* pos_u, const Grid& g,
                           uint32_t pad_key, uint32_t* keys, uint32_t* idx, uint32_t* start, uint32_t* end, void* temp,
                           hipStream_t st);
hipError_t cell_sort_finish(int n, int num_host, const int* d_num, uint32_t pad_key, const Grid& g,
                            uint32_t* start, uint32_t* end, uint32_t* sub, uint32_t* keys, uint32_t* idx,
                            const float4* pu, const float4* vu, const float4* eu, float4* ps, float4* vs, float4* es,
                            void* temp, hipStream_t st, const float4* cu = nullptr, float4* cs = nullptr,
                            int* left = nullptr);

// ---- bucket sort of the step's cell keys (bucket_sort.hip) ----
// True when hash_bucket_sort takes n keys of key_bits bits.
bool bucket_sort_fits(int n, int key_bits);
// Temp bytes of hash_bucket_sort for every count up to n (at least
// sort_temp_bytes(n, key_bits)).
size_t bucket_temp_bytes(int n, int key_bits);
// hash_sort_pairs's result (keys of pos_u, pad_key past num, start[0..n_clear)
// cleared, (keys, idx) sorted stably) always left in (keys, vals).
hipError_t hash_bucket_sort(int n, int key_bits, const float4* pos_u, int num_host, const int* d_num, uint32_t pad_key,
                            const Grid& g, int sub_bits, uint32_t* start_clear, int n_clear, uint32_t* keys,
                            uint32_t* vals, void* temp, hipStream_t st);

}  // namespace rtps
