// Density and force of small launches: nine waves per 64 particles, one row of
// cells of the neighbourhood each (density.cl, force.cl as in sph_kernels.hip,
// and the same bits).
//
// A wave that takes nine rows one after the other waits nine times for a
// window's lookup and for its candidates, 1.7 us a row, and up to 65,536
// particles the chip has no second wave on a SIMD to cover that.  Here the nine
// rows wait at the same time: each wave looks its row's window up (or reads its
// record), copies the candidates to LDS, tests them and works out the first
// terms of every particle into registers.  Then the rows take turns in
// their order, each adding its terms to the sums it takes over from the row
// before, through LDS: the additions are those of one wave walking the rows, at
// a few instructions per term.  Terms beyond those are worked out in the turn.

#include <hip/hip_runtime.h>

#include "rtps_internal.h"
#include "sph_device.h"

namespace rtps {

namespace {

constexpr int kRowWaves = 9, kRowBlock = 64 * kRowWaves;
constexpr int kRowCap = 192;        // candidates per LDS copy of a row; more are read from memory
constexpr int kAheadDensity = 20;    // a row of resting particles has 14 to 20 candidates
// and up to 7 neighbours, of a settled pool's up to 14: what 168 registers hold
// (three waves on one of the CU's SIMDs), fewer where positions are scaled or
// there are three chains
constexpr int keep_force(bool scaled, bool planes) { return scaled || planes ? 8 : 12; }
constexpr int kChunk = 32;          // candidates per word of rejection bits

// Turn of a wave and the chain of sums it belongs to: one chain over the nine
// rows, or (PLANES) one per plane of three, added afterwards.
template <bool PLANES>
struct Turn {
    static constexpr int kChains = PLANES ? 3 : 1, kTurns = PLANES ? 3 : 9;
    static __device__ __forceinline__ int chain(int w) { return PLANES ? w / 3 : 0; }
    static __device__ __forceinline__ int turn(int w) { return PLANES ? w % 3 : w; }
};

// The candidates of a row for the wave's particles: two runs of sorted
// particles, as the wave's end may lie in the next row of cells (the shorter
// the pool's rows, the more often), far from where its beginning looks.
// `later`: the particle lies in another row of cells than the wave's first one.
struct RowCopy {
    uint32_t A[2], n[2];   // first particle and length of each run
    __device__ __forceinline__ uint32_t size() const { return n[0] + n[1]; }
    // LDS slot of particle 0 for a lane of either run (wraps; slots of the run's particles do not)
    __device__ __forceinline__ uint32_t base(bool later) const { return later ? n[0] - A[1] : 0u - A[0]; }
    // the particle in LDS slot q
    __device__ __forceinline__ uint32_t particle(uint32_t q) const { return q < n[0] ? A[0] + q : A[1] + (q - n[0]); }
};
__device__ __forceinline__ RowCopy row_copy(uint32_t a, uint32_t b, bool later) {
    RowCopy r;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bool in = a < b && later == (k != 0);
        r.A[k] = __ockl_wfred_min_u32(in ? a : 0xFFFFFFFFu);
        const uint32_t B = __ockl_wfred_max_u32(in ? b : 0u);
        r.n[k] = B > r.A[k] ? B - r.A[k] : 0u;
    }
    return r;
}
__device__ __forceinline__ bool in_later_row(int3 c) {
    return c.y != __builtin_amdgcn_readfirstlane(c.y) || c.z != __builtin_amdgcn_readfirstlane(c.z);
}

template <bool SCALED, bool PLANES>
__global__ __launch_bounds__(kRowBlock) void k_density_rows(int num_host, const int* __restrict__ d_num,
                                                            const float4* __restrict__ pos_s,
                                                            const uint32_t* __restrict__ start,
                                                            const uint32_t* __restrict__ end, rtps_sph_params sp,
                                                            Grid g, Win win, float4* __restrict__ packed) {
    using T = Turn<PLANES>;
    __shared__ float4 stage[kRowWaves][kRowCap];
    __shared__ float chain[T::kChains][64];
    const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int first = remap_tile(win.remap, (int)blockIdx.x, (int)gridDim.x) * 64;
    int num = d_num ? *d_num : num_host;
    if (d_num) effective_num(num, start, g.nb_cells, num);
    if (first >= num) return;
    const bool live = first + lane < num;
    const int i = live ? first + lane : num - 1;   // the copies take whole waves
    const float scale = sp.simulation_scale, h = sp.smoothing_distance, h2 = h * h;
    float4 pi = pos_s[i];
    if (SCALED) { pi.x *= scale; pi.y *= scale; pi.z *= scale; }
    const int3 c = grid_cell(pi.x, pi.y, pi.z, g);
    const WindowCtx wc = window_ctx(pi.x, pi.y, pi.z, g, c, h, win.keys, win.rx, win.ry, win.rz);
    uint32_t a, b;
    row_window(wc, c, w % 3 - 1, w / 3 - 1, h2, g, start, end, win.keys, a, b, 0u, win.sub);
    const uint32_t A = __ockl_wfred_min_u32(a < b ? a : 0xFFFFFFFFu);
    const uint32_t B = __ockl_wfred_max_u32(a < b ? b : 0u);
    const uint32_t n = a < b ? b - a : 0u, nmax = __ockl_wfred_max_u32(n);
    const bool later = in_later_row(c);
    const RowCopy copy = row_copy(a, b, later);
    const bool staged = copy.size() <= (uint32_t)kRowCap;
    float4* __restrict__ my = stage[w];
    if (staged)
        for (uint32_t q = lane; q < copy.size(); q += 64u) my[q] = pos_s[copy.particle(q)];
    __builtin_amdgcn_wave_barrier();   // the copies before any lane reads them
    auto u_of = [&](float4 pj) {
        if (SCALED) { pj.x *= scale; pj.y *= scale; pj.z *= scale; }
        return h2_minus_r2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z, h2);
    };
    float t[kAheadDensity];
    uint32_t rej = 0u;
    auto tests = [&](auto&& at) {   // at(k): candidate k of the window
#pragma unroll
        for (int k0 = 0; k0 < kAheadDensity; k0 += 4) {
            if ((uint32_t)k0 < nmax) {
                float4 p[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) p[k] = at(min((uint32_t)(k0 + k), n ? n - 1u : 0u));
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float u = u_of(p[k]);
                    const bool in = (uint32_t)(k0 + k) < n;
                    t[k0 + k] = in ? fmaxf(u, 0.0f) : 0.0f;
                    rej = in ? rej_bit(rej, u) : rej;
                }
            }
        }
        for (uint32_t k = kAheadDensity; k < n; ++k) rej = rej_bit(rej, u_of(at(k)));
    };
    float sum = 0.0f;
    auto rest = [&](auto&& at) {
        for (uint32_t k = kAheadDensity; k < n; ++k) {
            const float v = fmaxf(u_of(at(k)), 0.0f);
            sum = fmaf(v * v, v, sum);
        }
    };
    // where the window is; an idle lane reads the row's first candidate
    const float4* __restrict__ lds = my + (n ? copy.base(later) + a : 0u);
    const float4* __restrict__ mem = pos_s + (n ? a : (B > A ? A : 0u));
    if (staged && B > A) tests([&](uint32_t k) { return lds[k]; });
    else if (B > A) tests([&](uint32_t k) { return mem[k]; });
    for (int s = 0; s < T::kTurns; ++s) {
        if (T::turn(w) == s) {
            sum = s ? chain[T::chain(w)][lane] : 0.0f;
            if (B > A) {
#pragma unroll
                for (int k0 = 0; k0 < kAheadDensity; k0 += 4)
                    if ((uint32_t)k0 < nmax) {
#pragma unroll
                        for (int k = k0; k < k0 + 4; ++k) sum = fmaf(t[k] * t[k], t[k], sum);
                    }
                if (nmax > (uint32_t)kAheadDensity) {
                    if (staged) rest([&](uint32_t k) { return lds[k]; });
                    else rest([&](uint32_t k) { return mem[k]; });
                }
            }
            chain[T::chain(w)][lane] = sum;
        }
        __syncthreads();
    }
    if (win.rows) {
        uint32_t* __restrict__ o = win.rows + 3 * ((size_t)w * win.rows_stride + (size_t)i);
        if (live) {
            o[0] = a;
            o[1] = b;
            o[2] = rej;
        }
        if (lane == 0) {
            uint32_t* __restrict__ wrec =
                win.rows + 27 * (size_t)win.rows_stride + 18 * (size_t)(first >> 6) + 2 * w;
            wrec[0] = A;
            wrec[1] = B;
        }
    }
    if (w == kRowWaves - 1 && live) {
        sum = chain[0][lane];
        if constexpr (PLANES) sum = (sum + chain[1][lane]) + chain[2][lane];
        packed[i].w = sp.wpoly6_coef * sp.mass * sum;
    }
}

// force_pair_r in two parts, its terms and their addition, which lie apart here.
// The fused multiply-adds that the compiler makes of force_pair_r's expressions
// are written out, so that the roundings are its own.  (The tile kernels keep
// force_pair_r: through this form they take 83 registers instead of 79, five
// waves per SIMD instead of six, and 8% more time at 4,000,000 particles.)
struct PairTerms {
    float rx, ry, rz, kern;        // force += r kern
    float dvx, dvy, dvz, lv, w6;   // viscosity += dv lv, xsph += dv w6
};

__device__ __forceinline__ PairTerms force_pair_terms(float rx, float ry, float rz, float r2, float h, float h2,
                                                      float eps, float K, float rho0, float Pi, float di, float4 vi,
                                                      float4 vj, float dj, float idj) {
    const float r2c = __int_as_float(max(__float_as_int(r2), __float_as_int(eps * eps)));
    const float rinv = __builtin_amdgcn_rsqf(r2c);
    const float hr = fmaf(-rinv, r2c, h);           // h - rlen
    const float dW = hr * hr * rinv;                // Wspiky_dr, cl_sph_kernels.h:81-97
    PairTerms p;
    p.rx = rx; p.ry = ry; p.rz = rz;
    p.kern = dW * fmaf(K, dj - rho0, Pi) * idj;     // :84-85 (Pi + Pj), :97
    p.dvx = vj.x - vi.x; p.dvy = vj.y - vi.y; p.dvz = vj.z - vi.z;
    p.lv = hr * idj;                                // Wvisc_lapl * idj, :109-112
    float t = h2 - r2;                              // Wpoly6, cl_sph_kernels.h:29-45
    p.w6 = t * t * t * fast_rcp(di + dj);           // :129-133
    return p;
}

__device__ __forceinline__ void add_pair(ForceAcc& acc, const PairTerms& p) {
    acc.vx = fmaf(p.dvx, p.lv, acc.vx);
    acc.vy = fmaf(p.dvy, p.lv, acc.vy);
    acc.vz = fmaf(p.dvz, p.lv, acc.vz);
    acc.xx = fmaf(p.dvx, p.w6, acc.xx);
    acc.xy = fmaf(p.dvy, p.w6, acc.xy);
    acc.xz = fmaf(p.dvz, p.w6, acc.xz);
    acc.fx = fmaf(p.rx, p.kern, acc.fx);            // :136
    acc.fy = fmaf(p.ry, p.kern, acc.fy);
    acc.fz = fmaf(p.rz, p.kern, acc.fz);
}

__device__ __forceinline__ ForceAcc load_acc(const float (*p)[64], int lane) {
    return ForceAcc{p[0][lane], p[1][lane], p[2][lane], p[3][lane], p[4][lane],
                    p[5][lane], p[6][lane], p[7][lane], p[8][lane]};
}
__device__ __forceinline__ void store_acc(float (*p)[64], int lane, const ForceAcc& a) {
    p[0][lane] = a.fx; p[1][lane] = a.fy; p[2][lane] = a.fz;
    p[3][lane] = a.vx; p[4][lane] = a.vy; p[5][lane] = a.vz;
    p[6][lane] = a.xx; p[7][lane] = a.xy; p[8][lane] = a.xz;
}

template <bool SCALED, bool FUSED, bool PLANES>
__global__ __launch_bounds__(kRowBlock) void k_force_rows(int num_host, int* d_num, const float4* __restrict__ pos_s,
                                                          const float4* __restrict__ ve,
                                                          const uint32_t* __restrict__ start, rtps_sph_params sp,
                                                          Grid g, Win win, float4* __restrict__ force_out,
                                                          float4* __restrict__ xsph_out,
                                                          // FUSED only:
                                                          const float4* __restrict__ vel_s,
                                                          const uint32_t* __restrict__ idx, GravitySources gsrc,
                                                          int collision, rtps_float4 bmin, rtps_float4 bmax, float dt,
                                                          float4* __restrict__ pos_u, float4* __restrict__ vel_u,
                                                          float4* __restrict__ veleval_u,
                                                          const float4* __restrict__ color_s,
                                                          float4* __restrict__ color_u) {
    using T = Turn<PLANES>;
    constexpr int kKeep = keep_force(SCALED, PLANES);
    __shared__ float4 stage[kRowWaves][2 * kRowCap];   // positions (1 / density in w), then veleval|density
    __shared__ float chain[T::kChains][9][64];
    const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int tile = remap_tile(win.remap, (int)blockIdx.x, (int)gridDim.x), first = tile * 64;
    int num = d_num ? *d_num : num_host;
    bool deleted = false;
    if (d_num) deleted = effective_num(num, start, g.nb_cells, num);
    if (FUSED && deleted && tile == 0 && threadIdx.x == 0) *d_num = num;   // the count for the next step (k_force)
    if (first >= num) return;
    const bool live = first + lane < num;
    const int i = live ? first + lane : num - 1;
    const uint32_t* __restrict__ rec = win.rows + 3 * ((size_t)w * win.rows_stride + (size_t)i);
    const uint32_t* __restrict__ wrec = win.rows + 27 * (size_t)win.rows_stride + 18 * (size_t)(first >> 6) + 2 * w;
    const uint32_t a = rec[0], b = rec[1], rej_last = rec[2];
    const uint32_t A = __builtin_amdgcn_readfirstlane(wrec[0]), B = __builtin_amdgcn_readfirstlane(wrec[1]);
    const float4 p_unscaled = pos_s[i], vi = ve[i];
    const bool last = w == kRowWaves - 1;   // finishes the particles
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t o = (uint32_t)i;
    if (FUSED && last) {
        v = vel_s[i];
        if (!deleted) o = idx[i];
    }
    const float scale = sp.simulation_scale, h = sp.smoothing_distance, h2 = h * h;
    const float eps = sp.EPSILON, K = sp.K, rho0 = sp.rest_density;
    float4 pi = p_unscaled;
    if (SCALED) { pi.x *= scale; pi.y *= scale; pi.z *= scale; }
    const float di = vi.w, Pi = K * (di - rho0);
    float4* __restrict__ my_p = stage[w];
    float4* __restrict__ my_v = my_p + kRowCap;
    const bool later = in_later_row(grid_cell(pi.x, pi.y, pi.z, g));
    const RowCopy copy = row_copy(a, b, later);
    const bool staged = copy.size() <= (uint32_t)kRowCap;
    const uint32_t base = copy.base(later);
    if (staged)
        for (uint32_t q = lane; q < copy.size(); q += 64u) {
            const uint32_t j = copy.particle(q);
            const float4 p = pos_s[j], e = ve[j];
            my_p[q] = make_float4(p.x, p.y, p.z, fast_rcp(e.w));
            my_v[q] = make_float4(e.x, e.y, e.z, e.w);
        }
    __builtin_amdgcn_wave_barrier();   // the copies before any lane reads them
    // The window in chunks, the first one ragged (1 to 32 candidates), as in
    // force_planes: the last one's tests are in the record.
    auto accepted = [&](uint32_t j0, uint32_t n, auto&& pos) {
        uint32_t rej = rej_last;
        if (j0 + n != b) {
            rej = 0u;
            for (uint32_t k = 0; k < n; ++k) {
                float4 pj = pos(j0 + k);
                if (SCALED) { pj.x *= scale; pj.y *= scale; pj.z *= scale; }
                rej = rej_bit(rej, h2_minus_r2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z, h2));
            }
        }
        uint32_t m = __builtin_bitreverse32(~rej) >> (32u - n);
        const uint32_t self = (uint32_t)i - j0;   // the particle itself passes (r = 0): drop it
        return self < n ? m & ~(1u << self) : m;
    };
    auto terms = [&](const float4& pq, const float4& vj, bool inv_w) {
        float4 pj = pq;
        if (SCALED) { pj.x *= scale; pj.y *= scale; pj.z *= scale; }
        const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        const float r2 = rx * rx + ry * ry + rz * rz;
        return force_pair_terms(rx, ry, rz, r2, h, h2, eps, K, rho0, Pi, di, vi, vj, vj.w,
                                inv_w ? pq.w : fast_rcp(vj.w));
    };
    const uint32_t n0 = a < b ? ((b - a - 1u) & (uint32_t)(kChunk - 1)) + 1u : 0u;
    uint32_t m = 0u, kept = 0u, kmax = 0u;   // the first chunk's accepted candidates not yet worked out
    PairTerms keep[kKeep];
    // A wave's first kKeep pairs four at a time, without branches: their
    // reads are issued together and their arithmetic overlaps.
    auto work = [&](auto&& pos, auto&& vel, bool inv_w, uint32_t idle) {   // idle: a particle to read in place of none
        if (n0) m = accepted(a, n0, pos);
        kept = min((uint32_t)__builtin_popcount(m), (uint32_t)kKeep);
        kmax = __ockl_wfred_max_u32(kept);
#pragma unroll
        for (int k0 = 0; k0 < kKeep; k0 += 4) {
            if ((uint32_t)k0 >= kmax) break;
            float4 p[4], e[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t j = m != 0u ? a + (uint32_t)__builtin_ctz(m) : idle;
                p[k] = pos(j);
                e[k] = vel(j);
                m &= m - 1u;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const PairTerms q = terms(p[k], e[k], inv_w);
                const bool in = (uint32_t)(k0 + k) < kept;   // idle slots add nothing, whatever was read
                PairTerms& t = keep[k0 + k];
                t.rx = in ? q.rx : 0.f; t.ry = in ? q.ry : 0.f; t.rz = in ? q.rz : 0.f;
                t.dvx = in ? q.dvx : 0.f; t.dvy = in ? q.dvy : 0.f; t.dvz = in ? q.dvz : 0.f;
                t.kern = in ? q.kern : 0.f; t.lv = in ? q.lv : 0.f; t.w6 = in ? q.w6 : 0.f;
            }
        }
    };
    ForceAcc acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto rest = [&](auto&& pos, auto&& vel, bool inv_w) {
        for (uint32_t j0 = a, n = n0; j0 < b;) {
            while (m != 0u) {
                const uint32_t j = j0 + (uint32_t)__builtin_ctz(m);
                add_pair(acc, terms(pos(j), vel(j), inv_w));
                m &= m - 1u;
            }
            j0 += n;
            n = (uint32_t)kChunk;
            if (j0 < b) m = accepted(j0, n, pos);
        }
    };
    auto ldsp = [&](uint32_t j) { return my_p[base + j]; };
    auto ldsv = [&](uint32_t j) { return my_v[base + j]; };
    auto memp = [&](uint32_t j) { return pos_s[j]; };
    auto memv = [&](uint32_t j) { return ve[j]; };
    if (B > A) {
        if (staged) work(ldsp, ldsv, true, 0u - base);
        else work(memp, memv, false, A);
    }
    const bool more = __ballot(m != 0u || (a < b && b - a > (uint32_t)kChunk)) != 0ull;
    for (int s = 0; s < T::kTurns; ++s) {
        if (T::turn(w) == s) {
            if (s) acc = load_acc(chain[T::chain(w)], lane);
            if (B > A) {
#pragma unroll
                for (int k = 0; k < kKeep; ++k)
                    if ((uint32_t)k < kmax) add_pair(acc, keep[k]);
                if (more) {
                    if (staged) rest(ldsp, ldsv, true);
                    else rest(memp, memv, false);
                }
            }
            store_acc(chain[T::chain(w)], lane, acc);
        }
        __syncthreads();
    }
    if (!last || !live) return;
    if constexpr (PLANES) {
        acc = load_acc(chain[0], lane);
        add_acc(acc, load_acc(chain[1], lane));
        add_acc(acc, load_acc(chain[2], lane));
    }
    float4 F, X;
    force_epilogue(acc, di, sp, F, X);
    if (force_out) force_out[i] = F;
    if (xsph_out) xsph_out[i] = X;
    if (FUSED) {
        gravity_sources(F, p_unscaled, gsrc, scale);
        if (collision) collision_wall(F, p_unscaled, v, sp, bmin, bmax);
        float4 po, vo, eo;
        leapfrog(p_unscaled, v, F, X, sp, dt, po, vo, eo, SCALED);
        pos_u[o] = po;
        vel_u[o] = vo;
        veleval_u[o] = eo;
        if (deleted && color_u) color_u[i] = color_s[i];   // leapfrog.cl:107, for renumbered survivors (k_force)
    }
}

}  // namespace

hipError_t launch_density_rows(int num, const int* d_num, const float4* pos_s, const uint32_t* start,
                               const uint32_t* end, const rtps_sph_params& sp, const Grid& g, const Win& win,
                               float4* packed, hipStream_t st) {
    const int nb = (num + 63) / 64;
    const bool scaled = sp.simulation_scale != 1.0f, planes = win.split != Win::kNever;
#define RTPS_ROWS(S, P) k_density_rows<S, P><<<nb, kRowBlock, 0, st>>>(num, d_num, pos_s, start, end, sp, g, win, packed)
    if (scaled) { if (planes) RTPS_ROWS(true, true); else RTPS_ROWS(true, false); }
    else { if (planes) RTPS_ROWS(false, true); else RTPS_ROWS(false, false); }
#undef RTPS_ROWS
    return hipGetLastError();
}

hipError_t launch_force_rows(int num, int* d_num, const float4* pos_s, const float4* ve, const uint32_t* start,
                             const rtps_sph_params& sp, const Grid& g, const Win& win, float4* force, float4* xsph,
                             bool fused, const float4* vel_s, const uint32_t* idx, const GravitySources& gsrc,
                             int collision, const rtps_float4& bmin, const rtps_float4& bmax, float dt, float4* pos_u,
                             float4* vel_u, float4* veleval_u, const float4* color_s, float4* color_u,
                             hipStream_t st) {
    const int nb = (num + 63) / 64;
    const bool scaled = sp.simulation_scale != 1.0f, planes = win.split != Win::kNever;
#define RTPS_ROWS(S, F, P)                                                                                            \
    k_force_rows<S, F, P><<<nb, kRowBlock, 0, st>>>(num, d_num, pos_s, ve, start, sp, g, win, force, xsph, vel_s, idx, \
                                                    gsrc, collision, bmin, bmax, dt, pos_u, vel_u, veleval_u, color_s, \
                                                    color_u)
#define RTPS_ROWS_F(S, F) do { if (planes) RTPS_ROWS(S, F, true); else RTPS_ROWS(S, F, false); } while (0)
    if (scaled) { if (fused) RTPS_ROWS_F(true, true); else RTPS_ROWS_F(true, false); }
    else { if (fused) RTPS_ROWS_F(false, true); else RTPS_ROWS_F(false, false); }
#undef RTPS_ROWS_F
#undef RTPS_ROWS
    return hipGetLastError();
}

}  // namespace rtps
