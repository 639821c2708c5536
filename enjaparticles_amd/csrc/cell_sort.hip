// Sort of the step's particles by cell key, with the cell tables and the
// permute (System::hash_and_sort of the reference: hash.cl, the bitonic sort of
// System.cpp:407-480, cellindices.cl, permute.cl), as one counting sort over
// the grid's cells.  The order is the stable sort's: keys (cell << 4 | x
// sixteenth) ascending, equal keys by particle index.
//
// Up to 4,096 particles on grids whose counters fit LDS (some 24,000 cells at
// 4,096 particles) k_cell_sort_one makes the order and launch_cells_permute the
// rest, above these four do:
//
//   k_cell_count    the key of every particle (hash_key) and its arrival rank
//                   in its cell: one atomic on the cell's counter.
//   k_cell_scan     counters to cell starts and ends (the start/end tables of
//                   cellindices.cl); the counters are zero again.
//   k_cell_place    (key, index) pairs to cell start + rank: cells together,
//                   any order inside a cell.
//   k_cell_finish   each pair's place in its cell is the number of the cell's
//                   pairs that precede it (x sixteenth, then index); the pair,
//                   the particle's records and its entries of the sub-cell
//                   table go there.
//
// Against digit passes this reads and writes the keys once, needs no look-back
// between tiles, and writes the cell tables on the way.  A cell holds 8
// particles at rest and 20 to 40 in a settled pool, so the counting inside a
// cell is short; a cell of m particles costs m^2 comparisons, 9,000 stacked in
// one cell 0.3 ms, which their pair sums then exceed.  The particles outside the
// grid, in one cell more, have no pair sums and may be any number: their keys
// are equal, so their order is that of the indices, and count leaves a bit for
// each slot that holds one, from which place counts (outside_rank).  A step of
// which 95% are outside takes 0.15 ms at 327,680 particles and 0.21 in a batch of
// 400,000; 47 and 78 where they are compared in pairs.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "batch_types.h"
#include "rtps_internal.h"
#include "sort_layout.h"
#include "sph_device.h"

namespace rtps {

constexpr int kCsThreads = 256;
constexpr int kScanThreads = 1024, kScanWaves = kScanThreads / 64;
constexpr int kScanTile = 4 * kScanThreads;   // counters per round of a scanning block
constexpr int kScanBlocks = 256;              // at most: a block adds up every earlier block's total

static inline int cs_blocks(long n) { return (int)((n + kCsThreads - 1) / kCsThreads); }

// Layout of the temp: the counters (zero between sorts), the scan's status
// words, the slots' bits of particles outside the grid, the pairs.
struct CellTemp {
    uint32_t* count;
    unsigned long long* status;
    uint64_t* outside;
    uint2* pairs;
};
static size_t cell_layout(int n, int nb_cells, CellTemp* t, char* p) {
    size_t off = 0;
    if (t) t->count = (uint32_t*)(p + off);
    off += (((size_t)nb_cells + 1) * 4 + 255) & ~(size_t)255;
    if (t) t->status = (unsigned long long*)(p + off);
    off += kScanBlocks * sizeof(unsigned long long);
    if (t) t->outside = (uint64_t*)(p + off);
    off += (size_t)cs_blocks(std::max(n, kScanBlocks)) * (kCsThreads / 64) * sizeof(uint64_t);   // one per wave of the count
    if (t) t->pairs = (uint2*)(p + off);
    return off + (size_t)std::max(n, 1) * sizeof(uint2);
}

size_t cell_sort_temp_bytes(int n, int nb_cells) { return cell_layout(n, nb_cells, nullptr, nullptr); }

hipError_t cell_sort_clear_temp(void* temp, int nb_cells, hipStream_t st) {
    return hipMemsetAsync(temp, 0, ((size_t)nb_cells + 1) * 4, st);
}

// The line: one atomic per particle costs more than the bucket sort's one per
// bucket that a tile touches where consecutive particles are neighbours, and
// less where they are not.  Measured for sort + cells (us, bucket / counting; at
// rest, then in a settled pool whose order is mixed): 22 / 16 and 21 / 16 at
// 2,048 particles, 31 / 24 and 37 / 29 at 99,991, 34 / 33 and 58 / 49 at
// 262,144, 42 / 45 and 94 / 81 at 524,288, 58 / 77 and 175 / 147 at 1,048,576
// (digit passes: 91 and 137).  At rest the two meet near 330,000.
// Grids with many more cells than particles take a sort of the keys instead:
// the scan reads every cell's counter.
bool cell_sort_fits(int n, int nb_cells) { return n <= kCellSortMax && (long)nb_cells <= 16L * n + (1 << 20); }

// Batches: the other way there is hash, four or five digit passes, cellindices
// and permute, nine launches in all.  Measured for all of it (us, digits /
// counting; settled scenes, then at rest): 43 / 27 and 41 / 25 at 2,574 slots,
// 76 / 51 and 70 / 39 at 216,557, 110 / 105 and 110 / 76 at 840,154, 155 / 159 and
// 159 / 125 at 1,356,782, 331 / 389 and 301 / 290 at 3,534,703.  The line, 2^20
// slots, is where settled scenes still gain.
bool cell_sort_fits_b(long T, long total_cells) { return T <= 1 << 20 && total_cells <= 16 * T + (1 << 20); }

// The place of lane `lane` of a wave over the slots [first, first + 64) among the
// particles outside the grid of its scene, which begins at slot `off`: those in
// the scene's slots before it.  same: the wave's lanes that hold one of that
// scene.  Called by whole waves.
__device__ __forceinline__ uint32_t outside_rank(const uint64_t* __restrict__ outside, int off, int first, int lane,
                                                 uint64_t same) {
    uint32_t before = 0u;
    for (int w = (off >> 6) + lane; w < first >> 6; w += 64) {
        const uint64_t m = w == off >> 6 ? ~0ull << (off & 63) : ~0ull;   // the scene's part of its first word
        before += (uint32_t)__popcll(outside[w] & m);
    }
    before = __shfl(wave_incl_scan(before), 63);
    return before + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
}

__global__ __launch_bounds__(kCsThreads) void k_cell_count(int num_host, const int* __restrict__ d_num,
                                                           const float4* __restrict__ pos_u, Grid g,
                                                           uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                                           uint32_t* __restrict__ count,
                                                           uint64_t* __restrict__ outside,
                                                           unsigned long long* __restrict__ status) {
    const int i = blockIdx.x * kCsThreads + threadIdx.x;
    if (i < kScanBlocks) status[i] = 0ull;
    const int num = d_num ? *d_num : num_host;
    const bool valid = i < num;
    const uint32_t key = valid ? hash_key(pos_u[i], g, kSubBits) : 0u, cell = key >> kSubBits;
    const bool out = valid && cell >= (uint32_t)g.nb_cells;
    const uint64_t outs = __ballot(out);
    if ((threadIdx.x & 63) == 0) {
        outside[i >> 6] = outs;
        if (outs != 0ull) atomicAdd(&count[g.nb_cells], (uint32_t)__popcll(outs));
    }
    if (valid) keys[i] = key;
    if (valid && !out) rank[i] = atomicAdd(&count[cell], 1u);
}

// Block b scans the cells [b * chunk, (b + 1) * chunk) of the n_cells = nb_cells
// + 1 counters (the last one: particles outside the grid).  It publishes its
// total first and then adds up those of every earlier block, which have come
// in by the time its own counters are read (blocks start in order and publish
// before they wait).
__global__ __launch_bounds__(kScanThreads) void k_cell_scan(int n_cells, int chunk, uint32_t* __restrict__ count,
                                                            uint32_t* __restrict__ start, uint32_t* __restrict__ end,
                                                            unsigned long long* status) {
    __shared__ uint32_t wsum[kScanWaves];
    __shared__ uint32_t prior[kScanBlocks / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int c0 = blockIdx.x * chunk, c1 = min(c0 + chunk, n_cells);
    auto load = [&](int base, uint32_t (&v)[4]) {   // four counters of the thread (c0 and chunk are multiples of 4)
        if (base + 4 <= c1) {
            const uint4 q = *(const uint4*)(count + base);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = base + k < c1 ? count[base + k] : 0u;
        }
    };
    // the block's sum of s over its threads (every thread)
    auto block_sum = [&](uint32_t s) {
        s = wave_incl_scan(s);
        __syncthreads();
        if (lane == 63) wsum[w] = s;
        __syncthreads();
        uint32_t t = 0;
#pragma unroll
        for (int q = 0; q < kScanWaves; ++q) t += wsum[q];
        return t;
    };
    uint32_t v[4], sum = 0;
    for (int t0 = c0; t0 < c1; t0 += kScanTile) {
        load(t0 + 4 * tid, v);
        sum += v[0] + v[1] + v[2] + v[3];
    }
    const uint32_t total = block_sum(sum);
    if (tid == 0)
        __hip_atomic_store(&status[blockIdx.x], (1ull << 63) | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t before = 0;
    if (tid < (int)blockIdx.x) {
        unsigned long long s;
        do {
            s = __hip_atomic_load(&status[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } while (!(s >> 63));
        before = (uint32_t)s;
    }
    if (tid < kScanBlocks) {
        before = wave_incl_scan(before);
        if (lane == 63) prior[w] = before;
    }
    __syncthreads();
    uint32_t run = 0;
#pragma unroll
    for (int q = 0; q < kScanBlocks / 64; ++q) run += prior[q];
    for (int t0 = c0; t0 < c1; t0 += kScanTile) {
        const int base = t0 + 4 * tid;
        if (c1 - c0 > kScanTile) load(base, v);   // one round: still in registers
        const uint32_t s = v[0] + v[1] + v[2] + v[3], inc = wave_incl_scan(s);
        __syncthreads();   // the former round's sums are read
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        uint32_t at = run + inc - s, all = 0;
#pragma unroll
        for (int q = 0; q < kScanWaves; ++q) {
            if (q < w) at += wsum[q];
            all += wsum[q];
        }
        run += all;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (base + k < c1) {
                start[base + k] = v[k] ? at : kEmpty;
                at += v[k];
                if (v[k]) {   // end[] of empty cells is left as it is (cellindices.cl)
                    end[base + k] = at;
                    count[base + k] = 0u;
                }
            }
        }
    }
}

__global__ __launch_bounds__(kCsThreads) void k_cell_place(int num_host, const int* __restrict__ d_num,
                                                           const uint32_t* __restrict__ keys,
                                                           const uint32_t* __restrict__ rank,
                                                           const uint32_t* __restrict__ start, int nb_cells,
                                                           const uint64_t* __restrict__ outside,
                                                           uint2* __restrict__ pairs) {
    const int i = blockIdx.x * kCsThreads + threadIdx.x, lane = (int)threadIdx.x & 63;
    const int num = d_num ? *d_num : num_host;
    const bool valid = i < num;
    const uint32_t key = valid ? keys[i] : 0u, cell = key >> kSubBits;
    uint32_t order = valid ? rank[i] : 0u;   // outside the grid not yet one
    const bool out = valid && cell >= (uint32_t)nb_cells;
    const uint64_t outs = __ballot(out);
    if (outs != 0ull) {
        const uint32_t r = outside_rank(outside, 0, i - lane, lane, outs);
        order = out ? r : order;
    }
    if (!valid) return;
    const uint32_t at = start[cell] + order;
    if (at < (uint32_t)num) pairs[at] = make_uint2(key, (uint32_t)i);
}

// How many of the cell's pairs [a, b) precede kv (by x sixteenth, then index),
// and the x sixteenth of the last of them in `prev_xq`.
__device__ __forceinline__ uint32_t rank_in_cell(const uint2* __restrict__ pairs, uint2 kv, uint32_t a, uint32_t b,
                                                 uint32_t& prev_xq) {
    // x sixteenth and index as one number: the order inside a cell
    auto order = [](const uint2& q) { return (q.x << 28) | q.y; };
    const uint32_t mine = order(kv);
    uint32_t before = 0u, prev = 0u;   // pairs that precede this one; the last of them
    auto member = [&](uint32_t o) {
        const bool less = o < mine;
        before += less ? 1u : 0u;
        prev = max(prev, less ? o : 0u);
    };
    uint32_t j = a;
    for (; j + 4 <= b; j += 4) {
        uint2 q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = pairs[j + k];
#pragma unroll
        for (int k = 0; k < 4; ++k) member(order(q[k]));
    }
    for (; j < b; ++j) member(order(pairs[j]));
    prev_xq = prev >> 28;
    return before;
}

// The cell's sub-cell starts that the pair at `to` writes: entry q = first
// index of the cell with x sixteenth >= q (the cell's end when none), each
// written by the pair that starts it.
__device__ __forceinline__ void write_sub_starts(uint32_t* __restrict__ row, uint32_t xq, uint32_t before,
                                                 uint32_t prev_xq, uint32_t to, uint32_t b) {
    for (uint32_t q = before ? prev_xq + 1u : 0u; q <= xq; ++q) row[q] = to;
    if (to + 1 == b)
        for (uint32_t q = xq + 1; q < (uint32_t)kSubCells; ++q) row[q] = b;
}

__global__ __launch_bounds__(kCsThreads) void k_cell_finish(int n, int num_host, const int* __restrict__ d_num,
                                                            uint32_t pad_key, const uint2* __restrict__ pairs,
                                                            int nb_cells, const uint32_t* __restrict__ start,
                                                            const uint32_t* __restrict__ end,
                                                            uint32_t* __restrict__ sub, uint32_t* __restrict__ keys,
                                                            uint32_t* __restrict__ idx, const float4* __restrict__ pu,
                                                            const float4* __restrict__ vu,
                                                            const float4* __restrict__ eu, float4* __restrict__ ps,
                                                            float4* __restrict__ vs, float4* __restrict__ es,
                                                            const float4* __restrict__ cu, float4* __restrict__ cs,
                                                            int* __restrict__ left) {
    const int i = blockIdx.x * kCsThreads + threadIdx.x;
    const int num = d_num ? *d_num : num_host;
    if (i >= num) {
        if (i < n) {   // slots past the device's count: the pad key, as the stable sort leaves them
            keys[i] = pad_key;
            idx[i] = (uint32_t)i;
        }
        return;
    }
    const uint2 kv = pairs[i];
    const float4 p = pu[kv.y], v = vu[kv.y], e = eu[kv.y];
    const uint32_t cell = kv.x >> kSubBits;
    uint32_t to = (uint32_t)i;   // outside the grid: in order already
    if (cell < (uint32_t)nb_cells) {
        const uint32_t a = start[cell], b = end[cell];
        uint32_t prev_xq;
        const uint32_t before = rank_in_cell(pairs, kv, a, b, prev_xq);
        to = a + before;
        if (sub)
            write_sub_starts(sub + (size_t)cell * kSubCells, kv.x & (kSubCells - 1), before, prev_xq, to, b);
    }
    keys[to] = kv.x;
    idx[to] = kv.y;
    ps[to] = p;
    vs[to] = v;
    es[to] = e;
    if (cu) cs[to] = cu[kv.y];   // permute.cl:41 (colours, when the system keeps them)
    if (left && cell >= (uint32_t)nb_cells) *left = 1;
}

// The order in one block, for small launches: the counters (16 bits each, two to
// a word) and the order inside the cells in LDS, the particles' keys and ranks in
// registers; launch_cells_permute does the rest.  Up to some thousand particles
// the count, the scan and the placing each do little but start and wait for
// memory; one CU alone takes 4 to 8 us for them.  A step takes (us, one block /
// three launches; settled pools) 23 / 27 with 100 particles, 34 / 38 with 1,000,
// 41 / 45 with 2,048, 46 / 48 with 4,096, 55 / 53 with 6,000, 61 / 55 with 8,192.
constexpr int kOneThreads = 1024, kOnePer = kCellSortOneMax / kOneThreads;
constexpr size_t kOneLds = 63 << 10;   // dynamic; the waves' sums come on top
static size_t one_lds(int n, int nb_cells) {   // counters of nb_cells + 1 cells and the end, then the orders
    return (((size_t)nb_cells + 3) / 2 + (size_t)n) * 4;
}
static bool one_block(int n, int nb_cells) { return n <= kCellSortOneMax && one_lds(n, nb_cells) <= kOneLds; }

__global__ __launch_bounds__(kOneThreads) void k_cell_sort_one(int n, int num_host, const int* __restrict__ d_num,
                                                               const float4* __restrict__ pu, Grid g,
                                                               uint32_t pad_key, uint32_t* __restrict__ start,
                                                               uint32_t* __restrict__ keys,
                                                               uint32_t* __restrict__ idx) {
    extern __shared__ uint32_t lds[];
    constexpr int kWaves = kOneThreads / 64;
    __shared__ uint32_t wsum[kWaves], wout[kOnePer * kWaves];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int nc = g.nb_cells + 1, words = (nc + 2) / 2;   // the last entry: the end of the last cell
    uint32_t* order = lds + words;
    const int num = min(d_num ? *d_num : num_host, n);
    auto at = [&](uint32_t c) { return (lds[c >> 1] >> (16u * (c & 1u))) & 0xFFFFu; };
    for (int q = tid; q < words; q += kOneThreads) lds[q] = 0u;
    uint32_t key[kOnePer], rank[kOnePer];
    float3 p[kOnePer];
#pragma unroll
    for (int k = 0; k < kOnePer; ++k) {
        const float4 q = pu[min(tid + k * kOneThreads, max(num - 1, 0))];   // no branch: the loads are issued together
        p[k] = make_float3(q.x, q.y, q.z);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kOnePer; ++k) {
        const int i = tid + k * kOneThreads;
        if (i < num) {
            key[k] = hash_key(make_float4(p[k].x, p[k].y, p[k].z, 0.f), g, kSubBits);
            const uint32_t c = key[k] >> kSubBits, sh = 16u * (c & 1u);
            rank[k] = (atomicAdd(&lds[c >> 1], 1u << sh) >> sh) & 0xFFFFu;   // counts stay below 2^16: no carry
        }
    }
    __syncthreads();
    // exclusive scan of the counters in place: an odd run of words per thread (LDS banks)
    const int per = ((words + kOneThreads - 1) / kOneThreads) | 1, w0 = min(tid * per, words), w1 = min(w0 + per, words);
    uint32_t sum = 0;
    for (int q = w0; q < w1; ++q) sum += (lds[q] & 0xFFFFu) + (lds[q] >> 16);
    const uint32_t inc = wave_incl_scan(sum);
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) run += q < w ? wsum[q] : 0u;
    for (int q = w0; q < w1; ++q) {
        const uint32_t v = lds[q], mid = run + (v & 0xFFFFu);
        lds[q] = run | mid << 16;
        run = mid + (v >> 16);
    }
    __syncthreads();
    const uint32_t inside = at((uint32_t)g.nb_cells);   // particles in the grid
    auto order_of = [](uint32_t key, int i) { return key << 28 | (uint32_t)i; };   // x sixteenth, then index
#pragma unroll
    for (int k = 0; k < kOnePer; ++k) {
        const int i = tid + k * kOneThreads;
        if (i < num) order[at(key[k] >> kSubBits) + rank[k]] = order_of(key[k], i);
    }
    for (int c = tid; c < nc; c += kOneThreads) start[c] = kEmpty;   // the occupied ones follow (launch_cells_permute)
    // The particles outside the grid, where they are more than a cell's usual
    // number: their places by counting the flags in index order.
    const bool many_out = num - __builtin_amdgcn_readfirstlane((int)inside) > 64;   // of the block
    uint32_t out_before[kOnePer];
    if (many_out) {
#pragma unroll
        for (int k = 0; k < kOnePer; ++k) {
            const bool out = tid + k * kOneThreads < num && key[k] >> kSubBits >= (uint32_t)g.nb_cells;
            const uint64_t outs = __ballot(out);
            out_before[k] = (uint32_t)__popcll(outs & ((1ull << lane) - 1ull));
            if (lane == 0) wout[k * kWaves + w] = (uint32_t)__popcll(outs);
        }
    }
    __syncthreads();
    if (many_out) {
#pragma unroll
        for (int k = 0; k < kOnePer; ++k)
            for (int q = 0; q < k * kWaves + w; ++q) out_before[k] += wout[q];
    }
#pragma unroll
    for (int k = 0; k < kOnePer; ++k) {
        const int i = tid + k * kOneThreads;
        if (i >= num) {
            if (i < n) {   // slots past the device's count: the pad key, as the stable sort leaves them
                keys[i] = pad_key;
                idx[i] = (uint32_t)i;
            }
            continue;
        }
        const uint32_t cell = key[k] >> kSubBits, a = at(cell), b = at(cell + 1), mine = order_of(key[k], i);
        if (many_out && cell >= (uint32_t)g.nb_cells) {
            keys[a + out_before[k]] = key[k];
            idx[a + out_before[k]] = (uint32_t)i;
            continue;
        }
        uint32_t before = 0u;   // of the cell
        uint32_t j = a;
        for (; j + 8 <= b; j += 8) {
            uint32_t o[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) o[u] = order[j + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) before += o[u] < mine ? 1u : 0u;
        }
#pragma unroll
        for (int u = 0; u < 7; ++u) {   // past the cell's end: not counted
            const uint32_t o = order[min(j + u, b - 1u)];
            before += j + u < b && o < mine ? 1u : 0u;
        }
        keys[a + before] = key[k];
        idx[a + before] = (uint32_t)i;
    }
}

// The same for the scenes of a batch: the cells of all scenes, counted
// together, each scene's followed by one more that counts its unused slots (so
// that every scene starts at its own slots).  Keys (scene << 24) | cell << 4 | x
// sixteenth; unused slots keep their place and get (scene << 24) | 0xFFFFFF.
// The blocks go over the slots in XCD order (xcd_tile): a scene's gathers and its
// counters stay in one L2, which its pair kernels' items use as well.  finish at
// 216,557 settled slots: 16 -> 11 us, 48 -> 26 at 840,154.
constexpr uint32_t kPadLocal = (1u << kSceneShift) - 1u;

__device__ __forceinline__ uint32_t cell_of_key(const SceneDev& S, uint32_t key) {
    return (uint32_t)S.cell_base + ((key & kPadLocal) >> kSubBits);
}

__global__ __launch_bounds__(kCsThreads) void k_cell_count_b(int T, const uint16_t* __restrict__ sid,
                                                             const SceneDev* __restrict__ scenes,
                                                             const int* __restrict__ d_num,
                                                             const float4* __restrict__ pos_u,
                                                             uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                                             uint32_t* __restrict__ count,
                                                             uint64_t* __restrict__ outside,
                                                             unsigned long long* __restrict__ status) {
    const int i = xcd_tile(blockIdx.x, gridDim.x) * kCsThreads + threadIdx.x, lane = (int)threadIdx.x & 63;
    if (i < kScanBlocks) status[i] = 0ull;
    const int s = i < T ? sid[i] : 0;
    const SceneDev& S = scenes[s];
    const int num = d_num[s], at = i - S.off;
    const bool valid = i < T && at < num;
    if (i < T && at == num) count[S.cell_base + S.g.nb_cells + 1] = (uint32_t)(S.cap - num);
    const uint32_t key = valid ? ((uint32_t)s << kSceneShift) | hash_key(pos_u[i], S.g, kSubBits) : 0u;
    const uint32_t cell = cell_of_key(S, key), past = (uint32_t)(S.cell_base + S.g.nb_cells);
    const bool out = valid && cell >= past;
    const uint64_t outs = __ballot(out);
    if (lane == 0) outside[i >> 6] = outs;
    for (uint64_t left = outs; left != 0ull;) {   // scene by scene
        const int lead = __builtin_ctzll(left), s0 = __builtin_amdgcn_readlane(s, lead);
        const uint64_t same = __ballot(out && s == s0);
        if (lane == lead) atomicAdd(&count[past], (uint32_t)__popcll(same));
        left &= ~same;
    }
    if (valid) keys[i] = key;
    if (valid && !out) rank[i] = atomicAdd(&count[cell], 1u);
}

__global__ __launch_bounds__(kCsThreads) void k_cell_place_b(int T, const uint16_t* __restrict__ sid,
                                                             const SceneDev* __restrict__ scenes,
                                                             const int* __restrict__ d_num,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint32_t* __restrict__ rank,
                                                             const uint32_t* __restrict__ start,
                                                             const uint64_t* __restrict__ outside,
                                                             uint2* __restrict__ pairs) {
    const int i = xcd_tile(blockIdx.x, gridDim.x) * kCsThreads + threadIdx.x, lane = (int)threadIdx.x & 63;
    const int s = i < T ? sid[i] : 0;
    const SceneDev& S = scenes[s];
    const bool valid = i < T && i - S.off < d_num[s];
    const uint32_t key = valid ? keys[i] : 0u, cell = cell_of_key(S, key);
    uint32_t order = valid ? rank[i] : 0u;   // outside the grid not yet one
    const bool out = valid && cell >= (uint32_t)(S.cell_base + S.g.nb_cells);
    for (uint64_t left = __ballot(out); left != 0ull;) {   // scene by scene
        const int lead = __builtin_ctzll(left), s0 = __builtin_amdgcn_readlane(s, lead);
        const uint64_t same = __ballot(out && s == s0);
        const uint32_t r = outside_rank(outside, scenes[s0].off, i - lane, lane, same);
        if ((same >> lane) & 1ull) order = r;
        left &= ~same;
    }
    if (!valid) return;
    const uint32_t at = start[cell] + order;
    if (at < (uint32_t)T) pairs[at] = make_uint2(key, (uint32_t)i);
}

__global__ __launch_bounds__(kCsThreads) void k_cell_finish_b(int T, const uint16_t* __restrict__ sid,
                                                              const SceneDev* __restrict__ scenes,
                                                              const int* __restrict__ d_num,
                                                              const uint2* __restrict__ pairs,
                                                              const uint32_t* __restrict__ start,
                                                              const uint32_t* __restrict__ end,
                                                              uint32_t* __restrict__ sub, uint32_t* __restrict__ keys,
                                                              uint32_t* __restrict__ idx,
                                                              const float4* __restrict__ pu,
                                                              const float4* __restrict__ vu,
                                                              const float4* __restrict__ eu, float4* __restrict__ ps,
                                                              float4* __restrict__ vs, float4* __restrict__ es) {
    const int i = xcd_tile(blockIdx.x, gridDim.x) * kCsThreads + threadIdx.x;
    if (i >= T) return;
    const int s = sid[i];
    const SceneDev& S = scenes[s];
    uint2 kv = make_uint2(((uint32_t)s << kSceneShift) | kPadLocal, (uint32_t)i);
    uint32_t to = (uint32_t)i;
    if (i - S.off < d_num[s]) {
        kv = pairs[i];
        const uint32_t cell = cell_of_key(S, kv.x);
        if (cell < (uint32_t)(S.cell_base + S.g.nb_cells)) {   // outside the grid: in order already
            const uint32_t a = start[cell], b = end[cell];
            uint32_t prev_xq;
            const uint32_t before = rank_in_cell(pairs, kv, a, b, prev_xq);
            to = a + before;
            if (sub)
                write_sub_starts(sub + (size_t)cell * kSubCells, kv.x & (kSubCells - 1), before, prev_xq, to, b);
        }
    }
    const float4 p = pu[kv.y], v = vu[kv.y], e = eu[kv.y];
    keys[to] = kv.x;
    idx[to] = kv.y;
    ps[to] = p;
    vs[to] = v;
    es[to] = e;
}

static void launch_cell_scan(int n_cells, const CellTemp& t, uint32_t* start, uint32_t* end, hipStream_t st) {
    const int want = std::min(kScanBlocks, (n_cells + kScanTile - 1) / kScanTile);
    const int chunk = ((n_cells + want - 1) / want + 3) & ~3;
    k_cell_scan<<<(n_cells + chunk - 1) / chunk, kScanThreads, 0, st>>>(n_cells, chunk, t.count, start, end, t.status);
}

hipError_t cell_sort_place_b(int T, const uint16_t* sid, const SceneDev* scenes, const int* d_num,
                             const float4* pos_u, int total_cells, uint32_t* keys, uint32_t* idx, uint32_t* start,
                             uint32_t* end, void* temp, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (T <= 0) return hipSuccess;
    CellTemp t;
    cell_layout(T, total_cells - 1, &t, (char*)temp);
    k_cell_count_b<<<cs_blocks(std::max(T, kScanBlocks)), kCsThreads, 0, st>>>(T, sid, scenes, d_num, pos_u, keys,
                                                                               idx, t.count, t.outside, t.status);
    launch_cell_scan(total_cells, t, start, end, st);
    k_cell_place_b<<<cs_blocks(T), kCsThreads, 0, st>>>(T, sid, scenes, d_num, keys, idx, start, t.outside,
                                                            t.pairs);
    return hipGetLastError();
}

hipError_t cell_sort_finish_b(int T, const uint16_t* sid, const SceneDev* scenes, const int* d_num, int total_cells,
                              const uint32_t* start, const uint32_t* end, uint32_t* sub, uint32_t* keys,
                              uint32_t* idx, const float4* pu, const float4* vu, const float4* eu, float4* ps,
                              float4* vs, float4* es, void* temp, hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (T <= 0) return hipSuccess;
    CellTemp t;
    cell_layout(T, total_cells - 1, &t, (char*)temp);
    k_cell_finish_b<<<cs_blocks(T), kCsThreads, 0, st>>>(T, sid, scenes, d_num, t.pairs, start, end, sub, keys, idx,
                                                         pu, vu, eu, ps, vs, es);
    return hipGetLastError();
}

hipError_t cell_sort_place(int n, int num_host, const int* d_num, const float4* pos_u, const Grid& g,
                           uint32_t pad_key, uint32_t* keys, uint32_t* idx, uint32_t* start, uint32_t* end, void* temp,
                           hipStream_t st) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (n <= 0) return hipSuccess;
    if (one_block(n, g.nb_cells)) {
        k_cell_sort_one<<<1, kOneThreads, one_lds(n, g.nb_cells), st>>>(n, num_host, d_num, pos_u, g, pad_key, start,
                                                                       keys, idx);
        return hipGetLastError();
    }
    CellTemp t;
    cell_layout(n, g.nb_cells, &t, (char*)temp);
    k_cell_count<<<cs_blocks(std::max(n, kScanBlocks)), kCsThreads, 0, st>>>(num_host, d_num, pos_u, g, keys, idx,
                                                                             t.count, t.outside, t.status);
    launch_cell_scan(g.nb_cells + 1, t, start, end, st);
    k_cell_place<<<cs_blocks(n), kCsThreads, 0, st>>>(num_host, d_num, keys, idx, start, g.nb_cells, t.outside,
                                                          t.pairs);
    return hipGetLastError();
}

hipError_t cell_sort_finish(int n, int num_host, const int* d_num, uint32_t pad_key, const Grid& g,
                            uint32_t* start, uint32_t* end, uint32_t* sub, uint32_t* keys, uint32_t* idx,
                            const float4* pu, const float4* vu, const float4* eu, float4* ps, float4* vs, float4* es,
                            void* temp, hipStream_t st, const float4* cu, float4* cs, int* left) {
    (void)hipGetLastError();   // drop a stale error left by unrelated earlier HIP calls
    if (n <= 0) return hipSuccess;
    if (one_block(n, g.nb_cells))   // place has made the order
        return launch_cells_permute(num_host, d_num, keys, g.nb_cells, start, end, kSubBits, sub, idx, pu, vu, eu, ps,
                                    vs, es, st, cu, cs, left);
    CellTemp t;
    cell_layout(n, g.nb_cells, &t, (char*)temp);
    k_cell_finish<<<cs_blocks(n), kCsThreads, 0, st>>>(n, num_host, d_num, pad_key, t.pairs, g.nb_cells, start, end, sub,
                                                       keys, idx, pu, vu, eu, ps, vs, es, cu, cs, left);
    return hipGetLastError();
}

}  // namespace rtps
