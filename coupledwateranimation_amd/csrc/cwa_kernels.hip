// cwa_kernels.hip — CDNA4 (gfx950) kernels of the coupled SPH +
// heightfield-wave step.
//
// Data layout in HBM (one scene):
//   particles  SoA float4 pos / vel / force + int id, in cell-sorted order;
//              two copies (A = state, B = this step's reorder target)
//   work       rho_w (float), pw (float2: pressure, 1/rho), flux (float),
//              packed points (uint32 per sorted particle, large scenes)
//   grid       key (int per particle), count and head (int per cell), link
//              (int2 per run), offset (int per cell + 1), list (int per particle)
//   wave       three W*H fp32 fields (newest, previous, write)
//
// Reference kernels replaced (paths relative to the reference root):
//   ugrid_particles_cs.glsl (hash / count / insert)  -> k_hash_count,
//       k_stable_reorder
//   prefix_sum_cs.glsl + ParallelScan.cpp            -> k_scan_*
//   rho_pres_comp.glsl                               -> k_density
//   force_comp.glsl + integrate_comp.glsl            -> k_force_integrate
//   wave_comp.glsl (EVOLVE, INIT)                    -> k_wave, k_init_wave
//   particle -> heightfield flux (no reference)      -> column blocks of
//                                                       k_force_integrate
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>

#include "cwa_device.hpp"
#include "cwa_kernels.hpp"

namespace cwa {

static std::atomic<long long> g_lane_split{kLaneSplitDefault};
long long lane_split_limit() { return g_lane_split.load(std::memory_order_relaxed); }
long long set_lane_split_limit(long long max_n) { return g_lane_split.exchange(max_n); }

// ---------------------------------------------------------------------------
// utilities
// ---------------------------------------------------------------------------
__global__ void k_fill_i32(int* __restrict__ p, int n, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Zeroes up to five int arrays of n (the first: n + 1) in one launch.
struct ClearList {
    int* p[5];
};
__global__ void __launch_bounds__(256) k_clear_cells(ClearList l, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 && l.p[0]) l.p[0][n] = 0;
    if (i >= n) return;
#pragma unroll
    for (int k = 0; k < 5; ++k)
        if (l.p[k]) l.p[k][i] = 0;
}

// ---------------------------------------------------------------------------
// Exclusive scan of int32 (replaces the Blelloch tree of
// prefix_sum_cs.glsl:18-43, which needs 2 log2(n) dispatches and a
// power-of-two n).  Reduce-then-scan over tiles of kScanTile elements:
//   k_scan_reduce  tile sums
//   (recursive scan of the tile sums)
//   k_scan_down    tile-local exclusive scan + tile prefix
// Block-level scans are wave64 shuffle scans plus one LDS exchange of the
// four wave totals.
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 256;

// Lists the run of counted item i (every lane of the wave calls it).
__device__ __forceinline__ void link_runs(int i, const LinkRuns& lr) {
    const bool valid = i < lr.n;
    push_runs<false, true>(valid ? lr.key[i] : -1, valid, i, CellRuns{nullptr, lr.head, lr.link});
}
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;  // 2048
constexpr int kScanDirectTiles = 1024;  // tile prefixes summed in-kernel up to here

__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// The kScanItems (8) consecutive values of a thread: two 16-byte loads when
// the whole chunk is in range and the array is 16-byte aligned (a chunk
// starts at a multiple of 8 ints), element loads otherwise.
__device__ __forceinline__ bool aligned16(const void* p) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

__device__ __forceinline__ void load_items(const int* __restrict__ in, int base, int n,
                                           int v[kScanItems]) {
    if (base + kScanItems <= n && aligned16(in)) {
        const int4 a = *reinterpret_cast<const int4*>(in + base);
        const int4 b = *reinterpret_cast<const int4*>(in + base + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
        v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) v[k] = (base + k < n) ? in[base + k] : 0;
    }
}

__device__ __forceinline__ void store_items(int* __restrict__ out, int base, int n,
                                            const int v[kScanItems]) {
    if (base + kScanItems <= n && aligned16(out)) {
        *reinterpret_cast<int4*>(out + base) = make_int4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<int4*>(out + base + 4) = make_int4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (base + k < n) out[base + k] = v[k];
    }
}

__device__ __forceinline__ int wave_sum_i32(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Exclusive scan of one value per thread across the block; returns the
// exclusive prefix and the block total.
__device__ __forceinline__ int block_excl_scan(int v, int& total) {
    __shared__ int wsum[kScanThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int incl = wave_incl_scan(v);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    int before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        const int s = wsum[w];
        before += (w < wid) ? s : 0;
        tot += s;
    }
    __syncthreads();
    total = tot;
    return before + incl - v;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_apply(const int* __restrict__ in, int n,
                                                             const int* __restrict__ tile_prefix,
                                                             int* __restrict__ out,
                                                             int* __restrict__ zero_out,
                                                             int* __restrict__ zero_out2) {
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    load_items(in, base, n, v);
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    int total;
    int run = block_excl_scan(s, total) + tile_prefix[blockIdx.x];
    int o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        o[k] = run;
        run += v[k];
    }
    store_items(out, base, n, o);
    const int z[kScanItems] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (zero_out) store_items(zero_out, base, n, z);
    if (zero_out2) store_items(zero_out2, base, n, z);
}

// Sum of one tile per block.  With runs listed (lr.n > 0) the blocks past the
// tiles do k_link_runs' work: both passes only read what is there before them, and
// a launch of its own takes about as long as either's work (MI355X, runs + sums -> one
// launch: 300 007 particles 5.2 + 4.5 -> 5.3 us, 1 048 576 6.7 + 4.9 -> 7.2; 24 steps at
// 300 007 1 416 -> 1 386 us).
__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(const int* __restrict__ in, int n,
                                                              int* __restrict__ part, int tiles,
                                                              LinkRuns lr) {
    static_assert(kScanThreads == 256, "the item passes' blocks");
    if ((int)blockIdx.x >= tiles) {
        link_runs(((int)blockIdx.x - tiles) * kScanThreads + (int)threadIdx.x, lr);
        return;
    }
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    load_items(in, base, n, v);
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    __shared__ int wsum[kScanThreads / 64];
    s = wave_sum_i32(s);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < kScanThreads / 64; ++w) t += wsum[w];
        part[blockIdx.x] = t;
    }
}

// Exclusive scan of one tile per block.  The tile's prefix is the sum of
// the tile sums before it (part[0 .. blockIdx.x), summed by the block
// itself; null part: single tile).  total_out (optional) receives the grand
// total, written by the last block.  zero_out and zero_out2 (optional) are
// cleared over the same index range (the other halves of the double-buffered
// cell counters and run-list heads).
__global__ void __launch_bounds__(kScanThreads) k_scan_down(const int* __restrict__ in, int n,
                                                            const int* __restrict__ part,
                                                            int* __restrict__ out,
                                                            int* __restrict__ total_out,
                                                            int* __restrict__ zero_out,
                                                            int* __restrict__ zero_out2) {
    int prefix = 0;
    if (part) {
        int s = 0;
        for (int t = threadIdx.x; t < (int)blockIdx.x; t += kScanThreads) s += part[t];
        int tot;
        (void)block_excl_scan(s, tot);
        prefix = tot;
    }
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    load_items(in, base, n, v);
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    int total;
    int run = block_excl_scan(s, total) + prefix;
    int o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        o[k] = run;
        run += v[k];
    }
    store_items(out, base, n, o);
    const int z[kScanItems] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (zero_out) store_items(zero_out, base, n, z);
    if (zero_out2) store_items(zero_out2, base, n, z);
    if (total_out && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *total_out = total + prefix;
}

// The whole scan in one launch, for inputs of up to kScanOneTiles tiles of
// kScanOneTile: each block sums the elements before its tile itself (from the
// L2, kScanOneAhead 16-byte loads in flight per thread) instead of waiting for
// a launch that has summed them.  Quadratic reads, so only while a block's
// share is a few rounds (MI355X, us a step, two launches -> one: 15 625 cells 14.0
// -> 13.6 with three scenes in flight, 46 656 25.6 -> 22.6; at 157 464 cells 22.5
// -> 24.0, at 202 612 the scan itself 9.4 -> 11.6); the input must not change
// during the launch, so it must not overlap what is written.
constexpr int kScanOneThreads = 1024;
constexpr int kScanOneTile = kScanOneThreads * kScanItems;  // 8192
constexpr int kScanOneTiles = 8;
constexpr int kScanOneAhead = 8;

__global__ void __launch_bounds__(kScanOneThreads)
    k_scan_one(const int* __restrict__ in, int n, int* __restrict__ out,
               int* __restrict__ total_out, int* __restrict__ zero_out,
               int* __restrict__ zero_out2) {
    const int first = blockIdx.x * kScanOneTile;
    int pre = 0;
    if (aligned16(in)) {
        const int4* __restrict__ q = reinterpret_cast<const int4*>(in);
        const int end = first / 4;  // a multiple of 2 * kScanOneThreads
        for (int t = threadIdx.x; t < end; t += kScanOneAhead * kScanOneThreads) {
            int4 a[kScanOneAhead];
#pragma unroll
            for (int u = 0; u < kScanOneAhead; ++u) {
                const int k = t + u * kScanOneThreads;
                a[u] = k < end ? q[k] : make_int4(0, 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < kScanOneAhead; ++u) pre += a[u].x + a[u].y + a[u].z + a[u].w;
        }
    } else {
        for (int t = threadIdx.x; t < first; t += kScanOneThreads) pre += in[t];
    }
    const int base = first + threadIdx.x * kScanItems;
    int v[kScanItems];
    load_items(in, base, n, v);
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    // one exchange for both: the waves' tile totals and their shares of the prefix
    constexpr int kWaves = kScanOneThreads / 64;
    __shared__ int wsum[kWaves], wpre[kWaves];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int incl = wave_incl_scan(s);
    pre = wave_sum_i32(pre);
    if (lane == 63) {
        wsum[wid] = incl;
        wpre[wid] = pre;
    }
    __syncthreads();
    int run = incl - s, total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        run += wpre[w] + (w < wid ? wsum[w] : 0);
        total += wpre[w] + wsum[w];
    }
    int o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        o[k] = run;
        run += v[k];
    }
    store_items(out, base, n, o);
    const int z[kScanItems] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (zero_out) store_items(zero_out, base, n, z);
    if (zero_out2) store_items(zero_out2, base, n, z);
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *total_out = total;
}

__global__ void k_scan_total(const int* __restrict__ src, int* __restrict__ dst) {
    if (threadIdx.x == 0) *dst = *src;
}

// Workspace per recursion level with t tiles: tile sums (t) followed by
// their exclusive scan (t + 1, the last entry being the level total).
size_t scan_workspace_ints(int n) {
    size_t ws = 0;
    int m = n;
    while (m > kScanTile * kScanDirectTiles) {
        const int tiles = (m + kScanTile - 1) / kScanTile;
        ws += 2 * (size_t)tiles + 1;
        m = tiles;
    }
    return ws + (size_t)(m + kScanTile - 1) / kScanTile + 1;
}

// Runs of items that are already counted.
__global__ void __launch_bounds__(256) k_link_runs(LinkRuns lr) {
    link_runs(blockIdx.x * blockDim.x + threadIdx.x, lr);
}

// Whether the int arrays [a, a + na) and [b, b + nb) share memory (null: no).
static bool overlap(const int* a, size_t na, const int* b, size_t nb) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(a), q = reinterpret_cast<uintptr_t>(b);
    return a && b && p < q + nb * sizeof(int) && q < p + na * sizeof(int);
}

static bool takes_one_launch(const int* in, const int* out, int n, const int* zero_out,
                             const int* zero_out2) {
    return n <= kScanOneTile * kScanOneTiles && !overlap(in, n, out, (size_t)n + 1) &&
           !overlap(in, n, zero_out, n) && !overlap(in, n, zero_out2, n);
}

// out has n+1 entries; out[n] = total.  ws holds scan_workspace_ints(n).
// One launch where k_scan_one takes the input, unless it is scanned in place.
// Otherwise, up to kScanDirectTiles tiles the tile prefixes are summed inside
// k_scan_down (two launches); larger inputs recurse on the tile sums.
hipError_t launch_scan(const int* in, int* out, int n, int* ws, hipStream_t st,
                       int* zero_out, int* zero_out2, const LinkRuns& lr) {
    const int link_blocks = (lr.n + kScanThreads - 1) / kScanThreads;
    const bool reduces = n > kScanTile && !takes_one_launch(in, out, n, zero_out, zero_out2);
    if (lr.n > 0 && !reduces) k_link_runs<<<link_blocks, kScanThreads, 0, st>>>(lr);
    if (n <= 0) {
        k_fill_i32<<<1, 64, 0, st>>>(out, 1, 0);
        return hipGetLastError();
    }
    if (takes_one_launch(in, out, n, zero_out, zero_out2)) {
        k_scan_one<<<(n + kScanOneTile - 1) / kScanOneTile, kScanOneThreads, 0, st>>>(
            in, n, out, out + n, zero_out, zero_out2);
        return hipGetLastError();
    }
    const int tiles = (n + kScanTile - 1) / kScanTile;
    if (tiles == 1) {
        k_scan_down<<<1, kScanThreads, 0, st>>>(in, n, nullptr, out, out + n, zero_out,
                                                    zero_out2);
        return hipGetLastError();
    }
    int* part = ws;
    k_scan_reduce<<<tiles + link_blocks, kScanThreads, 0, st>>>(in, n, part, tiles, lr);
    if (tiles <= kScanDirectTiles) {
        k_scan_down<<<tiles, kScanThreads, 0, st>>>(in, n, part, out, out + n, zero_out,
                                                    zero_out2);
        return hipGetLastError();
    }
    int* part_ex = ws + tiles;  // tiles + 1 entries
    hipError_t e = launch_scan(part, part_ex, tiles, ws + 2 * (size_t)tiles + 1, st, nullptr,
                               nullptr);
    if (e != hipSuccess) return e;
    k_scan_apply<<<tiles, kScanThreads, 0, st>>>(in, n, part_ex, out, zero_out, zero_out2);
    k_scan_total<<<1, 64, 0, st>>>(part_ex + tiles, out + n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Uniform grid: a stable counting sort of keyed items (particle slots, or
// (box, cell) pairs).  Replaces the atomicAdd insertion of
// ugrid_particles_cs.glsl:90-117 (whose order within a cell is not
// deterministic) with the UniformGrid2D::Build order (UniformGrid2D.cpp:
// 75-91: items ascending within each cell):
//   count    one atomicAdd per run of equal keys in a wave (lane order),
//            issued by the run's first lane, its result unused.  The same lane
//            pushes the run on its cell's run list: head[c] (first item + 1 of
//            the newest run, 0 for an empty list) is exchanged, and link[first
//            item] records (the older head, the run's length)
//   scan     exclusive scan of the counts -> offsets
//   reorder  the run head walks its cell's run list (one link per run, not one
//            per item) and counts the items of the runs that start before
//            its own; the lanes of the run take that rank plus their
//            distance to the head.  The particle positions and ids move to
//            their sorted slots in the same pass.
// The rank is right because a listed run that starts before a run's head also
// ends before it.  Runs end where the key changes and at the ends of the listing
// wave's items: 64, in step with the reorder's waves, or the 16 of k_force_split,
// whose finer runs still end with the reorder's.  The lists need no offsets, so
// whoever counts the keys can also list the runs; builds of up to
// kFuseLinksMax particles do.  In larger ones k_link_runs lists them, and in large
// builds outside a scene k_place_runs puts them side by side in their cell's
// segment instead (kFuseLinksMax and kListRunsMax give both sides' times).
// ---------------------------------------------------------------------------
// Cell hash + count of particle slots (ComputeCellIndex / Index / ComputeCounts,
// ugrid_particles_cs.glsl:90-108, with the y-fastest linearisation).
template <bool kLink>
__global__ void __launch_bounds__(256) k_hash_count(const float4* __restrict__ pos, int n,
                                                    GridDesc g, int* __restrict__ key,
                                                    CellRuns runs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    int c = -1;
    if (valid) {
        const float4 p = pos[i];
        const int ix = cell_axis(p.x, g.gmin[0], g.cell, g.dims[0]);
        const int iy = cell_axis(p.y, g.gmin[1], g.cell_y, g.dims[1]);
        const int iz = cell_axis(p.z, g.gmin[2], g.cell, g.dims[2]);
        c = lin_cell(g.dims, ix, iy, iz);
        key[i] = c;
    }
    push_runs<true, kLink>(c, valid, i, runs);
}

// Count and runs of items whose keys are already known.
template <bool kLink>
__global__ void __launch_bounds__(256) k_key_count(const int* __restrict__ key, int n,
                                                   CellRuns runs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    push_runs<true, kLink>(valid ? key[i] : -1, valid, i, runs);
}

// The runs of counted items at a place in their cells' segments: (first item, length)
// at the place of the run's first lane, which leaves as many free as the run has
// items.  fill: zero on entry.
__global__ void __launch_bounds__(256) k_place_runs(const int* __restrict__ key,
                                                    const int* __restrict__ offset,
                                                    int* __restrict__ fill, int n,
                                                    int2* __restrict__ runs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const int c = valid ? key[i] : -1;
    const RunInfo r = wave_runs(c);
    if (valid && r.head) {
        const int len = r.run_end - (int)(threadIdx.x & 63);
        runs[offset[c] + atomicAdd(&fill[c], len)] = make_int2(i, len);
    }
}

// Stable destination of every item; list[d] = item_of[item] (or the item
// itself), and the particle positions and ids move to their sorted slots
// when pos_out is set (the passes that follow read velocities and forces in
// their pre-sort slots through list).  The walk ends with the cell's count,
// whatever the links hold.  kLists: the cells' run lists, else the runs placed in
// their segments (link; head is not used).
template <bool kLists>
__global__ void __launch_bounds__(256) k_stable_reorder(
    const int* __restrict__ key, const int* __restrict__ offset, const int* __restrict__ head,
    const int2* __restrict__ link, int n, const int* __restrict__ item_of,
    int* __restrict__ list, const float4* __restrict__ pos_in,
    const int* __restrict__ id_in, float4* __restrict__ pos_out, int* __restrict__ id_out,
    const DevParams* __restrict__ Pd, uint32_t* __restrict__ packed_out) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool valid = s < n;
    const int c = valid ? key[s] : -1;
    const RunInfo r = wave_runs(c);
    int rank = 0;
    if (valid && r.head) {
        const int b = offset[c];
        const int e = offset[c + 1];
        if (kLists) {
            int left = e - b;
            for (int q = head[c]; q > 0 && left > 0;) {
                const int2 u = link[q - 1];
                if (q - 1 < s) rank += u.y;
                left -= max(u.y, 1);
                q = u.x;
            }
        } else {
            for (int q = b; q < e;) {
                const int2 u = link[q];
                if (u.x < s) rank += u.y;
                q += max(u.y, 1);
            }
        }
        rank += b;
    }
    const int d = __shfl(rank, r.my_head, 64) + (lane - r.my_head);
    if (!valid || d < 0 || d >= n) return;  // out of range only on inconsistent run lists
    list[d] = item_of ? item_of[s] : s;
    if (pos_out) {
        // read once (nt): the previous force pass's output leaves the L2 to the
        // sorted copy this pass writes and the next passes gather from (A/B
        // on one box: step 0.2606 -> 0.2548 ms, the force pass 109.6 -> 104.6 us)
        const float4 p = load_once(&pos_in[s]);
        pos_out[d] = p;
        id_out[d] = load_once(&id_in[s]);
        if (packed_out) packed_out[d] = pack_point(*Pd, p);
    }
}

// Boxes (UniformGridPbdGpu3D, uniform_grid_pbd_3D_cs.glsl:145-206): the
// cells a box overlaps are ComputeCellIndex(x - hw) .. ComputeCellIndex(x + hw)
// per axis, with a cell size per axis.
struct BoxGrid {
    float gmin[3];
    float cell[3];
    int dims[3];
};

__device__ __forceinline__ void box_cells(const BoxGrid& g, float4 x, float4 hw, int lo[3],
                                          int hi[3]) {
#pragma clang fp contract(off)
    const float a[3] = {x.x - hw.x, x.y - hw.y, x.z - hw.z};
    const float b[3] = {x.x + hw.x, x.y + hw.y, x.z + hw.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lo[k] = cell_axis(a[k], g.gmin[k], g.cell[k], g.dims[k]);
        hi[k] = cell_axis(b[k], g.gmin[k], g.cell[k], g.dims[k]);
    }
}

// Number of cells each box overlaps (0 for a box whose corners cross).
__global__ void __launch_bounds__(256) k_box_cover(const float4* __restrict__ x,
                                                   const float4* __restrict__ hw, int n,
                                                   BoxGrid g, int* __restrict__ ncov) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int lo[3], hi[3];
    box_cells(g, x[i], hw[i], lo, hi);
    long long m = 1;
#pragma unroll
    for (int k = 0; k < 3; ++k) m *= (long long)max(hi[k] - lo[k] + 1, 0);
    ncov[i] = (int)m;
}

// 64-bit sum of n ints (one atomic per wave), for totals an int scan would wrap.
__global__ void __launch_bounds__(256) k_sum_i64(const int* __restrict__ a, int n,
                                                 unsigned long long* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    long long v = i < n ? (long long)a[i] : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(out, (unsigned long long)v);
}

// The (box, cell) pairs in box order, the cells of a box x-outer, then y,
// then z (InsertBox's loop order): pair p = first[i] + t.
__global__ void __launch_bounds__(256) k_box_pairs(const float4* __restrict__ x,
                                                   const float4* __restrict__ hw, int n,
                                                   BoxGrid g, const int* __restrict__ first,
                                                   int* __restrict__ pkey,
                                                   int* __restrict__ pbox) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int lo[3], hi[3];
    box_cells(g, x[i], hw[i], lo, hi);
    int p = first[i];
    for (int a = lo[0]; a <= hi[0]; ++a)
        for (int b = lo[1]; b <= hi[1]; ++b)
            for (int c = lo[2]; c <= hi[2]; ++c) {
                pkey[p] = (a * g.dims[2] + c) * g.dims[1] + b;  // untiled, y fastest
                pbox[p] = i;
                ++p;
            }
}

// ---------------------------------------------------------------------------
// Neighbour columns: candidate column c = 0..8 is (dx, dz) = (c/3 - 1,
// c%3 - 1) (dx outer, dz inner, the oracle's order); its candidates are the
// contiguous sorted range of cells iy-1..iy+1 of that column.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool coupled(const DevParams& P, float y, float H) {
    return !(P.band > 0.0f) || fabsf(y - H) < P.band;
}

// One density candidate: w = max(T - r2, 0) with T the exact threshold
// (r < h  <=>  r2 < T), so w > 0 exactly for neighbours; accumulates w^3 and
// sets mask bit k for a neighbour.
__device__ __forceinline__ void density_candidate(const float4 pi, const float4 pj, float T,
                                                  float& acc, uint32_t& word, int k) {
    const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const float r2 = dist2_fma(dx, dy, dz);
    const float w = fmaxf(T - r2, 0.0f);
    acc = fmaf(w * w, w, acc);
    word |= min(__float_as_uint(w), 1u) << k;
}

// What both density kernels do with a particle's kernel sum and the surface
// height above it: EOS, wave term, rest-density clamp, the neighbour record
// and the particle flux.
__device__ __forceinline__ void density_finish(const DevParams& P, int i, float4 pi, float4 vi,
                                               float acc, float height,
                                               float* __restrict__ rho_w,
                                               float2* __restrict__ pw, float* __restrict__ flux,
                                               float4* __restrict__ nrec,
                                               float* __restrict__ rho_raw) {
    float rho = P.m_poly6 * acc;
    if (rho_raw) rho_raw[i] = rho;  // taped for the adjoint
    float pressure = fmaxf(P.k * (rho - P.rho0), 0.0f);
    if (coupled(P, pi.y, height)) {
        const float wf = height * rho;
        pressure += wf;
        rho += wf / P.k_rp;
    }
    rho = fmaxf(P.rho0, rho);
    const float irho = 1.0f / rho;
    rho_w[i] = rho;
    if (pw) pw[i] = make_float2(pressure, irho);  // taped for the adjoint
    // the 32-byte record the force pass reads for this particle as a neighbour
    nrec[2 * (size_t)i] = make_float4(pi.x, pi.y, pi.z, pressure);
    nrec[2 * (size_t)i + 1] = make_float4(vi.x, vi.y, vi.z, irho);
    float fl = 0.0f;
    if (P.band > 0.0f) {
        const float d = fabsf(pi.y - height);
        if (d < P.band) {
            const float qq = d / P.band;
            const float w = (1.0f - qq * qq) * (1.0f - qq * qq);
            fl = P.m_rho0 * vi.y * w;
        }
    }
    flux[i] = fl;
}

// ---------------------------------------------------------------------------
// Density / pressure (rho_pres_comp.glsl:49-81) + particle flux term.
// Also records the exact neighbour set of every particle as neighbour words
// (the packed non-empty words of each candidate column's 32-candidate
// chunks, the particle itself left out; layout at kNbEntries).
//
// One lane per particle, in two stages.  The first goes over the candidate
// columns (rows within h of the particle) and tests the candidates' packed
// points, 4 bytes and 3 VALU instructions a candidate, which leaves the
// neighbours and a few more as words in LDS.  The second visits only those, in
// one flat loop, by the exact distance, and takes the others out of the words.
// Neighbours are summed in candidate order.
//
// What bounds it is the address unit (77 % busy at 1 048 576 particles), by
// the bytes its loads hand to the lanes: testing all ~120 candidates of a
// particle by their 16-byte positions took 125.7 us at 1 048 576 particles and
// 44.5 at 300 007 (3 780 VALU instructions a wave), this takes 87.1 and 33.5
// (2 490).  Measured at 1 048 576: kPackFirst 16, 20, 24: 102, 88.4, 90.8;
// kDensityBatch 3, 4, 6, 8: 87.1, 88.4, 91.2, 94.5; batches that end with their
// word (fewer instructions, more idle loads) 94.9; rows cut to the support
// sphere per column cost what their candidates save.
// ---------------------------------------------------------------------------
struct alignas(4) PackedQuad {
    uint32_t v[4];
};
// Bits kFrom .. kTo - 1: which of the points q[kFrom .. kTo) may be a neighbour.
template <int kFrom, int kTo>
__device__ __forceinline__ uint32_t pack_chunk(const uint32_t* __restrict__ q, uint32_t own,
                                               int bias) {
    constexpr int kNum = kTo - kFrom;
    PackedQuad v[kNum / 4];
#pragma unroll
    for (int k = 0; k < kNum / 4; ++k)
        v[k] = *reinterpret_cast<const PackedQuad*>(q + kFrom + 4 * k);
    uint32_t bits = 0;
#pragma unroll
    for (int k = 0; k < kNum; ++k) pack_test(own, v[k / 4].v[k % 4], bias, bits);
    return __brev(bits) >> (32 - kTo);
}
constexpr int kPackFirst = 20;  // candidates of a chunk tested without a look at their number
constexpr int kDensityBatch = 3;  // exact tests whose loads are in flight together

__global__ void __launch_bounds__(256) k_density(
    const DevParams* __restrict__ Pd, const float4* __restrict__ pos,
    const uint32_t* __restrict__ packed, const float4* __restrict__ vel,
    const int* __restrict__ list, const int* __restrict__ offset, int n,
    const float* __restrict__ H0, float* __restrict__ rho_w, float2* __restrict__ pw,
    float* __restrict__ flux, uint2* __restrict__ nbw, float4* __restrict__ nrec,
    float* __restrict__ rho_raw, float4* __restrict__ vel_out, float* __restrict__ vpad) {
    const DevParams& P = *Pd;
    const int i = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 pi = pos[i];
    const float4 vi = vel[list[i]];  // the state's velocity, in its pre-sort slot
    if (vel_out) vel_out[i] = vi;
    vpad[i] = vi.w;
    const int ix = cell_axis(pi.x, P.gmin[0], P.cell, P.dims[0]);
    const int iz = cell_axis(pi.z, P.gmin[2], P.cell, P.dims[2]);
    const float T = P.r2_lt;
    float acc = 0.0f;
    __shared__ uint2 s_held[kNbHeld][256];
    uint2* const held = &s_held[0][threadIdx.x];
    int w = 0;    // words in LDS
    int out = 0;  // words given out
    uint2* plane = nbw + i;
    // second stage: the words in LDS
    const auto flush = [&]() {
        uint32_t cur = 0, base = 0;
        const int end = w * 256;
        int t = 0;  // the word after cur's, as an index into held
        for (;;) {
            uint32_t j[kDensityBatch], bit[kDensityBatch];
            int at[kDensityBatch];
#pragma unroll
            for (int u = 0; u < kDensityBatch; ++u) {
                if (cur == 0u && t < end) {
                    const uint2 v = held[t];
                    cur = v.x;
                    base = v.y;
                    t += 256;
                }
                bit[u] = cur & (0u - cur);
                at[u] = t - 256;
                j[u] = base + (uint32_t)__builtin_ctz(max(cur, 1u));
                cur &= cur - 1u;
            }
            if (bit[0] == 0u) break;
            float4 a[kDensityBatch];
#pragma unroll
            for (int u = 0; u < kDensityBatch; ++u) a[u] = pos[j[u]];
#pragma unroll
            for (int u = 0; u < kDensityBatch; ++u) {
                const float r2 = dist2_fma(pi.x - a[u].x, pi.y - a[u].y, pi.z - a[u].z);
                // > 0 exactly for neighbours; slots past the last word count nothing
                const float ww = fmaxf((u == 0 || bit[u] ? T : 0.0f) - r2, 0.0f);
                acc = fmaf(ww * ww, ww, acc);
                if (!(ww > 0.0f)) atomicAnd(&held[at[u]].x, ~bit[u]);
            }
        }
#pragma unroll
        for (int k = 0; k < kNbHeld; ++k) {
            if (k < w) {
                uint2 v = held[k * 256];
                const uint32_t self = (uint32_t)i - v.y;
                if (self < 32u) v.x &= ~(1u << self);
                if (v.x) {
                    if (out < kNbEntries) {
                        *plane = v;
                        plane += n;
                    }
                    ++out;
                }
            }
        }
        w = 0;
    };
    const int ylo = cell_axis(pi.y - P.h - P.grid_eps, P.gmin[1], P.cell_y, P.dims[1]);
    const int yhi = cell_axis(pi.y + P.h + P.grid_eps, P.gmin[1], P.cell_y, P.dims[1]);
    const uint32_t own = packed[i];
    const int bias = __any(pack_far(P, pi)) ? INT32_MIN : -kPackLt;
    // first cell of column (ix - 1, iz - 1 + k), and the step to the next ix
    int first[3], step[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int cz = min(max(iz + k - 1, 0), P.dims[2] - 1);
        first[k] = grid_column(P.dims, ix, cz) * P.dims[1];
        step[k] = grid_column(P.dims, ix + 1, cz) * P.dims[1] - first[k];
        first[k] -= step[k];
    }
#pragma unroll 1
    for (int dx = 0; dx < 3; ++dx) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int cx = ix + dx - 1, cz = iz + k - 1;
            int b = 0, e = 0;
            if (cx >= 0 && cx < P.dims[0] && cz >= 0 && cz < P.dims[2]) {
                b = offset[first[k] + ylo];
                e = offset[first[k] + yhi + 1];
            }
            first[k] += step[k];
            for (; b < e; b += 32) {
                const int len = e - b;
                uint32_t bits = pack_chunk<0, kPackFirst>(packed + b, own, bias);
                if (len > kPackFirst) bits |= pack_chunk<kPackFirst, 32>(packed + b, own, bias);
                if (len < 32) bits &= ~(~0u << len);
                if (bits) held[w++ * 256] = make_uint2(bits, (uint32_t)b);
                if (__any(w == kNbHeld)) flush();
            }
        }
    }
    flush();
    nb_count(nbw, n)[i] = out > kNbEntries ? -1 : out;
    const float u = (pi.x - P.org[0]) * P.uvs[0];
    const float v = (pi.z - P.org[1]) * P.uvs[1];
    density_finish(P, i, pi, vi, acc, tex_sample(H0, P.W, P.H, u, v), rho_w, pw, flux, nrec,
                   rho_raw);
}

// Density for scenes of up to lane_split_limit() particles: kDensitySplit
// consecutive lanes per particle, each testing every kDensitySplit-th
// candidate of each column, so a scene of some ten thousand particles still
// keeps several waves per SIMD busy.  The group's neighbour bits are OR-ed
// together (k_density's neighbours, in its order), its partial sums added in a
// fixed tree, and the group's first lane finishes the particle.
//
// At these sizes the pass is one dependent chain per wave, not throughput: nine
// columns, each an offset load, then candidate loads a few at a time.  So the
// lanes of a group look up all nine column ranges at once (three each), a
// column's first kAhead candidates are loaded while the column before is
// summed, and the surface taps are loaded first.  Each lane still adds its
// candidates in the same order.  MI355X, before -> after: 4 096 particles 21.4
// -> 12.1 us, 65 536 25.5 -> 17.9, 130 000 32.1 -> 24.5, 250 000 55.6 -> 42.4
// (kAhead 16, 20, 24, 32 at 65 536: 18.9, 19.2, 17.9, 18.8; at 250 000: 44.9,
// 40.2, 42.4, 50.2; slots guarded by branches instead of filled: 20.6 / 62.2).
constexpr int kDensitySplit = 4;
constexpr int kAhead = 24;  // candidates of a column loaded ahead
constexpr int kSplitAhead = kAhead / kDensitySplit;

// The lane's first U candidates of slots [b, e), every kDensitySplit-th; slots past the end
// hold a point infinitely far away.
template <int U>
struct SplitAhead {
    float4 a[U];
    __device__ __forceinline__ void load(const float4* __restrict__ pos, int b, int e, int sub) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = make_float4(INFINITY, 0.0f, 0.0f, 0.0f);
            const int j = b + sub + u * kDensitySplit;
            if (j < e) a[u] = pos[j];
        }
    }
};

__global__ void __launch_bounds__(256) k_density_split(
    const DevParams* __restrict__ Pd, const float4* __restrict__ pos,
    const float4* __restrict__ vel, const int* __restrict__ list,
    const int* __restrict__ offset, int n, const float* __restrict__ H0,
    float* __restrict__ rho_w, float2* __restrict__ pw, float* __restrict__ flux,
    uint2* __restrict__ nbw, float4* __restrict__ nrec, float* __restrict__ rho_raw,
    float4* __restrict__ vel_out, float* __restrict__ vpad) {
    const DevParams& P = *Pd;
    const int sub = threadIdx.x & (kDensitySplit - 1);
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kDensitySplit);
    if (i >= n) return;  // whole groups: the lanes of a group share i
    const float4 pi = pos[i];
    const int src = list[i];
    const int ix = cell_axis(pi.x, P.gmin[0], P.cell, P.dims[0]);
    const int iz = cell_axis(pi.z, P.gmin[2], P.cell, P.dims[2]);
    int rb[3], re[3];  // columns sub, sub + 4, sub + 8
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        rb[q] = re[q] = 0;
        const int c = sub + q * kDensitySplit;
        if (c < 9) column_range(P, offset, pi.x, pi.y, pi.z, ix, iz, c, rb[q], re[q]);
    }
    const TexTaps taps = tex_taps(H0, P.W, P.H, (pi.x - P.org[0]) * P.uvs[0],
                                  (pi.z - P.org[1]) * P.uvs[1]);
    const float4 vi = vel[src];  // the state's velocity, in its pre-sort slot
    const float T = P.r2_lt;
    float acc = 0.0f;
    // words kept by the group's first lane
    __shared__ uint2 s_held[kNbHeld][256 / kDensitySplit];
    NbWriter wr(&s_held[0][threadIdx.x / kDensitySplit], 256 / kDensitySplit);
    bool tail = false;  // a column longer than kNbMaxColumn candidates
    const auto column = [&](const SplitAhead<kSplitAhead>& cur, int b, int e) {
        const int len = e - b;
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int u = 0; u < kSplitAhead; ++u)
            density_candidate(pi, cur.a[u], T, acc, lo, sub + u * kDensitySplit);
        if (len > kAhead) {  // uniform in the group
            SplitAhead<8 - kSplitAhead> rest;
            rest.load(pos, b + kAhead, e, sub);
#pragma unroll
            for (int u = 0; u < 8 - kSplitAhead; ++u)
                density_candidate(pi, rest.a[u], T, acc, lo, kAhead + sub + u * kDensitySplit);
        }
        lo = quad_or(lo);
        if (len > 32) {  // uniform in the group
            uint32_t none = 0;
            int k = 32 + sub;
            for (; k < len && k < 64; k += kDensitySplit)
                density_candidate(pi, pos[b + k], T, acc, hi, k - 32);
            for (; k < len; k += kDensitySplit) density_candidate(pi, pos[b + k], T, acc, none, 0);
            hi = quad_or(hi);
            tail |= len > kNbMaxColumn;
        }
        const uint32_t self = (uint32_t)(i - b);  // i is a candidate of one column
        if (self < 32u) lo &= ~(1u << self);
        else if (self < 64u) hi &= ~(1u << (self - 32u));
        if (sub == 0) {
            wr.put(nbw, n, i, lo, (uint32_t)b);
            wr.put(nbw, n, i, hi, (uint32_t)b + 32u);
        }
    };
    SplitAhead<kSplitAhead> A, B;
    const int b0 = quad_bcast<0>(rb[0]), e0 = quad_bcast<0>(re[0]);
    const int b1 = quad_bcast<1>(rb[0]), e1 = quad_bcast<1>(re[0]);
    const int b2 = quad_bcast<2>(rb[0]), e2 = quad_bcast<2>(re[0]);
    const int b3 = quad_bcast<3>(rb[0]), e3 = quad_bcast<3>(re[0]);
    const int b4 = quad_bcast<0>(rb[1]), e4 = quad_bcast<0>(re[1]);
    const int b5 = quad_bcast<1>(rb[1]), e5 = quad_bcast<1>(re[1]);
    const int b6 = quad_bcast<2>(rb[1]), e6 = quad_bcast<2>(re[1]);
    const int b7 = quad_bcast<3>(rb[1]), e7 = quad_bcast<3>(re[1]);
    const int b8 = quad_bcast<0>(rb[2]), e8 = quad_bcast<0>(re[2]);
    A.load(pos, b0, e0, sub);
    B.load(pos, b1, e1, sub);
    column(A, b0, e0);
    A.load(pos, b2, e2, sub);
    column(B, b1, e1);
    B.load(pos, b3, e3, sub);
    column(A, b2, e2);
    A.load(pos, b4, e4, sub);
    column(B, b3, e3);
    B.load(pos, b5, e5, sub);
    column(A, b4, e4);
    A.load(pos, b6, e6, sub);
    column(B, b5, e5);
    B.load(pos, b7, e7, sub);
    column(A, b6, e6);
    A.load(pos, b8, e8, sub);
    column(B, b7, e7);
    column(A, b8, e8);
    acc = quad_sum(acc);
    if (sub != 0) return;
    wr.finish(nbw, n, i, tail);
    if (vel_out) vel_out[i] = vi;
    vpad[i] = vi.w;
    density_finish(P, i, pi, vi, acc, taps.value(), rho_w, pw, flux, nrec, rho_raw);
}

// Pressure + viscosity contribution of one neighbour (force_comp.glsl:85-86).
struct PairAcc {
    float pfx, pfy, pfz, vfx, vfy, vfz;
};

// Neighbour record written by the density pass: (x, y, z, p), (vx, vy, vz, 1/rho),
// one 32-byte block per particle so a neighbour costs one cache line.
struct Nbr {
    float4 a;
    float4 b;
};

__device__ __forceinline__ Nbr load_nbr(const float4* __restrict__ nrec, int j) {
    return Nbr{nrec[2 * (size_t)j], nrec[2 * (size_t)j + 1]};
}

// The value of the other lane of a pair (lane ^ 1, both active).
__device__ __forceinline__ int pair_swap(int v) {
    return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);
}
__device__ __forceinline__ float4 pair_swap(float4 v) {
    const auto f = [](float x) { return __int_as_float(pair_swap(__float_as_int(x))); };
    return make_float4(f(v.x), f(v.y), f(v.z), f(v.w));
}
__device__ __forceinline__ float4 select4(bool c, float4 a, float4 b) {
    return make_float4(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w);
}

// load_nbr by the two lanes of a pair together: each load instruction takes
// both halves of one lane's record, so a record costs the cache one access
// instead of two, and the lanes swap the halves they loaded for each other.
// The even lane's record comes with the first half in the even lane, the odd
// lane's with the first half in the odd lane: what is swapped is always a
// second half.  The force pass is bound by those accesses (address unit 81 %
// busy, 45 cache accesses a load instruction): 1 048 576 particles 105 -> 94
// us, 300 007 38.4 -> 33.8, for 17 VALU instructions more a record.
__device__ __forceinline__ Nbr load_nbr_pair(const float4* __restrict__ nrec, int j) {
    const bool odd = threadIdx.x & 1;
    const int other = pair_swap(j);
    const float4 x = nrec[2 * (size_t)(odd ? other : j) + (odd ? 1 : 0)];
    const float4 y = nrec[2 * (size_t)(odd ? j : other) + (odd ? 0 : 1)];
    return Nbr{select4(odd, y, x), pair_swap(select4(odd, x, y))};
}

__device__ __forceinline__ void force_pair(float h, float4 pi, float4 vi, float p_i,
                                           float m_spiky_half, float m_lap, const Nbr& nb,
                                           PairAcc& a) {
    const float dx = pi.x - nb.a.x, dy = pi.y - nb.a.y, dz = pi.z - nb.a.z;
    const float r2 = dist2_fma(dx, dy, dz);
    // an exactly coincident pair (possible after boundary clamping) has no
    // pressure direction: rinv = 0 drops that term
    const float rinv = r2 > 0.0f ? __builtin_amdgcn_rsqf(r2) : 0.0f;
    const float r = r2 * rinv;
    const float hr = h - r;
    const float s = m_spiky_half * (p_i + nb.a.w) * nb.b.w * hr * hr * rinv;
    a.pfx -= s * dx;
    a.pfy -= s * dy;
    a.pfz -= s * dz;
    const float t = m_lap * nb.b.w * hr;
    a.vfx += t * (nb.b.x - vi.x);
    a.vfy += t * (nb.b.y - vi.y);
    a.vfz += t * (nb.b.z - vi.z);
}

// ---------------------------------------------------------------------------
// Texels of the wave EVOLVE (wave_comp.glsl:171-206; the kernels are further
// down).  Arithmetic is not contracted, so every kernel gives the oracle's
// result bit for bit.  The column flux is read through cf(ix, iz), indices
// inside the column grid.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_texel(const DevParams& P, float C0, float C1, float nn,
                                            float ss, float ee, float ww, int i, bool flux,
                                            float S, float dt) {
#pragma clang fp contract(off)
    float o = P.wc0 * C0 + P.lx * (ee + ww) + P.lz * (nn + ss) - P.wc1 * C1;
    o *= P.atten;
    if (flux) o += P.kappa * dt * (S * P.inv_area);
    if (P.wake && o > P.wake_thr && i == P.W / 2) o += P.wake_amt;
    return o;
}

// Column coordinates of texel i / row j, and the floor()ed coordinate as the
// sampler clamps it.
__device__ __forceinline__ float column_x(const DevParams& P, int i) {
#pragma clang fp contract(off)
    return P.ax * (float)i + P.bx;
}
__device__ __forceinline__ float column_z(const DevParams& P, int j) {
#pragma clang fp contract(off)
    return P.az * (float)j + P.bz;
}
__device__ __forceinline__ int floor_index(float g, int n) {
    return (int)fminf(fmaxf(floorf(g), -2.0f), (float)(n + 1));
}

// bilerp() of the column grid at (gx, gz).
template <class Col>
__device__ __forceinline__ float colflux_at(const DevParams& P, const Col& cf, float gx, float gz) {
#pragma clang fp contract(off)
    const int w = P.dims[0], h = P.dims[2];
    TexTaps t;
    t.a = gx - floorf(gx);
    t.b = gz - floorf(gz);
    const int i0 = floor_index(gx, w), j0 = floor_index(gz, h);
    const int ia = min(max(i0, 0), w - 1), ib = min(max(i0 + 1, 0), w - 1);
    const int ja = min(max(j0, 0), h - 1), jb = min(max(j0 + 1, 0), h - 1);
    t.t00 = cf(ia, ja);
    t.t10 = cf(ib, ja);
    t.t01 = cf(ia, jb);
    t.t11 = cf(ib, jb);
    return t.value();
}

// Column-flux source of texels i0..i0+3 of row j: bilerp of the column grid
// at each texel's (gx, gz), with the same values and arithmetic as bilerp.
// The four samples share gz and, when they fall in at most two adjacent x
// cells (the column grid is much coarser than the texels), also their six
// grid values, loaded once.
template <class Col>
__device__ __forceinline__ void colflux_quad(const DevParams& P, const Col& cf, int i0, int j,
                                             float S[4]) {
#pragma clang fp contract(off)
    const int w = P.dims[0], h = P.dims[2];
    const float gz = column_z(P, j);
    float a[4];
    int ix[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const float gx = column_x(P, i0 + t);
        a[t] = gx - floorf(gx);
        ix[t] = floor_index(gx, w);
    }
    if (ix[3] - ix[0] > 1 || ix[3] < ix[0]) {  // a grid finer than the texels, or mirrored
#pragma unroll
        for (int t = 0; t < 4; ++t) S[t] = colflux_at(P, cf, column_x(P, i0 + t), gz);
        return;
    }
    const float b = gz - floorf(gz);
    const int j0 = floor_index(gz, h);
    const int ra = min(max(j0, 0), h - 1), rb = min(max(j0 + 1, 0), h - 1);
    float r0[3], r1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int ik = min(max(ix[0] + k, 0), w - 1);
        r0[k] = cf(ik, ra);
        r1[k] = cf(ik, rb);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const bool d = ix[t] != ix[0];
        const float t00 = d ? r0[1] : r0[0], t10 = d ? r0[2] : r0[1];
        const float t01 = d ? r1[1] : r1[0], t11 = d ? r1[2] : r1[1];
        const float q0 = (1.0f - a[t]) * t00 + a[t] * t10;
        const float q1 = (1.0f - a[t]) * t01 + a[t] * t11;
        S[t] = (1.0f - b) * q0 + b * q1;
    }
}

// One texel, and four texels along u (W % 4 == 0, i0 % 4 == 0).
template <class Col>
__device__ __forceinline__ void wave_single(const DevParams& P, const float* __restrict__ h0,
                                            const float* __restrict__ h1, float* __restrict__ out,
                                            int i, int j, bool flux, const Col& cf, float dt) {
    const int W = P.W, H = P.H;
    const size_t c = (size_t)j * W + i;
    const float C0 = h0[c];
    const float C1 = h1[c];
    const float nn = h0[(size_t)min(j + 1, H - 1) * W + i];
    const float ss = h0[(size_t)max(j - 1, 0) * W + i];
    const float ee = h0[(size_t)j * W + min(i + 1, W - 1)];
    const float ww = h0[(size_t)j * W + max(i - 1, 0)];
    const float S = flux ? colflux_at(P, cf, column_x(P, i), column_z(P, j)) : 0.0f;
    out[c] = wave_texel(P, C0, C1, nn, ss, ee, ww, i, flux, S, dt);
}

template <class Col>
__device__ __forceinline__ void wave_quad(const DevParams& P, const float* __restrict__ h0,
                                          const float* __restrict__ h1, float* __restrict__ out,
                                          int i0, int j, bool flux, const Col& cf, float dt) {
    const int W = P.W, H = P.H;
    const size_t row = (size_t)j * W;
    const float4 c0 = *reinterpret_cast<const float4*>(h0 + row + i0);
    // the older level is read once, here (nt; A/B on one box: step -0.75 %)
    const float4 c1 = load_once(reinterpret_cast<const float4*>(h1 + row + i0));
    const float4 nn = *reinterpret_cast<const float4*>(h0 + (size_t)min(j + 1, H - 1) * W + i0);
    const float4 ss = *reinterpret_cast<const float4*>(h0 + (size_t)max(j - 1, 0) * W + i0);
    const float west = h0[row + max(i0 - 1, 0)];
    const float east = h0[row + min(i0 + 4, W - 1)];
    float S[4] = {0.f, 0.f, 0.f, 0.f};
    if (flux) colflux_quad(P, cf, i0, j, S);
    float4 o;
    o.x = wave_texel(P, c0.x, c1.x, nn.x, ss.x, c0.y, west, i0, flux, S[0], dt);
    o.y = wave_texel(P, c0.y, c1.y, nn.y, ss.y, c0.z, c0.x, i0 + 1, flux, S[1], dt);
    o.z = wave_texel(P, c0.z, c1.z, nn.z, ss.z, c0.w, c0.y, i0 + 2, flux, S[2], dt);
    o.w = wave_texel(P, c0.w, c1.w, nn.w, ss.w, east, c0.z, i0 + 3, flux, S[3], dt);
    *reinterpret_cast<float4*>(out + row + i0) = o;
}

// ---------------------------------------------------------------------------
// Particle -> wave flux per vertical column of grid cells.  Each column is
// one contiguous sorted range; one wave64 sums memory column `wave`
// (lane-strided partial sums, then a fixed xor tree: deterministic) and
// stores it at [iz*nx + ix] of its (ix, iz).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_sum_f32(float s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

__device__ __forceinline__ void column_flux_sum(const int* __restrict__ offset,
                                                const float* __restrict__ flux, int nx, int ny,
                                                int nz, float* __restrict__ colflux, int wave,
                                                int lane) {
    if (wave >= nx * nz) return;  // uniform across the wave
    const int b = offset[wave * ny], e = offset[(wave + 1) * ny];
    float s = 0.0f;
    for (int k = b + lane; k < e; k += 64) s += flux[k];
    s = wave_sum_f32(s);
    if (lane == 0) {
        const int dims[3] = {nx, ny, nz};
        int ix, iz;
        grid_column_xz(dims, wave, ix, iz);
        colflux[iz * nx + ix] = s;
    }
}

// ---------------------------------------------------------------------------
// The wave EVOLVE as blocks of the force launch (both read only the density
// pass's output and the heightfields): a block of 256 threads advances one
// tile of the heightfield.  It first sums the flux of the columns its texels
// sample (column_flux_sum's order, so the same bits) into LDS, kTileColBatch
// columns of a wave at a time; tiles are small enough that this takes a few
// rounds (wave_tiles_for gives the rule).
//
// That rule went by the parameters of the launch.  A graph replayed with others
// keeps its tiles, so how much of a tile is advanced at once is decided here,
// by the columns it samples with the parameters the kernel reads: the whole
// tile while their sums fit in the LDS, else parts of half the side, a quarter,
// ... (a single texel samples at most four columns).
// ---------------------------------------------------------------------------
constexpr int kTileColBatch = 4;
// Column sums a block has room for, the neighbour words' LDS; colflux_quad may
// load one more (the column east of the last), whose value it does not use.
constexpr int kTileColumnsHeld = kNbStage * 256 * 2 - 1;

__device__ __forceinline__ void wave_tile(const DevParams& P, const WaveTiles& w, int tile,
                                          const int* __restrict__ offset,
                                          const float* __restrict__ pflux, float dt,
                                          float* __restrict__ s_col) {
    const int tx = tile % w.nx, ty = tile / w.nx;
    if (ty * w.side >= P.H) return;  // padding blocks
    const int nx = P.dims[0], ny = P.dims[1], nz = P.dims[2];
    const bool flux = pflux != nullptr;
    for (int side = w.side, level = 0, part = 0; part >> (2 * level) == 0; ++part) {
        const int i_lo = tx * w.side + (part & ((1 << level) - 1)) * side;
        const int j_lo = ty * w.side + (part >> level) * side;
        if (i_lo >= P.W || j_lo >= P.H) continue;
        const int i_hi = min(i_lo + side, P.W) - 1, j_hi = min(j_lo + side, P.H) - 1;
        int x0 = 0, z0 = 0, ncx = 0;
        if (flux) {
            // column coordinates are monotone in the texel index, so the part's
            // first and last texels bound what it samples
            const int xa = floor_index(column_x(P, i_lo), nx);
            const int xb = floor_index(column_x(P, i_hi), nx);
            const int za = floor_index(column_z(P, j_lo), nz);
            const int zb = floor_index(column_z(P, j_hi), nz);
            x0 = min(max(min(xa, xb), 0), nx - 1);
            z0 = min(max(min(za, zb), 0), nz - 1);
            ncx = min(max(max(xa, xb) + 1, 0), nx - 1) - x0 + 1;
            const int ncz = min(max(max(za, zb) + 1, 0), nz - 1) - z0 + 1;
            if ((long long)ncx * ncz > kTileColumnsHeld) {  // again, in parts of half the side
                side >>= 1;
                ++level;
                part = -1;
                continue;
            }
            const int nc = ncx * ncz;
            const int lane = threadIdx.x & 63;
            if (level > 0) __syncthreads();  // the part before has read its columns
            for (int q0 = ((int)threadIdx.x >> 6) * kTileColBatch; q0 < nc;
                 q0 += 4 * kTileColBatch) {
                int k[kTileColBatch], e[kTileColBatch], longest = 0;
                float s[kTileColBatch];
#pragma unroll
                for (int u = 0; u < kTileColBatch; ++u) {
                    s[u] = 0.0f;
                    k[u] = e[u] = 0;
                    if (q0 + u < nc) {
                        const int c = grid_column(P.dims, x0 + (q0 + u) % ncx, z0 + (q0 + u) / ncx);
                        k[u] = offset[c * ny];
                        e[u] = offset[(c + 1) * ny];
                    }
                }
#pragma unroll
                for (int u = 0; u < kTileColBatch; ++u) {
                    longest = max(longest, e[u] - k[u]);
                    k[u] += lane;
                }
                for (; longest > 0; longest -= 64) {
#pragma unroll
                    for (int u = 0; u < kTileColBatch; ++u) {
                        if (k[u] < e[u]) s[u] += pflux[k[u]];
                        k[u] += 64;
                    }
                }
#pragma unroll
                for (int u = 0; u < kTileColBatch; ++u) {
                    s[u] = wave_sum_f32(s[u]);
                    if (lane == 0 && q0 + u < nc) s_col[q0 + u] = s[u];
                }
            }
            __syncthreads();
        }
        const auto cf = [&](int ix, int iz) { return s_col[(iz - z0) * ncx + (ix - x0)]; };
        const int per = P.W % 4 == 0 && side % 4 == 0 ? 4 : 1;  // texels per thread along u
        const int across = side / per;  // a power of two; across * side <= 256 threads
        const int i = i_lo + ((int)threadIdx.x & (across - 1)) * per;
        const int j = j_lo + ((int)threadIdx.x >> __builtin_ctz(across));
        if (i <= i_hi && j <= j_hi) {
            if (per == 4) wave_quad(P, w.h0, w.h1, w.out, i, j, flux, cf, dt);
            else wave_single(P, w.h0, w.h1, w.out, i, j, flux, cf, dt);
        }
    }
}

// What the force pass writes (fpre: only for the adjoint tape).
struct ForceOut {
    float4* __restrict__ pos;
    float4* __restrict__ vel;
    float4* __restrict__ force;
    int* __restrict__ id;
    float* __restrict__ rho;
    float* __restrict__ prs;
    float4* __restrict__ fpre;
};

// What a particle needs after its neighbour sums, loaded where it is used:
// the surface above it and beside it, its density and id.
struct LateInputs {
    const DevParams& P;
    const float* __restrict__ H0;
    const float* __restrict__ rho_w;
    const int* __restrict__ bid;
    float u, v;
    int i;
    __device__ __forceinline__ float height() const { return tex_sample(H0, P.W, P.H, u, v); }
    __device__ __forceinline__ float east_du() const {
        return tex_sample(H0, P.W, P.H, u + P.du, v);
    }
    __device__ __forceinline__ float north_du() const {
        return tex_sample(H0, P.W, P.H, u, v + P.du);
    }
    __device__ __forceinline__ float east() const { return tex_sample(H0, P.W, P.H, u + 1.0f, v); }
    __device__ __forceinline__ float north() const { return tex_sample(H0, P.W, P.H, u, v + 1.0f); }
    __device__ __forceinline__ float rho() const { return load_once(&rho_w[i]); }
    __device__ __forceinline__ int id() const { return load_once(&bid[i]); }
};

// Everything of the force pass after the neighbour sums: crest, viscosity,
// torque, drag and wave force, integration, foam, surface and boundary, and
// the next step's cell key (returned; -1 with key null).
template <class In>
__device__ __forceinline__ int force_finish(const DevParams& P, float dt, int i, float4 pi,
                                            float4 vi, float4 fp, float p_i, const PairAcc& a,
                                            const In& in, const float* __restrict__ H0,
                                            const ForceOut& o, int* __restrict__ key) {
    float vfx = a.vfx, vfy = a.vfy, vfz = a.vfz;
    if (pi.y > P.crest) {
        fp.x /= P.brk_mass;
        fp.y /= P.brk_mass;
        fp.z /= P.brk_mass;
        fp.w /= P.brk_mass;
        vfx *= P.brk_visc;
        vfy *= P.brk_visc;
        vfz *= P.brk_visc;
    }
    vfx *= P.visc;
    vfy *= P.visc;
    vfz *= P.visc;
    const float height = in.height();
    float tqx = (pi.y * fp.z - pi.z * fp.y) * P.torque;
    float tqy = (pi.z * fp.x - pi.x * fp.z) * P.torque;
    float tqz = (pi.x * fp.y - pi.y * fp.x) * P.torque;
    float drx = 0.f, dry = 0.f, drz = 0.f, wfx = 0.f, wfy = 0.f, wfz = 0.f;
    if (coupled(P, pi.y, height)) {
        // WaveVelocity (force_comp.glsl:117-128)
        const float hx = in.east_du();
        const float hy = in.north_du();
        const float wvx = (hx - height) / dt, wvy = (hy - height) / dt, wvz = (hx - hy) / P.du;
        drx = -P.drag * (vi.x - wvx);
        dry = -P.drag * (vi.y - wvy);
        drz = -P.drag * (vi.z - wvz);
        // WaveNormal (force_comp.glsl:131-139) = (H(u+1)-H, H(v+1)-H, -1)
        const float nx = in.east() - height;
        const float ny = in.north() - height;
        wfx = -height * nx * P.wforce;
        wfy = -height * ny * P.wforce;
        wfz = -height * -1.0f * P.wforce;
    }
    float rho = in.rho();
    float prs = p_i;
    float Fx = a.pfx + vfx + rho * P.g[0] + tqx + drx + wfx;
    float Fy = a.pfy + vfy + rho * P.g[1] + tqy + dry + wfy;
    float Fz = a.pfz + vfz + rho * P.g[2] + tqz + drz + wfz;
    float Fw = fp.w;
    if (o.fpre) o.fpre[i] = make_float4(Fx, Fy, Fz, 0.0f);  // taped for the adjoint

    // integrate_comp.glsl:56-92
    float nvx = vi.x + dt * (Fx / rho), nvy = vi.y + dt * (Fy / rho), nvz = vi.z + dt * (Fz / rho);
    float npx = pi.x + dt * nvx, npy = pi.y + dt * nvy, npz = pi.z + dt * nvz;
    const float damp = 1.0f - P.vdamp * dt;
    nvx *= damp;
    nvy *= damp;
    nvz *= damp;
    if (sqrtf(dist2_fma(nvx, nvy, nvz)) > P.foam_speed) {
        Fx *= P.foam_f;
        Fy *= P.foam_f;
        Fz *= P.foam_f;
        Fw *= P.foam_f;
        rho *= P.foam_rho;
        prs *= P.foam_p;
        nvx *= P.foam_v;
        nvy *= P.foam_v;
        nvz *= P.foam_v;
    }
    const float th = tex_sample(H0, P.W, P.H, (npx - P.org[0]) * P.uvs[0],
                                (npz - P.org[1]) * P.uvs[1]);
    if (npy < th) npy = th - P.rp;
    // CheckBoundary (integrate_comp.glsl:135-178)
    if (npx < P.lo[0]) { npx = P.lo[0]; nvx *= -P.bounce; }
    else if (npx > P.up[0]) { npx = P.up[0]; nvx *= -P.bounce; }
    if (npy < P.lo[1]) { npy = P.lo[1]; nvy *= -P.bounce; }
    else if (npy > P.up[1]) { npy = P.up[1]; nvy *= -P.bounce; }
    if (npz < P.lo[2]) { npz = P.lo[2]; nvz *= -P.bounce; }
    else if (npz > P.up[2]) { npz = P.up[2]; nvz *= -P.bounce; }
    if (P.wake) {
        if (npy > P.up[1] + P.ceil_extra) { npy = P.up[1] + P.ceil_extra; nvy *= -P.bounce; }
    }
    o.pos[i] = make_float4(npx, npy, npz, pi.w);
    o.vel[i] = make_float4(nvx, nvy, nvz, vi.w);
    o.force[i] = make_float4(Fx, Fy, Fz, Fw);
    o.id[i] = in.id();
    store_once(&o.rho[i], rho);  // not read by the next step (A/B: step -0.7 %)
    store_once(&o.prs[i], prs);
    if (!key) return -1;
    const int ix = cell_axis(npx, P.gmin[0], P.cell, P.dims[0]);
    const int iy = cell_axis(npy, P.gmin[1], P.cell_y, P.dims[1]);
    const int iz = cell_axis(npz, P.gmin[2], P.cell, P.dims[2]);
    const int cell = lin_cell(P.dims, ix, iy, iz);
    key[i] = cell;
    return cell;
}

// Neighbour records in flight per lane.  At 1 048 576 particles 4, 5, 6, 7, 8, 10
// -> 98.3, 93.8, 94.1, 99.6, 98.9, 101.8 us; at 300 007 6, 8, 10 -> 33.8, 35.9,
// 36.6; the next batch loaded while one is summed, batches of 2, 3, 4: 104.3,
// 97.3, 97.7.
constexpr int kForceBatch = 6;

// ---------------------------------------------------------------------------
// Forces (force_comp.glsl:62-139) fused with symplectic Euler + boundary
// (integrate_comp.glsl:56-92, 135-178).  Visits only the neighbours the
// density pass recorded (its neighbour words, in candidate order).  Reads
// the particle's own record from the density pass (position, pressure,
// velocity), its id from the sorted copy and its previous force from the
// state in its pre-sort slot (list[i]); writes the next state in the sorted
// slot order.  When `next` is set it also hashes the new position into the
// next step's grid (cell key, count and run lists, ComputeCounts of
// ugrid_particles_cs.glsl:90-95), so that step needs no hash pass of its own.
// The grid's last blocks, from nfb on, sum the particle flux per column (one
// wave per column; they read only the density pass's output and run in the
// force blocks' tail).  With kWave the first wt.nblk blocks advance the
// heightfield (wave_tile), which small scenes would otherwise wait on a launch
// for (wave_tiles_for gives the rule and both sides); their number is a
// multiple of eight, so the force blocks keep the density pass's XCDs.
// ---------------------------------------------------------------------------
template <bool kLink, bool kWave>
__global__ void __launch_bounds__(256) k_force_integrate(
    const DevParams* __restrict__ Pd, float dt, const float4* __restrict__ bpos,
    const int* __restrict__ bid, const float* __restrict__ vpad,
    const float4* __restrict__ force, const int* __restrict__ list,
    const int* __restrict__ offset, int n, const float* __restrict__ rho_w,
    const uint2* __restrict__ nbw, const float4* __restrict__ nrec,
    const float* __restrict__ H0, ForceOut out, int nfb, const float* __restrict__ pflux, float* __restrict__ colflux, NextKeys next, WaveTiles wt) {
    const DevParams& P = *Pd;
    __shared__ uint2 s_nb[kNbStage][256];
    static_assert(sizeof(s_nb) >= (kTileColumnsHeld + 1) * sizeof(float), "a tile's column sums");
    if (kWave && (int)blockIdx.x < wt.nblk) {
        wave_tile(P, wt, blockIdx.x, offset, colflux ? pflux : nullptr, dt,
                  reinterpret_cast<float*>(&s_nb[0][0]));
        return;
    }
    const int blk = (int)blockIdx.x - (kWave ? wt.nblk : 0);
    if (blk >= nfb) {
        column_flux_sum(offset, pflux, P.dims[0], P.dims[1], P.dims[2], colflux,
                        ((blk - nfb) * (int)blockDim.x + (int)threadIdx.x) >> 6,
                        threadIdx.x & 63);
        return;
    }
    const int i = xcd_block(blk, nfb) * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    // lanes past the end stay for their partner's loads, without neighbours
    const int slot = min(i, n - 1);
    const float4 own_a = nrec[2 * (size_t)slot];      // (x, y, z, p)
    const float4 own_b = nrec[2 * (size_t)slot + 1];  // (vx, vy, vz, 1/rho)
    const int src = load_once(&list[slot]);           // the particle's slot in the state
    // the previous force is used only after the neighbour loop; issued
    // here, its load is in flight while the loop runs
    float4 fp = load_once(&force[src]);
    const float4 pi = make_float4(own_a.x, own_a.y, own_a.z, load_once(&bpos[slot].w));
    const float4 vi = make_float4(own_b.x, own_b.y, own_b.z, load_once(&vpad[slot]));
    const float p_i = own_a.w;
    const float h = P.h;
    const float m_spiky_half = P.m * P.spiky * 0.5f;
    const float m_lap = P.m * P.lap;
    PairAcc a{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    uint2* st = &s_nb[0][threadIdx.x];
    const int nw = valid ? stage_nb_words(nbw, n, i, st, 256) : 0;
    {
        // kForceBatch neighbours per iteration: every record is loaded
        // before any pair is evaluated (slots past the end of the list hold
        // the particle's own record and are evaluated with zero weight); pairs
        // are accumulated in order
        NbCursor nb(st, 256, nw);
        for (;;) {
            int j[kForceBatch];
            j[0] = nb.next();
            if (max(j[0], pair_swap(j[0])) < 0) break;
#pragma unroll
            for (int u = 1; u < kForceBatch; ++u) j[u] = nb.next();
            Nbr r[kForceBatch];
#pragma unroll
            for (int u = 0; u < kForceBatch; ++u) r[u] = load_nbr_pair(nrec, j[u] < 0 ? slot : j[u]);
#pragma unroll
            for (int u = 0; u < kForceBatch; ++u) {
                const bool live = j[u] >= 0;
                force_pair(h, pi, vi, p_i, live ? m_spiky_half : 0.0f, live ? m_lap : 0.0f, r[u],
                           a);
            }
        }
    }
    // a particle without neighbours that loaded for its partner: its own record
    // has no weight, but may hold an infinity or NaN
    if (nw <= 0) a = PairAcc{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int cell = -1;
    if (valid) {
        if (nw < 0)
            for_each_candidate_neighbour(P, offset, bpos, i, pi, [&](int j) {
                force_pair(h, pi, vi, p_i, m_spiky_half, m_lap, load_nbr(nrec, j), a);
            });
        const float u = (pi.x - P.org[0]) * P.uvs[0];
        const float v = (pi.z - P.org[1]) * P.uvs[1];
        const LateInputs in{P, H0, rho_w, bid, u, v, i};
        cell = force_finish(P, dt, i, pi, vi, fp, p_i, a, in, H0, out, next.key);
    }
    if (next.key) push_runs<true, kLink>(cell, valid, i, next.runs);
}

// The force pass of scenes of up to kForceSplitMax particles (and
// lane_split_limit()): kForceSplit consecutive lanes per particle.  There the
// pass is one chain of latencies per wave: own record and words, then the
// neighbours a few at a time, then the surface samples and the stores.  So
// each lane takes the neighbours whose word bits are its own mod kForceSplit,
// kSplitBatch records in flight; the first words are loaded without waiting
// for their count; and everything the end needs (the surface samples, each by
// one lane of the group, density, id) is loaded before the neighbours.  The
// group's sums are added in a fixed tree and its first lane finishes the
// particle.
// MI355X, one lane -> four, three scenes in flight / alone: 4 096 particles 13.6
// / 39.0 -> 12.2 / 34.8 us a step, 20 011 (eager) 42.0 -> 37.2 alone, 30 000
// 15.7 / 38.9 -> 15.3 / 33.8; 65 536 24.3 -> 25.8, 120 000 34.1 -> 37.4 and
// 240 000 60.1 -> 70.3 in flight, where the chip has enough waves without it.
constexpr int kForceSplit = 4;
constexpr int kSplitWords = 8;  // words loaded ahead of their count
constexpr int kSplitBatch = 8;

// What force_finish reads, all of it already loaded.
struct EarlyInputs {
    float h, hx, hy, h1x, h1y, r;
    int own_id;
    __device__ __forceinline__ float height() const { return h; }
    __device__ __forceinline__ float east_du() const { return hx; }
    __device__ __forceinline__ float north_du() const { return hy; }
    __device__ __forceinline__ float east() const { return h1x; }
    __device__ __forceinline__ float north() const { return h1y; }
    __device__ __forceinline__ float rho() const { return r; }
    __device__ __forceinline__ int id() const { return own_id; }
};

template <bool kLink, bool kWave>
__global__ void __launch_bounds__(256) k_force_split(
    const DevParams* __restrict__ Pd, float dt, const float4* __restrict__ bpos,
    const int* __restrict__ bid, const float* __restrict__ vpad,
    const float4* __restrict__ force, const int* __restrict__ list,
    const int* __restrict__ offset, int n, const float* __restrict__ rho_w,
    const uint2* __restrict__ nbw, const float4* __restrict__ nrec,
    const float* __restrict__ H0, ForceOut out, int nfb, const float* __restrict__ pflux,
    float* __restrict__ colflux, NextKeys next, WaveTiles wt) {
    const DevParams& P = *Pd;
    __shared__ uint2 s_nb[kNbStage][256];
    if (kWave && (int)blockIdx.x < wt.nblk) {
        wave_tile(P, wt, blockIdx.x, offset, colflux ? pflux : nullptr, dt,
                  reinterpret_cast<float*>(&s_nb[0][0]));
        return;
    }
    const int blk = (int)blockIdx.x - (kWave ? wt.nblk : 0);
    if (blk >= nfb) {
        column_flux_sum(offset, pflux, P.dims[0], P.dims[1], P.dims[2], colflux,
                        ((blk - nfb) * (int)blockDim.x + (int)threadIdx.x) >> 6,
                        threadIdx.x & 63);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int sub = threadIdx.x & (kForceSplit - 1);
    const int i = (blk * 256 + (int)threadIdx.x) / kForceSplit;  // a group shares i
    int cell = -1;
    if (i < n) {
        const int nw_all = load_once(&nb_count(nbw, n)[i]);
        uint2 w[kSplitWords];
#pragma unroll
        for (int k = 0; k < kSplitWords; ++k) w[k] = nbw[(size_t)k * n + i];
        const float4 own_a = nrec[2 * (size_t)i];      // (x, y, z, p)
        const float4 own_b = nrec[2 * (size_t)i + 1];  // (vx, vy, vz, 1/rho)
        const int src = list[i];
        const float pad = bpos[i].w, vw = vpad[i];
        EarlyInputs in;
        in.r = rho_w[i];
        in.own_id = bid[i];
        const float4 fp = force[src];
        const float4 pi = make_float4(own_a.x, own_a.y, own_a.z, pad);
        const float4 vi = make_float4(own_b.x, own_b.y, own_b.z, vw);
        // the surface: above the particle, and the sample of this lane
        const float u = (pi.x - P.org[0]) * P.uvs[0];
        const float v = (pi.z - P.org[1]) * P.uvs[1];
        const float du = (sub & 2) ? 1.0f : P.du;
        const TexTaps here = tex_taps(H0, P.W, P.H, u, v);
        const TexTaps mine = tex_taps(H0, P.W, P.H, (sub & 1) ? u : u + du, (sub & 1) ? v + du : v);
        const float p_i = own_a.w;
        const float h = P.h;
        const float m_spiky_half = P.m * P.spiky * 0.5f;
        const float m_lap = P.m * P.lap;
        PairAcc a{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (nw_all >= 0) {
            // this lane's bits of the particle's words, the empty ones left out
            uint2* st = &s_nb[0][threadIdx.x];
            const uint32_t own_bits = 0x11111111u << sub;
            int nw = 0;
#pragma unroll
            for (int k = 0; k < kSplitWords; ++k) {
                const uint32_t bits = k < nw_all ? w[k].x & own_bits : 0u;
                if (bits) st[256 * nw++] = make_uint2(bits, w[k].y);
            }
            for (int k = kSplitWords; k < nw_all; ++k) {
                const uint2 x = nbw[(size_t)k * n + i];
                if (x.x & own_bits) st[256 * nw++] = make_uint2(x.x & own_bits, x.y);
            }
            const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
            NbCursor nb(st, 256, nw);
            for (;;) {
                int j[kSplitBatch];
                j[0] = nb.next();
                if (j[0] < 0) break;
#pragma unroll
                for (int q = 1; q < kSplitBatch; ++q) j[q] = nb.next();
                Nbr r[kSplitBatch];
#pragma unroll
                for (int q = 0; q < kSplitBatch; ++q) {
                    r[q] = Nbr{zero, zero};
                    if (j[q] >= 0) r[q] = load_nbr(nrec, j[q]);
                }
#pragma unroll
                for (int q = 0; q < kSplitBatch; ++q) {
                    const bool live = j[q] >= 0;
                    force_pair(h, pi, vi, p_i, live ? m_spiky_half : 0.0f, live ? m_lap : 0.0f,
                               r[q], a);
                }
            }
        } else {
            int t = 0;
            for_each_candidate_neighbour(P, offset, bpos, i, pi, [&](int j) {
                if ((t++ & (kForceSplit - 1)) == sub)
                    force_pair(h, pi, vi, p_i, m_spiky_half, m_lap, load_nbr(nrec, j), a);
            });
        }
        a.pfx = quad_sum(a.pfx);
        a.pfy = quad_sum(a.pfy);
        a.pfz = quad_sum(a.pfz);
        a.vfx = quad_sum(a.vfx);
        a.vfy = quad_sum(a.vfy);
        a.vfz = quad_sum(a.vfz);
        const float s = mine.value();
        in.h = here.value();
        in.hx = quad_bcast_f<0>(s);
        in.hy = quad_bcast_f<1>(s);
        in.h1x = quad_bcast_f<2>(s);
        in.h1y = quad_bcast_f<3>(s);
        if (sub == 0) cell = force_finish(P, dt, i, pi, vi, fp, p_i, a, in, H0, out, next.key);
    }
    if (next.key) {
        // the wave's 16 particles on its first lanes, in slot order
        constexpr int kPer = 64 / kForceSplit;
        cell = __shfl(cell, (lane * kForceSplit) & 63, 64);
        if (lane >= kPer) cell = -1;
        push_runs<true, kLink>(cell, cell >= 0, i - lane / kForceSplit + lane, next.runs);
    }
}

// ---------------------------------------------------------------------------
// Neighbour count of every slot as the last density pass found it (the
// particle itself included, as the density sum of rho_pres_comp.glsl:60-68
// counts it): popcounts of its neighbour words, or the re-search by distance
// for a particle whose words are flagged incomplete.  pos / offset: that
// pass's sorted positions and cell offsets.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_neighbour_counts(const DevParams* __restrict__ Pd,
                                                          const float4* __restrict__ pos,
                                                          const int* __restrict__ offset,
                                                          const uint2* __restrict__ nbw, int n,
                                                          int* __restrict__ out) {
    const DevParams& P = *Pd;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int k = 1;  // the particle itself
    const int nw = nb_count(nbw, n)[i];
    if (nw < 0) {
        for_each_candidate_neighbour(P, offset, pos, i, pos[i], [&](int) { ++k; });
    } else {
        for (int w = 0; w < nw; ++w) k += __popc(nbw[(size_t)w * n + i].x);
    }
    out[i] = k;
}

// ---------------------------------------------------------------------------
// Wave EVOLVE (wave_comp.glsl:171-206), lambda split per axis, clamped
// neighbours, optional particle flux source, wake line, as a launch of its
// own (steps without particles, grids too fine for wave_tile, profiled steps).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_wave(const DevParams* __restrict__ Pd, const float* __restrict__ h0,
                                              const float* __restrict__ h1,
                                              float* __restrict__ out,
                                              const float* __restrict__ colflux, float dt) {
    const DevParams& P = *Pd;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= P.W || j >= P.H) return;
    const int nx = P.dims[0];
    const auto cf = [&](int ix, int iz) { return colflux[(size_t)iz * nx + ix]; };
    wave_single(P, h0, h1, out, i, j, colflux != nullptr, cf, dt);
}

// The same EVOLVE, four texels per thread along u (W % 4 == 0).
__global__ void __launch_bounds__(256) k_wave4(const DevParams* __restrict__ Pd, const float* __restrict__ h0,
                                               const float* __restrict__ h1,
                                               float* __restrict__ out,
                                               const float* __restrict__ colflux, float dt) {
    const DevParams& P = *Pd;
    const int i0 = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i0 >= P.W || j >= P.H) return;
    const int nx = P.dims[0];
    const auto cf = [&](int ix, int iz) { return colflux[(size_t)iz * nx + ix]; };
    wave_quad(P, h0, h1, out, i0, j, colflux != nullptr, cf, dt);
}

// InitWave (wave_comp.glsl:82-140): peak * smoothstep(5, 0, d), d = distance
// to the nearest of 2 or 3 centres.
__global__ void k_init_wave(float* __restrict__ out, int W, int H, int c0x, int c0y, int c1x,
                            int c1y, int c2x, int c2y, int three, float peak) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    auto dist = [&](int cx, int cy) {
        const float dx = (float)(i - cx), dy = (float)(j - cy);
        return sqrtf(dx * dx + dy * dy);
    };
    float d = fminf(dist(c0x, c0y), dist(c1x, c1y));
    if (three) d = fminf(d, dist(c2x, c2y));
    float t = (d - 5.0f) / (0.0f - 5.0f);
    t = fminf(fmaxf(t, 0.0f), 1.0f);
    out[(size_t)j * W + i] = peak * (t * t * (3.0f - 2.0f * t));
}

// Non-finite detector for the optional per-step check.
__global__ void k_check_finite(const float* __restrict__ a, size_t n, int* __restrict__ flag) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    int bad = 0;
    for (; i < n; i += stride) bad |= !isfinite(a[i]);
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
static inline int blocks_for(long long n, int t) { return (int)((n + t - 1) / t); }

hipError_t launch_fill_i32(int* p, int n, int v, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_fill_i32<<<blocks_for(n, 256), 256, 0, st>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_clear_cells(int* offset, int* a, int* b, int* c, int* d, int n,
                              hipStream_t st) {
    if (n < 0) return hipErrorInvalidValue;
    k_clear_cells<<<blocks_for(std::max(n, 1), 256), 256, 0, st>>>(ClearList{{offset, a, b, c, d}},
                                                                   n);
    return hipGetLastError();
}

hipError_t launch_hash_count(const float4* pos, int n, const GridDesc& g, int* key,
                             const CellRuns& runs, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (runs.head)
        k_hash_count<true><<<blocks_for(n, 256), 256, 0, st>>>(pos, n, g, key, runs);
    else
        k_hash_count<false><<<blocks_for(n, 256), 256, 0, st>>>(pos, n, g, key, runs);
    return hipGetLastError();
}

hipError_t launch_key_count(const int* key, int n, const CellRuns& runs, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (runs.head) k_key_count<true><<<blocks_for(n, 256), 256, 0, st>>>(key, n, runs);
    else k_key_count<false><<<blocks_for(n, 256), 256, 0, st>>>(key, n, runs);
    return hipGetLastError();
}

hipError_t launch_link_runs(const int* key, int n, int* head, int2* link, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_link_runs<<<blocks_for(n, 256), 256, 0, st>>>(LinkRuns{key, n, head, link});
    return hipGetLastError();
}

hipError_t launch_place_runs(const int* key, const int* offset, int* fill, int n, int2* runs,
                             hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_place_runs<<<blocks_for(n, 256), 256, 0, st>>>(key, offset, fill, n, runs);
    return hipGetLastError();
}

hipError_t launch_stable_reorder(const int* key, const int* offset, const int* head,
                                 const int2* link, int n, const int* item_of, int* list,
                                 const float4* pos_in, const int* id_in, float4* pos_out,
                                 int* id_out, hipStream_t st, const DevParams* Pd,
                                 uint32_t* packed_out) {
    if (n <= 0) return hipSuccess;
    const auto kernel = head ? k_stable_reorder<true> : k_stable_reorder<false>;
    kernel<<<blocks_for(n, 256), 256, 0, st>>>(key, offset, head, link, n, item_of, list, pos_in,
                                               id_in, pos_out, id_out, Pd, packed_out);
    return hipGetLastError();
}

hipError_t launch_box_cover(const float4* x, const float4* hw, int n, const float gmin[3],
                            const float cell[3], const int dims[3], int* ncov, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    BoxGrid g{};
    for (int k = 0; k < 3; ++k) {
        g.gmin[k] = gmin[k];
        g.cell[k] = cell[k];
        g.dims[k] = dims[k];
    }
    k_box_cover<<<blocks_for(n, 256), 256, 0, st>>>(x, hw, n, g, ncov);
    return hipGetLastError();
}

hipError_t launch_sum_i64(const int* a, int n, unsigned long long* out, hipStream_t st) {
    k_fill_i32<<<1, 64, 0, st>>>(reinterpret_cast<int*>(out), 2, 0);
    if (n > 0) k_sum_i64<<<blocks_for(n, 256), 256, 0, st>>>(a, n, out);
    return hipGetLastError();
}

hipError_t launch_box_pairs(const float4* x, const float4* hw, int n, const float gmin[3],
                            const float cell[3], const int dims[3], const int* first,
                            int* pkey, int* pbox, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    BoxGrid g{};
    for (int k = 0; k < 3; ++k) {
        g.gmin[k] = gmin[k];
        g.cell[k] = cell[k];
        g.dims[k] = dims[k];
    }
    k_box_pairs<<<blocks_for(n, 256), 256, 0, st>>>(x, hw, n, g, first, pkey, pbox);
    return hipGetLastError();
}

hipError_t launch_density(const DevParams& P, const float4* bpos, const float4* state_vel,
                          const int* list, const int* offset, int n, const float* H0,
                          float* rho_w, float2* pw, float* flux, uint2* nbw, float4* nrec,
                          float* rho_raw, float4* vel_out, float* vpad, const uint32_t* packed,
                          hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (!packed)
        k_density_split<<<blocks_for((long long)n * kDensitySplit, 256), 256, 0, st>>>(
            P.dev, bpos, state_vel, list, offset, n, H0, rho_w, pw, flux, nbw, nrec, rho_raw,
            vel_out, vpad);
    else
        k_density<<<blocks_for(n, 256), 256, 0, st>>>(P.dev, bpos, packed, state_vel, list, offset,
                                                      n, H0, rho_w, pw, flux, nbw, nrec, rho_raw,
                                                      vel_out, vpad);
    return hipGetLastError();
}

hipError_t launch_force_integrate(const DevParams& P, float dt, const float4* bpos,
                                  const int* bid, const ParticleArrays& S, const int* list,
                                  const int* offset, int n, const float* rho_w, const uint2* nbw,
                                  const float4* nrec, const float* H0, ParticleArrays& N,
                                  float* rho, float* prs, float4* fpre, const float* flux,
                                  float* colflux, const float* vpad, const NextKeys& next,
                                  const WaveTiles& wt, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const long long ncol = colflux ? (long long)P.dims[0] * P.dims[2] : 0;
    const int ncb = blocks_for(ncol * 64, 256);
    const bool link = next.runs.head != nullptr;
    if (wt.nblk && !link) return hipErrorInvalidValue;  // kFuseWaveParticles <= kFuseLinksMax
    const bool split = link && n <= kForceSplitMax && n <= lane_split_limit();
    const int nfb = blocks_for(split ? (long long)n * kForceSplit : n, 256);
    const auto kernel = split     ? (wt.nblk ? k_force_split<true, true> : k_force_split<true, false>)
                        : wt.nblk ? k_force_integrate<true, true>
                        : link    ? k_force_integrate<true, false>
                                  : k_force_integrate<false, false>;
    const ForceOut out{N.pos, N.vel, N.force, N.id, rho, prs, fpre};
    kernel<<<wt.nblk + nfb + ncb, 256, 0, st>>>(P.dev, dt, bpos, bid, vpad, S.force, list, offset,
                                                n, rho_w, nbw, nrec, H0, out, nfb, flux, colflux,
                                                next, wt);
    return hipGetLastError();
}

// Tiles of 32 texels a side (four a thread; 16 and one where W % 4 != 0 or the
// grid is fine) whose samples touch at most kWaveTileColumns columns, up to
// kFuseWaveTiles of them, for scenes of up to kFuseWaveParticles particles;
// none (nblk 0) otherwise.  There the step is bound by its launches, and the
// tiles end before the force blocks do (MI355X, three scenes in flight / alone,
// launch of its own -> blocks of the force launch: 4 096 particles and 128^2
// texels 14.9 / 42.9 -> 14.0 / 40.0 us a step, 5 000 and 100^2 16.9 / 39.1 ->
// 15.2 / 36.1, 50 000 and 512^2 19.4 / 47.3 -> 19.1 / 44.7).  Larger fields
// stream better at the occupancy of the wave's own kernel (40 000 and 1000^2
// 19.6 -> 24.0 in flight, 10 000 and 501^2 39.6 -> 41.5 alone), larger scenes
// fill the chip without them (120 000 and 301^2 34.2 -> 35.3 in flight), and on
// a grid too fine for the texels a tile spends longer on its columns than a
// launch takes.
WaveTiles wave_tiles_for(const DevParams& P, int n, bool flux, const float* h0,
                         const float* h1, float* out) {
    WaveTiles w{h0, h1, out, 0, 1, 0};
    if (P.W <= 0 || P.H <= 0 || n > kFuseWaveParticles) return w;
    const auto spans = [](float per_texel, int texels, int n) {
        // floor(first) .. floor(last) + 1, one more for the rounding of the ends
        return std::min<double>((double)std::fabs(per_texel) * (texels - 1) + 3.0, n);
    };
    for (int side : {32, 16}) {
        if (side == 32 && P.W % 4 != 0) continue;  // one quad or one texel a thread
        if (flux && spans(P.ax, side, P.dims[0]) * spans(P.az, side, P.dims[2]) > kWaveTileColumns)
            continue;
        const int nx = (P.W + side - 1) / side, ny = (P.H + side - 1) / side;
        if ((long long)nx * ny > kFuseWaveTiles) continue;
        w.side = side;
        w.nx = nx;
        w.nblk = (nx * ny + 7) / 8 * 8;
        break;
    }
    return w;
}

hipError_t launch_neighbour_counts(const DevParams& P, const float4* pos, const int* offset,
                                  const uint2* nbw, int n, int* out, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_neighbour_counts<<<blocks_for(n, 256), 256, 0, st>>>(P.dev, pos, offset, nbw, n, out);
    return hipGetLastError();
}

hipError_t launch_wave(const DevParams& P, const float* h0, const float* h1, float* out,
                       const float* colflux, float dt, hipStream_t st) {
    if (P.W <= 0 || P.H <= 0) return hipSuccess;
    dim3 blk(64, 4);
    if (P.W % 4 == 0) {
        dim3 grd((P.W / 4 + 63) / 64, (P.H + 3) / 4);
        k_wave4<<<grd, blk, 0, st>>>(P.dev, h0, h1, out, colflux, dt);
    } else {
        dim3 grd((P.W + 63) / 64, (P.H + 3) / 4);
        k_wave<<<grd, blk, 0, st>>>(P.dev, h0, h1, out, colflux, dt);
    }
    return hipGetLastError();
}

hipError_t launch_init_wave(float* out, int W, int H, float type, hipStream_t st) {
    if (W <= 0 || H <= 0) return hipSuccess;
    int c0x, c0y, c1x, c1y, c2x = 0, c2y = 0, three = 1;
    float peak;
    if (type == 1.0f) {  // splash
        c0x = (int)(0.25f * (float)W);
        c0y = (int)(0.25f * (float)H);
        c1x = (int)(0.75f * (float)W);
        c1y = (int)(0.75f * (float)H);
        three = 0;
        peak = 0.5f;
    } else if (type == 0.0f) {  // wave
        c0x = (int)(0.25f * (float)W);
        c0y = H;
        c2x = (int)(0.5f * (float)W);
        c2y = H;
        c1x = (int)(0.75f * (float)W);
        c1y = H;
        peak = 1.0f;
    } else {  // wake
        c0x = (int)(0.5f * (float)W);
        c0y = (int)(0.1f * (float)H);
        c1x = c2x = c0x;
        c1y = c2y = c0y;
        peak = 0.1f;
    }
    dim3 blk(64, 4);
    dim3 grd((W + 63) / 64, (H + 3) / 4);
    k_init_wave<<<grd, blk, 0, st>>>(out, W, H, c0x, c0y, c1x, c1y, c2x, c2y, three, peak);
    return hipGetLastError();
}

hipError_t launch_check_finite(const float* a, size_t n, int* flag, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const int blocks = (int)std::min<size_t>((n + 255) / 256, 2048);
    k_check_finite<<<blocks, 256, 0, st>>>(a, n, flag);
    return hipGetLastError();
}

}  // namespace cwa
