// cwa_batch2d.hip — the batched 2D coupled step: many independent scenes of
// 2D SPH (Koschier cubic kernel, WCSPH gamma = 3, box SDF) each coupled to
// its own 1D wave column, advanced by one launch per kernel per step.
//
// Reference, per scene (SphWave2D/):
//   SphUgrid::Compute            StencilBuffer.cpp:150-179
//   UniformGridSph2D::CollisionQuery  UniformGridGpu2D.cpp:220-265 and
//                                uniform_grid_sph_cs.glsl:112-183 (hash, count,
//                                insert; here a stable counting sort)
//   ComputeDensityPressure       SphWaveKoschier2D_grid_cs.glsl:393-487
//   ComputeForces (+ Euler)      SphWaveKoschier2D_grid_cs.glsl:490-628
//   ImageStencil::Compute        StencilImage2D.cpp:141-164 with
//                                Wave1D_cs.glsl IterateWave :120-130, FreeBC :139-157
//
// Packing.  Scene s owns the slot range [pbeg_s, pbeg_s + n_s) and the
// global cells [s*C, (s+1)*C) (C = nx*ny cells of size H/2, y fastest), so
// one counting sort over all cells keeps every scene inside its own slot
// range.  A step is at most 7 launches for any number of scenes:
//   k2_hash      cell keys, counts and run lists of a call's first step
//   scan         exclusive offsets over all cells (cwa_kernels.hip)
//   k2_reorder   stable rank from the run lists; state A -> B, sorted
//   k2_density   tiles; B -> q, (rho, p), (p/rho^2, 1/rho)
//   k2_force     tiles; q -> A (forward Euler), and the next step's keys
//   k2_wave      one workgroup per scene: column flux sums, the wave
//                substeps in LDS, flux source; levels updated in place
// The state ends every step in A, so a captured step replays as is.
//
// Tiles.  A tile is up to one block of consecutive slots of one scene.  Workgroup
// i runs on XCD i mod 8, so entry e of the tile table belongs to XCD e mod 8:
// scenes, the costly ones cut into pieces, are bound to XCDs by longest-
// processing-time assignment of their cost (neighbours per particle grow with
// n_s in a fixed box), costly tiles first.  With one block per tile, block e
// takes entry e, and the hardware hands out the blocks of an XCD as its CUs free
// up.  Fewer, persistent blocks take their XCD's entries from a queue counter
// and then the other XCDs' (static shares left them unbalanced: 256 scenes at
// 1 024 blocks of 512, density 803 -> 972 us).  The counter is a serial chain of
// atomics, which bound the passes when every tile came from it (MI355X, one
// block of 256 per tile, queue -> table: 256 scenes of 4 M particles, density
// 1 099 -> 700 us, force 1 558 -> 1 310; 100 scenes of 678 000, 139 -> 54 and
// 173 -> 91; 24 scenes of 20 000, 17.0 -> 14.0 and 20.8 -> 17.3).
//
// Arithmetic follows the float restatement of the oracle
// (oracle/cwa_oracle2d.hpp) expression by expression, with contraction
// off, so results are bit-identical to it and independent of the launch
// configuration.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <numeric>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/cwa2d.h"
#include "cwa_device.hpp"
#include "cwa_kernels.hpp"
#include "cwa_modules.hpp"

#pragma clang fp contract(off)

namespace cwa {

int guarded_call(void (*fn)(void*), void* ctx);

namespace b2d {

constexpr int kNumXcd = 8;      // XCDs of an MI355X
constexpr int kPiecesPerXcd = 8;  // a scene is cut into pieces of at most this share of an XCD
// Candidates loaded ahead in the density / force loops (the lanes of a tile
// walk the same candidates, so each load is one address per wave).  Measured
// on the 256-scene workload (MI355X): density 2, 4, 6, 8 -> 689, 663, 657, 660
// us; force 2, 4, 6 -> 1 511, 1 480, 1 497 us.
constexpr int kDensityBatch2D = 6;
constexpr int kForceBatch2D = 4;
// Batches of up to this many particles run density and force with four lanes per
// particle (quad_candidates): there a pass is one chain of candidates per wave,
// on a chip with waves to spare.  With more, the four lanes' 16 additions a round
// cost more than they hide.  MI355X, us a step, one lane -> four: 24 scenes of 20
// 324 particles 55.9 -> 45.6, 8 of 32 768 59.7 -> 49.4, one of 30 000 140 -> 92, 4 of
// 50 287 97.5 -> 68.5, 64 of 68 236 54.8 -> 51.7, 4 of 120 000 149 -> 158, 40 of 141 448
// 73 -> 74, 10 of 254 690 189 -> 239, 160 of 700 520 150 -> 208.
constexpr int kQuadMax2D = 80000;
// Batches with more cells than this per particle clear the run lists of the cells that
// hold particles, in a launch of its own; others clear all of them beside the
// density pass.  MI355X, us a call of 6 steps, all -> the particles' cells: 64 scenes
// of 100 particles with 1 600 cells a particle 476 -> 450, with 10 000 1 945 -> 1 595, with
// 40 000 6 246 -> 5 334 (5 827 before builds had lists); one of 500 with 2 000 301 -> 286.
// With few cells a particle the launch costs more than it saves.
constexpr int kSparseCells = 1024;
constexpr int kReadPast2D = 8;  // points a batch may load past the end of an array
static_assert(kDensityBatch2D % 2 == 0 && kForceBatch2D % 2 == 0, "points are loaded in pairs");
static_assert(kDensityBatch2D <= kReadPast2D && kForceBatch2D <= kReadPast2D, "padding");
// Terms of a flux column a lane loads together (256 scenes, 256 threads each: one
// -> eight 137 -> 59 us; columns of a wave side by side instead: 149 us, and at
// 1 024 threads 77 against 23).
constexpr int kFluxAhead = 8;

// Per-scene table (device).
struct Scene2D {
    int pbeg, n, wbeg, L;
    int nsub, model;
    float mass, lambda, dx;
};

// Kernel-side parameters (derived constants in float, as the oracle).
struct Dev2 {
    float H, HSQ, invH, T;          // T: sqrt_rn(r2) < H  <=>  r2 < T
    float k2, k2x2, c6k2, m6k2, c01, ga, gb;  // ga, gb: c6k2 / H, m6k2 / H
    float rho0, k, visc_pre, psi, gx, gy;
    float lox, loy, hix, hiy, walls[4];
    float thr, wref, wpress, wdy, wmask, atten, beta, band, kappa;
    float hc;            // grid cell edge H/2
    float eps;           // margin of the trimmed candidate rows
    int nx, ny, ncell;   // grid cells (H/2) per axis, per scene
    int nxc;             // flux columns (H wide): cell columns 2c, 2c + 1
    int nsph;
};

// ---------------------------------------------------------------------------
// device helpers (each mirrors the oracle function of the same name)
// ---------------------------------------------------------------------------
// Called with r = sqrt of an r2 < HSQ (pairs) or r = d < H (walls); both
// give q = r (1/H) <= 1 (the largest such r times the rounded 1/H rounds to
// at most 1), and at q == 1 the second piece is +0, as the shader's early
// return.  Hence no q >= 1 test here.
__device__ __forceinline__ float W_cubic(const Dev2& c, float r) {
    const float q = r * c.invH;
    if (q <= 0.5f) return c.k2 * (6.0f * q * q * (q - 1.0f) + 1.0f);
    const float q1 = 1.0f - q;
    return c.k2x2 * q1 * q1 * q1;
}

// Called with r < H only (pairs with r2 < T, walls with d < H).  Then
// q = r (1/H) <= 1: the largest float below H times the rounded 1/H is at
// most 1 before rounding.  q >= 1 would be q == 1 exactly, where the second
// piece gives -0 and the shader's early return +0; the sums that take W'
// never hold -0, so both add the same.  Hence no q >= 1 test here.
__device__ __forceinline__ float W_cubic_grad(const Dev2& c, float r) {
    const float q = r * c.invH;
    if (q <= 0.5f) return c.ga * q * (3.0f * q - 2.0f);
    const float q1 = 1.0f - q;
    return c.gb * (q1 * q1);
}

__device__ __forceinline__ float smoothstep(float e0, float e1, float x) {
    float t = (x - e0) / (e1 - e0);
    t = fminf(fmaxf(t, 0.0f), 1.0f);
    return t * t * (3.0f - 2.0f * t);
}

__device__ __forceinline__ float box_sdf(const Dev2& c, float x, float y, float& nx, float& ny) {
    const float d0 = y - c.walls[0], d1 = x - c.walls[1], d2 = c.walls[2] - x,
                d3 = c.walls[3] - y;
    float d = d0;
    nx = 0.0f;
    ny = 1.0f;
    if (!(d < d1)) { d = d1; nx = 1.0f; ny = 0.0f; }
    if (!(d < d2)) { d = d2; nx = -1.0f; ny = 0.0f; }
    if (!(d < d3)) { d = d3; nx = 0.0f; ny = -1.0f; }
    return d;
}

// floor()ed coordinate clamped to [lo, hi], NaN -> lo (fmaxf drops NaN).
__device__ __forceinline__ float clampf_nan(float f, float lo, float hi) {
    return fminf(fmaxf(f, lo), hi);
}

__device__ __forceinline__ float wave_at(const Dev2& c, const float* __restrict__ w, int L,
                                         float sL, float x) {
    const float t = (x - c.lox) * sL - 0.5f;
    const float f0 = floorf(t);
    const float a = t - f0;
    const float f = clampf_nan(f0, -2.0f, (float)(L + 1));
    const int i0 = min(max((int)f, 0), L - 1);
    const int i1 = min(max((int)f + 1, 0), L - 1);
    return (1.0f - a) * w[i0] + a * w[i1];
}

// The wave's coupling velocity at x: uh/h for a shallow-water column (the
// reference's xvel = w[1]/w[0], :362), (h^n - h^(n-1))/dt_sub for a leapfrog
// column.
__device__ __forceinline__ float wave_velocity(const Dev2& c, const Scene2D& S,
                                               const float* __restrict__ w0,
                                               const float* __restrict__ w1, float sL, float x,
                                               float dt) {
    if (S.model == CWA2D_WAVE_SHALLOW)
        return wave_at(c, w1, S.L, sL, x) / wave_at(c, w0, S.L, sL, x);
    const float dts = dt / (float)S.nsub;
    return (wave_at(c, w0, S.L, sL, x) - wave_at(c, w1, S.L, sL, x)) / dts;
}

// Correctly rounded square root of x >= 0, as sqrtf: the hardware square
// root (within 1 ulp) followed by the two residual tests that round it --
// the sequence the compiler emits for sqrtf, without its input scaling for
// x < 2^-96 and its select for 0 and inf, which change nothing for
// x in [2^-96, inf) and at 0.  Inputs in (0, 2^-96) take sqrtf itself.
__device__ __forceinline__ float sqrt_rn(float x) {
    if (__builtin_expect(x < 0x1p-96f && x > 0.0f, 0)) return sqrtf(x);
    const float s = __builtin_amdgcn_sqrtf(x);
    const float sm = __int_as_float(__float_as_int(s) - 1);
    const float sp = __int_as_float(__float_as_int(s) + 1);
    float r = fmaf(-sm, s, x) <= 0.0f ? sm : s;
    r = fmaf(-sp, s, x) > 0.0f ? sp : r;
    return r;
}

// 1 / b correctly rounded (bit-identical to IEEE division) for
// 2^-40 <= b <= 2^40, from a start y within 3 ulp of it: two Newton-Raphson
// steps y + y (1 - b y), each with two fused multiply-adds.  These give the
// correctly rounded reciprocal for every b in that range but one kind, a
// mantissa of all ones, b = (2 - 2^-23) 2^e: there 1 / b lies just above
// the midpoint 2^-(e+1) (1 + 2^-24), the step lands exactly on it and
// rounds to the even 2^-(e+1), whose last mantissa bit is the one missing.
// The carry out of mantissa + 1 is that bit.  Checked
// exhaustively over all 81 binades for starts up to 3 ulp either side.
__device__ __forceinline__ float recip_rn(float b, float y) {
    y = fmaf(fmaf(-b, y, 1.0f), y, y);
    y = fmaf(fmaf(-b, y, 1.0f), y, y);
    const unsigned ub = __float_as_uint(b);
    return __uint_as_float(__float_as_uint(y) | (((ub & 0x7FFFFFu) + 1u) >> 23));
}

// sqrt(x) correctly rounded for 2^-96 <= x <= 2^96, without compares:
// the hardware reciprocal square root y, g = x y and h = y / 2, one coupled
// Newton step on both and Markstein's correction g + (x - g g) h.  2h is
// then within 2 ulp of 1 / sqrt(x) rounded (checked exhaustively), a start
// for recip_rn that saves the hardware reciprocal.
__device__ __forceinline__ float sqrt_rn_mid(float x, float& half_rsqrt) {
    const float y = __builtin_amdgcn_rsqf(x);
    float g = x * y, h = 0.5f * y;
    const float e = fmaf(-g, h, 0.5f);
    g = fmaf(g, e, g);
    h = fmaf(h, e, h);
    half_rsqrt = h;
    return fmaf(fmaf(-g, g, x), h, g);
}

// r = sqrt(max(x, 2^-80)) correctly rounded, for 0 <= x < 2^38: the density
// pass's r.  The clamp (r = 2^-40 for x <= 2^-80) leaves W(r) unchanged:
// with H >= 2^-16, q = r / H <= 2^-24 there, 6 q^2 (q - 1) stays below half
// an ulp of 1 and W rounds to k2 for every such r, 0 included.
__device__ __forceinline__ float sqrt_rn_clamped(float x) {
    // max on the bit patterns: the same as fmaxf for x >= 0, one instruction
    float h;
    return sqrt_rn_mid(__uint_as_float(max(__float_as_uint(x), 0x17800000u)), h);
}

__device__ __forceinline__ int cell2(float p, float lo, float H, int dim) {
    const float f = clampf_nan(floorf((p - lo) / H), -1.0f, (float)dim);
    return min(max((int)f, 0), dim - 1);
}

// Candidate slot range [b, e) of cell column cx for a query at (x, y) in
// cell column ix: the rows of the column the disc of radius H reaches,
// widened by a margin far above the rounding of the float bounds, or an
// empty range when the column lies H or more away -- the oracle's
// column_rows, operation for operation (so both see the same candidates,
// in the same order, also for a neighbour moved out of its cell by the
// density pass's un-penetration).
__device__ __forceinline__ void column_rows(const Dev2& P, const int* __restrict__ off, int cb,
                                            float x, float y, int ix, int cx, int& b, int& e) {
    float dx = 0.0f;
    if (cx < ix) dx = x - (P.lox + (float)(cx + 1) * P.hc);
    else if (cx > ix) dx = (P.lox + (float)cx * P.hc) - x;
    dx = fmaxf(dx - P.eps, 0.0f);
    b = e = 0;
    const float d2 = dx * dx;
    if (!(d2 < P.T)) return;
    const float ry = sqrt_rn(P.T - d2) + P.eps;
    const int ylo = cell2(y - ry, P.loy, P.hc, P.ny);
    const int yhi = cell2(y + ry, P.loy, P.hc, P.ny);
    b = off[cb + cx * P.ny + ylo];
    e = off[cb + cx * P.ny + yhi + 1];
}

// ---------------------------------------------------------------------------
// grid: hash / count.  The keys, counts and run lists (cwa_kernels.hip) of a
// build come from k2_hash, or within one call of several steps or substeps
// from the force pass before, which hashes the positions it writes (key null:
// it does not).  A call's last pass leaves counts and lists empty, as the next
// call may start from positions the caller has written.
// Small batches are bound by their launches: two fewer a substep (the hash, and
// the pass that placed the runs in their cells) took 20 eager steps of 24 small
// scenes from 637 to 474 us and 10 steps of the application's scene, eight
// copies, from 331 to 288, three batches in flight; 256 scenes unchanged.
// ---------------------------------------------------------------------------
struct Keys2D {
    int* key;
    CellRuns runs;
};

// Cell of a point of scene s.
__device__ __forceinline__ int cell_of(const Dev2& P, int s, float x, float y) {
    return s * P.ncell + cell2(x, P.lox, P.hc, P.nx) * P.ny + cell2(y, P.loy, P.hc, P.ny);
}

__global__ void __launch_bounds__(256)
    k2_hash(Dev2 P, const Scene2D* __restrict__ sc, const int* __restrict__ blk_scene,
            const float4* __restrict__ xv, int ntot, Keys2D out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < ntot;
    int c = -1;
    if (valid) {
        int s = blk_scene[blockIdx.x];
        while (i >= sc[s].pbeg + sc[s].n) ++s;
        const float4 p = xv[i];
        c = cell_of(P, s, p.x, p.y);
        out.key[i] = c;
    }
    push_runs<true, true>(c, valid, i, out.runs);
}

// Stable destination: a run's first lane walks its cell's run list and counts
// the items before its own slot; the run itself is contiguous.  Also clears
// the counts for the next build (the density pass clears the lists) and the
// tile queues.
__global__ void __launch_bounds__(256)
    k2_reorder(Keys2D in, const int* __restrict__ offset, int ntot,
               const float4* __restrict__ xvA, const float2* __restrict__ rpA,
               const int* __restrict__ idfA, float2* __restrict__ xyB, float2* __restrict__ velB,
               float2* __restrict__ rpB, int* __restrict__ idfB, int ncells,
               int* __restrict__ queues) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    if (s < 2 * kNumXcd) queues[s] = 0;
    if (s < ncells) in.runs.count[s] = 0;
    const bool valid = s < ntot;
    const int c = valid ? in.key[s] : -1;
    const RunInfo r = wave_runs(c);
    int rank = 0;
    if (valid && r.head) {
        const int b = offset[c];
        int left = offset[c + 1] - b;
        for (int q = in.runs.head[c]; q > 0 && left > 0;) {
            const int2 u = in.runs.link[q - 1];
            // a run the force pass listed may go on past this one's first slot
            if (q - 1 < s) rank += min(u.y, s - (q - 1));
            left -= max(u.y, 1);
            q = u.x;
        }
        rank += b;
    }
    const int d = __shfl(rank, r.my_head, 64) + (lane - r.my_head);
    if (!valid || d < 0 || d >= ntot) return;  // out of range only on inconsistent lists
    const float4 p = xvA[s];
    xyB[d] = make_float2(p.x, p.y);
    velB[d] = make_float2(p.z, p.w);
    rpB[d] = rpA[s];
    idfB[d] = idfA[s];
}

// Empties the run lists of the cells that hold particles, for the next build.
__global__ void __launch_bounds__(256) k2_clear_lists(Keys2D in, int ntot) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ntot) in.runs.head[in.key[i]] = 0;
}

// ---------------------------------------------------------------------------
// tiles
// ---------------------------------------------------------------------------
struct TileTable {
    const int4* entry;  // scene (-1: none), first slot, end slot
    int n;              // entries, a multiple of nq
    int nq;             // XCDs the entries are dealt to in turn
    int* queue;         // persistent blocks: entries of each XCD already taken,
    const int* len;     // and how many it has (the others of its n / nq are empty)
};

// Next entry of a persistent block: its XCD's first, then the others' in
// order.  Every queue is finite, so every block ends.
__device__ __forceinline__ int next_entry(const TileTable& T) {
    const int home = (int)(blockIdx.x % T.nq);
    for (int k = 0; k < T.nq; ++k) {
        int q = home + k;
        if (q >= T.nq) q -= T.nq;
        const int cnt = T.len[q];
        if (__hip_atomic_load(&T.queue[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= cnt)
            continue;
        const int idx = atomicAdd(&T.queue[q], 1);
        if (idx < cnt) return idx * T.nq + q;
    }
    return -1;
}

// How a pass is laid out on the chip.
enum class Form {
    tiles,       // a block per tile, a lane per particle
    quads,       // four blocks per tile, four lanes per particle
    persistent,  // blocks that take their tiles from the queues, a lane per particle
};

// Runs body(tile, slot of the thread's particle) for the block's tiles.
template <Form kForm, class Body>
__device__ __forceinline__ void for_each_tile(const TileTable& T, Body&& body) {
    if (kForm == Form::tiles) {
        const int4 t = T.entry[blockIdx.x];
        if (t.x >= 0) body(t, t.y + (int)threadIdx.x);
        return;
    }
    if (kForm == Form::quads) {  // a tile's four blocks on the XCD of its entry
        const int b = blockIdx.x, q = T.nq;
        const int4 t = T.entry[b / (4 * q) * q + b % q];
        if (t.x >= 0) body(t, t.y + (int)((b / q % 4 * blockDim.x + threadIdx.x) / 4));
        return;
    }
    __shared__ int s_entry;
    for (;;) {
        if (threadIdx.x == 0) s_entry = next_entry(T);
        __syncthreads();
        const int e = __builtin_amdgcn_readfirstlane(s_entry);
        __syncthreads();
        if (e < 0) return;
        const int4 t = T.entry[e];
        body(t, t.y + (int)threadIdx.x);
    }
}

// ---------------------------------------------------------------------------
// density / pressure (ComputeDensityPressure, :393-487)
// ---------------------------------------------------------------------------
// N consecutive points, two to a 16-byte load: a load keeps the address unit
// busy for 16 cycles or more whatever its width, and with one load a candidate
// the density pass kept it busy 93 % of the time (256 scenes of 4 M particles:
// 773 -> 657 us).
template <int N>
struct Points {
    struct alignas(8) Two {
        float x0, y0, x1, y1;
    };
    Two v[N / 2];
    __device__ __forceinline__ void load(const float2* __restrict__ p) {
#pragma unroll
        for (int k = 0; k < N / 2; ++k) v[k] = *reinterpret_cast<const Two*>(p + 2 * k);
    }
    __device__ __forceinline__ float2 operator[](int u) const {
        return u % 2 ? make_float2(v[u / 2].x1, v[u / 2].y1)
                     : make_float2(v[u / 2].x0, v[u / 2].y0);
    }
};

// The candidates of a particle shared by four lanes, in rounds of four
// consecutive ones: load(j) gives what a lane needs of its candidate, and
// sum(candidate, whether there is one) is called in all four lanes, round by
// round, so that each can add the terms of the four in candidate order: the same
// sums as one lane's, to the bit.  The lanes look up the five column ranges
// at once, and a column's first kQuadAhead rounds are loaded while the column
// before is summed (1, 2, 3, 4 rounds: 24 scenes 45.3, 45.6, 46.1, 46.8 us a step, 4
// dense scenes of 120 000 particles 166, 158, 161, 166).  Force / density at 24 small
// scenes 14.7 / 13.1 -> 9.0 / 8.5 us.
constexpr int kQuadAhead = 2;
template <class Load, class Sum>
__device__ __forceinline__ void quad_candidates(const Dev2& P, const int* __restrict__ off, int cb,
                                                float x, float y, int sub, Load&& load,
                                                Sum&& sum) {
    const int ix = cell2(x, P.lox, P.hc, P.nx);
    int rb[2] = {0, 0}, re[2] = {0, 0};  // cell columns ix - 2 + sub, ix + 2 (first lane)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int cx = ix - 2 + sub + 4 * q;
        if ((q == 0 || sub == 0) && cx >= 0 && cx < P.nx)
            column_rows(P, off, cb, x, y, ix, cx, rb[q], re[q]);
    }
    int b[5] = {quad_bcast<0>(rb[0]), quad_bcast<1>(rb[0]), quad_bcast<2>(rb[0]),
                quad_bcast<3>(rb[0]), quad_bcast<0>(rb[1])};
    int e[5] = {quad_bcast<0>(re[0]), quad_bcast<1>(re[0]), quad_bcast<2>(re[0]),
                quad_bcast<3>(re[0]), quad_bcast<0>(re[1])};
    using Cand = decltype(load(0));
    Cand next[kQuadAhead];
    const auto ahead = [&](int first, int end) {
#pragma unroll
        for (int u = 0; u < kQuadAhead; ++u)
            if (first + 4 * u < end) next[u] = load(min(first + 4 * u + sub, end - 1));
    };
    ahead(b[0], e[0]);
#pragma unroll 1
    for (int c = 0; c < 5; ++c) {
        const int first = b[0], end = e[0];
        Cand cur[kQuadAhead];
#pragma unroll
        for (int u = 0; u < kQuadAhead; ++u) cur[u] = next[u];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            b[k] = b[k + 1];
            e[k] = e[k + 1];
        }
        if (c < 4) ahead(b[0], e[0]);
        for (int j = first; j < end;) {
#pragma unroll
            for (int u = 0; u < kQuadAhead; ++u)
                if (j + 4 * u < end) sum(cur[u], j + 4 * u + sub < end);
            j += 4 * kQuadAhead;
#pragma unroll
            for (int u = 0; u < kQuadAhead; ++u)
                if (j + 4 * u < end) cur[u] = load(min(j + 4 * u + sub, end - 1));
        }
    }
}

struct DensityArgs {
    const Scene2D* sc;
    TileTable tiles;
    const float2* xyB;
    const float2* velB;
    const float2* rpB;
    const int* idfB;
    const int* off;
    const float* h0;
    const float* h1;
    float2* qxy;
    float4* qva;
    float2* rpA;
    int* idfA;
    float* flux;
    int* head;  // run lists of the grid, cleared for the next build
    int ncells;  // (0: k2_clear_lists does)
};

template <int BS, Form kForm>
__global__ void __launch_bounds__(BS) k2_density(Dev2 P, float dt, DensityArgs A) {
    for (int c = blockIdx.x * BS + threadIdx.x; c < A.ncells; c += gridDim.x * BS) A.head[c] = 0;
    for_each_tile<kForm>(A.tiles, [&](const int4 t, const int i) {
        if (i >= t.z) return;  // with quads the four lanes of a particle
        constexpr bool kQuads = kForm == Form::quads;
        const int sub = kQuads ? threadIdx.x & 3 : 0;
        const Scene2D S = A.sc[t.x];
        const float* w0 = A.h0 + S.wbeg;
        const float* w1 = A.h1 + S.wbeg;
        const float sL = (float)S.L / (P.hix - P.lox);
        const float2 p0 = A.xyB[i], v0 = A.velB[i];
        float x = p0.x, y = p0.y, vx = v0.x, vy = v0.y;
        int idf = A.idfB[i];
        int en = (idf >> 30) & 1;
        // enable flag (:400-415); with a zero threshold an enabled particle
        // stays enabled, so the samples are skipped
        if (!(en == 1 && P.thr == 0.0f)) {
            const float vw = wave_velocity(P, S, w0, w1, sL, x, dt);
            if (en == 0 && fabsf(vw) > P.thr) en = 1;
            if (en == 1 && fabsf(vw) < P.thr) en = 0;
        }
        float bnx, bny;
        const float d = box_sdf(P, x, y, bnx, bny);
        if (d < 0.0f) {  // un-penetrate (:417-423)
            x -= 0.75f * d * bnx;
            y -= 0.75f * d * bny;
            const float vn = fminf(0.0f, vx * bnx + vy * bny);
            vx -= 1.75f * vn * bnx;
            vy -= 1.75f * vn * bny;
        }
        if (sub == 0) A.qxy[i] = make_float2(x, y);
        float f = 0.0f;
        if (P.band > 0.0f) {
            const float dd = fabsf(y - wave_at(P, w0, S.L, sL, x));
            if (dd < P.band) {
                const float qq = dd / P.band;
                const float tq = 1.0f - qq * qq;
                f = S.mass / P.rho0 * vy * tq * tq;
            }
        }
        if (sub == 0) A.flux[i] = f;
        float2 rp = A.rpB[i];
        float rho = rp.x, p = rp.y;
        if (!(y > P.hiy)) {
            const int cb = t.x * P.ncell;
            float acc = 0.0f;
            const auto add = [&](float w) { acc += w; };
            // a candidate's W, given to `to` when it is a neighbour
            const auto near = [&](const float2 pj, auto&& to) {
                const float dx = x - pj.x, dy = y - pj.y;
                const float r2 = fmaf(dy, dy, dx * dx);
                if (r2 < P.HSQ) to(W_cubic(P, sqrt_rn_clamped(r2)));
            };
            if constexpr (kQuads) {
                quad_candidates(
                    P, A.off, cb, x, y, sub, [&](int j) { return A.xyB[j]; },
                    [&](const float2 pj, bool some) {
                        float w = 0.0f;
                        if (some) near(pj, [&](float v) { w = v; });
                        add(quad_bcast_f<0>(w));
                        add(quad_bcast_f<1>(w));
                        add(quad_bcast_f<2>(w));
                        add(quad_bcast_f<3>(w));
                    });
            } else {
                const auto cand = [&](const float2 pj) { near(pj, add); };
                const int ix = cell2(x, P.lox, P.hc, P.nx);
                for (int cx = max(ix - 2, 0); cx <= min(ix + 2, P.nx - 1); ++cx) {
                    int b, e;
                    column_rows(P, A.off, cb, x, y, ix, cx, b, e);
                    // kDensityBatch2D candidates loaded before the first is
                    // tested; tested in order
                    const float2* q = A.xyB + b;
                    int left = e - b;
                    for (; left >= kDensityBatch2D; left -= kDensityBatch2D, q += kDensityBatch2D) {
                        Points<kDensityBatch2D> pj;
                        pj.load(q);
#pragma unroll
                        for (int u = 0; u < kDensityBatch2D; ++u) cand(pj[u]);
                    }
                    if (left > 0) {
                        Points<kDensityBatch2D> pj;
                        pj.load(q);
#pragma unroll
                        for (int u = 0; u < kDensityBatch2D - 1; ++u)
                            if (u < left) cand(pj[u]);
                    }
                }
            }
            rho = S.mass * acc;
            if (d < P.H) rho += P.psi * W_cubic(P, fmaxf(0.0f, d));
            rho = fmaxf(P.rho0, rho);
            const float tr = rho / P.rho0;
            p = P.k * (tr * tr * tr - 1.0f);
        }
        if (sub != 0) return;
        A.rpA[i] = make_float2(rho, p);
        A.qva[i] = make_float4(vx, vy, p / (rho * rho), 1.0f / rho);
        A.idfA[i] = (idf & ~(1 << 30)) | (en << 30);
    });
}

// ---------------------------------------------------------------------------
// forces + forward Euler (ComputeForces, :490-628)
// ---------------------------------------------------------------------------
struct ForceArgs {
    const Scene2D* sc;
    TileTable tiles;
    const float2* qxy;
    const float4* qva;
    const int* idfA;
    const int* off;
    const float* h0;
    const float* h1;
    float4* xvA;
    Keys2D next;
};

template <int BS, Form kForm>
__global__ void __launch_bounds__(BS) k2_force(Dev2 P, float dt, ForceArgs A) {
    constexpr bool kQuads = kForm == Form::quads;
    const int sub = kQuads ? threadIdx.x & 3 : 0;
    // The new position of particle i (with quads in the first of its four lanes).
    const auto advance = [&](const int4 t, const int i) {
        const float2 xyi = A.qxy[i];
        const float4 vai = A.qva[i];
        const float x = xyi.x, y = xyi.y, vx = vai.x, vy = vai.y;
        const int idf = A.idfA[i];
        if (((idf >> 30) & 1) == 0) {  // disabled: pass through (:494-498)
            if (sub == 0) A.xvA[i] = make_float4(x, y, vx, vy);
            return xyi;
        }
        const Scene2D S = A.sc[t.x];
        const float ai = vai.z;
        float apx = 0.0f, apy = 0.0f, avx = 0.0f, avy = 0.0f;
        const int cb = t.x * P.ncell;
        // A candidate's terms; false (and nothing written) for one that is no
        // neighbour.
        struct Terms {
            float px = 0.0f, py = 0.0f, vx = 0.0f, vy = 0.0f;
        };
        const auto terms = [&](const float2 qj, const float4 va, Terms& w) {
            const float dx = x - qj.x, dy = y - qj.y;
            const float r2 = fmaf(dy, dy, dx * dx);
            if (!(r2 < P.T && r2 > 0.0f)) return false;  // r2 > 0 also excludes j == i
            // r2 < T <= 2^38 (h <= 2^19); below 2^-80 the library square
            // root and division
            const bool wide = r2 < 0x1p-80f;
            float r, inv;
            if (__builtin_expect(wide, 0)) {
                r = sqrtf(r2);
                inv = 1.0f / r;
            } else {
                float h;
                r = sqrt_rn_mid(r2, h);
                inv = recip_rn(r, h + h);  // 2h: within 2 ulp of 1 / r
            }
            const float wg = W_cubic_grad(P, r);
            const float ux = dx * inv, uy = dy * inv;
            const float s = (ai + va.z) * wg;
            w.px = s * ux;
            w.py = s * uy;
            const float vdr = (vx - va.x) * dx + (vy - va.y) * dy;
            // dot(vij, rij) / (r^2 + 0.01 H^2) as dot * (1 / ...); the
            // denominator lies in [2^-40, 2^40] for 2^-16 <= H <= 2^19
            const float den = r2 + P.c01;
            const float tv = va.w * vdr * recip_rn(den, __builtin_amdgcn_rcpf(den)) * wg;
            w.vx = tv * ux;
            w.vy = tv * uy;
            return true;
        };
        const auto add = [&](float px, float py, float wx, float wy) {
            apx -= px;
            apy -= py;
            avx -= wx;
            avy -= wy;
        };
        if constexpr (kQuads) {
            struct Cand {
                float2 xy;
                float4 va;
            };
            // a term of +0 leaves a sum as it is (the sums never hold -0)
            quad_candidates(
                P, A.off, cb, x, y, sub, [&](int j) { return Cand{A.qxy[j], A.qva[j]}; },
                [&](const Cand& c, bool some) {
                    Terms w;
                    if (some) (void)terms(c.xy, c.va, w);
                    add(quad_bcast_f<0>(w.px), quad_bcast_f<0>(w.py), quad_bcast_f<0>(w.vx),
                        quad_bcast_f<0>(w.vy));
                    add(quad_bcast_f<1>(w.px), quad_bcast_f<1>(w.py), quad_bcast_f<1>(w.vx),
                        quad_bcast_f<1>(w.vy));
                    add(quad_bcast_f<2>(w.px), quad_bcast_f<2>(w.py), quad_bcast_f<2>(w.vx),
                        quad_bcast_f<2>(w.vy));
                    add(quad_bcast_f<3>(w.px), quad_bcast_f<3>(w.py), quad_bcast_f<3>(w.vx),
                        quad_bcast_f<3>(w.vy));
                });
            if (sub != 0) return xyi;
        } else {
            const auto pair = [&](const float2 qj, const float4 va) {
                Terms w;
                if (terms(qj, va, w)) add(w.px, w.py, w.vx, w.vy);
            };
            const int ix = cell2(x, P.lox, P.hc, P.nx);
            for (int cx = max(ix - 2, 0); cx <= min(ix + 2, P.nx - 1); ++cx) {
                int b, e;
                column_rows(P, A.off, cb, x, y, ix, cx, b, e);
                // kForceBatch2D candidates (position; velocity, pressure term and
                // 1/rho) loaded before the first is tested; tested and accumulated in
                // order.  Loading all of every candidate, not only of the
                // neighbours, trades a few cached loads for the latency each
                // neighbour otherwise waits on.
                int j = b;
                for (; j + kForceBatch2D <= e; j += kForceBatch2D) {
                    Points<kForceBatch2D> pj;
                    pj.load(A.qxy + j);
                    float4 va[kForceBatch2D];
#pragma unroll
                    for (int u = 0; u < kForceBatch2D; ++u) va[u] = A.qva[j + u];
#pragma unroll
                    for (int u = 0; u < kForceBatch2D; ++u) pair(pj[u], va[u]);
                }
                if (j < e) {
                    Points<kForceBatch2D> pj;
                    pj.load(A.qxy + j);
                    float4 va[kForceBatch2D - 1];
#pragma unroll
                    for (int u = 0; u < kForceBatch2D - 1; ++u) va[u] = A.qva[j + u];
#pragma unroll
                    for (int u = 0; u < kForceBatch2D - 1; ++u)
                        if (j + u < e) pair(pj[u], va[u]);
                }
            }
        }
        const float cv = P.visc_pre * S.mass;
        avx *= cv;
        avy *= cv;
        apx *= S.mass;
        apy *= S.mass;
        float bnx, bny;
        const float d = box_sdf(P, x, y, bnx, bny);
        if (d < P.H) {  // boundary pressure (:553-562)
            const float wg = W_cubic_grad(P, fmaxf(0.0f, d));
            apx += P.psi * ai * wg * -bnx;
            apy += P.psi * ai * wg * -bny;
        }
        float aty = 0.0f;
        if ((idf & 0x3FFFFFFF) % 5 < 4) {  // wave pressure (:586-603)
            const float sL = (float)S.L / (P.hix - P.lox);
            const float hw = wave_at(P, A.h0 + S.wbeg, S.L, sL, x);
            const float vw = wave_velocity(P, S, A.h0 + S.wbeg, A.h1 + S.wbeg, sL, x, dt);
            const float dh = hw - P.wref;
            const float mask = smoothstep(0.0f, P.wmask, fabsf(vw));
            float dyw = y - hw;
            dyw -= 0.5f * dh;
            aty = 0.0f - mask * P.wpress * smoothstep(0.0f, P.wdy, dyw);
        }
        const float ax = apx + avx + P.gx + 0.0f;
        const float ay = apy + avy + P.gy + aty;
        const float v1x = vx + dt * ax, v1y = vy + dt * ay;
        const float2 x1 = make_float2(x + dt * v1x, y + dt * v1y);
        A.xvA[i] = make_float4(x1.x, x1.y, v1x, v1y);
        return x1;
    };
    for_each_tile<kForm>(A.tiles, [&](const int4 t, int i) {
        int c = -1;
        if (i < t.z) {  // with quads the same in the four lanes of a particle
            const float2 p = advance(t, i);
            if (A.next.key && sub == 0) {
                c = cell_of(P, t.x, p.x, p.y);
                A.next.key[i] = c;
            }
        }
        if (!A.next.key) return;
        if (kQuads) {  // the wave's 16 particles on its first lanes, in slot order
            const int lane = threadIdx.x & 63;
            c = __shfl(c, (lane * 4) & 63, 64);
            if (lane >= 16) c = -1;
            i += lane - lane / 4;
        }
        push_runs<true, true>(c, c >= 0, i, A.next.runs);
    });
}

// ---------------------------------------------------------------------------
// wave column: flux sums, substeps in LDS, flux source (one block per scene)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
    k2_wave(Dev2 P, float dt, const Scene2D* __restrict__ sc, const int* __restrict__ off,
            const float* __restrict__ flux, float* __restrict__ h0, float* __restrict__ h1,
            int lds_stride) {
    extern __shared__ float sm[];
    const Scene2D S = sc[blockIdx.x];
    const int L = S.L, tid = threadIdx.x, bd = blockDim.x;
    float* A = sm;
    float* B = sm + lds_stride;
    float* O = sm + 2 * lds_stride;
    float* col = sm + 4 * lds_stride;
    float* g0 = h0 + S.wbeg;
    float* g1 = h1 + S.wbeg;
    for (int k = tid; k < L; k += bd) {
        A[k] = g0[k];
        B[k] = g1[k];
    }
    const bool couple = P.band > 0.0f;
    if (couple) {
        // column sums in the fixed order: lane-strided partials, xor butterfly
        const int lane = tid & 63, wv = tid >> 6, nw = bd >> 6;
        const int cb = blockIdx.x * P.ncell;
        for (int cx = wv; cx < P.nxc; cx += nw) {  // flux column = cell columns 2cx, 2cx + 1
            const int b = off[cb + 2 * cx * P.ny], e = off[cb + min(2 * cx + 2, P.nx) * P.ny];
            float s = 0.0f;
            // kFluxAhead terms of the lane loaded before the first is added
            for (int k = b + lane; k < e; k += 64 * kFluxAhead) {
                float f[kFluxAhead];
#pragma unroll
                for (int u = 0; u < kFluxAhead; ++u) f[u] = k + 64 * u < e ? flux[k + 64 * u] : 0.0f;
#pragma unroll
                for (int u = 0; u < kFluxAhead; ++u)
                    if (k + 64 * u < e) s += f[u];
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            if (lane == 0) col[cx] = s;
        }
    }
    __syncthreads();
    const float lam = S.lambda;
    if (S.model == CWA2D_WAVE_SHALLOW) {
        // Shallow1D (Shallow1D_cs.glsl:133-167): A = h, B = uh, O = h at
        // i + 1/2, M = uh at i + 1/2; each phase ends with FreeBC's copy of
        // cells 1 and L-2 (all four channels) to the edges.
        float* M = sm + 3 * lds_stride;
        const float G = 9.8f, hg = 0.5f * G, l2 = lam / 2.0f, dx = S.dx;
        auto edges = [&] {
            if (tid == 0) {
                A[0] = A[1], B[0] = B[1], O[0] = O[1], M[0] = M[1];
                A[L - 1] = A[L - 2], B[L - 1] = B[L - 2], O[L - 1] = O[L - 2],
                      M[L - 1] = M[L - 2];
            }
        };
        for (int s = 0; s < S.nsub; ++s) {
            for (int k = 1 + tid; k < L - 1; k += bd) {
                const int e = k + 1;
                O[k] = (A[k] + A[e]) / 2.0f - l2 * (B[e] - B[k]) / dx;
                M[k] = (B[k] + B[e]) / 2.0f -
                       l2 * (B[e] * B[e] / A[e] + hg * A[e] * A[e] - B[k] * B[k] / A[k] -
                             hg * A[k] * A[k]) / dx;
            }
            __syncthreads();
            edges();
            __syncthreads();
            for (int k = 1 + tid; k < L - 1; k += bd) {
                const int w = k - 1;
                const float h = A[k] - lam * (M[k] - M[w]) / dx;
                const float uh = B[k] - lam * (M[k] * M[k] / O[k] + hg * O[k] * O[k] -
                                               M[w] * M[w] / O[w] - hg * O[w] * O[w]) / dx;
                A[k] = h;
                B[k] = uh;
            }
            __syncthreads();
            edges();
            __syncthreads();
        }
    } else {
        const float ca = 2.0f - 2.0f * lam - P.beta, cb1 = 1.0f - P.beta;
        for (int s = 0; s < S.nsub; ++s) {
            for (int k = 1 + tid; k < L - 1; k += bd) {
                const float v = P.atten * (ca * A[k] + lam * (A[k + 1] + A[k - 1]) - cb1 * B[k]);
                O[k] = v;
                if (k == 1) O[0] = v;          // free boundary (FreeBC :139-157)
                if (k == L - 2) O[L - 1] = v;
            }
            __syncthreads();
            float* tmp = B;
            B = A;
            A = O;
            O = tmp;
        }
    }
    if (couple) {
        const float cw = (P.hix - P.lox) / (float)L;
        const float kd = P.kappa * (dt * (float)P.nsph);
        for (int k = tid; k < L; k += bd) {
            const float gx = ((float)k + 0.5f) * cw * P.invH - 0.5f;
            const float f0 = floorf(gx);
            const float al = gx - f0;
            const float f = clampf_nan(f0, -2.0f, (float)(P.nxc + 1));
            const int c0 = min(max((int)f, 0), P.nxc - 1);
            const int c1 = min(max((int)f + 1, 0), P.nxc - 1);
            const float Sx = (1.0f - al) * col[c0] + al * col[c1];
            A[k] = A[k] + kd * Sx * P.invH;
        }
    }
    for (int k = tid; k < L; k += bd) {
        g0[k] = A[k];
        g1[k] = B[k];
    }
}

// Splash (Shallow1D_cs.glsl:101-115) on the shallow-water scenes (scene < 0)
// or on one: h += -0.1 V exp(-xc^2/0.005), uh += 0.2 |dh| sign(xc).
__global__ void __launch_bounds__(256) k2_splash(const Scene2D* __restrict__ sc, int only,
                                                 float view_height, float* __restrict__ h,
                                                 float* __restrict__ uh) {
    const int s = blockIdx.y;
    if (only >= 0 && s != only) return;
    const Scene2D S = sc[s];
    if (S.model != CWA2D_WAVE_SHALLOW) return;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < S.L; k += gridDim.x * blockDim.x) {
        const float x = (float)k / (float)(S.L - 1);
        const float xc = x - 0.5f;
        const float dh = -view_height * 0.1f * expf(-xc * xc / 0.005f);
        const float sg = xc > 0.0f ? 1.0f : (xc < 0.0f ? -1.0f : 0.0f);
        h[S.wbeg + k] += dh;
        uh[S.wbeg + k] += 0.2f * fabsf(dh) * sg;
    }
}

// Render copy: (x, y) of every slot into a caller buffer.
__global__ void __launch_bounds__(256) k2_points(const float4* __restrict__ xv, int n,
                                                 float2* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float4 p = xv[i];
        out[i] = make_float2(p.x, p.y);
    }
}

inline int blocks_for(long long n, int bs) { return (int)((n + bs - 1) / bs); }

static float exact_r2_threshold(float h) {
    float x = h * h;
    while (x > 0.0f && std::sqrt(x) >= h) x = std::nextafter(x, 0.0f);
    while (!(std::sqrt(x) >= h)) x = std::nextafter(x, INFINITY);
    return x;
}

static int grid_dim(float lo, float hi, float h) {
    const float w = (hi - lo) / h;
    return std::max(1, (int)std::ceil(w));
}

static Dev2 make_dev2(const cwa2d_params& p) {
    Dev2 d{};
    d.H = p.h;
    d.HSQ = d.H * d.H;
    d.invH = 1.0f / d.H;
    d.T = exact_r2_threshold(p.h);
    d.k2 = 40.0f / (7.0f * (float)3.14159265 * d.HSQ);
    d.k2x2 = d.k2 * 2.0f;
    d.c6k2 = 6.0f * d.k2;
    d.m6k2 = -6.0f * d.k2;
    d.ga = d.c6k2 * d.invH;
    d.gb = d.m6k2 * d.invH;
    d.c01 = 0.01f * d.HSQ;
    d.rho0 = p.rest_rho;
    d.k = p.gas_const;
    d.visc_pre = -p.visc * 8.0f;
    d.psi = p.psi;
    d.gx = p.gravity[0];
    d.gy = p.gravity[1];
    d.lox = p.lo[0];
    d.loy = p.lo[1];
    d.hix = p.hi[0];
    d.hiy = p.hi[1];
    for (int i = 0; i < 4; ++i) d.walls[i] = p.walls[i];
    d.thr = p.enable_vel;
    d.wref = p.wave_ref;
    d.wpress = p.wave_press;
    d.wdy = p.wave_dy;
    d.wmask = p.wave_maskv;
    d.atten = p.atten;
    d.beta = p.beta;
    d.band = p.couple_band;
    d.kappa = p.couple_strength;
    d.hc = 0.5f * p.h;
    d.nx = grid_dim(p.lo[0], p.hi[0], d.hc);
    d.ny = grid_dim(p.lo[1], p.hi[1], d.hc);
    d.ncell = d.nx * d.ny;
    d.nxc = grid_dim(p.lo[0], p.hi[0], p.h);
    {   // margin of the trimmed rows: far above the rounding of the bounds
        const float ext = std::max({std::fabs(p.lo[0]), std::fabs(p.hi[0]), std::fabs(p.lo[1]),
                                    std::fabs(p.hi[1]), p.h});
        d.eps = 4e-6f * ext;
    }
    d.nsph = std::max(1, (int)p.sph_substeps);
    return d;
}

static void validate(const cwa2d_params& p) {
    auto fin = [](float v) { return std::isfinite(v); };
    // the pair loops' square root and reciprocals are exact in this range
    if (!(p.h >= 0x1p-16f) || !(p.h <= 0x1p19f)) throw Error(CWA_EINVAL, "h must be in [2^-16, 2^19]");
    if (!(p.rest_rho > 0.0f) || !fin(p.rest_rho)) throw Error(CWA_EINVAL, "rest_rho must be positive");
    if (!(p.hi[0] > p.lo[0]) || !(p.hi[1] > p.lo[1]) || !fin(p.lo[0]) || !fin(p.hi[0]) ||
        !fin(p.lo[1]) || !fin(p.hi[1]))
        throw Error(CWA_EINVAL, "domain needs hi > lo");
    if (!(p.wave_maskv > 0.0f) || !(p.wave_dy > 0.0f))
        throw Error(CWA_EINVAL, "wave_maskv and wave_dy must be positive");
    if (p.sph_substeps < 1 || p.sph_substeps > 64) throw Error(CWA_EINVAL, "sph_substeps in 1..64");
    const double cells = (double)grid_dim(p.lo[0], p.hi[0], 0.5f * p.h) *
                         grid_dim(p.lo[1], p.hi[1], 0.5f * p.h);
    if (cells > (double)(1 << 24)) throw Error(CWA_EINVAL, "grid too fine for the domain (cells per scene > 2^24)");
    if (grid_dim(p.lo[0], p.hi[0], p.h) > 4096) throw Error(CWA_EINVAL, "more than 4096 grid columns");
}

// ---------------------------------------------------------------------------
// Batch2D: the batch as a Module (SphUgrid + ImageStencil per scene)
// ---------------------------------------------------------------------------
enum K2Slot { B_HASH, B_SCAN, B_SCATTER, B_REORDER, B_DENSITY, B_FORCE, B_WAVE };
static const char* kNames[CWA2D_NUM_KERNELS] = {"hash", "scan", "scatter", "reorder",
                                                "density", "force", "wave"};

struct TileSet {
    DeviceBuffer<int4> tiles;
    DeviceBuffer<int> len;  // entries per XCD
    int ntiles = 0;  // table entries, empty ones included
};

class Batch2D {
   public:
    Batch2D(const cwa2d_params& p, int nscenes, const cwa2d_scene* scenes) {
        validate(p);
        if (nscenes < 1) throw Error(CWA_EINVAL, "nscenes must be >= 1");
        params_ = p;
        dev_ = make_dev2(p);
        long long po = 0, wo = 0;
        host_sc_.resize(nscenes);
        lmax_ = 3;
        for (int s = 0; s < nscenes; ++s) {
            const cwa2d_scene& q = scenes[s];
            if (q.n < 1) throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": n < 1");
            if (q.wave_len < 3 || q.wave_len > CWA2D_MAX_WAVE_LEN)
                throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": wave_len out of range");
            if (q.wave_substeps < 1 || q.wave_substeps > 1024)
                throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": wave_substeps in 1..1024");
            if (!(q.mass > 0.0f) || !std::isfinite(q.mass) || !std::isfinite(q.lambda))
                throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": bad mass or lambda");
            if (q.wave_model != CWA2D_WAVE_LEAPFROG && q.wave_model != CWA2D_WAVE_SHALLOW)
                throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": unknown wave model");
            if (q.wave_model == CWA2D_WAVE_SHALLOW && (!(q.wave_dx > 0.0f) || !std::isfinite(q.wave_dx)))
                throw Error(CWA_EINVAL, "scene " + std::to_string(s) + ": wave_dx must be positive");
            Scene2D& d = host_sc_[s];
            d.pbeg = (int)po;
            d.n = q.n;
            d.wbeg = (int)wo;
            d.L = q.wave_len;
            d.nsub = q.wave_substeps;
            d.model = q.wave_model;
            d.mass = q.mass;
            d.lambda = q.lambda;
            d.dx = q.wave_dx;
            po += q.n;
            wo += q.wave_len;
            lmax_ = std::max(lmax_, q.wave_len);
        }
        if (po > CWA2D_MAX_PARTICLES) throw Error(CWA_EINVAL, "too many particles in the batch");
        ns_ = nscenes;
        ntot_ = (int)po;
        wtot_ = (int)wo;
        const long long cells = (long long)nscenes * dev_.ncell;
        if (cells + 1 > (1ll << 30)) throw Error(CWA_EINVAL, "too many cells in the batch");
        ncells_ = (int)cells;
        lds_bytes_ = (size_t)(4 * lmax_ + dev_.nxc) * sizeof(float);
        if (lds_bytes_ > 160 * 1024) throw Error(CWA_EINVAL, "wave column and grid exceed LDS");

        hip_check(hipStreamCreateWithFlags(&st_, hipStreamNonBlocking), "stream");
        int dev = 0;
        hip_check(hipGetDevice(&dev), "device");
        hip_check(hipDeviceGetAttribute(&num_cu_, hipDeviceAttributeMultiprocessorCount, dev), "cu count");
        if (lds_bytes_ > 65536)
            hip_check(hipFuncSetAttribute((const void*)k2_wave,
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          (int)lds_bytes_),
                      "wave lds");

        sc_.resize(ns_);
        hip_check(hipMemcpy(sc_.get(), host_sc_.data(), sizeof(Scene2D) * ns_, hipMemcpyHostToDevice), "scenes");
        std::vector<int> bsc(blocks_for(ntot_, 256));
        {
            int s = 0;
            for (size_t b = 0; b < bsc.size(); ++b) {
                const long long i = (long long)b * 256;
                while (i >= host_sc_[s].pbeg + host_sc_[s].n) ++s;
                bsc[b] = s;
            }
        }
        blk_scene_.resize(bsc.size());
        hip_check(hipMemcpy(blk_scene_.get(), bsc.data(), sizeof(int) * bsc.size(), hipMemcpyHostToDevice), "block scenes");
        std::vector<int> pb(ns_), wb(ns_);
        for (int s = 0; s < ns_; ++s) {
            pb[s] = host_sc_[s].pbeg;
            wb[s] = host_sc_[s].wbeg;
        }
        pbeg_.resize(ns_);
        wbeg_.resize(ns_);
        hip_check(hipMemcpy(pbeg_.get(), pb.data(), sizeof(int) * ns_, hipMemcpyHostToDevice), "pbeg");
        hip_check(hipMemcpy(wbeg_.get(), wb.data(), sizeof(int) * ns_, hipMemcpyHostToDevice), "wbeg");

        for (int k = 0; k < 2; ++k) {
            rp_[k].resize(ntot_);
            idf_[k].resize(ntot_);
        }
        xv_.resize(ntot_);
        xy_.resize(ntot_ + kReadPast2D);
        vel_.resize(ntot_);
        qxy_.resize(ntot_ + kReadPast2D);
        qva_.resize(ntot_ + kReadPast2D);
        flux_.resize(ntot_);
        key_.resize(ntot_);
        link_.resize(ntot_);
        head_.resize(ncells_ + 1);
        count_.resize(ncells_ + 1);
        offset_.resize(ncells_ + 1);
        ws_.resize(scan_workspace_ints(ncells_ + 1));
        queue_.resize(2 * kNumXcd);
        h0_.resize(wtot_);
        h1_.resize(wtot_);
        finite_.resize(1);
        ZeroLists();
        hip_check(hipMemset(offset_.get(), 0, sizeof(int) * (ncells_ + 1)), "offset zero");
        hip_check(hipMemset(key_.get(), 0, sizeof(int) * ntot_), "key zero");

        tune_.block_density = 256;
        tune_.block_force = 256;
        tune_.grid_density = 0;
        tune_.grid_force = 0;
        tune_.xcd_queues = 1;
        // the largest block, for a scene's column sums and substeps (MI355X, 256
        // threads -> 1 024: 256 scenes 59 -> 23 us, 24 small ones 16.3 -> 9.3, the
        // application's scene 6.2 both)
        tune_.wave_block = 1024;
        tune_.ms_per_step = 0.0f;
        for (auto& e : ev_)
            for (auto& x : e) hip_check(hipEventCreate(&x), "event");
    }

    ~Batch2D() {
        for (auto& g : graphs_)
            if (g.second) (void)hipGraphExecDestroy(g.second);
        for (auto& e : ev_)
            for (auto& x : e)
                if (x) (void)hipEventDestroy(x);
        if (st_) {
            (void)hipStreamSynchronize(st_);
            (void)hipStreamDestroy(st_);
        }
    }

    void Reinit(const float* xv, const int32_t* en, const float* h0, const float* h1) {
        if (!xv) throw Error(CWA_EINVAL, "xv is required");
        std::vector<float2> rp(ntot_, make_float2(params_.rest_rho, 0.0f));
        std::vector<int> idf(ntot_);
        for (int s = 0; s < ns_; ++s)
            for (int i = 0; i < host_sc_[s].n; ++i) {
                const int g = host_sc_[s].pbeg + i;
                const int e = en ? (en[g] != 0) : 1;
                idf[g] = i | (e << 30);
            }
        for (long long i = 0; i < 4ll * ntot_; ++i)
            if (!std::isfinite(xv[i])) throw Error(CWA_EINVAL, "non-finite particle state");
        hip_check(hipStreamSynchronize(st_), "sync");
        hip_check(hipMemcpy(xv_.get(), xv, sizeof(float4) * ntot_, hipMemcpyHostToDevice), "xv");
        hip_check(hipMemcpy(rp_[0].get(), rp.data(), sizeof(float2) * ntot_, hipMemcpyHostToDevice), "rp");
        hip_check(hipMemcpy(idf_[0].get(), idf.data(), sizeof(int) * ntot_, hipMemcpyHostToDevice), "idf");
        std::vector<float> z(wtot_, 0.0f);
        hip_check(hipMemcpy(h0_.get(), h0 ? h0 : z.data(), sizeof(float) * wtot_, hipMemcpyHostToDevice), "h0");
        hip_check(hipMemcpy(h1_.get(), h1 ? h1 : z.data(), sizeof(float) * wtot_, hipMemcpyHostToDevice), "h1");
        ZeroLists();
        hip_check(hipDeviceSynchronize(), "reinit");
    }

    void SetParams(const cwa2d_params& p) {
        validate(p);
        const Dev2 d = make_dev2(p);
        if (d.nx != dev_.nx || d.ny != dev_.ny)
            throw Error(CWA_EINVAL, "parameters change the grid dimensions of the batch");
        if ((size_t)(4 * lmax_ + d.nxc) * sizeof(float) > lds_bytes_)
            throw Error(CWA_EINVAL, "grid exceeds the wave pass's LDS");
        params_ = p;
        dev_ = d;
        InvalidateGraph();
    }
    const cwa2d_params& Params() const { return params_; }

    void SetTuning(const cwa2d_tuning& t) {
        auto okb = [](int b) { return b == 64 || b == 128 || b == 256 || b == 512 || b == 1024; };
        if (!okb(t.block_density) || !okb(t.block_force) || !okb(t.wave_block))
            throw Error(CWA_EINVAL, "block sizes must be 64, 128, 256, 512 or 1024");
        if (t.grid_density < 0 || t.grid_force < 0) throw Error(CWA_EINVAL, "grid must be >= 0");
        tune_ = t;
        tune_.xcd_queues = t.xcd_queues ? 1 : 0;
        InvalidateGraph();
    }
    const cwa2d_tuning& Tuning() const { return tune_; }

    // The launches of a call.  Between its steps the counts and run lists hold the
    // next step's keys; a call that fails there leaves them so, and the next
    // one, which hashes afresh, clears them first.
    template <class F>
    void WithLists(F&& launches) {
        if (lists_left_)
            hip_check(launch_clear_cells(nullptr, count_.get(), head_.get(), nullptr, nullptr,
                                         ncells_, st_),
                      "clear lists");
        lists_left_ = true;
        launches();
        lists_left_ = false;
    }

    // --- one step on the stream (optionally with events around kernels) ---
    // keyed: the force pass of the step before hashed its positions; key_next:
    // this one's does for the next.
    void Step(float dt, bool profile, bool keyed = false, bool key_next = false) {
        const int nq = tune_.xcd_queues ? kNumXcd : 1;
        const TileSet& td = Tiles(tune_.block_density, nq);
        const TileSet& tf = Tiles(tune_.block_force, nq);
        auto mark = [&](int slot, int which) {
            if (profile) hip_check(hipEventRecord(ev_[slot][which], st_), "event");
        };
        const Keys2D keys{key_.get(), {count_.get(), head_.get(), link_.get()}};
        for (int sub = 0; sub < dev_.nsph; ++sub) {
            const bool first = sub == 0;
            const bool last = sub == dev_.nsph - 1;
            const bool hash_next = last ? key_next : true;
            mark(B_HASH, first ? 0 : 2);
            if (!keyed) {
                k2_hash<<<blocks_for(ntot_, 256), 256, 0, st_>>>(
                    dev_, sc_.get(), blk_scene_.get(), xv_.get(), ntot_, keys);
                hip_check(hipGetLastError(), "hash");
            }
            mark(B_HASH, first ? 1 : 3);
            mark(B_SCAN, first ? 0 : 2);
            hip_check(launch_scan(count_.get(), offset_.get(), ncells_, ws_.get(), st_, nullptr), "scan");
            mark(B_SCAN, first ? 1 : 3);
            mark(B_SCATTER, first ? 0 : 2);  // the runs are listed where the keys are counted
            mark(B_SCATTER, first ? 1 : 3);
            mark(B_REORDER, first ? 0 : 2);
            k2_reorder<<<blocks_for(std::max(ntot_, ncells_), 256), 256, 0, st_>>>(
                keys, offset_.get(), ntot_, xv_.get(), rp_[0].get(), idf_[0].get(), xy_.get(),
                vel_.get(), rp_[1].get(), idf_[1].get(), ncells_, queue_.get());
            hip_check(hipGetLastError(), "reorder");
            mark(B_REORDER, first ? 1 : 3);

            DensityArgs da{sc_.get(), {td.tiles.get(), td.ntiles, nq, queue_.get(), td.len.get()}, xy_.get(), vel_.get(), rp_[1].get(), idf_[1].get(), offset_.get(),
                           h0_.get(), h1_.get(), qxy_.get(), qva_.get(), rp_[0].get(), idf_[0].get(), flux_.get(),
                           head_.get(), sparse() ? 0 : ncells_};
            mark(B_DENSITY, first ? 0 : 2);
            if (sparse()) {
                k2_clear_lists<<<blocks_for(ntot_, 256), 256, 0, st_>>>(keys, ntot_);
                hip_check(hipGetLastError(), "clear lists");
            }
            LaunchDensity(da, dt);
            mark(B_DENSITY, first ? 1 : 3);
            ForceArgs fa{sc_.get(), {tf.tiles.get(), tf.ntiles, nq, queue_.get() + kNumXcd, tf.len.get()}, qxy_.get(), qva_.get(), idf_[0].get(), offset_.get(), h0_.get(), h1_.get(),
                         xv_.get(), hash_next ? keys : Keys2D{}};
            mark(B_FORCE, first ? 0 : 2);
            LaunchForce(fa, dt);
            mark(B_FORCE, first ? 1 : 3);
            keyed = hash_next;
        }
        mark(B_WAVE, 0);
        k2_wave<<<ns_, tune_.wave_block, lds_bytes_, st_>>>(dev_, dt, sc_.get(), offset_.get(),
                                                             flux_.get(), h0_.get(), h1_.get(), lmax_);
        hip_check(hipGetLastError(), "wave");
        mark(B_WAVE, 1);
    }

    void StepN(float dt, int steps) {
        WithLists([&] {
            for (int k = 0; k < steps; ++k) Step(dt, false, k > 0, k + 1 < steps);
        });
        if (params_.check_finite) CheckFinite();
    }

    // Steps of a captured run: whether its keys come from the step before it, and
    // whether it hashes for a step after it (Step).
    struct GraphForm {
        bool keyed, next;
        int steps;
        bool operator<(const GraphForm& o) const {
            return std::tie(keyed, next, steps) < std::tie(o.keyed, o.next, o.steps);
        }
    };
    // Steps a graph holds: what a capture costs the first call grows with its
    // launches, what a longer run saves does not (a call of 6 steps of 32 substeps,
    // captures included: 7.1 ms from graphs of one step, 11.1 of six).
    static constexpr int kGraphSteps = 8, kGraphLaunches = 176;
    int graph_steps() const {
        return std::min(std::max(kGraphLaunches / (5 * dev_.nsph + 1), 1), kGraphSteps);
    }

    // Graphs of up to graph_steps() steps, captured when first needed: a call of that
    // many is one of them, a longer one a first step, runs of that many and the
    // rest.  Every replay between two steps costs the host a launch and the GPU
    // a gap (MI355X, three batches in flight, a graph a step -> these: 6 steps of 19
    // scenes of 6 601 particles 203 -> 122 us a call, 60 steps 1 260 -> 766, 10 steps of
    // the application's scene, eight copies, 311 -> 237; graphs of 4 and 16 steps: 161 and
    // 128, 784 and 757, 238 and 236).
    void StepGraph(float dt, int steps) {
        if (graph_dt_ != dt) InvalidateGraph();
        graph_dt_ = dt;
        const int most = graph_steps();
        const auto each_run = [&](auto&& f) {
            for (int done = 0; done < steps;) {
                const int left = steps - done;
                const int n = left <= most ? left : done == 0 ? 1 : most;
                f(GraphForm{done > 0, left > n, n});
                done += n;
            }
        };
        // all of them before the first runs: a capture that fails leaves the state as it was
        each_run([&](const GraphForm& form) {
            hipGraphExec_t& exec = graphs_[form];
            if (!exec) CaptureGraph(exec, dt, form);
        });
        WithLists([&] {
            each_run([&](const GraphForm& form) {
                hip_check(hipGraphLaunch(graphs_[form], st_), "graph launch");
            });
        });
        if (params_.check_finite) CheckFinite();
    }

    void CaptureGraph(hipGraphExec_t& exec, float dt, const GraphForm& f) {
        // tile tables allocate: build them before the capture
        const int nq = tune_.xcd_queues ? kNumXcd : 1;
        Tiles(tune_.block_density, nq);
        Tiles(tune_.block_force, nq);
        hipGraph_t g = nullptr;
        hip_check(hipStreamBeginCapture(st_, hipStreamCaptureModeThreadLocal), "capture");
        try {
            for (int k = 0; k < f.steps; ++k)
                Step(dt, false, f.keyed || k > 0, f.next || k + 1 < f.steps);
        } catch (...) {
            (void)hipStreamEndCapture(st_, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        hip_check(hipStreamEndCapture(st_, &g), "end capture");
        const hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) exec = nullptr;
        hip_check(e, "graph instantiate");
    }

    void StepProfiled(float dt, cwa2d_kernel_times* t) {
        WithLists([&] { Step(dt, true); });
        hip_check(hipStreamSynchronize(st_), "sync");
        for (int k = 0; k < CWA2D_NUM_KERNELS; ++k) {
            float ms = 0.0f;
            hip_check(hipEventElapsedTime(&ms, ev_[k][0], ev_[k][1]), "elapsed");
            if (dev_.nsph > 1 && k != B_WAVE) {
                float m2 = 0.0f;
                hip_check(hipEventElapsedTime(&m2, ev_[k][2], ev_[k][3]), "elapsed");
                ms += m2 * (float)(dev_.nsph - 1);  // later substeps: last one, scaled
            }
            if (t) t->ms[k] = ms;
        }
        if (params_.check_finite) CheckFinite();
    }

    void CheckFinite() {
        hip_check(hipMemsetAsync(finite_.get(), 0, sizeof(int), st_), "finite zero");
        hip_check(launch_check_finite(reinterpret_cast<const float*>(xv_.get()), 4ull * ntot_,
                                      finite_.get(), st_), "finite xv");
        hip_check(launch_check_finite(h0_.get(), (size_t)wtot_, finite_.get(), st_), "finite h0");
        int flag = 0;
        hip_check(hipMemcpyAsync(&flag, finite_.get(), sizeof(int), hipMemcpyDeviceToHost, st_), "finite copy");
        hip_check(hipStreamSynchronize(st_), "sync");
        if (flag) throw Error(CWA_ENONFINITE, "non-finite particle or wave state after the step");
    }

    void Splash(int scene, float view_height) {
        if (scene >= ns_) throw Error(CWA_EINVAL, "scene index out of range");
        dim3 grd(blocks_for(lmax_, 256), ns_);
        k2_splash<<<grd, 256, 0, st_>>>(sc_.get(), scene, view_height, h0_.get(), h1_.get());
        hip_check(hipGetLastError(), "splash");
    }

    void Render(float* points_xy, float* wave) {
        if (points_xy) {
            k2_points<<<blocks_for(ntot_, 256), 256, 0, st_>>>(
                xv_.get(), ntot_, reinterpret_cast<float2*>(points_xy));
            hip_check(hipGetLastError(), "render points");
        }
        if (wave)
            hip_check(hipMemcpyAsync(wave, h0_.get(), sizeof(float) * wtot_,
                                     hipMemcpyDeviceToDevice, st_),
                      "render wave");
    }

    void Sync() { hip_check(hipStreamSynchronize(st_), "sync"); }
    hipStream_t stream() const { return st_; }

    void Views(cwa2d_views* v) {
        v->nscenes = ns_;
        v->n_total = ntot_;
        v->wave_total = wtot_;
        v->grid_nx = dev_.nx;
        v->grid_ny = dev_.ny;
        v->cells_total = ncells_;
        v->xv = reinterpret_cast<float*>(xv_.get());
        v->rp = reinterpret_cast<float*>(rp_[0].get());
        v->idf = idf_[0].get();
        v->key = key_.get();
        v->offset = offset_.get();
        v->h0 = h0_.get();
        v->h1 = h1_.get();
        v->scene_begin = pbeg_.get();
        v->wave_begin = wbeg_.get();
    }

    void Readback(float* xv, float* rp, int32_t* en, float* h0, float* h1) {
        Sync();
        std::vector<float4> x(ntot_);
        std::vector<float2> r(ntot_);
        std::vector<int> idf(ntot_);
        hip_check(hipMemcpy(x.data(), xv_.get(), sizeof(float4) * ntot_, hipMemcpyDeviceToHost), "xv");
        hip_check(hipMemcpy(r.data(), rp_[0].get(), sizeof(float2) * ntot_, hipMemcpyDeviceToHost), "rp");
        hip_check(hipMemcpy(idf.data(), idf_[0].get(), sizeof(int) * ntot_, hipMemcpyDeviceToHost), "idf");
        for (int s = 0; s < ns_; ++s) {
            const Scene2D& S = host_sc_[s];
            for (int k = 0; k < S.n; ++k) {
                const int slot = S.pbeg + k;
                const int id = idf[slot] & 0x3FFFFFFF;
                if (id >= S.n) throw Error(CWA_ESTATE, "particle id out of range");
                const int g = S.pbeg + id;
                if (xv) std::memcpy(xv + 4ll * g, &x[slot], sizeof(float4));
                if (rp) std::memcpy(rp + 2ll * g, &r[slot], sizeof(float2));
                if (en) en[g] = (idf[slot] >> 30) & 1;
            }
        }
        if (h0) hip_check(hipMemcpy(h0, h0_.get(), sizeof(float) * wtot_, hipMemcpyDeviceToHost), "h0");
        if (h1) hip_check(hipMemcpy(h1, h1_.get(), sizeof(float) * wtot_, hipMemcpyDeviceToHost), "h1");
    }

    // --- autotuner -------------------------------------------------------
    cwa2d_tuning Tune(float dt, int steps) {
        if (steps < 1) throw Error(CWA_EINVAL, "tune steps must be >= 1");
        Snapshot snap(*this);
        const cwa2d_tuning start = tune_;
        const int blocks[] = {64, 128, 256, 512};
        const int mults[] = {0, 1, 2, 4, 8};  // persistent blocks per CU (0: one per tile)
        struct Cand {
            cwa2d_tuning t;
            double dens = 0, force = 0;
        };
        std::vector<Cand> cands;
        for (int xq = 0; xq < 2; ++xq)
            for (int b : blocks)
                for (int m : mults) {
                    Cand c;
                    c.t = start;
                    c.t.block_density = c.t.block_force = b;
                    c.t.grid_density = c.t.grid_force = m * num_cu_;
                    c.t.xcd_queues = xq;
                    cands.push_back(c);
                }
        cwa2d_kernel_times kt{};
        for (auto& c : cands) {
            snap.Restore(*this);
            SetTuning(c.t);
            WithLists([&] { Step(dt, false); });  // warm caches and tiles for this setting
            snap.Restore(*this);
            for (int k = 0; k < steps; ++k) {
                StepProfiled(dt, &kt);
                c.dens += kt.ms[B_DENSITY];
                c.force += kt.ms[B_FORCE];
            }
        }
        cwa2d_tuning best = start;
        double bd = 1e30, bf = 1e30;
        for (auto& c : cands) {
            if (c.dens < bd) {
                bd = c.dens;
                best.block_density = c.t.block_density;
                best.grid_density = c.t.grid_density;
                best.xcd_queues = c.t.xcd_queues;
            }
        }
        for (auto& c : cands) {
            if (c.t.xcd_queues != best.xcd_queues) continue;  // one queue layout for both
            if (c.force < bf) {
                bf = c.force;
                best.block_force = c.t.block_force;
                best.grid_force = c.t.grid_force;
            }
        }
        double bw = 1e30;
        for (int wbk : {128, 256, 512, 1024}) {
            cwa2d_tuning t = best;
            t.wave_block = wbk;
            snap.Restore(*this);
            SetTuning(t);
            double w = 0;
            for (int k = 0; k < steps; ++k) {
                StepProfiled(dt, &kt);
                w += kt.ms[B_WAVE];
            }
            if (w < bw) {
                bw = w;
                best.wave_block = wbk;
            }
        }
        // the chosen setting, timed as graph replays: the same call before, for its captures
        snap.Restore(*this);
        SetTuning(best);
        StepGraph(dt, steps);
        Sync();
        snap.Restore(*this);
        hipEvent_t a = ev_[0][0], b = ev_[0][1];
        hip_check(hipEventRecord(a, st_), "event");
        StepGraph(dt, steps);
        hip_check(hipEventRecord(b, st_), "event");
        Sync();
        float ms = 0.0f;
        hip_check(hipEventElapsedTime(&ms, a, b), "elapsed");
        best.ms_per_step = ms / (float)steps;
        tune_.ms_per_step = best.ms_per_step;
        snap.Restore(*this);
        return tune_;
    }

   private:
    struct Snapshot {
        DeviceBuffer<float4> xv;
        DeviceBuffer<float2> rp;
        DeviceBuffer<int> idf;
        DeviceBuffer<float> h0, h1;
        explicit Snapshot(Batch2D& b) {
            b.Sync();
            xv.resize(b.ntot_);
            rp.resize(b.ntot_);
            idf.resize(b.ntot_);
            h0.resize(b.wtot_);
            h1.resize(b.wtot_);
            copy(b, false);
        }
        void copy(Batch2D& b, bool restore) {
            auto cp = [&](void* dst, const void* src, size_t bytes) {
                hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, b.st_), "snapshot");
            };
            if (!restore) {
                cp(xv.get(), b.xv_.get(), sizeof(float4) * b.ntot_);
                cp(rp.get(), b.rp_[0].get(), sizeof(float2) * b.ntot_);
                cp(idf.get(), b.idf_[0].get(), sizeof(int) * b.ntot_);
                cp(h0.get(), b.h0_.get(), sizeof(float) * b.wtot_);
                cp(h1.get(), b.h1_.get(), sizeof(float) * b.wtot_);
            } else {
                cp(b.xv_.get(), xv.get(), sizeof(float4) * b.ntot_);
                cp(b.rp_[0].get(), rp.get(), sizeof(float2) * b.ntot_);
                cp(b.idf_[0].get(), idf.get(), sizeof(int) * b.ntot_);
                cp(b.h0_.get(), h0.get(), sizeof(float) * b.wtot_);
                cp(b.h1_.get(), h1.get(), sizeof(float) * b.wtot_);
            }
            b.Sync();
        }
        void Restore(Batch2D& b) { copy(b, true); }
    };

    void InvalidateGraph() {
        if (graphs_.empty()) return;
        (void)hipStreamSynchronize(st_);
        for (auto& g : graphs_)
            if (g.second) (void)hipGraphExecDestroy(g.second);
        graphs_.clear();
    }

    // The tile table for blocks of `bs` slots, its entries dealt to nq XCDs in
    // turn (1: one list in order of cost).
    const TileSet& Tiles(int bs, int nq) {
        const int key = bs * 16 + nq;
        auto it = tiles_.find(key);
        if (it != tiles_.end()) return it->second;
        // a particle's cost: its neighbours grow with n_s, the rest does not
        const auto cost = [&](int s) { return (double)host_sc_[s].n + 4096.0; };
        double total = 0.0;
        for (const Scene2D& S : host_sc_) total += (double)S.n * ((double)S.n + 4096.0);
        const double most = std::max(total / (nq * kPiecesPerXcd), 1.0);
        std::vector<int> order(ns_);
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(),
                         [&](int a, int b) { return host_sc_[a].n > host_sc_[b].n; });
        std::vector<double> load(nq, 0.0);
        std::vector<std::vector<int4>> per(nq);
        for (int s : order) {
            const Scene2D& S = host_sc_[s];
            const int end = S.pbeg + S.n;
            // whole tiles per piece
            const int piece =
                (int)std::min<double>((std::floor(most / (cost(s) * bs)) + 1.0) * bs, S.n);
            for (int p = S.pbeg; p < end; p += piece) {
                const int stop = std::min(p + piece, end);
                const int q = (int)(std::min_element(load.begin(), load.end()) - load.begin());
                load[q] += (double)(stop - p) * cost(s);
                for (int b = p; b < stop; b += bs)
                    per[q].push_back(make_int4(s, b, std::min(b + bs, stop), 0));
            }
        }
        size_t longest = 0;
        for (const auto& v : per) longest = std::max(longest, v.size());
        std::vector<int4> tl(longest * nq, make_int4(-1, 0, 0, 0));
        for (int q = 0; q < nq; ++q)
            for (size_t k = 0; k < per[q].size(); ++k) tl[k * nq + q] = per[q][k];
        TileSet& t = tiles_[key];
        t.ntiles = (int)tl.size();
        t.tiles.resize(tl.size());
        t.len.resize(nq);
        std::vector<int> len(nq);
        for (int q = 0; q < nq; ++q) len[q] = (int)per[q].size();
        hip_check(hipMemcpy(t.len.get(), len.data(), sizeof(int) * nq, hipMemcpyHostToDevice), "tile counts");
        hip_check(hipMemcpy(t.tiles.get(), tl.data(), sizeof(int4) * tl.size(), hipMemcpyHostToDevice), "tiles");
        return t;
    }

    // One block per tile, or g persistent blocks when those are fewer.
    // kQuadMax2D's rule; persistent blocks are a tuning choice
    bool quads() const { return ntot_ <= kQuadMax2D; }
    bool sparse() const { return ncells_ / kSparseCells > ntot_; }
    void ZeroLists() {
        hip_check(hipMemset(count_.get(), 0, sizeof(int) * (ncells_ + 1)), "count zero");
        hip_check(hipMemset(head_.get(), 0, sizeof(int) * (ncells_ + 1)), "list zero");
        lists_left_ = false;
    }
    template <int BS>
    void LaunchDensityOf(const DensityArgs& a, float dt) {
        const int g = tune_.grid_density;
        if (g > 0 && g < a.tiles.n)
            k2_density<BS, Form::persistent><<<g, BS, 0, st_>>>(dev_, dt, a);
        else if (quads())
            k2_density<BS, Form::quads><<<4 * a.tiles.n, BS, 0, st_>>>(dev_, dt, a);
        else
            k2_density<BS, Form::tiles><<<a.tiles.n, BS, 0, st_>>>(dev_, dt, a);
    }
    template <int BS>
    void LaunchForceOf(const ForceArgs& a, float dt) {
        const int g = tune_.grid_force;
        if (g > 0 && g < a.tiles.n)
            k2_force<BS, Form::persistent><<<g, BS, 0, st_>>>(dev_, dt, a);
        else if (quads())
            k2_force<BS, Form::quads><<<4 * a.tiles.n, BS, 0, st_>>>(dev_, dt, a);
        else
            k2_force<BS, Form::tiles><<<a.tiles.n, BS, 0, st_>>>(dev_, dt, a);
    }
    void LaunchDensity(const DensityArgs& a, float dt) {
        switch (tune_.block_density) {
            case 64: LaunchDensityOf<64>(a, dt); break;
            case 128: LaunchDensityOf<128>(a, dt); break;
            case 256: LaunchDensityOf<256>(a, dt); break;
            case 512: LaunchDensityOf<512>(a, dt); break;
            default: LaunchDensityOf<1024>(a, dt); break;
        }
        hip_check(hipGetLastError(), "density");
    }
    void LaunchForce(const ForceArgs& a, float dt) {
        switch (tune_.block_force) {
            case 64: LaunchForceOf<64>(a, dt); break;
            case 128: LaunchForceOf<128>(a, dt); break;
            case 256: LaunchForceOf<256>(a, dt); break;
            case 512: LaunchForceOf<512>(a, dt); break;
            default: LaunchForceOf<1024>(a, dt); break;
        }
        hip_check(hipGetLastError(), "force");
    }

    cwa2d_params params_{};
    Dev2 dev_{};
    int ns_ = 0, ntot_ = 0, wtot_ = 0, ncells_ = 0, lmax_ = 3, num_cu_ = 256;
    size_t lds_bytes_ = 0;
    std::vector<Scene2D> host_sc_;
    DeviceBuffer<Scene2D> sc_;
    DeviceBuffer<int> blk_scene_, pbeg_, wbeg_;
    DeviceBuffer<float4> xv_;
    DeviceBuffer<float2> xy_, vel_;  // sorted copy, read in order by the density pass
    DeviceBuffer<float2> rp_[2];
    DeviceBuffer<int> idf_[2];
    DeviceBuffer<float2> qxy_;  // what the force pass reads: positions, and velocity,
    DeviceBuffer<float4> qva_;  // pressure term and 1/rho
    DeviceBuffer<float> flux_;
    DeviceBuffer<int> key_, count_, head_, offset_, ws_, queue_, finite_;
    DeviceBuffer<int2> link_;
    DeviceBuffer<float> h0_, h1_;
    std::map<int, TileSet> tiles_;
    cwa2d_tuning tune_{};
    bool lists_left_ = false;  // a call ended before its last step (WithLists)
    hipStream_t st_ = nullptr;
    std::map<GraphForm, hipGraphExec_t> graphs_;
    float graph_dt_ = 0.0f;
    hipEvent_t ev_[CWA2D_NUM_KERNELS][4] = {};
};

}  // namespace b2d
}  // namespace cwa

// ===========================================================================
// C ABI
// ===========================================================================
using cwa::Error;
using cwa::b2d::Batch2D;

struct cwa2d_batch {
    Batch2D* impl;
};

namespace {
template <class F>
int guarded2(F&& f) {
    return cwa::guarded_call([](void* c) { (*static_cast<F*>(c))(); }, &f);
}
Batch2D* impl(cwa2d_batch* b) {
    if (!b || !b->impl) throw Error(CWA_EINVAL, "null batch");
    return b->impl;
}
}  // namespace

extern "C" {

int cwa2d_abi_version(void) { return CWA2D_ABI_VERSION; }

int cwa2d_struct_size(int which) {
    switch (which) {
        case 0: return (int)sizeof(cwa2d_params);
        case 1: return (int)sizeof(cwa2d_scene);
        case 2: return (int)sizeof(cwa2d_tuning);
        case 3: return (int)sizeof(cwa2d_views);
        case 4: return (int)sizeof(cwa2d_kernel_times);
        default: return -1;
    }
}

const char* cwa2d_kernel_name(int k) {
    if (k < 0 || k >= CWA2D_NUM_KERNELS) return "";
    return cwa::b2d::kNames[k];
}

int cwa2d_params_reference(cwa2d_params* p) {
    return guarded2([&] {
        if (!p) throw Error(CWA_EINVAL, "null params");
        std::memset(p, 0, sizeof(*p));
        const float prad = 0.025f;                     // PARTICLE_RADIUS
        const float H = 4.0f * prad;                    // :120
        const float view = 2.0f * 4.8f;                 // VIEW_WIDTH/HEIGHT :132-133
        const float k2 = 40.0f / (7.0f * (float)3.14159265 * (H * H));
        p->h = H;
        p->rest_rho = 1000.0f;
        p->gas_const = 35000.0f;
        p->visc = 0.05f;
        p->psi = 1000.0f / (1.5f * k2);                 // :136
        p->gravity[0] = 0.0f;
        p->gravity[1] = -9.8f;
        p->lo[0] = p->lo[1] = 0.0f;
        p->hi[0] = p->hi[1] = view;
        p->walls[0] = 0.5f * view - 15.0f * prad + prad - 0.3f;  // plane0, bottom = 0.3
        p->walls[1] = prad;
        p->walls[2] = view - prad;
        p->walls[3] = view - prad;
        p->enable_vel = 0.05f;
        p->wave_ref = 0.5f * view;
        p->wave_press = 500000.0f;
        p->wave_dy = 10.0f;
        p->wave_maskv = 0.2f;
        p->atten = 0.9995f;
        p->beta = 0.001f;
        p->couple_band = 0.0f;
        p->couple_strength = 0.0f;
        p->sph_substeps = 2;                            // SphWave2D/Main.cpp
        p->check_finite = 0;
    });
}

int cwa2d_wave_init_reference(int32_t L, float* h0, float* h1) {
    return guarded2([&] {
        if (L < 3 || !h0 || !h1) throw Error(CWA_EINVAL, "wave_init: L >= 3 and two outputs");
        for (int mode = 0; mode < 2; ++mode) {
            float* out = mode == 0 ? h1 : h0;
            const int cen = (int)(0.25f * (float)L) + mode;
            for (int k = 0; k < L; ++k) {
                const int x = cen - k;
                out[k] = 0.0f + 0.1f * std::exp((float)(-x * x) / 5000.0f);
            }
        }
    });
}

int cwa2d_wave_init_shallow(int32_t L, float view_height, float* h, float* uh) {
    return guarded2([&] {
        if (L < 3 || !h || !uh) throw Error(CWA_EINVAL, "wave_init_shallow: L >= 3 and two outputs");
        for (int k = 0; k < L; ++k) {
            const float x = (float)k / (float)(L - 1);
            const float xc = x - 0.5f;
            const float h_free = view_height * 0.5f;
            const float bump = view_height * 0.1f * std::exp(-xc * xc / 0.005f);
            const float sg = xc > 0.0f ? 1.0f : (xc < 0.0f ? -1.0f : 0.0f);
            h[k] = h_free + bump;
            uh[k] = 0.5f * std::fabs(bump) * sg;
        }
    });
}

int cwa2d_batch_splash(cwa2d_batch* b, int32_t scene, float view_height) {
    return guarded2([&] { impl(b)->Splash(scene, view_height); });
}

int cwa2d_batch_render(cwa2d_batch* b, float* points_xy, float* wave) {
    return guarded2([&] { impl(b)->Render(points_xy, wave); });
}

int cwa2d_batch_create(const cwa2d_params* p, int32_t nscenes, const cwa2d_scene* scenes,
                       const float* xv, const int32_t* enabled, const float* h0, const float* h1,
                       cwa2d_batch** out) {
    return guarded2([&] {
        if (!p || !scenes || !xv || !out) throw Error(CWA_EINVAL, "null argument");
        *out = nullptr;
        auto* b = new cwa2d_batch{nullptr};
        try {
            b->impl = new Batch2D(*p, nscenes, scenes);
            b->impl->Reinit(xv, enabled, h0, h1);
        } catch (...) {
            delete b->impl;
            delete b;
            throw;
        }
        *out = b;
    });
}

int cwa2d_batch_destroy(cwa2d_batch* b) {
    return guarded2([&] {
        if (!b) return;
        delete b->impl;
        delete b;
    });
}

int cwa2d_batch_reinit(cwa2d_batch* b, const float* xv, const int32_t* enabled, const float* h0,
                       const float* h1) {
    return guarded2([&] { impl(b)->Reinit(xv, enabled, h0, h1); });
}

int cwa2d_batch_set_params(cwa2d_batch* b, const cwa2d_params* p) {
    return guarded2([&] {
        if (!p) throw Error(CWA_EINVAL, "null params");
        impl(b)->SetParams(*p);
    });
}

int cwa2d_batch_get_params(cwa2d_batch* b, cwa2d_params* p) {
    return guarded2([&] {
        if (!p) throw Error(CWA_EINVAL, "null params");
        *p = impl(b)->Params();
    });
}

int cwa2d_batch_step(cwa2d_batch* b, float dt, int32_t steps) {
    return guarded2([&] {
        if (!(dt > 0.0f) || !std::isfinite(dt) || steps < 0) throw Error(CWA_EINVAL, "dt > 0, steps >= 0");
        impl(b)->StepN(dt, steps);
    });
}

int cwa2d_batch_step_graph(cwa2d_batch* b, float dt, int32_t steps) {
    return guarded2([&] {
        if (!(dt > 0.0f) || !std::isfinite(dt) || steps < 0) throw Error(CWA_EINVAL, "dt > 0, steps >= 0");
        impl(b)->StepGraph(dt, steps);
    });
}

int cwa2d_batch_step_profiled(cwa2d_batch* b, float dt, cwa2d_kernel_times* t) {
    return guarded2([&] {
        if (!(dt > 0.0f) || !std::isfinite(dt)) throw Error(CWA_EINVAL, "dt > 0");
        impl(b)->StepProfiled(dt, t);
    });
}

int cwa2d_batch_sync(cwa2d_batch* b) {
    return guarded2([&] { impl(b)->Sync(); });
}

int cwa2d_batch_stream(cwa2d_batch* b, void** s) {
    return guarded2([&] {
        if (!s) throw Error(CWA_EINVAL, "null output");
        *s = (void*)impl(b)->stream();
    });
}

int cwa2d_batch_views(cwa2d_batch* b, cwa2d_views* v) {
    return guarded2([&] {
        if (!v) throw Error(CWA_EINVAL, "null output");
        impl(b)->Views(v);
    });
}

int cwa2d_batch_readback(cwa2d_batch* b, float* xv, float* rp, int32_t* enabled, float* h0,
                         float* h1) {
    return guarded2([&] { impl(b)->Readback(xv, rp, enabled, h0, h1); });
}

int cwa2d_batch_tune(cwa2d_batch* b, float dt, int32_t steps, cwa2d_tuning* best) {
    return guarded2([&] {
        if (!(dt > 0.0f) || !std::isfinite(dt)) throw Error(CWA_EINVAL, "dt > 0");
        const cwa2d_tuning t = impl(b)->Tune(dt, steps);
        if (best) *best = t;
    });
}

int cwa2d_batch_get_tuning(cwa2d_batch* b, cwa2d_tuning* t) {
    return guarded2([&] {
        if (!t) throw Error(CWA_EINVAL, "null output");
        *t = impl(b)->Tuning();
    });
}

int cwa2d_batch_set_tuning(cwa2d_batch* b, const cwa2d_tuning* t) {
    return guarded2([&] {
        if (!t) throw Error(CWA_EINVAL, "null tuning");
        impl(b)->SetTuning(*t);
    });
}

}  // extern "C"
