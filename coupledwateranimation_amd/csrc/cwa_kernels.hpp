// cwa_kernels.hpp — launch wrappers of the coupled-step kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "cwa_device.hpp"

namespace cwa {

struct GridDesc {
    float gmin[3];
    float cell;    // x and z cell edge
    float cell_y;  // y cell edge
    int dims[3];
};

// One copy of the particle state (SoA, device).
struct ParticleArrays {
    float4* pos = nullptr;
    float4* vel = nullptr;
    float4* force = nullptr;
    int* id = nullptr;
};

size_t scan_workspace_ints(int n);
// Items that are counted, whose runs are still to be listed (n 0: none).
struct LinkRuns {
    const int* key;
    int n;
    int* head;
    int2* link;
};
// zero_out and zero_out2 (optional, n ints each) are cleared in the same pass;
// lr's runs are listed in it or beside it.
hipError_t launch_scan(const int* in, int* out, int n, int* ws, hipStream_t st,
                       int* zero_out = nullptr, int* zero_out2 = nullptr,
                       const LinkRuns& lr = LinkRuns{});
hipError_t launch_fill_i32(int* p, int n, int v, hipStream_t st);
// Zeroes offset[0..n] and a, b, c, d[0..n) (each may be null).
hipError_t launch_clear_cells(int* offset, int* a, int* b, int* c, int* d, int n,
                              hipStream_t st);
// Stable counting sort of keyed items: count (keys of particle positions, or
// given keys) with the cells' run lists, scan, reorder.
hipError_t launch_hash_count(const float4* pos, int n, const GridDesc& g, int* key,
                             const CellRuns& runs, hipStream_t st);
hipError_t launch_key_count(const int* key, int n, const CellRuns& runs, hipStream_t st);
hipError_t launch_link_runs(const int* key, int n, int* head, int2* link, hipStream_t st);
hipError_t launch_place_runs(const int* key, const int* offset, int* fill, int n, int2* runs,
                             hipStream_t st);
// Builds of up to this many particles list their runs in the pass that counts
// the keys, larger ones in a pass of their own: each run's push waits for its
// exchange, at the end of waves that hold the force pass's LDS.  A launch less
// pays where launches count (MI355X, step without the pass against with it,
// three scenes in flight: 4 096 particles 17.7 / 18.3 us, 65 536 25.9 /
// 27.2 us, 300 007 71.0 / 71.1 us, 1 048 576 285 / 276 us; the first step's
// hash pass at 1 048 576 particles 51 / 32 us).
constexpr int kFuseLinksMax = 1 << 18;
// Grid builds outside a scene, whose items come in any order, place their runs in
// the cells' segments (launch_place_runs) above these numbers of points and of
// (box, cell) pairs.  With a run per item, a list is one load from anywhere for
// every item of the cell; placed runs lie side by side (MI355X, listed ->
// placed, random points in 100^3, 50^3 and 25^3 cells: 700 000 points 117 -> 112,
// 126 -> 132, 241 -> 234 us, 1 000 000 158 -> 150, 200 -> 180, 472 -> 412, 2 000 000
// 339 -> 297, 632 -> 480, 2 751 -> 1 907; points nearly in order, 1 000 000: 57 -> 54,
// 73 -> 75, 144 -> 151.  Pairs of boxes: 540 000 144 -> 172, 2 160 000 554 -> 559,
// 3 240 000 1 059 -> 1 011, 5 400 000 3 143 -> 2 746).
constexpr int kListRunsMax = 3 << 18;
constexpr int kListPairsMax = 1 << 21;
// list[d] = item_of ? item_of[s] : s at each item's stable destination d;
// head null: link holds the runs placed in the cells' segments.  With pos_out
// set, pos_out[d] = pos_in[s] and id_out[d] = id_in[s], and with
// packed_out set also (Pd: the device parameters) packed_out[d] =
// pack_point(pos_in[s]).
hipError_t launch_stable_reorder(const int* key, const int* offset, const int* head,
                                 const int2* link, int n, const int* item_of, int* list,
                                 const float4* pos_in, const int* id_in, float4* pos_out,
                                 int* id_out, hipStream_t st, const DevParams* Pd = nullptr,
                                 uint32_t* packed_out = nullptr);
// Boxes: cells covered per box (ncov, n ints), then the (box, cell) pairs at
// first[i] = exclusive scan of ncov (pkey: cell, pbox: box index).
hipError_t launch_box_cover(const float4* x, const float4* hw, int n, const float gmin[3],
                            const float cell[3], const int dims[3], int* ncov, hipStream_t st);
// *out = sum of a[0..n) in 64 bits (non-negative values).
hipError_t launch_sum_i64(const int* a, int n, unsigned long long* out, hipStream_t st);
hipError_t launch_box_pairs(const float4* x, const float4* hw, int n, const float gmin[3],
                            const float cell[3], const int dims[3], const int* first,
                            int* pkey, int* pbox, hipStream_t st);
// The density pass: sorted positions bpos, the state's velocities read in
// their pre-sort slots state_vel[list[i]].  nbw (nb_buffer_uint2(n) uint2:
// neighbour words and counts) and nrec (2*n float4: position and pressure,
// velocity and 1/rho) and vpad (the velocity's fourth component, carried
// through the step) are written for the force pass.  pw (pressure, 1/rho),
// rho_raw (density before the wave term and the rest-density clamp) and
// vel_out (the sorted velocities) are optional outputs for the adjoint tape
// (null: not written).  packed: the packed points of bpos[0..n) followed by
// kPackPad readable words for the one-lane pass, null for the four-lane pass.
// Scenes of up to this many particles run the density pass (and a tape's
// pair adjoint, and up to kForceSplitMax the force pass) with four lanes per
// particle, larger ones with one lane; read at each launch and at tape
// creation.  Default kLaneSplitDefault.
constexpr long long kLaneSplitDefault = 1 << 18;
long long lane_split_limit();
long long set_lane_split_limit(long long max_n);  // returns the previous limit

hipError_t launch_density(const DevParams& P, const float4* bpos, const float4* state_vel,
                          const int* list, const int* offset, int n, const float* H0,
                          float* rho_w, float2* pw, float* flux, uint2* nbw, float4* nrec,
                          float* rho_raw, float4* vel_out, float* vpad, const uint32_t* packed,
                          hipStream_t st);
// Where the force pass hashes the next step's grid, or key == null for no
// fused hash.
struct NextKeys {
    int* key;
    CellRuns runs;
};
// The heightfield's EVOLVE as blocks of the force launch: nblk tiles of
// side x side texels, nx a row (nblk 0: none, the wave takes its own launch).
struct WaveTiles {
    const float* h0;
    const float* h1;
    float* out;
    int nblk, nx, side;
};
constexpr int kWaveTileColumns = 128;  // columns a tile's samples may touch when it is chosen
constexpr int kFuseWaveParticles = 1 << 16;
constexpr int kFuseWaveTiles = 512;
static_assert(kFuseWaveParticles <= kFuseLinksMax, "tiles go with the fused run lists");
// n particles; flux: the step couples (the tiles sum the columns they sample).
WaveTiles wave_tiles_for(const DevParams& P, int n, bool flux, const float* h0, const float* h1,
                         float* out);
// Scenes of up to this many particles (and lane_split_limit()) run the force
// pass with four lanes per particle (k_force_split gives both sides' times).
constexpr int kForceSplitMax = 1 << 15;
static_assert(kForceSplitMax <= kFuseLinksMax, "the split force pass lists its runs");
// Forces + integration: own record from nrec, id from bid and the velocity
// pad from vpad (sorted), previous force from the state S in its pre-sort
// slot list[i]; writes the next state N in sorted order.  The launch also
// sums the column flux (colflux set) and advances the heightfield (wt).  fpre (force before
// the foam branch) is an optional output for the adjoint tape.
hipError_t launch_force_integrate(const DevParams& P, float dt, const float4* bpos,
                                  const int* bid, const ParticleArrays& S, const int* list,
                                  const int* offset, int n, const float* rho_w, const uint2* nbw,
                                  const float4* nrec, const float* H0, ParticleArrays& N,
                                  float* rho, float* prs, float4* fpre, const float* flux,
                                  float* colflux, const float* vpad, const NextKeys& next,
                                  const WaveTiles& wt, hipStream_t st);
// Neighbour counts (self included) of the last density pass, per sorted slot.
hipError_t launch_neighbour_counts(const DevParams& P, const float4* pos, const int* offset,
                                   const uint2* nbw, int n, int* out, hipStream_t st);
hipError_t launch_wave(const DevParams& P, const float* h0, const float* h1, float* out,
                       const float* colflux, float dt, hipStream_t st);
hipError_t launch_init_wave(float* out, int W, int H, float type, hipStream_t st);
hipError_t launch_check_finite(const float* a, size_t n, int* flag, hipStream_t st);

}  // namespace cwa
