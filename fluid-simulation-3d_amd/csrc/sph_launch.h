// sph_launch.h -- host-callable launchers of the gfx950 kernels in
// sph_kernels.hip.  Every launcher enqueues on `stream` and returns the
// launch status; none of them synchronises or allocates.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sph_device.h"
#include "sph_generate.h"
#include "sph_types.h"

namespace sph {

// buckets per workgroup of the one-pass count scan: a chain status word and a
// ticket (one atomic on a single counter) per chunk
constexpr uint32_t kCountChunkBuckets = 4096;
// words of the fused update's grid barrier (counters on cache lines of their own)
constexpr uint32_t kFusedBarWords = 64 + 16 * 64;

struct DevState {
    // engine descriptors
    const EngineDesc *ed;
    const SceneDesc *sd;
    const uint32_t *scene_of;  // [n] scene of each slot (unused when single)
    bool multi;                // more than one scene
    bool grid;                 // cell-grid bucket key (SceneDesc::grid of every scene)
    // particle state in the resident order: slot k holds particle ids[k]
    // (the sorted order of the last update; any order gives the same results)
    float4 *pos;    // x,y,z, w = 0.34 after an update (OutPositions layout, cc:107)
    float4 *vel;    // x,y,z, w unused
    uint32_t *ids;  // particle index (engine-wide) of each resident slot
    // bucket sort: keys[0] bucket key and keys[1] ticket by resident slot
    // (recorded by the previous update's viscosity pass, or by predict);
    // order the (resident slot, particle index) pairs of each bucket in
    // ticket order
    uint32_t *keys[2];
    uint2 *order;
    uint32_t *count;   // [count_size = table_capacity + scene capacity] bucket counts, then
                       // scene flags: the next update's records, or zero
    uint32_t count_size;
    uint64_t *chain;   // [count_blocks + 1] chunk status words of the one-pass scan, then
                       // its chunk counter; zero between updates
    uint32_t count_blocks;
    // radix sort of the Morton work order
    uint32_t *hist;        // [radix * radix_blocks] counts, then [radix] digit totals
    uint32_t radix_blocks;
    // sorted order
    float4 *xps;   // predicted position, w = float(hash) (the reference record's .y)
    float4 *vs;    // velocity after stage A, sorted
    float4 *vs2;   // velocity after the pressure stage, sorted
    float4 *dens;  // rho, rho_near, RN(1/rho), RN(1/rho_near) (reciprocals 0 out of range)
    float4 *ps;    // position before the update, w = bits of the exact u32 hash
    uint32_t *sids;  // particle index of each sorted slot
    uint32_t *bounds;  // [table_total + 1] bucket b holds sorted slots [bounds[b], bounds[b+1])
    // work order of the gather kernels
    uint32_t *wkeys[2];  // Morton ordering keys (sort buffers)
    uint32_t *wvals[2];  // particle ids (sort buffers); the sorted ones are the work order
    const uint32_t *work;  // = wvals[result] of the last rebuild
    uint32_t *rank;      // [capacity] sorted slot of each particle id
    float4 *colors;      // [capacity] speed colours, particle order (null: not written)
    float4 *rpos;        // [capacity] render positions, particle order (null: not written)
    uint32_t *sflags;    // [scenes] grid key: 1 when a particle's cell lies outside the grid's box
                         // (copied from the count flags by the bucket sort)
    uint32_t *nbr;       // [capacity * nbr_words] neighbour rows by work index (nbr mode)
    uint32_t nbr_words;  // words per particle of nbr
    uint32_t *spare;     // at least nbr_words words that are written and never read
    uint32_t *ncnt;      // [capacity] neighbour count per row
    uint32_t *scan_err;  // [1] (host memory in an engine) raised when a bounded wait gave up (count scan, grid barrier)
    uint32_t *uneven;    // [2] nonzero: density found particles without a usable mask record in this update,
                         // in the last one (gather_index; null: not recorded)
    uint32_t *fbar;      // [kFusedBarWords] grid barrier of the fused update (zero between launches)
    uint32_t fused_grid[2]; // workgroups of the fused update (fast, IEEE) that the device holds resident at once
    uint32_t capacity;       // particle slots allocated
    uint32_t table_capacity; // bucket slots allocated
};

// Result-identical variants of a gather kernel (sph_kernels.hip explains them).
struct GatherVariant {
    bool work = false;  // Morton work order + XCD-contiguous workgroups
    bool list = false;  // two phases through a per-lane LDS list
    int block = 256;    // work-items per workgroup (64..256)
    bool rows = false;  // pressure / viscosity: read the density pass's neighbour rows
};

struct LaunchCfg {
    // defaults: the autotuner's usual picks on the benchmark scenes
    GatherVariant density{false, false, 64};
    GatherVariant pressure{true, true, 64};
    GatherVariant viscosity{false, false, 64};
    // nbr mode: density (in the work order) stores neighbour rows; pressure
    // and viscosity read them when their `rows` is set (then in the work order)
    bool nbr = false;
    // grid key, neighbour masks in all three gathers: a steady update (buckets
    // recorded) is one persistent launch with grid barriers between its
    // stages (launch_fused_update) instead of one launch per stage
    bool fused = false;
    // one work-item per particle at every size, also where the variants are the
    // defaults (whose form else follows the scene's size, coop_slots)
    bool pinned = false;
    // > 0: the gathers run with several work-items per particle, over a grid
    // of this many slots (follows_size, set per update by the engine)
    uint32_t coop_n = 0;
    // the bucket sort is one launch, and the density pass clears its counts
    // (with coop_n only; small_sort_ok, set per update by the engine)
    bool small_sort = false;
    // the mask kernels use IEEE roots and divisions (a scene is outside the fast
    // arithmetic's range; set per update by limit_launch_cfg)
    bool ieee = false;
    int block_stream = 256;  // threads per block of streaming kernels
    bool needs_work() const { return nbr || density.work || pressure.work || viscosity.work; }
};

// Defaults per bucket key.  Under the cell-grid key the sorted order is
// already spatially coherent: the kernels run in it (no Morton work order),
// and the row mode records neighbour masks instead of neighbour rows.
inline LaunchCfg sanitize_launch_cfg(LaunchCfg c, bool grid)
{
    if (grid)
        for (GatherVariant *v : {&c.density, &c.pressure, &c.viscosity}) v->work = false;
    return c;
}

inline LaunchCfg default_launch_cfg(bool grid)
{
    LaunchCfg c;
    if (grid) {
        // the autotuner's usual picks: neighbour masks for all three kernels
        c.density = GatherVariant{false, false, 256, true};
        c.pressure = GatherVariant{false, false, 256, true};
        // (viscosity with workgroups of 128 / 256, us: uniform 1,048,576 113 / 110,
        // 64 scenes 349 / 333, colliding 1,000,000 164 / 159.5: a workgroup's waves
        // share more of what the L1 holds; 512 loses on the colliding scene)
        c.viscosity = GatherVariant{false, false, 256, true};
        c.nbr = true;
    }
    return sanitize_launch_cfg(c, grid);
}

// The same variants (whatever pinned and coop_n say).
inline bool same_variants(const LaunchCfg &a, const LaunchCfg &b)
{
    auto same = [](const GatherVariant &x, const GatherVariant &y) {
        return x.work == y.work && x.list == y.list && x.block == y.block && x.rows == y.rows;
    };
    return same(a.density, b.density) && same(a.pressure, b.pressure) && same(a.viscosity, b.viscosity) &&
           a.nbr == b.nbr && a.fused == b.fused;
}

// The form of the gathers follows the scene's size.
inline bool follows_size(const LaunchCfg &c, bool grid)
{
    return !c.pinned && same_variants(c, default_launch_cfg(grid));
}

// The mask kernels and those with several work-items per particle take square
// roots and quotients by methods that are exact for every usual radius.  Where
// a scene lies outside that range (scene_fast), all of its layout's scenes run
// with IEEE operations instead: the mask kernels' own IEEE forms, or the walks,
// which know no others.
inline bool scene_fast(const SceneDesc &d) { return radius_fast(d.h) && d.thr >= 0x1p-60f; }

inline LaunchCfg limit_launch_cfg(LaunchCfg c, bool all_fast)
{
    if (!all_fast) {
        c.coop_n = 0;
        c.small_sort = false;
        c.ieee = true;
    }
    return c;
}

// Largest particle count for which the gathers run with several work-items per
// particle (sph_coop.hip).  Under the grid key one work-item per particle fills
// the chip above it, and tests each candidate cheaper.  Under the reference key
// density is cheaper so too, but only several work-items leave lists that
// pressure and viscosity can read instead of walking, at every size measured;
// the limit is the last of them, and where the reference's own float indices
// end.  us per steady update (all kernels; from 1,200,000 on the three gathers)
// with one / several work-items per particle:
//   grid key       1,000: 64 / 27   16,384: 77 / 34   65,536: 85 / 60
//                  131,072: 94 / 94   200,000: 115 / 127
//   reference key  4,000: 153 / 30   50,000: 195 / 64   200,000: 318 / 163
//                  1,200,000: 1,233 / 1,017   2,000,000: 2,001 / 1,660
//                  6,000,000: 6,662 / 5,202   16,700,000: 19,477 / 15,160
// Compressed fluid, whose lists overflow their rows or the LDS (mean of a run of
// 60 steps of two blocks colliding, and one state of 24 particles a cell):
//   grid key       70,000: 216 / 84   131,072: 356 / 147; 24 a cell 662 / 282
//   reference key  200,000: 668 / 351   1,000,000: 2,460 / 2,060; 24 a cell
//                  3,714 / 3,435 (at 40 a cell, five times the rest density, 5,688 /
//                  5,904)   4,000,000: 3,888 / 3,679
// Calm scenes near the line, one / several: dam break of 120,000 100 / 94, 124,000
// 145 / 99, 128,000 96 / 99, 131,072 97.5 / 100; 16 scenes 120,000 107 / 84,
// 124,000 113 / 93, 128,000 92 / 92; 64 scenes 128,000 107 / 90, 131,072 87 / 94:
// whole waves per scene favour one work-item, and round sizes have them.  Sparse
// fluid takes fewer tests, so its line lies lower: 4 particles a cell 127,000:
// 82 / 82, 2 a cell 100,000: 64 / 63, 1 a cell 80,000: 54 / 52, 127,000: 59 / 69.
constexpr uint32_t kCoopMaxGrid = 127000;
constexpr uint32_t kCoopMaxReference = 1u << 24;
// The same for the density pass of InitializeData under the reference key, which
// no pressure follows; us of sph_initialize with one / several work-items:
// 200,000: 198 / 165   700,000: 462 / 431   1,000,000: 684 / 729   2,500,000 (40 a
// cell): 2,294 / 4,777.
constexpr uint32_t kCoopMaxReferencePrime = 700000;

// Slots that the several-work-item gathers' grid covers for n particles in a
// layout of `capacity` slots, or 0 when the one-work-item forms run.
inline uint32_t coop_slots(bool grid, uint32_t n, uint32_t capacity)
{
    const uint32_t most = grid ? kCoopMaxGrid : kCoopMaxReference;
    return n > most ? 0u : (capacity < most ? capacity : most);
}

// Their form for n slots: work-items per particle, and what an entry of a
// neighbour list is: 16 a slot in 16 bits, -16 the low 16 of 17 bits, 32 a slot in
// 32 bits.  Up to kCoopWide slots a particle has 16 lanes,
// above 8: twice the particles per wave, fewer idle lanes in runs of 24 slots.
// us per steady update with 16 / 8 lanes: 1,000: 26.5 / 30.4, 8,000: 29.8 / 32.0,
// 16,384: 33.8 / 34.2, 32,768: 46.0 / 40.5, 131,072: 113.7 / 93.7.
constexpr uint32_t kCoopWide = 16384;
struct CoopForm {
    int lanes, entry;
};
inline CoopForm coop_form(bool grid, uint32_t n, uint32_t capacity)
{
    if (n <= kCoopWide && capacity <= 65536u) return CoopForm{16, 16};
    return CoopForm{8, capacity <= 65536u ? 16 : grid ? -16 : 32};
}

// Rows per strip of the grid key's bucket order, log2 (grid_row), for a scene
// of n particles.  A gather reads three planes around its own, and an XCD works
// on a window of some 40,000 slots (32 CUs of 16 to 24 waves).  Once planes hold
// more than about 24,000 slots (768 KiB of positions and velocities), window
// and neighbours no longer fit the XCD's 4 MiB L2 and every plane is fetched
// for each of its neighbours; in strips of eight rows they fit again, for two
// rows at a strip's edge that are fetched once more.  us of pressure + viscosity
// per update without strips / with 16 / 8 / 4 rows:
//   uniform 2,097,152 (21,000 slots a plane)       488 / 476 / 483 / -
//   two blocks 3,000,000 (26,000, 34,000 inside)   612 / - / 559 / -
//   two blocks 4,194,304 (32,000, 42,000 inside)   904 / 800 / 798 / 837
//   uniform 4,194,304 (33,000)                     1,193 / - / 1,047 / -
//   uniform 8,388,608 (52,000)                     2,474 / 2,277 / 2,219 / 2,490
//   two blocks 16,777,216 (82,000, 105,000 inside) 3,574 / 3,276 / 3,223 / 3,395
// (density gains nothing and loses up to 1%).  Scenes that the gathers with
// several work-items per particle may take have none: their fast walk counts on rows
// in plane order.
constexpr uint32_t kStripPlane = 24576, kStripShift = 3;
inline uint32_t grid_strips(uint32_t n, const uint32_t g[3])
{
    return n > kCoopMaxGrid && n / g[0] > kStripPlane && g[1] > (1u << kStripShift) ? kStripShift : kNoStrips;
}

// The one-launch bucket sort (k_small_sort) for one scene of n particles and
// `table` buckets.  Every workgroup reads all keys, so above some 20,000
// particles the three launches are faster.  us per steady update with three
// launches / with one: 1,000: 25.9 / 21.9, 4,000: 28.1 / 24.9, 10,000: 31.6 /
// 29.5, 16,384: 33.6 / 32.6, 24,000: 37.7 / 38.4, 50,000: 52.9 / 58.5.  The
// table's limit is what 16 workgroups' buckets in LDS cover.
constexpr uint32_t kSmallSortMax = 16384, kSmallSortTable = 65536;
inline bool small_sort_ok(bool multi, uint32_t n, uint32_t table)
{
    return !multi && n <= kSmallSortMax && table <= kSmallSortTable;
}

// Stage A + B1 when the previous update did not record the buckets: clears
// the counts, then predict, cell, hash, bucket key and ticket of every particle.
hipError_t launch_predict(const DevState &s, const LaunchCfg &c, hipStream_t st);
// The same for one scene in particle order (ids not read), counts at zero, its
// descriptors written to s.ed and s.sd by the kernel.
hipError_t launch_predict_first(const DevState &s, const EngineDesc &e, const SceneDesc &d, hipStream_t st);
// A steady update (buckets recorded by the previous one) as one launch of
// s.fused_grid[c.ieee] persistent workgroups: count scan, scatter, reorder, density,
// pressure, viscosity+integrate, separated by grid barriers.  Grid key with
// neighbour masks only (c.fused; see LaunchCfg).
hipError_t launch_fused_update(const DevState &s, const LaunchCfg &c, hipStream_t st);
// Workgroups of the fused update that fit on the device at once (its
// occupancy x compute units, a multiple of 8), or 0 when none does.
uint32_t fused_update_grid(bool multi, bool ieee, int device);
// Stages B2 + B3: counting sort into (bucket, particle index) order, bucket
// bounds, gather of xp, v into sorted order; clears the counts.
hipError_t launch_bucket_sort(const DevState &s, const LaunchCfg &c, hipStream_t st);
// Stable LSD radix sort of (keys, vals) over `bits` key bits (Morton work
// order); the input values are first_vals (null: the input slot indices).
// Returns the index (0/1) of the buffer pair holding the result.
hipError_t launch_radix_sort(const DevState &s, uint32_t *const keys[2], uint32_t *const vals[2],
                             const uint32_t *first_vals, uint32_t bits, hipStream_t st,
                             int *result_buf);
// Stage C, D, E+F.
hipError_t launch_density(const DevState &s, const LaunchCfg &c, hipStream_t st);
hipError_t launch_pressure(const DevState &s, const LaunchCfg &c, hipStream_t st);
hipError_t launch_viscosity_integrate(const DevState &s, const LaunchCfg &c, hipStream_t st);

// The same stages with several work-items per particle (sph_coop.hip), over the
// first n slots (n >= the live particles).
hipError_t launch_coop_density(const DevState &s, uint32_t n, bool clear_counts, hipStream_t st);
hipError_t launch_coop_pressure(const DevState &s, uint32_t n, hipStream_t st);
hipError_t launch_coop_viscosity_integrate(const DevState &s, uint32_t n, hipStream_t st);
// Its last stage writing the new state (and, unless null, the densities) in
// particle order only: no resident state, no buckets of a next update.
hipError_t launch_coop_viscosity_out(const DevState &s, uint32_t n, float4 *pos, float4 *vel, float2 *dens,
                                     hipStream_t st);

// Particles off .. off + n - 1 (one scene) into particle order: positions and
// velocities from the resident slots [off, off + n), densities (rho, rho_near)
// from the sorted ones; a null destination is left out.  corrupt[0] / [1] (unless
// null) are set to 1 when the particle index of a resident / sorted slot lies
// outside the scene; such a slot is not written.
hipError_t launch_download(const DevState &s, uint32_t off, uint32_t n, float4 *pos, float4 *vel, float2 *dens,
                           uint32_t *corrupt, hipStream_t st);
// Resident slots [off, off + n) of one scene (particles off .. off + n - 1)
// into particle order: dst_pos[i] / dst_vel[i] = state of particle off + i.
hipError_t launch_unpermute_state(const DevState &s, uint32_t off, uint32_t n, float4 *dst_pos,
                                  float4 *dst_vel, hipStream_t st);
// a[k] = first + k for k < n.
hipError_t launch_iota(uint32_t *a, uint32_t n, uint32_t first, hipStream_t st);
// scene_of of every slot of the first n_scenes scenes, from the device scene
// table (max_n: the largest scene's particle count)
hipError_t launch_scene_map(const SceneDesc *sd, uint32_t *scene_of, uint32_t n_scenes, uint32_t max_n,
                            hipStream_t st);
// a[k] = 0 for k < n, by a fill kernel (no memset node when captured).
hipError_t launch_clear_words(uint32_t *a, uint32_t n, hipStream_t st);
// Neighbour lists for parity checks (particle order, walk order, self included).
hipError_t launch_neighbour_count(const DevState &s, uint32_t *counts, hipStream_t st);
hipError_t launch_neighbour_fill(const DevState &s, const uint64_t *offs,
                                 uint32_t *list, hipStream_t st);
// Initial state of one scene from its plan (sph_generate.h), n = g.n slots
// starting at pos / vel.
hipError_t launch_generate(const GenPlan &g, float4 *pos, float4 *vel, hipStream_t st);
// Count of floats with bit patterns in [lo, hi] whose kernel reciprocal
// (recip_rn) differs from IEEE 1/x, and the smallest such pattern (atomic
// min into *first_bad, which the caller sets first).
hipError_t launch_recip_check(uint32_t lo, uint32_t hi, unsigned long long *bad,
                              uint32_t *first_bad, hipStream_t st);
// The same for the kernel square root (root_rn) and IEEE sqrt.
hipError_t launch_root_check(uint32_t lo, uint32_t hi, unsigned long long *bad,
                             uint32_t *first_bad, hipStream_t st);
// Plain copy of n float4 (HBM counter calibration).
hipError_t launch_copy(const float4 *src, float4 *dst, size_t n, hipStream_t st);
// Count of non-finite position/velocity components (error flag).
hipError_t launch_count_nonfinite(const DevState &s, uint32_t *counter, hipStream_t st);

}  // namespace sph
