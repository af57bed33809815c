// sph_coop.hip -- the gather stages with G = 16 or 8 work-items per particle,
// for scenes too small to fill the chip with one work-item per particle, and
// for the reference key.
//
// One work-item per particle makes 16,384 particles 256 waves on 1,024 SIMDs,
// each a serial chain of some 240 candidate tests and 35 to 50 pair bodies: the
// stages take that chain's latency (density 36, pressure 21, viscosity 13 us)
// whatever the size below about 100,000 particles.  Here a group of G lanes
// takes a particle, and at 16,384 particles they take 8.4, 6.1 and 7.2 us:
//   - the candidates of a neighbour row are tested G at a time, in slot order
//     (one coalesced load per group), and the passing ones go to a list in LDS
//     at the place a ballot gives them, so the list has walk order;
//   - the pair terms of the list's entries are computed G at a time and put in
//     LDS, and one lane per component adds them up in list order.
// What bounds them then is the chain of dependent loads (bounds, records,
// neighbours), each a few hundred ns, and from about 30,000 particles on the
// vector issue of the tests (a list entry costs about 30 instructions per
// candidate where one work-item per particle spends 11).
// The sums therefore add the same terms in the same order as the one-work-item
// form, and the results agree with it to the bit; entries past the list's end
// add +0, which leaves a sum that began at +0 as it is.
//
// The density stage also writes each particle's list (its own slot among it) to
// the neighbour-row buffer, and the pressure and viscosity stages take it from
// there; a wave with a particle of more neighbours than a row holds walks again.
//
// Reference: Allkams/Fluid-Simulation-3D, engine/physics/physicsWorld.cc:304-464
// (stages C, D, E), cc:80-108 (stage F).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sph_kernel_common.h"

namespace sph {

namespace {

constexpr int kCoopBlock = 256;  // work-items per workgroup
constexpr uint32_t kList = 96;   // list entries per particle held in LDS

// Mean particles of the cells that one lane looks up (of a row's three, under
// the grid key) from which the wave's lists are expected to overflow: a 1 / 6.4 of the
// candidates pass, and 27 cells of 24 then give kList entries.
constexpr uint32_t kCrowded = 24;

// Eight lanes, grid key: where no row of the wave's particles holds more slots
// than this, two loads of eight a row instead of four (and a third where it
// holds more than 16).  us per update, four / two: 127,000 particles at 4 a cell
// 88 / 82, at 1 a cell 77 / 69; 40,000 at 1 a cell 38 / 35; unchanged at 8 a cell.
constexpr uint32_t kSparse = 22;

// G lanes per particle.
template <uint32_t G>
struct Group {
    static constexpr uint32_t kParticles = kCoopBlock / G;  // per workgroup
    static constexpr uint32_t kChunk = 3 * G;               // entries whose pair terms are held at once
};

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// Lane L of the own group's value, in all its lanes: a DPP broadcast where the
// group is a DPP row, else through the LDS crossbar.
template <uint32_t G, int L>
__device__ __forceinline__ uint32_t group_bcast(uint32_t x)
{
    static_assert(L < (int)G, "lane of the group");
#if __HIP_DEVICE_COMPILE__
    if constexpr (G == 16) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + L, 0xf, 0xf, false);
    else return (uint32_t)__builtin_amdgcn_ds_bpermute((int)((threadIdx.x & 63u & ~(G - 1u)) * 4u) + 4 * L, (int)x);
#else
    return x;
#endif
}

template <uint32_t G, int L>
__device__ __forceinline__ float group_bcast(float x)
{
    return __uint_as_float(group_bcast<G, L>(__float_as_uint(x)));
}

// Orders the wave's LDS writes before its later LDS reads (one wave runs its
// LDS operations in order; this keeps the compiler to that order).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ bool wave_any(bool x) { return __ballot(x) != 0; }

// The slot that a group handles: workgroups are numbered so that each XCD
// takes one contiguous run of the live slots (as the one-work-item stages do).
template <uint32_t G>
__device__ __forceinline__ uint32_t coop_slot(uint32_t n)
{
    constexpr uint32_t N = Group<G>::kParticles;
    const uint32_t live = (n + N - 1) / N;
    const uint32_t per = (live + 7u) >> 3, x = blockIdx.x & 7u, j = blockIdx.x >> 3;
    const uint32_t lb = j < per ? x * per + j : live + j;
    return lb * N + threadIdx.x / G;
}

// MULTI: the slot, opaque to the optimiser at each pass of run_scene's loop, so
// that the addresses derived from it are formed where used, not hoisted out of
// the loop and kept in registers.
template <bool MULTI>
__device__ __forceinline__ uint32_t opaque_slot(uint32_t k)
{
#if __HIP_DEVICE_COMPILE__
    if (MULTI) asm volatile("" : "+v"(k));
#endif
    return k;
}

// The walk of the neighbour cells (cc:331-363) by a group: every candidate of
// the 27 cells in the reference's order, ascending slot within a cell, tested
// with the one-work-item walk's expressions.  put(at, m, d2): slot m goes to
// entry `at` of the group's list; entry kList is where everything else goes.
// flush(cnt) consumes the lists (cnt entries of the own group's) when one could
// overflow, and at the end.
//
// No branch in here depends on a lane: a candidate that fails is written to the
// entry that nobody reads.  (With `if (pass) put(...)` before and inside a loop
// whose condition is a ballot, the compiler merges the two stores and sends
// the lanes that do not store around the loop by themselves, so its ballots
// miss the others.)
//
// FAST: first an unrolled walk, its loads in flight together, for the common
// case (no float-hash test needed under the grid key, no list overflow).  Where a
// list overflows in it or is expected to (kCrowded), and first where !FAST,
// batches of runs go in a loop that flushes the lists on the way: a third of the
// general walk's time for them (131,072 particles at 24 a cell: 619 -> 282 us an
// update; 1,000,000 under the reference key 4,739 -> 3,435, where one work-item
// per particle takes 3,714).  The
// general walk takes one chunk of G slots of one bucket at a time: for what is
// left where one batch alone overflows, and under the grid key for waves that
// need the float-hash test.
template <uint32_t G, bool GRID, bool FAST, typename Put, typename Flush>
__device__ __forceinline__ void coop_walk(const SceneDesc &S, const float4 *__restrict__ xps,
                                          const uint32_t *__restrict__ bounds, uint32_t k, const float4 &pi,
                                          bool clean, Put &&put_at, Flush &&flush)
{
    const uint32_t lane = threadIdx.x & 63u, gl = lane & (G - 1u);
    const uint32_t below = (1u << gl) - 1u;  // the group's lanes below this one
    const float thr = S.thr;
    uint32_t cnt = 0;  // entries of the group's list
    bool done = false;
    auto put = [&](bool pass, uint32_t p, uint32_t m, float d2) __attribute__((always_inline)) {
        put_at(pass ? min(p, kList) : kList, m, d2);
    };
    auto near = [&](float x, float y, float z, float &d2) __attribute__((always_inline)) {
        const float ox = x - pi.x, oy = y - pi.y, oz = z - pi.z;
        d2 = ox * ox + oy * oy + oz * oz;  // glm::dot order
        return d2 < thr;
    };
    // one candidate per lane
    auto test = [&](const float4 &r, uint32_t m, bool in) __attribute__((always_inline)) {
        float d2;
        const bool pass = near(r.x, r.y, r.z, d2) & in;
        const uint64_t b = __ballot(pass);
        const uint32_t half = (lane & 32u) ? (uint32_t)(b >> 32) : (uint32_t)b;
        const uint32_t mine = (half >> (lane & (32u - G))) & ((1u << G) - 1u);
        put(pass, cnt + (uint32_t)__popc(mine & below), m, d2);
        cnt += (uint32_t)__popc(mine);
    };
    const int cx = cell_coord(pi.x, S.h), cy = cell_coord(pi.y, S.h), cz = cell_coord(pi.z, S.h);
    const uint32_t h0 = hash_cell(cx, cy, cz);
    auto cell_hash = [&](uint32_t o) {  // of the o-th cell in the reference's order
        return h0 + (o / 9u - 1u) * 15823u + ((o / 3u) % 3u - 1u) * 9737333u + (o % 3u - 1u) * 440817757u;
    };
    auto half_of = [&](uint64_t b) { return (lane & 32u) ? (uint32_t)(b >> 32) : (uint32_t)b; };
    // The candidates of N runs [b, e) of slots, in order: a run's first COVER
    // slots by COVER / G loads, the loads of all N runs in flight together;
    // the run's passing bits form one word per group, in slot order.  HASH: a
    // record's float hash (w) must equal the run's.
    auto runs = [&](auto nr, auto cover, auto hash, const uint32_t *b, const uint32_t *e, auto &&hash_of)
        __attribute__((always_inline)) {
        constexpr int N = decltype(nr)::value, NP = decltype(cover)::value / (int)G;
        constexpr bool HASH = decltype(hash)::value;
        constexpr uint32_t COVER = decltype(cover)::value;
        static_assert(NP == 1 || NP == 2 || NP == 4, "parts");
        // v_perm selectors: the group's bits of each part's ballot half
        const uint32_t q8 = (lane >> 3) & 3u;
        const uint32_t sel0 = G == 16 ? ((lane & 16u) ? 0x07060302u : 0x05040100u) : 0x0c0c0400u + q8 * 0x0101u;
        const uint32_t sel1 = 0x04000c0cu + q8 * 0x01010000u;
        float4 rec[N][NP];
#pragma unroll
        for (int q = 0; q < N; ++q)
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                const uint32_t m = b[q] + G * c + gl;
                const float4 *at = xps + (m < e[q] ? m : k);
                if (HASH) {
                    rec[q][c] = *at;
                } else {
                    const float3 t = *reinterpret_cast<const float3 *>(at);
                    rec[q][c] = make_float4(t.x, t.y, t.z, 0.0f);
                }
            }
        static_for<N>([&](auto Q) __attribute__((always_inline)) {
            constexpr int q = decltype(Q)::value;
            const float f = HASH ? hash_of(Q) : 0.0f;
            bool pass[NP];
            float d2[NP];
            uint32_t w[NP];
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                pass[c] = near(rec[q][c].x, rec[q][c].y, rec[q][c].z, d2[c]) & (b[q] + G * c + gl < e[q]) &
                          (!HASH | (rec[q][c].w == f));
                w[c] = half_of(__ballot(pass[c]));
            }
            uint32_t bits;
            if constexpr (NP == 1) bits = (w[0] >> (lane & (32u - G))) & ((1u << G) - 1u);
            else bits = __builtin_amdgcn_perm(w[1], w[0], sel0);
            if constexpr (NP == 4) bits |= __builtin_amdgcn_perm(w[3], w[2], sel1);
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                const uint32_t under = (below << (G * c)) | ((1u << (G * c)) - 1u);  // candidates before this lane's
                put(pass[c], cnt + (uint32_t)__popc(bits & under), b[q] + G * c + gl, d2[c]);
            }
            cnt += (uint32_t)__popc(bits);
            for (uint32_t m0 = b[q] + COVER; wave_any(m0 < e[q]); m0 += G) {
                const bool in = m0 + gl < e[q];
                const float4 r = xps[in ? m0 + gl : k];
                test(r, m0 + gl, in & (!HASH | (r.w == f)));
            }
        });
    };
    // grid key, plain: the wave's particles' 27 cells lie inside the grid without
    // wrapping and no particle's cell lies outside it, so every record of a row's
    // run belongs to the row (walk_grid); base: the bucket of the particle's cell
    bool plain = true;
    uint32_t base = 0;
    const uint32_t gy = S.gdim[1], gz = S.gdim[2];
    if constexpr (GRID) {
        const uint32_t ux = (uint32_t)cx - (uint32_t)S.cell_lo[0];
        const uint32_t uy = (uint32_t)cy - (uint32_t)S.cell_lo[1];
        const uint32_t uz = (uint32_t)cz - (uint32_t)S.cell_lo[2];
        auto inside = [](uint32_t u, uint32_t g) { return u < g && u - 1u < g && u + 1u < g; };
        const bool interior = inside(ux, S.gdim[0]) && inside(uy, gy) && inside(uz, gz);
        plain = !wave_any(!(clean && interior));
        base = S.key_off + (ux * gy + uy) * gz + uz;
    }
    if constexpr (FAST && GRID) {
        if (plain) {
            // the lanes fetch the bounds of the group's nine runs together
            // (G = 8: the ninth by all)
            const uint32_t row = min(gl, 8u);
            const uint32_t mine = base + ((row / 3u - 1u) * gy + (row % 3u - 1u)) * gz;
            const uint32_t rb = bounds[mine - 1u], re = bounds[mine + 2u];
            uint32_t b8 = 0, e8 = 0;
            if constexpr (G == 8) {
                b8 = bounds[base + (gy + 1u) * gz - 1u];
                e8 = bounds[base + (gy + 1u) * gz + 2u];
            }
            auto rows = [&](auto cover) __attribute__((always_inline)) {
                constexpr int kRows = 3;  // runs in flight together (nine: 122 registers, 0.4 us more at 16,384)
                static_for<9 / kRows>([&](auto Q) __attribute__((always_inline)) {
                    uint32_t b[kRows], e[kRows];
                    static_for<kRows>([&](auto R) __attribute__((always_inline)) {
                        constexpr int q = decltype(R)::value, r = decltype(Q)::value * kRows + q;
                        if constexpr (r < (int)G) {
                            b[q] = group_bcast<G, r>(rb);
                            e[q] = group_bcast<G, r>(re);
                        } else {
                            b[q] = b8;
                            e[q] = e8;
                        }
                    });
                    runs(std::integral_constant<int, kRows>{}, cover, std::false_type{}, b, e,
                         [](auto) { return 0.0f; });
                });
                done = !wave_any(cnt > kList);
            };
            if (G == 8 && !wave_any(re - rb > kSparse)) rows(std::integral_constant<int, 16>{});
            else if (!wave_any(re - rb > 3u * kCrowded)) rows(std::integral_constant<int, 32>{});
        }
    }
    if constexpr (FAST && !GRID) {
        // The lanes fetch the buckets of cells gl, gl + G, ... together.  Cells in
        // flight together: with nine of them eight lanes a particle need 128
        // registers and spill, 95 us on 200,003 particles, with three 72 registers
        // and 75 us (one: 91).  Sixteen lanes hold nine in 80 registers: 7.8 us on
        // 3,000 particles, 8.5 with three.
        constexpr int kFetch = (27 + G - 1) / G, kCells = G == 16 ? 9 : 3;
        uint32_t fb[kFetch], fe[kFetch], all = 0;
#pragma unroll
        for (int c = 0; c < kFetch; ++c) {
            const uint32_t o = min(gl + G * c, 26u);
            const uint32_t key = S.key_off + fastmod(cell_hash(o), S.mod_m, S.table);
            fb[c] = bounds[key];
            fe[c] = bounds[key + 1u];
            all += fe[c] - fb[c];
        }
        if (!wave_any(all > (uint32_t)kFetch * kCrowded)) {
            static_for<27 / kCells>([&](auto H) __attribute__((always_inline)) {
                uint32_t b[kCells], e[kCells];
                static_for<kCells>([&](auto P) __attribute__((always_inline)) {
                    constexpr int q = decltype(P)::value, A = decltype(H)::value * kCells + q;
                    b[q] = group_bcast<G, A % G>(fb[A / G]);
                    e[q] = group_bcast<G, A % G>(fe[A / G]);
                });
                runs(std::integral_constant<int, kCells>{}, std::integral_constant<int, 16>{}, std::true_type{}, b, e,
                     [&](auto P) { return (float)cell_hash((uint32_t)(decltype(H)::value * kCells + decltype(P)::value)); });
            });
            done = !wave_any(cnt > kList);
        }
    }
    if (!done) cnt = 0;
    // The rest: cell o is the next one.  In batches: a row of cells at a time
    // under the grid key, else three cells (12 to 24 registers of records; three
    // rows leave fewer waves).  Then the general walk of bucket o, its slots from
    // m0 on (each bucket by itself, so the grid's wrap seam needs no case of its
    // own).
    constexpr uint32_t kRuns = GRID ? 1 : 3, kRun = GRID ? 3 : 1;  // runs, cells of a run
    static_assert(27 % (kRuns * kRun) == 0, "whole batches");
    bool batches = plain;
    uint32_t o = 0, m0 = 0, e = 0;
    float f = 0.0f;
    auto bucket = [&]() {
        const uint32_t dx = o / 9u - 1u, dy = (o / 3u) % 3u - 1u, dz = o % 3u - 1u;
        uint32_t key;
        if constexpr (GRID)
            key = S.key_off + grid_key(cx + (int)dx, cy + (int)dy, cz + (int)dz, S.cell_lo, S.gdim, S.gmod, S.strip_shift);
        else
            key = S.key_off + fastmod(cell_hash(o), S.mod_m, S.table);
        m0 = bounds[key];
        e = bounds[key + 1u];
        f = (float)cell_hash(o);
    };
    if (!done && !batches) bucket();
#pragma unroll 1
    for (;;) {
        bool full = done;
        if (!done && batches) {
            uint32_t rb[kRuns], re[kRuns];
#pragma unroll
            for (uint32_t q = 0; q < kRuns; ++q) {
                const uint32_t c = o + q * kRun;
                if constexpr (GRID) {
                    const uint32_t mid = base + ((c / 9u - 1u) * gy + ((c / 3u) % 3u - 1u)) * gz;
                    rb[q] = bounds[mid - 1u];
                    re[q] = bounds[mid + 2u];
                } else {
                    const uint32_t key = S.key_off + fastmod(cell_hash(c), S.mod_m, S.table);
                    rb[q] = bounds[key];
                    re[q] = bounds[key + 1u];
                }
            }
            const uint32_t before = cnt;
            runs(std::integral_constant<int, kRuns>{}, std::integral_constant<int, GRID ? 32 : 16>{},
                 std::integral_constant<bool, !GRID>{}, rb, re,
                 [&](auto P) { return (float)cell_hash(o + (uint32_t)decltype(P)::value); });
            if (!wave_any(cnt > kList)) {
                o += kRuns * kRun;
                full = done = o == 27u;
            } else {  // a list is full: what it held before, then this batch again
                cnt = before;
                full = wave_any(cnt != 0u);
                if (!full) {  // (one batch alone fills it)
                    batches = false;
                    bucket();
                }
            }
        } else if (!done) {
            full = wave_any(cnt + G > kList);
        }
        if (full) {
            flush(cnt);
            cnt = 0;
        }
        if (done) break;
        if (batches) continue;
        const uint32_t m = m0 + gl;
        const bool in = m < e;
        const float4 r = xps[in ? m : k];
        test(r, m, in & (r.w == f));
        m0 += G;
        if (!wave_any(m0 < e)) {
            if (++o == 27u) done = true;
            else bucket();
        }
    }
}

// acc + plane[0] + plane[1] + ..., in order: the first m entries, rounded up to
// a multiple of 4 (entries past the list's end hold +0).
__device__ __forceinline__ float ordered_sum(float acc, const float *plane, uint32_t m)
{
    for (uint32_t q = 0; wave_any(q < m); q += 4u) {
        const float4 t = *reinterpret_cast<const float4 *>(plane + q);
        acc += t.x;
        acc += t.y;
        acc += t.z;
        acc += t.w;
    }
    return acc;
}

// Rows of the neighbour lists: entry t of slot k at [k * cap + t].  uint16_t:
// slots, while every slot fits.  int16_t: the low 16 bits of slots below 131,072
// (grid key).  The walk meets slots in ascending order, but for cells that wrap
// around the grid, so a list's first `split` entries are those below 65,536; the
// split lies beside the count, and a list that is not so counts as too long for
// its row.  uint32_t: slots.  In 16 bits a row holds twice as many (70,000
// colliding particles, mean of 60 steps: 128 us an update with rows of 64, 84 of
// 128, and the walk in batches).
template <typename T>
struct Rows {
    static constexpr bool kSplit = std::is_signed<T>::value;
    T *rows, *spare;  // spare: a row that nobody reads
    uint32_t cap;
    __device__ __forceinline__ uint32_t get(uint32_t k, uint32_t t, uint32_t split) const
    {
        const T e = rows[(size_t)k * cap + t];
        return kSplit ? (uint32_t)(uint16_t)e + (t < split ? 0u : 65536u) : (uint32_t)e;
    }
};
static_assert(kCoopMaxGrid <= 131072u, "17 bits of slots");

struct CoopArgs {
    const EngineDesc *ed;
    const SceneDesc *sd;
    const uint32_t *scene_of;
    const uint32_t *sids;
    const float4 *xps;
    const uint32_t *bounds;
    const uint32_t *sflags;
    uint32_t *ncnt;
    uint32_t *clear;  // counts to clear for the next update (table_total + n_scenes), or null
};

template <uint32_t G, bool MULTI, bool GRID, typename T>
__global__ __launch_bounds__(kCoopBlock, 5) void k_coop_density(const CoopArgs A, const Rows<T> out,
                                                                float4 *__restrict__ dens)
{
    constexpr uint32_t kChunk = Group<G>::kChunk;
    __shared__ uint2 lists[Group<G>::kParticles][kList + 1];                // (slot, d2)
    __shared__ __align__(16) float terms[Group<G>::kParticles][2][kChunk];  // the two sums' terms
    const uint32_t n = A.ed->n_total, slot = coop_slot<G>(n);
    if (A.clear) {
        const uint32_t nc = A.ed->table_total + A.ed->n_scenes;
        for (uint32_t i = blockIdx.x * kCoopBlock + threadIdx.x; i < nc; i += gridDim.x * kCoopBlock) A.clear[i] = 0u;
    }
    if (slot >= n) return;
    const uint32_t gl = threadIdx.x & (G - 1u), gq = threadIdx.x / G;
    uint2 *const lst = lists[gq];
    float *const t0p = terms[gq][0], *const t1p = terms[gq][1];
    const float4 pi = A.xps[slot];
    auto scene = [&](const SceneDesc &S) __attribute__((always_inline)) {
        const uint32_t k = opaque_slot<MULTI>(slot);
        const bool clean = GRID && A.sflags[S.index] == 0u;
        const float h = S.h, w2c = S.w2c, w3c = S.w3c;
        float acc = 0.0f;    // lane 0: rho, lane 1: near rho
        uint32_t total = 0;  // neighbours flushed so far
        uint32_t split = 0;  // neighbours below slot 65,536
        bool mixed = false;  // one of them after a slot past it
        auto flush = [&](uint32_t cnt) {
            wave_sync();
            for (uint32_t c0 = 0; wave_any(c0 < cnt); c0 += kChunk) {
#pragma unroll
                for (uint32_t r = 0; r < kChunk; r += G) {
                    if (!wave_any(c0 + r < cnt)) break;
                    const uint32_t t = c0 + r + gl;
                    const bool have = t < cnt;
                    // a lane without an entry repeats entry 0 (its row entry
                    // too; an empty list's goes to the spare row)
                    const uint32_t at = have ? t : 0u;
                    const uint2 e = lst[at];
                    float a, b;
                    density_pair<true>(h, w2c, w3c, __uint_as_float(e.y), true, a, b);
                    t0p[r + gl] = have ? a : 0.0f;
                    t1p[r + gl] = have ? b : 0.0f;
                    T *const row = cnt ? out.rows + (size_t)k * out.cap : out.spare;
                    row[min(total + at, out.cap - 1u)] = (T)e.x;
                    if constexpr (Rows<T>::kSplit) {
                        const uint32_t lane = threadIdx.x & 63u;
                        const uint64_t b = __ballot(have & (e.x < 65536u));
                        const uint32_t half = (lane & 32u) ? (uint32_t)(b >> 32) : (uint32_t)b;
                        const uint32_t low = (half >> (lane & (32u - G))) & ((1u << G) - 1u);
                        mixed |= low != 0u && (split != total + c0 + r || (low & (low + 1u)) != 0u);
                        split += (uint32_t)__popc(low);
                    }
                }
                wave_sync();
                acc = ordered_sum(acc, gl == 0u ? t0p : t1p, cnt > c0 ? min(kChunk, cnt - c0) : 0u);
                wave_sync();
            }
            total += cnt;
        };
        coop_walk<G, GRID, true>(
            S, A.xps, A.bounds, k, pi, clean,
            [&](uint32_t at, uint32_t m, float d2) { lst[at] = make_uint2(m, __float_as_uint(d2)); }, flush);
        if constexpr (Rows<T>::kSplit) total = mixed || total > out.cap ? out.cap + 1u : total | split << 16;
        const float rho = group_bcast<G, 0>(acc), rhon = group_bcast<G, 1>(acc);
        if (gl == 0u) {
            A.ncnt[k] = total;
            dens[k] = make_float4(rho, rhon, reciprocal_or_zero(rho), reciprocal_or_zero(rhon));
        }
    };
    run_scene<MULTI>(A.sd, A.scene_of, slot, scene);
}

// The sum over a particle's neighbours of NT three-component terms each (added
// one after the other), from its row, or by walking again where the row does
// not hold them all.  pair(m, d2, ox, oy, oz, aux, out): the 3 * NT terms of
// neighbour m, component fastest.  Lane c < 3 of the group returns component c.
template <uint32_t G, bool GRID, int NT, typename T, typename Pair>
__device__ __forceinline__ float coop_sum(const CoopArgs &A, const SceneDesc &S, const Rows<T> &in,
                                          const float4 *__restrict__ aux, uint32_t k, const float4 &pi, bool clean,
                                          uint32_t *lst, float *planes, Pair &&pair)
{
    constexpr uint32_t kChunk = Group<G>::kChunk;
    constexpr uint32_t kPlane = kChunk * NT;  // floats per component: entry t's terms at [NT t, NT t + NT)
    const uint32_t gl = threadIdx.x & (G - 1u);
    const float *const mine = planes + min(gl, 2u) * kPlane;
    float acc = 0.0f;
    const uint32_t found = A.ncnt[k], split = found >> 16, total = Rows<T>::kSplit ? found & 0xffffu : found;
    // (the two ways share nothing: most waves take the first, which then needs
    // neither the cell nor the registers of the walk)
    auto take = [&](auto from_rows, uint32_t cnt) __attribute__((always_inline)) {
        wave_sync();
#pragma unroll 1
        for (uint32_t c0 = 0; wave_any(c0 < cnt); c0 += kChunk) {
            constexpr uint32_t R = kChunk / G;
            uint32_t m[R];
            float4 x[R], a[R];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t t = c0 + r * G + gl, at = t < cnt ? t : 0u;
                const uint32_t e = decltype(from_rows)::value ? in.get(k, at, split) : lst[at];
                m[r] = t < cnt ? e : k;
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                x[r] = A.xps[m[r]];
                a[r] = aux[m[r]];
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                if (!wave_any(c0 + r * G < cnt)) break;
                float out[3 * NT];
                const float ox = x[r].x - pi.x, oy = x[r].y - pi.y, oz = x[r].z - pi.z;
                const bool have = m[r] != k;  // not the particle itself, nor past the end
                // (at distance 0 the terms would take their slow path)
                pair(have ? ox * ox + oy * oy + oz * oz : 0.25f * S.thr, ox, oy, oz, a[r], out);
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int q = 0; q < NT; ++q)
                        planes[c * kPlane + (r * G + gl) * NT + q] = have ? out[3 * q + c] : 0.0f;
            }
            wave_sync();
            acc = ordered_sum(acc, mine, cnt > c0 ? NT * min(kChunk, cnt - c0) : 0u);
            wave_sync();
        }
    };
    if (!wave_any(total > in.cap)) take(std::true_type{}, total);
    else
        coop_walk<G, GRID, false>(S, A.xps, A.bounds, k, pi, clean,
                                  [&](uint32_t at, uint32_t m, float) { lst[at] = m; },
                                  [&](uint32_t cnt) { take(std::false_type{}, cnt); });
    return acc;
}

template <uint32_t G, bool MULTI, bool GRID, typename T>
__global__ __launch_bounds__(kCoopBlock, 5) void k_coop_pressure(const CoopArgs A, const Rows<T> in,
                                                                 const float4 *__restrict__ dens,
                                                                 const float4 *__restrict__ vs,
                                                                 float4 *__restrict__ vs2)
{
    __shared__ uint32_t lists[Group<G>::kParticles][kList + 1];
    __shared__ __align__(16) float terms[Group<G>::kParticles][3][2 * Group<G>::kChunk];
    const uint32_t n = A.ed->n_total, slot = coop_slot<G>(n);
    if (slot >= n) return;
    const uint32_t gl = threadIdx.x & (G - 1u), gq = threadIdx.x / G;
    const float4 pi = A.xps[slot], di = dens[slot];
    float4 v = vs[slot];
    auto scene = [&](const SceneDesc &S) __attribute__((always_inline)) {
        const uint32_t k = opaque_slot<MULTI>(slot);
        const bool clean = GRID && A.sflags[S.index] == 0u;
        const PressureSelf self = pressure_self<true>(S, pi, di);
        const float f = coop_sum<G, GRID, 2>(
            A, S, in, dens, k, pi, clean, lists[gq], &terms[gq][0][0],
            [&](float d2, float ox, float oy, float oz, const float4 &dj, float out[6]) {
                const PressureTerms r = pressure_pair<true>(self, ox, oy, oz, d2, dj);
                out[0] = r.tx;
                out[1] = r.ty;
                out[2] = r.tz;
                out[3] = r.ux;
                out[4] = r.uy;
                out[5] = r.uz;
            });
        const float fx = group_bcast<G, 0>(f), fy = group_bcast<G, 1>(f), fz = group_bcast<G, 2>(f);
        const float dt = S.dt, rho = di.x;
        v.x = v.x + (fx / rho) * dt;  // cc:421
        v.y = v.y + (fy / rho) * dt;
        v.z = v.z + (fz / rho) * dt;
        if (gl == 0u) vs2[k] = v;
    };
    run_scene<MULTI>(A.sd, A.scene_of, slot, scene);
}

struct CoopState {  // what the viscosity stage writes (see k_viscosity_integrate)
    const float4 *vs2, *ps;
    float4 *pos, *vel;
    uint32_t *ids;
    float4 *rpos, *colors;
    uint32_t *keys, *ticks, *count, *wkeys;
    // the state in particle order (sph_update_noalloc), or null; with them the
    // resident state and the next update's buckets (pos .. wkeys) are not written
    float4 *out_pos, *out_vel;
    float2 *out_dens;
    const float4 *dens;
};

// (waves per SIMD: what the LDS allows, 5 for density and pressure, 7 here; one
// scene fits 72 registers, and with 75, 6 waves, the reference key's stage takes
// 43.3 instead of 40.8 us on 200,003 particles; several scenes take 90)
template <uint32_t G, bool MULTI, bool GRID, typename T>
__global__ __launch_bounds__(kCoopBlock, MULTI ? 5 : 7) void k_coop_viscosity(const CoopArgs A, const Rows<T> in,
                                                                  const CoopState W)
{
    __shared__ uint32_t lists[Group<G>::kParticles][kList + 1];
    __shared__ uint32_t buckets[Group<G>::kParticles];
    __shared__ __align__(16) float terms[Group<G>::kParticles][3][Group<G>::kChunk];
    const uint32_t n = A.ed->n_total, slot = coop_slot<G>(n);
    const uint32_t gl = threadIdx.x & (G - 1u), gq = threadIdx.x / G;
    auto scene = [&](const SceneDesc &S) __attribute__((always_inline)) {
        const uint32_t k = opaque_slot<MULTI>(slot);
        const float4 pi = A.xps[k], vi = W.vs2[k], x0 = W.ps[k];
        const uint32_t g = A.sids[k];
        const bool clean = GRID && A.sflags[S.index] == 0u;
        const float hh = S.hh, c6 = S.poly6c;
        const float f = coop_sum<G, GRID, 1>(
            A, S, in, W.vs2, k, pi, clean, lists[gq], &terms[gq][0][0],
            [&](float d2, float, float, float, const float4 &vj, float out[3]) {
                const float w = viscosity_weight<true>(hh, c6, d2);
                out[0] = (vj.x - vi.x) * w;  // cc:460
                out[1] = (vj.y - vi.y) * w;
                out[2] = (vj.z - vi.z) * w;
            });
        float4 x, v;
        integrate_particle(S, vi, group_bcast<G, 0>(f), group_bcast<G, 1>(f), group_bcast<G, 2>(f), x0, x, v);
        if (gl != 0u) return;
        if (W.out_pos) {
            W.out_pos[g] = x;
            W.out_vel[g] = v;
            if (W.out_dens) {
                const float4 d = W.dens[k];
                W.out_dens[g] = make_float2(d.x, d.y);
            }
            return;
        }
        W.pos[k] = x;
        W.vel[k] = v;
        W.ids[k] = g;
        if (W.rpos) W.rpos[g] = x;
        if (W.colors) {
            float c[4];
            speed_color(v.x, v.y, v.z, A.ed->stops, c);
            W.colors[g] = make_float4(c[0], c[1], c[2], c[3]);
        }
        // stage A + B1 of the next update, from the new state
        const Predicted P = predict_particle(S, x, v);
        buckets[gq] = bucket_key(*A.ed, S, P, W.count);
        if (W.wkeys) W.wkeys[k] = work_key(*A.ed, S, S.index, P.cx, P.cy, P.cz);
    };
    if (slot < n) run_scene<MULTI>(A.sd, A.scene_of, slot, scene);
    if (W.out_pos) return;
    // the tickets of the workgroup's particles, by one lane each: one atomic
    // per run of equal buckets
    __syncthreads();
    if (threadIdx.x >= Group<G>::kParticles) return;
    const uint32_t at = slot - gq + threadIdx.x;
    const bool valid = at < n;
    const uint32_t key = valid ? buckets[threadIdx.x] : 0xffffffffu;
    const uint32_t ticket = bucket_ticket(valid, key, W.count);
    if (valid) {
        W.keys[at] = key;
        W.ticks[at] = ticket;
    }
}

template <uint32_t G>
inline uint32_t coop_grid(uint32_t n)
{
    constexpr uint32_t N = Group<G>::kParticles;
    return ((n + N - 1) / N + 7u) & ~7u;  // XCD numbering: a multiple of 8
}

CoopArgs coop_args(const DevState &s)
{
    return CoopArgs{s.ed, s.sd, s.scene_of, s.sids, s.xps, s.bounds, s.sflags, s.ncnt, nullptr};
}

// Rows of nbr_words words per particle: whole groups of entries.
template <typename T>
Rows<T> coop_rows(const DevState &s)
{
    const uint32_t cap = s.nbr_words * (uint32_t)(sizeof(uint32_t) / sizeof(T));
    return Rows<T>{reinterpret_cast<T *>(s.nbr), reinterpret_cast<T *>(s.spare), cap < 128u ? cap & ~15u : 128u};
}

// Launches KER<G, MULTI, GRID, T> over n particle slots.
#define SPH_COOP_LAUNCH_T(KER, G, GRID, T, n, st, ...)                                             \
    do {                                                                                           \
        const Rows<T> r_ = coop_rows<T>(s);                                                        \
        const uint32_t g_ = coop_grid<G>(n);                                                       \
        if (s.multi) KER<G, true, GRID><<<g_, kCoopBlock, 0, st>>>(a, r_, __VA_ARGS__);            \
        else KER<G, false, GRID><<<g_, kCoopBlock, 0, st>>>(a, r_, __VA_ARGS__);                   \
    } while (0)
#define SPH_COOP_LAUNCH(KER, n, st, ...)                                                           \
    do {                                                                                           \
        const CoopForm f_ = coop_form(s.grid, n, s.capacity);                                      \
        if (s.grid && f_.lanes == 16) SPH_COOP_LAUNCH_T(KER, 16, true, uint16_t, n, st, __VA_ARGS__);       \
        else if (s.grid && f_.entry == 16) SPH_COOP_LAUNCH_T(KER, 8, true, uint16_t, n, st, __VA_ARGS__);   \
        else if (s.grid) SPH_COOP_LAUNCH_T(KER, 8, true, int16_t, n, st, __VA_ARGS__);                      \
        else if (f_.lanes == 16) SPH_COOP_LAUNCH_T(KER, 16, false, uint16_t, n, st, __VA_ARGS__);           \
        else if (f_.entry == 16) SPH_COOP_LAUNCH_T(KER, 8, false, uint16_t, n, st, __VA_ARGS__);            \
        else SPH_COOP_LAUNCH_T(KER, 8, false, uint32_t, n, st, __VA_ARGS__);                                \
    } while (0)

}  // namespace

hipError_t launch_coop_density(const DevState &s, uint32_t n, bool clear_counts, hipStream_t st)
{
    CoopArgs a = coop_args(s);
    if (clear_counts) a.clear = s.count;
    SPH_COOP_LAUNCH(k_coop_density, n, st, s.dens);
    return hipGetLastError();
}

hipError_t launch_coop_pressure(const DevState &s, uint32_t n, hipStream_t st)
{
    const CoopArgs a = coop_args(s);
    SPH_COOP_LAUNCH(k_coop_pressure, n, st, s.dens, s.vs, s.vs2);
    return hipGetLastError();
}

hipError_t launch_coop_viscosity_integrate(const DevState &s, uint32_t n, hipStream_t st)
{
    const CoopArgs a = coop_args(s);
    const CoopState w{s.vs2, s.ps,     s.pos,     s.vel,     s.ids,   s.rpos,
                      s.colors, s.keys[0], s.keys[1], s.count, s.grid ? nullptr : s.wkeys[0],
                      nullptr,  nullptr,   nullptr,   nullptr};
    SPH_COOP_LAUNCH(k_coop_viscosity, n, st, w);
    return hipGetLastError();
}

hipError_t launch_coop_viscosity_out(const DevState &s, uint32_t n, float4 *pos, float4 *vel, float2 *dens,
                                     hipStream_t st)
{
    const CoopArgs a = coop_args(s);
    CoopState w{};
    w.vs2 = s.vs2;
    w.ps = s.ps;
    w.out_pos = pos;
    w.out_vel = vel;
    w.out_dens = dens;
    w.dens = s.dens;
    SPH_COOP_LAUNCH(k_coop_viscosity, n, st, w);
    return hipGetLastError();
}

}  // namespace sph
