// sph_kernel_common.h -- device functions shared by the gfx950 kernels of
// sph_kernels.hip (one work-item per particle) and sph_coop.hip (16 or 8
// work-items per particle): the scene loop, stage A, the bucket of a particle
// and the pair terms of stages C to F.  Every floating-point expression keeps
// the reference's operation order and rounding, so the two forms of a stage
// agree to the bit.
#pragma once
#include <hip/hip_runtime.h>

#include "sph_device.h"
#include "sph_launch.h"

namespace sph {

namespace {

__device__ __forceinline__ uint32_t grid_stride() { return gridDim.x * blockDim.x; }
__device__ __forceinline__ uint32_t global_id() { return blockIdx.x * blockDim.x + threadIdx.x; }

// Scene q's descriptor for a wave-uniform q, read through the constant
// address space: the table does not change while a kernel runs, so the reads
// are scalar loads into scalar registers wherever they are placed.
__device__ __forceinline__ SceneDesc scene_uniform(const SceneDesc *sd, uint32_t q)
{
#if __HIP_DEVICE_COMPILE__
    typedef const __attribute__((address_space(4))) uint32_t ConstWord;
    const ConstWord *w = (const ConstWord *)(sd + q);
    SceneDesc d;
    uint32_t *o = reinterpret_cast<uint32_t *>(&d);
#pragma unroll
    for (uint32_t j = 0; j < sizeof(SceneDesc) / 4; ++j) o[j] = w[j];
    return d;
#else
    return sd[q];  // (host pass: never called)
#endif
}

// Runs body(S) with slot k's scene.  MULTI: the wave takes its scenes one at
// a time (one pass unless it spans a scene boundary), the lanes of that scene
// active and its descriptor read with scalar loads into scalar registers.
// The loop runs on a wave-uniform mask, and a lane's membership is read back
// from a ballot, so the compiler keeps the body inside the loop with the
// uniform scene index (rather than substituting the per-lane one).
template <bool MULTI, typename Body>
__device__ __forceinline__ void run_scene(const SceneDesc *sd, const uint32_t *scene_of, uint32_t k,
                                          Body &body)
{
    if (!MULTI) {
        body(sd[0]);
        return;
    }
    const uint32_t q = scene_of[k], lane = threadIdx.x & 63u;
    uint64_t pending = __ballot(1);
    while (pending) {
        const uint32_t qq = (uint32_t)__builtin_amdgcn_readlane((int)q, (int)__builtin_ctzll(pending));
        const uint64_t mine = __ballot(q == qq);
        if ((mine >> lane) & 1u) body(scene_uniform(sd, qq));
        pending &= ~mine;
    }
}

template <bool MULTI>
__device__ __forceinline__ const SceneDesc &scene_of_slot(const SceneDesc *sd,
                                                          const uint32_t *scene_of, uint32_t k)
{
    return MULTI ? sd[scene_of[k]] : sd[0];
}

// PositionToCellCoord (cc:499-503): floor(pos / r) with IEEE division, then (int).
__device__ __forceinline__ int cell_coord(float x, float h) { return (int)floorf(x / h); }

// 10-bit Morton spread: bit i of x moves to bit 3i.
__device__ __forceinline__ uint32_t spread3(uint32_t x)
{
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// Ordering key of the gather kernels' work order: scene index in the top
// bits, then the Morton code of the cell (relative to the scene's box,
// clamped to 10 bits per axis).  It only decides WHICH work-item handles a
// particle, never a result, so clamping and truncation are harmless.
__device__ __forceinline__ uint32_t work_key(const EngineDesc &E, const SceneDesc &S, uint32_t s,
                                             int cx, int cy, int cz)
{
    const uint32_t ux = (uint32_t)min(max(cx - S.cell_lo[0], 0), 1023);
    const uint32_t uy = (uint32_t)min(max(cy - S.cell_lo[1], 0), 1023);
    const uint32_t uz = (uint32_t)min(max(cz - S.cell_lo[2], 0), 1023);
    const uint32_t m = spread3(ux) | (spread3(uy) << 1) | (spread3(uz) << 2);
    return E.scene_shift >= 32 ? m : ((s << E.scene_shift) | (m >> E.morton_drop));
}

// ---------------------------------------------------------------------------
// Stage A + B1
// ---------------------------------------------------------------------------
// Stage A of one particle (cc:42-48) and its cell (cc:499-503) and hash
// (cc:505-511).  Every kernel that needs them recomputes them from the same
// inputs with the same operations, so the values agree to the bit.
struct Predicted {
    float vx, vy, vz;  // velocity += CalculateExternalFoce(...) * deltatime (cc:45)
    float px, py, pz;  // predictedPositions = positions + velocity * (1/120) (cc:47)
    int cx, cy, cz;
    uint32_t hash;
};

__device__ __forceinline__ Predicted predict_particle(const SceneDesc &S, const float4 &x,
                                                      const float4 &v)
{
    Predicted P;
    const float dt = S.dt;
    P.vx = v.x + S.g[0] * dt;
    P.vy = v.y + S.g[1] * dt;
    P.vz = v.z + S.g[2] * dt;
    P.px = x.x + P.vx * S.lookahead;
    P.py = x.y + P.vy * S.lookahead;
    P.pz = x.z + P.vz * S.lookahead;
    P.cx = cell_coord(P.px, S.h);
    P.cy = cell_coord(P.py, S.h);
    P.cz = cell_coord(P.pz, S.h);
    P.hash = hash_cell(P.cx, P.cy, P.cz);
    return P;
}

// The bucket of a particle (GetKeyFromHash, cc:513-516, or the cell-grid key).
// Under the grid key a cell outside the grid's box wraps onto another cell's
// bucket: it raises the scene's flag, in count's tail.
__device__ __forceinline__ uint32_t bucket_key(const EngineDesc &E, const SceneDesc &S, const Predicted &P,
                                               uint32_t *__restrict__ count)
{
    if (S.grid && ((uint32_t)P.cx - (uint32_t)S.cell_lo[0] >= S.gdim[0] ||
                   (uint32_t)P.cy - (uint32_t)S.cell_lo[1] >= S.gdim[1] ||
                   (uint32_t)P.cz - (uint32_t)S.cell_lo[2] >= S.gdim[2]))
        count[E.table_total + S.index] = 1u;
    return S.key_off + (S.grid ? grid_key(P.cx, P.cy, P.cz, S.cell_lo, S.gdim, S.gmod, S.strip_shift)
                               : fastmod(P.hash, S.mod_m, S.table));
}

// A ticket in bucket `key`: a distinct place in the bucket in arbitrary order,
// from count (records per bucket).  One atomic per run of equal keys in
// consecutive lanes: in the resident order, nearly sorted, a wave's records
// fall in a few runs.  Every lane of the wave that has not exited calls this,
// the valid lanes a prefix of the wave.
__device__ __forceinline__ uint32_t bucket_ticket(bool valid, uint32_t key, uint32_t *__restrict__ count)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t upto = (2ull << lane) - 1ull;  // lanes 0..lane
    // runs of equal keys: a run starts at lane 0, after a different key, and
    // after a lane without a record (those come after every lane with one)
    const uint32_t prev = __shfl_up(key, 1u, 64);
    const uint64_t heads = __ballot(valid && (lane == 0u || prev != key)) | ~__ballot(valid);
    const uint32_t first = 63u - (uint32_t)__builtin_clzll(heads & upto);  // this run's head
    const uint64_t later = heads & ~upto;
    const uint32_t len = (later ? (uint32_t)__builtin_ctzll(later) : 64u) - lane;
    uint32_t base = 0;
    if (valid && first == lane) base = atomicAdd(&count[key], len);
    base = __shfl(base, (int)first, 64);
    return base + (lane - first);
}

// ---------------------------------------------------------------------------
// Pair terms of stages C to E, and stage F
// ---------------------------------------------------------------------------
// FAST: the scene's radius lies in radius_fast's range.
template <bool FAST>
__device__ __forceinline__ float pair_root(float d2)
{
    return FAST ? root_rn(d2) : sqrtf(d2);
}

// Density terms of a neighbour at squared distance d2 (kernels.h:31, 43); 0
// when !in.
template <bool FAST>
__device__ __forceinline__ void density_pair(float h, float w2c, float w3c, float d2, bool in, float &a, float &b)
{
    const float d = pair_root<FAST>(d2);
    const float v = in ? h - d : 0.0f;
    a = v * v * w2c;      // SmoothingPow2
    b = v * v * v * w3c;  // SmoothingPow3
}

// The particle's side of its pressure pairs.
struct PressureSelf {
    float h, dw2c, dw3c, rho0, kp, kn;
    float P, Pn;  // cc:371-372
    bool near_ok;
};

template <bool FAST>
__device__ __forceinline__ PressureSelf pressure_self(const SceneDesc &S, const float4 &pi, const float4 &di)
{
    PressureSelf p;
    p.h = S.h;
    p.dw2c = S.dw2c;
    p.dw3c = S.dw3c;
    p.rho0 = S.rho0;
    p.kp = S.k;
    p.kn = S.k_near;
    p.P = (di.x - p.rho0) * p.kp;
    p.Pn = di.y * p.kn;
    p.near_ok = coords_clear_of_zero(pi.x, pi.y, pi.z, FAST ? S.h * 0x1p-26f : 0x1p-60f);
    return p;
}

// The six terms of a pair's pressure force: t (cc:416), then u (cc:417).
// Every division is correctly rounded.  dj = (rho_j, rho_near_j,
// RN(1/rho_j), RN(1/rho_near_j)); the six divisions by rho_j / rho_near_j
// use those reciprocals and the three by d use RN(1/d), through quotient()
// (exact for divisors in [2^-26, 2^26] and numerators that are 0 or of
// magnitude in [2^-91, 2^100]), and fall back to IEEE division outside that
// range.  FAST proves the range from few values, for h in [2^-16, 2^26]:
//   - d in [2^-26, 2^26] from d2 >= 2^-52 and d < h, and a nonzero difference
//     is >= h 2^-51 (near_ok), so a nonzero component of the direction is of
//     magnitude in [2^-51 (1 - 2^-23), 1 + 2^-22];
//   - with |sp|, |snp| <= 2^30 and |a sp|, |b snp| >= 2^-38, |a| and |b| are
//     >= 2^-69, so no product dir * a or dir * b underflows (>= 2^-121), and
//     every nonzero term is >= 2^-91; |a| <= 15 / (pi h^4) and |b| <= 45 /
//     (pi h^4) are <= 2^68, so it is <= 2^100.
// The reciprocals are 0 when unusable and >= 2^-26 else, so one minimum over
// four values and one maximum over two decide (7 instructions, where testing
// the six terms takes 26): with root_rn, pressure 120 -> 103 us on 1,048,576
// uniform particles, where vector issue and the neighbour gathers (two loads a
// neighbour, 13 million L1 misses a launch) now take about as long as each
// other.  Pairs that fail it (weak forces, odd units) are tested term by term
// before IEEE division is taken.  Without FAST d's own range is tested (the
// differences are >= 2^-84 then, and h bounds nothing) and every pair's terms.
struct PressureTerms {
    float tx, ty, tz, ux, uy, uz;
};

template <bool FAST>
__device__ __forceinline__ PressureTerms pressure_pair(const PressureSelf &p, float ox, float oy, float oz,
                                                       float d2, const float4 &dj)
{
    const float pj = (dj.x - p.rho0) * p.kp, pnj = dj.y * p.kn;  // cc:407-408
    const float sp = (p.P + pj) * 0.5f;     // cc:410
    const float snp = (p.Pn + pnj) * 0.5f;  // cc:411
    float d = pair_root<FAST>(d2);
    float dirx, diry, dirz;
    const bool near_fast = p.near_ok & (FAST ? d2 >= 0x1p-52f : divisor_ok(d));
    if (near_fast) {
        const float yd = recip_rn(d);
        dirx = quotient(ox, d, yd);
        diry = quotient(oy, d, yd);
        dirz = quotient(oz, d, yd);
    } else {
        if (FAST) d = sqrtf(d2);
        const bool apart = d > 0.0f;  // (0, 1, 0) at d = 0, cc:414
        dirx = apart ? ox / d : 0.0f;
        diry = apart ? oy / d : 1.0f;
        dirz = apart ? oz / d : 0.0f;
    }
    const float v = p.h - d;
    const float a = -v * p.dw2c;      // SmoothingDerivativePow2, kernels.h:55
    const float b = -v * v * p.dw3c;  // SmoothingDerivativePow3, kernels.h:67
    const float tx = dirx * a * sp, ty = diry * a * sp, tz = dirz * a * sp;
    const float ux = dirx * b * snp, uy = diry * b * snp, uz = dirz * b * snp;
    bool fast = false;
    if (FAST) {
        const float as = fabsf(a * sp), bs = fabsf(b * snp);
        fast = ((int)near_fast & (int)(fminf(fminf(fminf(as, bs), dj.z), dj.w) >= 0x1p-38f) &
                (int)(fmaxf(fabsf(sp), fabsf(snp)) <= 0x1p30f)) != 0;
    }
    if (!fast)
        fast = ((int)(dj.z != 0.0f) & (int)(dj.w != 0.0f) & (int)quotients_ok(tx, ty, tz, ux, uy, uz)) != 0;
    PressureTerms r;
    if (fast) {
        r.tx = quotient(tx, dj.x, dj.z);
        r.ty = quotient(ty, dj.x, dj.z);
        r.tz = quotient(tz, dj.x, dj.z);
        r.ux = quotient(ux, dj.y, dj.w);
        r.uy = quotient(uy, dj.y, dj.w);
        r.uz = quotient(uz, dj.y, dj.w);
    } else {
        r.tx = tx / dj.x;
        r.ty = ty / dj.x;
        r.tz = tz / dj.x;
        r.ux = ux / dj.y;
        r.uy = uy / dj.y;
        r.uz = uz / dj.y;
    }
    return r;
}

// Viscosity weight of a neighbour at squared distance d2 (kernels.h:78-79).
template <bool FAST>
__device__ __forceinline__ float viscosity_weight(float hh, float c6, float d2)
{
    const float d = pair_root<FAST>(d2);
    const float v = hh - d * d;
    return v * v * v * c6;
}

// Stage E's end and stage F (cc:463, 84-107): velocity v (f: the viscosity
// sum), position x0 -> x.
__device__ __forceinline__ void integrate_particle(const SceneDesc &S, const float4 &vi, float fx, float fy, float fz,
                                                   const float4 &x0, float4 &x, float4 &v)
{
    const float dt = S.dt, mu = S.mu;
    v = vi;
    v.x = vi.x + fx * mu * dt;  // cc:463
    v.y = vi.y + fy * mu * dt;
    v.z = vi.z + fz * mu * dt;
    x = x0;
    x.x += v.x * dt;
    x.y += v.y * dt;
    x.z += v.z * dt;
    if (S.half[0] - fabsf(x.x) <= 0.0f) { x.x = S.half[0] * sign_f(x.x); v.x *= S.damp_neg; }
    if (S.half[1] - fabsf(x.y) <= 0.0f) { x.y = S.half[1] * sign_f(x.y); v.y *= S.damp_neg; }
    if (S.half[2] - fabsf(x.z) <= 0.0f) { x.z = S.half[2] * sign_f(x.z); v.z *= S.damp_neg; }
    x.w = 0.34f;  // OutPositions[i] = vec4(positions[i], 0.34f), cc:107
}

}  // namespace

}  // namespace sph
