// trace.hip - software sparse-voxel-DAG ray traversal for gfx950.
//
// One ray per lane. The traversal is the reference's walk (src/device/dag.zig:
// 160-351: octant mirroring, ESVO-style ascent through the highest changed
// coordinate bit, the two brick levels inside the 64-bit leaf) and must give
// the same hits and the same fp32 t bit for bit, so this file is compiled with
// -ffp-contract=off and every float expression keeps the reference's order of
// operations. The per-ray node stack (one word per level) lives in LDS,
// strided by lane so the 64 lanes of a wave hit distinct banks, and is sized
// by the launch to the DAG's edge (or the scene's largest), not to the
// largest edge the format allows, which keeps more waves resident.
//
// A hit's attribute needs its DFS rank (a second walk down the stack, one
// dependent load per earlier sibling). The walk computes it after the step
// loop, once the whole wave has left the loop, so all lanes of a wave that
// hit rank their voxels together; inside the loop every lane that hits in a
// different iteration would make the wave run the rank walk again with
// only that lane active.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include "common.h"
#include "internal.h"

namespace pyr {

constexpr int kTraceBlock = 128;  // rays per workgroup (types.zig:498 trace_block)
constexpr int kMaxLevels = 21;    // log2_size <= 20
constexpr uint32_t kMaxSteps = 65536;
// Scenes from this many instances on test their boxes against a whole wave
// first. (1920x1080 frames of instance grids: 3 and 6 instances are as fast
// either way, 16 take 325 us with the test and 330 without, 64 take 476 and
// 533, 1000 take 802 and 2429.)
constexpr uint32_t kCullInstances = 8;
// The most waves that a launch is spread over by halving its rays per wave: a
// chip with idle slots gains from waves that diverge less and whose boxes
// are smaller, a full one loses by the repeated lanes. (Rays that fill more than
// half as many waves are not spread.) The chip holds 8192 waves. One DAG (or a
// few instances): 1000 diffuse rays 55 -> 36 us, 16000 88 -> 73, 64000 84 -> 81;
// with up to 8192 waves the 64000 take 89 us, with up to 16384 115. Instances: a
// 640x360 frame of 64 takes 468 us with full waves, 383 with up to 8192, 340
// with 16384, 354 with 32768; of 1000: 633, 500, 432, 557.
constexpr uint32_t kRayWaves = 4096, kSceneWaves = 16384;
constexpr uint32_t kNotMoved = 4;  // added to the entry axis of a walk that has not left its first cell
constexpr uint32_t kHit = 32, kMiss = 64;  // values of a finished walk's scale

// Device memory by its address space: a pointer made from a number would be
// read with flat instructions, which also wait for the LDS; what a traversal
// kernel only reads at an index that all lanes share goes through the scalar
// cache.
#define PYR_GLOBAL __attribute__((address_space(1)))
#define PYR_CONSTANT __attribute__((address_space(4)))
typedef const PYR_GLOBAL uint32_t* Words;
typedef const PYR_GLOBAL uint64_t* Masks;

struct DagView {
    Words nodes;
    Masks leaves;
    Words attrs;    // null: default_attribute
    Words palette;  // non-null: attrs holds 4-bit indices into these 16 values
    uint32_t root, log2_size, default_attribute, attr_base;
};

// attributeAt (dag.zig:64-68): rank r's value, or its palette entry through
// the 4-bit index in bits 4 (r & 7) of word r >> 3
__device__ __forceinline__ uint32_t attribute_at(const DagView& g, uint32_t rank) {
    const uint32_t r = g.attr_base + rank;
    if (g.palette) return g.palette[(g.attrs[r >> 3] >> ((r & 7) * 4)) & 15u];
    return g.attrs[r];
}

struct DagHitD {
    float t;
    uint32_t face;
    uint32_t attribute;
    uint32_t inside;
    int32_t voxel[3];
};

__device__ __forceinline__ uint32_t bit_of(uint32_t v, uint32_t s) { return (v >> s) & 1u; }
__device__ __forceinline__ uint32_t brick_bit(uint32_t x, uint32_t y, uint32_t z) { return x + 4 * y + 16 * z; }

// Node word i, for an index every active lane shares: a scalar load (the
// node array does not change while a traversal kernel runs).
__device__ __forceinline__ uint32_t node_uniform(const DagView& g, uint32_t i) {
    return ((const PYR_CONSTANT uint32_t*)g.nodes)[i];
}

// attributeRank (dag.zig:70-87); stk[s * kTraceBlock] is the node whose
// children have edge 2^s
__device__ uint32_t attribute_rank(const DagView& g, const uint32_t* stk, const uint32_t v[3], uint64_t brick) {
    uint32_t rank = 0;
    for (uint32_t s = g.log2_size - 1; s >= 2; s--) {
        const uint32_t node = stk[s * kTraceBlock];
        const uint32_t mask = g.nodes[node] & 0xFFu;
        const uint32_t idx = bit_of(v[0], s) | (bit_of(v[1], s) << 1) | (bit_of(v[2], s) << 2);
        const uint32_t before = (uint32_t)__popc(mask & ((1u << idx) - 1));
        for (uint32_t k = 0; k < before; k++) {
            const uint32_t ref = g.nodes[node + 2 + k];
            rank += s == 2 ? (uint32_t)__popcll(g.leaves[ref]) : g.nodes[ref + 1];
        }
    }
    const uint32_t bit = brick_bit(v[0] & 3, v[1] & 3, v[2] & 3);
    return rank + (uint32_t)__popcll(brick & ((1ull << bit) - 1));
}

// skipped (dag.zig:153-157): bit (attribute & 0xFF) of a 256-bit material set
__device__ __forceinline__ bool skipped(const uint64_t* set, uint32_t attribute) {
    if (!set) return false;
    const uint32_t idx = attribute & 0xFFu;
    return ((set[idx >> 6] >> (idx & 63u)) & 1ull) != 0;
}

// cutHole (dag.zig:133-151) for a DAG at the origin of its object space: is
// the entry point p on face `axis` of the voxel in a hole of the material's
// fixed 3 x 3 pattern (about 30 % of the face)?
__device__ __forceinline__ bool cut_hole(const uint64_t* cut, uint32_t attribute, const int32_t voxel[3],
                                         const float p[3], uint32_t axis) {
    if (!skipped(cut, attribute)) return false;
    uint32_t sub[2] = {0, 0}, k = 0;
#pragma unroll
    for (uint32_t a = 0; a < 3; a++) {
        if (a == axis) continue;
        const float f = fminf(fmaxf(p[a] - (float)voxel[a], 0.0f), 0.999f);
        sub[k++] = (uint32_t)(f * 3.0f);
    }
    uint32_t h = (uint32_t)voxel[0] * 0x8da6b343u + (uint32_t)voxel[1] * 0xd8163841u + (uint32_t)voxel[2] * 0xcb1ab31fu +
                 (attribute >> 8) * 0x2545f491u + axis * 0x9e3779b9u + (sub[0] * 3 + sub[1]) * 0x632be5abu;
    h ^= h >> 15;
    h *= 0x2c1b3c6du;
    h ^= h >> 12;
    return (h & 0xFFu) < 77u;
}

// floor(p) clamped to [lo, hi]; a NaN gives lo. The hardware conversion
// truncates and saturates (negative and NaN to 0), which the C++ cast leaves
// undefined.
__device__ __forceinline__ uint32_t clamped_cell(float p, uint32_t lo, uint32_t hi) {
    uint32_t x, r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(x) : "v"(p));
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}

// the larger of two numbers (fmaxf would canonicalise both operands first)
__device__ __forceinline__ float max_f32(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// walk (dag.zig:160-351); stk points at this lane's column of the block's
// LDS stack. SKIPPING (traceSkipping, dag.zig:113-115, 236-289): voxels of a
// material in `skip` are passed, and voxels of a material in `cut` where the
// entry point lies in a hole of the material's pattern or the ray starts
// inside them; such a walk needs each candidate voxel's attribute inside the
// loop, so it ranks there, and its hits carry the attribute even when
// want_attr is false (as the reference's do).
template <bool SKIPPING>
__device__ bool walk(const DagView& g, const float o[3], const float d[3], float tmin, float tmax, bool want_attr,
                     uint32_t* stk, DagHitD* hit, const uint64_t* skip = nullptr, const uint64_t* cut = nullptr) {
    const uint32_t n = 1u << g.log2_size;
    const float nf = (float)n;
    uint32_t oct = 0;
    float od[3], dd[3], inv[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float oa = o[a], da = d[a];
        if (da < 0) {
            oa = nf - oa;
            da = -da;
            oct |= 1u << a;
        }
        od[a] = oa;
        dd[a] = da;
        inv[a] = 1.0f / fmaxf(da, 1e-30f);
    }
    uint32_t axis = 0;
    float tn = -od[0] * inv[0];
#pragma unroll
    for (int a = 1; a < 3; a++) {
        const float ta = -od[a] * inv[a];
        if (ta > tn) {
            tn = ta;
            axis = (uint32_t)a;
        }
    }
    const float tf = fminf(fminf((nf - od[0]) * inv[0], (nf - od[1]) * inv[1]), (nf - od[2]) * inv[2]);
    float t = fmaxf(tn, tmin);
    const float tend = fminf(tf, tmax);
    if (!(t < tend)) return false;
    const bool starts_inside = tn < tmin;
    // brick bit of a mirrored cell: its low two bits per axis, flipped on the
    // mirrored axes (3 - x for a voxel; the high bit of each pair alone for a
    // 2 x 2 x 2 block; n is a multiple of 4)
    const uint32_t flip1 = (oct & 1u ? 3u : 0u) | (oct & 2u ? 12u : 0u) | (oct & 4u ? 48u : 0u);

    // The point of the ray at t as whole coordinates, clamped to the current
    // cell (edge 2^scale): q[a] & ~(2^scale - 1) is the cell, and bit s of q
    // says in which half of its ancestor of edge 2^(s+1) the point lies. t
    // does not change while the ray enters children, and the reference's
    // "p - cell >= half" on a float p is the same test as "bit scale - 1 of
    // clamp(floor(p))" (the difference of p and a whole number below it is
    // exact, and above it only the sign counts), so one conversion per
    // advance serves every level entered after it, and entering a child costs
    // no arithmetic on the coordinates.
    axis |= kNotMoved;
    const uint32_t top = g.log2_size - 1;
    uint32_t scale = top;
    uint32_t q[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float p = fminf(fmaxf(floorf(od[a] + dd[a] * t), 0.0f), nf - 1.0f);
        q[a] = (uint32_t)p;
    }
    stk[scale * kTraceBlock] = g.root;
    // The levels that every lane of the wave enters the same way, node words
    // through the scalar cache: neighbouring primary and shadow rays share
    // most of the way down to their first cell (six poses over a 4096^3
    // landscape: 3840x2160 primary rays 671 -> 664 us a frame, 1920x1080 shadow
    // rays 182 -> 179, 1920x1080 primary rays 229 either way; 64 instances 459 ->
    // 456).
    {
        const uint32_t u0 = first_lane32(q[0]), u1 = first_lane32(q[1]), u2 = first_lane32(q[2]), uo = first_lane32(oct);
        const uint32_t apart = oct == uo ? (q[0] ^ u0) | (q[1] ^ u1) | (q[2] ^ u2) : ~0u;
        uint32_t node = g.root, us = top;
        while (us >= 3 && __ballot((apart >> us) != 0) == 0) {
            const uint32_t mask = node_uniform(g, node);
            const uint32_t idx = (((u0 >> us) & 1u) | (((u1 >> us) & 1u) << 1) | (((u2 >> us) & 1u) << 2)) ^ uo;
            const uint32_t bit = 1u << idx;
            if (!(mask & bit)) break;
            node = node_uniform(g, node + 2 + __popc(mask & (bit - 1)));
            us -= 1;
            stk[us * kTraceBlock] = node;
        }
        scale = us;
    }
    uint64_t brick = 0;
    // cells looked up so far, less the levels entered since the start (the
    // bound kMaxSteps counts every lookup; a ray cannot reach it below 2^13)
    const bool bounded = g.log2_size > 12;
    uint32_t steps = 0, iter = 0;
    // One iteration looks a cell up and enters it if it is filled, or leaves
    // it along the ray and ascends to the highest coordinate bit that changed.
    // The walk is bound by instruction issue (vector ALU busy 78 % of a primary
    // frame), the scalar unit's share included, which the masks of nested
    // branches and of flags kept across them load as much as the arithmetic
    // does the vector unit. So there are three branches in a row and no exits
    // from inside them: an empty cell's step is formed whole also when it ends
    // the walk, and the end of a walk is a value of `scale`, not a flag.
    // 1920x1080 frames of a 4096^3 landscape, mean of six poses, against the
    // form that converted and compared coordinates at every level entered and
    // left: primary 306 -> 229 us, shadow 236 -> 179 us; 1e6 diffuse rays 271 ->
    // 215 us. (Measured and left out: entering until a cell is empty before any
    // lane leaves one, primary 1.30 times as long; two lookups per iteration, 0.99,
    // but shadow rays 1.02; the child loaded for empty cells too to save a
    // branch, 1.02.)
    do {
        uint32_t filled = 1;
        if (scale >= 2) {
            const uint32_t node = stk[scale * kTraceBlock];
            const uint32_t mask = g.nodes[node];
            const uint32_t idx = (__builtin_amdgcn_ubfe(q[0], scale, 1) | (__builtin_amdgcn_ubfe(q[1], scale, 1) << 1) |
                                  (__builtin_amdgcn_ubfe(q[2], scale, 1) << 2)) ^ oct;
            filled = __builtin_amdgcn_ubfe(mask, idx, 1);
            if (filled) {
                const uint32_t child = (g.nodes + 2)[node + __popc(mask & ((1u << idx) - 1))];
                scale -= 1;
                stk[scale * kTraceBlock] = child;
                if (scale == 1) brick = g.leaves[child];
            }
        }
        if (scale < 2) {
            // a brick of 4^3 voxels: its 2 x 2 x 2 block, then the voxel
            const uint32_t b = brick_bit(q[0] & 3u, q[1] & 3u, q[2] & 3u) ^ flip1;
            filled = (uint32_t)(brick >> b) & 1u;
            const bool block = ((uint32_t)(brick >> (b & 0x2Au)) & 0x00330033u) != 0;
            if (scale == 1 && block) scale = 0;
            if constexpr (SKIPPING) {
                if (filled) {
                    uint32_t v[3];
                    int32_t vox[3];
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        v[k] = ((oct >> k) & 1u) ? n - 1 - q[k] : q[k];
                        vox[k] = (int32_t)v[k];
                    }
                    uint32_t attribute = g.default_attribute;
                    if ((want_attr || skip || cut) && g.attrs) attribute = attribute_at(g, attribute_rank(g, stk, v, brick));
                    bool through = false;
                    if (starts_inside && axis >= kNotMoved) {
                        through = skipped(cut, attribute);
                    } else if (cut) {
                        float p[3];
#pragma unroll
                        for (int k = 0; k < 3; k++) p[k] = o[k] + d[k] * t;
                        through = cut_hole(cut, attribute, vox, p, axis & (kNotMoved - 1));
                    }
                    // a passed voxel is left like an empty one
                    hit->attribute = attribute;
                    filled = skipped(skip, attribute) || through ? 0u : 1u;
                }
            }
            if (filled) scale = kHit;
        }
        if (!filled) {
            // leaving the cell: the nearest of its three far faces
            const uint32_t m = ~0u << scale;
            const uint32_t n0 = (q[0] | ~m) + 1, n1 = (q[1] | ~m) + 1, n2 = (q[2] | ~m) + 1;
            const float t0 = ((float)n0 - od[0]) * inv[0];
            const float t1 = ((float)n1 - od[1]) * inv[1];
            const float t2 = ((float)n2 - od[2]) * inv[2];
            // the first axis with the smallest exit (ties to the lower axis)
            const bool a1 = t1 < t0;
            const float t01 = a1 ? t1 : t0;
            const bool s2 = t2 < t01;
            const bool s1 = a1 && !s2, s0 = !a1 && !s2;
            const float tnext = s2 ? t2 : t01;
            const uint32_t c0 = s0 ? n0 : q[0], c1 = s1 ? n1 : q[1], c2 = s2 ? n2 : q[2];
            // highest changed bit; the grid's own bit when the ray leaves the grid
            const uint32_t diff = (c0 ^ q[0]) | (c1 ^ q[1]) | (c2 ^ q[2]);
            const uint32_t up = 31 - (uint32_t)__builtin_clz(diff);
            bool leave = !(tnext < tend) || diff >= n;
            t = max_f32(t, tnext);
            axis = s2 ? 2u : (a1 ? 1u : 0u);
            if (bounded) {
                asm volatile("");  // (opaque, so that this stays a block of its own: without it 229 -> 240 us)
                steps += up + 1 - scale;
                leave |= steps + top - up >= kMaxSteps;
            }
            scale = leave ? kMiss : up;
            const uint32_t um = ~0u << up;
            q[0] = clamped_cell(od[0] + dd[0] * t, c0 & um, c0 | ~um);
            q[1] = clamped_cell(od[1] + dd[1] * t, c1 & um, c1 | ~um);
            q[2] = clamped_cell(od[2] + dd[2] * t, c2 & um, c2 | ~um);
        }
    } while (scale < kHit && ++iter < kMaxSteps);
    // (a hit voxel whose lookup lies past the bound is none)
    if (scale != kHit || (bounded && steps + top >= kMaxSteps)) return false;
    // the hit: every value below is final when the loop leaves
    uint32_t v[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        v[a] = ((oct >> a) & 1u) ? n - 1 - q[a] : q[a];
        hit->voxel[a] = (int32_t)v[a];
    }
    hit->inside = starts_inside && axis >= kNotMoved;
    axis &= kNotMoved - 1;
    const bool mirrored = ((oct >> axis) & 1u) != 0;
    hit->t = t;
    hit->face = 2 * axis + (mirrored ? 0u : 1u);
    if constexpr (!SKIPPING) {
        uint32_t attribute = g.default_attribute;
        // the stack still holds the hit voxel's path and brick is its leaf
        if (want_attr && g.attrs) attribute = attribute_at(g, attribute_rank(g, stk, v, brick));
        hit->attribute = attribute;
    }
    return true;
}

__device__ __forceinline__ PyrHit to_hit(bool found, const DagHitD& h, uint32_t instance) {
    PyrHit r;
    if (found) {
        r.t = h.t;
        r.instance = instance;
        r.attribute = h.attribute;
        r.meta = h.face | (h.inside ? PYR_HIT_INSIDE : 0u);
    } else {
        r.t = PYR_FLT_MAX;
        r.instance = PYR_NO_HIT;
        r.attribute = 0;
        r.meta = 0;
    }
    return r;
}

// ---- scene traversal (trace.zig:56-113) -------------------------------------
__device__ __forceinline__ float safe_rcp(float x) {
    return 1.0f / (fabsf(x) < 1e-30f ? (x < 0 ? -1e-30f : 1e-30f) : x);
}

__device__ __forceinline__ void xform_point(const float* m, const float p[3], float r[3]) {
    r[0] = m[0] * p[0] + m[1] * p[1] + m[2] * p[2] + m[3];
    r[1] = m[4] * p[0] + m[5] * p[1] + m[6] * p[2] + m[7];
    r[2] = m[8] * p[0] + m[9] * p[1] + m[10] * p[2] + m[11];
}

__device__ __forceinline__ void xform_vector(const float* m, const float v[3], float r[3]) {
    r[0] = m[0] * v[0] + m[1] * v[1] + m[2] * v[2];
    r[1] = m[4] * v[0] + m[5] * v[1] + m[6] * v[2];
    r[2] = m[8] * v[0] + m[9] * v[1] + m[10] * v[2];
}

// anyCutout / cutoutHere (trace.zig:161-173): cutouts only where a voxel
// edge is at most about 1.4 world units (row 0 of world_to_object)
__device__ __forceinline__ bool any_cutout(const PyrScene& s) {
    return (s.cutout_materials[0] | s.cutout_materials[1] | s.cutout_materials[2] | s.cutout_materials[3]) != 0;
}
__device__ __forceinline__ bool cutout_here(const float world_to_object[12]) {
    float w2o = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; a++) w2o += world_to_object[a] * world_to_object[a];
    return w2o > 0.5f;
}

// Largest and smallest value of a wave's lanes (all of them active).
__device__ __forceinline__ float wave_max(float x) {
    const float u = __uint_as_float(first_lane32(__float_as_uint(x)));
    if (__ballot(x != u) == 0) return u;
    auto step = [&](float y) { x = fmaxf(x, y); };
    auto moved = [&](uint32_t y) { step(__uint_as_float(y)); };
    moved(dpp32<kDppRowShr1>(__float_as_uint(x), __float_as_uint(x)));
    moved(dpp32<kDppRowShr2>(__float_as_uint(x), __float_as_uint(x)));
    moved(dpp32<kDppRowShr4>(__float_as_uint(x), __float_as_uint(x)));
    moved(dpp32<kDppRowShr8>(__float_as_uint(x), __float_as_uint(x)));
    moved(dpp32<kDppRowBcast15, 0xa>(__float_as_uint(x), __float_as_uint(x)));
    moved(dpp32<kDppRowBcast31, 0xc>(__float_as_uint(x), __float_as_uint(x)));
    return __uint_as_float(lane_read32(__float_as_uint(x), kWave - 1));
}
struct Range {
    float lo, hi;
};
__device__ __forceinline__ Range wave_range(float x) { return {-wave_max(-x), wave_max(x)}; }

// SKIPPING: the launch found a material set that may apply (skip flag with
// transparent materials, or cutout materials); each variant holds one walk,
// which keeps the registers of the plain one at its own count. EXT: the best
// hit's point in its instance's object space goes to p_object (trace.zig:107).
template <bool SKIPPING, bool EXT = false>
__device__ PyrHit trace_scene(const PyrScene& s, const float o[3], const float d[3], float tmin, float tmax,
                              uint32_t ray_mask, uint32_t flags, uint32_t* stk, uint32_t levels,
                              float* p_object = nullptr) {
    const PYR_CONSTANT PyrInstanceData* inst = (const PYR_CONSTANT PyrInstanceData*)(uintptr_t)s.instances;
    const PYR_CONSTANT PyrGeometryData* geo = (const PYR_CONSTANT PyrGeometryData*)(uintptr_t)s.geometries;
    const float inv[3] = {safe_rcp(d[0]), safe_rcp(d[1]), safe_rcp(d[2])};
    const bool want_attr = (flags & PYR_TRACE_NO_ATTRIBUTE) == 0;
    float best = tmax;
    PyrHit result = to_hit(false, DagHitD{}, 0);
    // material sets of the traversal (trace.zig:80, 93-98)
    const uint64_t* skip = SKIPPING && (flags & PYR_TRACE_SKIP_TRANSPARENT) ? s.transparent_materials : nullptr;
    const uint64_t* cut = SKIPPING && any_cutout(s) ? s.cutout_materials : nullptr;
    auto visit = [&](uint32_t i) {
        const PYR_CONSTANT PyrInstanceData& in = inst[i];
        if (!(in.flags & PYR_INSTANCE_ACTIVE) || !(in.mask & ray_mask)) return;
        float lo[3], hi[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            lo[a] = (in.bounds_min[a] - o[a]) * inv[a];
            hi[a] = (in.bounds_max[a] - o[a]) * inv[a];
        }
        const float t0 = fmaxf(fmaxf(fminf(lo[0], hi[0]), fminf(lo[1], hi[1])), fminf(lo[2], hi[2]));
        const float t1 = fminf(fminf(fmaxf(lo[0], hi[0]), fmaxf(lo[1], hi[1])), fmaxf(lo[2], hi[2]));
        if (!(t0 <= t1)) return;
        if (!(fmaxf(t0, tmin) < fminf(t1, best))) return;
        const PYR_CONSTANT PyrGeometryData& g = geo[in.geometry];
        if (g.log2_size > levels) return;  // cannot happen: the stack is sized to the scene's largest edge
        DagView v;
        v.nodes = (Words)(uintptr_t)s.nodes + g.node_offset;
        v.leaves = (Masks)(uintptr_t)s.leaves + g.leaf_offset;
        v.attrs = (g.flags & PYR_GEOMETRY_HAS_ATTRIBUTES) ? (Words)(uintptr_t)s.attributes + g.attribute_offset
                                                         : nullptr;
        v.palette = (g.flags & PYR_GEOMETRY_PALETTE) ? (Words)(uintptr_t)s.attributes + g.palette_offset
                                                     : nullptr;
        v.root = g.root;
        v.log2_size = g.log2_size;
        v.default_attribute = g.default_attribute;
        v.attr_base = 0;
        float m[12], oo[3], dv[3];
#pragma unroll
        for (int k = 0; k < 12; k++) m[k] = in.world_to_object[k];
        xform_point(m, o, oo);
        xform_vector(m, d, dv);
        DagHitD h;
        // with both sets null the skipping walk returns what the plain one does
        const uint64_t* icut = cut && cutout_here(m) ? cut : nullptr;
        if (walk<SKIPPING>(v, oo, dv, tmin, best, want_attr, stk, &h, skip, icut)) {
            best = h.t;
            result = to_hit(true, h, i);
            if (EXT)
#pragma unroll
                for (int a = 0; a < 3; a++) p_object[a] = oo[a] + dv[a] * h.t;
            // (an any-hit ray is over: no box begins before minus infinity)
            if (flags & PYR_TRACE_ANY_HIT) best = -__builtin_inff();
        }
    };
    if (s.instance_count < kCullInstances) {
        for (uint32_t i = 0; i < s.instance_count; i++) visit(i);
        return result;
    }
    // The test of every box by every ray was most of a frame of many instances
    // (1000 instances, 1920x1080: 3.59 ms, 2.43 with the tables read through
    // the scalar cache, 0.80 with the test below; 64 instances 0.60, 0.53,
    // 0.48 ms). So each lane tests another instance's box against all rays of the wave at
    // once: the boxes' slab distances over the range of the wave's origins and
    // reciprocal directions. Subtraction and multiplication round monotonically,
    // so the range of the corners' products holds every ray's own product, and
    // an instance that fails the test fails it for each of the rays. Those that
    // pass are visited in their order. (Undefined and infinite numbers of an
    // origin or direction give no range: then every instance is a candidate. An
    // undefined limit of a ray is none, as in visit(): the larger and the smaller
    // of it and a number are the number.)
    Range ro[3], ri[3];
    bool finite = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        finite &= fabsf(o[a]) < __builtin_inff() && fabsf(inv[a]) < __builtin_inff() && inv[a] != 0.0f;
        ro[a] = wave_range(o[a]);
        ri[a] = wave_range(inv[a]);
    }
    const bool ranges = __ballot(!finite) == 0;
    const float near = -wave_max(tmin == tmin ? -tmin : __builtin_inff());
    for (uint32_t base = 0; base < s.instance_count; base += kWave) {
        const uint32_t j = base + lane_id();
        const float far = wave_max(best == best ? best : __builtin_inff());
        bool candidate = j < s.instance_count;
        if (candidate) {
            const PYR_CONSTANT PyrInstanceData& in = inst[j];
            candidate = (in.flags & PYR_INSTANCE_ACTIVE) && (in.mask & ray_mask);
            if (ranges) {
                float t0 = near, t1 = far;
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    const float b[4] = {in.bounds_min[a] - ro[a].lo, in.bounds_min[a] - ro[a].hi,
                                        in.bounds_max[a] - ro[a].lo, in.bounds_max[a] - ro[a].hi};
                    float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        lo = fminf(lo, fminf(b[k] * ri[a].lo, b[k] * ri[a].hi));
                        hi = fmaxf(hi, fmaxf(b[k] * ri[a].lo, b[k] * ri[a].hi));
                    }
                    t0 = fmaxf(t0, lo);
                    t1 = fminf(t1, hi);
                }
                candidate = candidate && t0 <= t1;
            }
        }
        for (uint64_t m = __ballot(candidate); m; m &= m - 1) visit(base + (uint32_t)__builtin_ctzll(m));
    }
    return result;
}

// ---- kernels -------------------------------------------------------------------
// Every kernel takes its stack from dynamic LDS: stack_bytes(levels) per block.
extern __shared__ uint32_t s_stk[];

__host__ __device__ constexpr uint32_t stack_bytes(uint32_t levels) { return levels * kTraceBlock * 4u; }

// A wave holds per_wave rays (a power of two); its other lanes repeat
// them, so every lane of a wave stays active (the instance test works on all).
__device__ __forceinline__ uint32_t shared_ray(uint32_t per_wave) {
    const uint32_t wave = blockIdx.x * (kTraceBlock / kWave) + threadIdx.x / kWave;
    return wave * per_wave + (lane_id() & (per_wave - 1));
}
// pixels of a frame: a wave holds a tile of 2^tile_x by 2^tile_y pixels, and
// the two waves of a workgroup lie one above the other
__device__ __forceinline__ void shared_pixel(uint32_t tile, uint32_t* x, uint32_t* y) {
    const uint32_t tx = tile & 0xFFu, ty = tile >> 8, i = lane_id() & ((1u << (tx + ty)) - 1);
    *x = (blockIdx.x << tx) + (i & ((1u << tx) - 1));
    *y = ((blockIdx.y * (kTraceBlock / kWave) + threadIdx.x / kWave) << ty) + (i >> tx);
}
__device__ __forceinline__ bool own_lane(uint32_t per_wave) { return lane_id() < per_wave; }

template <bool SKIPPING>
__global__ void __launch_bounds__(kTraceBlock) k_trace_scene(const PyrScene* scene, const PyrRay* rays, PyrHit* hits,
                                                              uint32_t count, uint32_t ray_mask, uint32_t flags,
                                                              uint32_t levels, uint32_t per_wave) {
    const uint32_t i = shared_ray(per_wave), k = min(i, count - 1);
    const PyrRay r = rays[k];
    const PyrHit h = trace_scene<SKIPPING>(*scene, r.origin, r.direction, r.tmin, r.tmax, ray_mask, flags,
                                           s_stk + threadIdx.x, levels);
    if (i < count && own_lane(per_wave)) hits[i] = h;
}

// extendedHit and hitNormal (trace.zig:125-157): the voxel from the object
// space hit point moved half a voxel inward on the hit face's axis (unless the
// ray started inside), the hit point o + d t in the rays' space, and the face
// normal through the transpose of world_to_object (vec.zig:43-49), normalised
// as v * (1 / sqrt((x x + y y) + z z)) (vec.zig:13-23). A miss is all zero
// but for the miss hit.
__device__ __forceinline__ void store_extended(const PyrScene& s, const float o[3], const float d[3], const PyrHit& h,
                                               const float po[3], PyrHitEx* out) {
    PyrHitEx r = {};
    r.hit = h;
    if (h.instance != PYR_NO_HIT) {
        const uint32_t face = h.meta & PYR_HIT_FACE_MASK, axis = face >> 1;
        const bool inside = (h.meta & PYR_HIT_INSIDE) != 0;
        float n[3];
#pragma unroll
        for (uint32_t a = 0; a < 3; a++) {
            float p = po[a];
            if (!inside && a == axis) p += (face & 1u) ? 0.5f : -0.5f;
            r.voxel[a] = (int32_t)floorf(p);
            r.position[a] = o[a] + d[a] * h.t;
            n[a] = a == axis ? ((face & 1u) ? -1.0f : 1.0f) : 0.0f;
        }
        const float* m = ((const PyrInstanceData*)(uintptr_t)s.instances)[h.instance].world_to_object;
        const float v0 = m[0] * n[0] + m[4] * n[1] + m[8] * n[2];
        const float v1 = m[1] * n[0] + m[5] * n[1] + m[9] * n[2];
        const float v2 = m[2] * n[0] + m[6] * n[1] + m[10] * n[2];
        const float il = 1.0f / sqrtf((v0 * v0 + v1 * v1) + v2 * v2);
        r.normal[0] = v0 * il;
        r.normal[1] = v1 * il;
        r.normal[2] = v2 * il;
    }
    *out = r;
}

// pyr_trace with PYR_TRACE_EXTENDED (gpu_kernels.zig:79-81): one PyrHitEx per ray
template <bool SKIPPING>
__global__ void __launch_bounds__(kTraceBlock) k_trace_scene_ex(const PyrScene* scene, const PyrRay* rays,
                                                                 PyrHitEx* hits, uint32_t count, uint32_t ray_mask,
                                                                 uint32_t flags, uint32_t levels, uint32_t per_wave) {
    const uint32_t i = shared_ray(per_wave), k = min(i, count - 1);
    const PyrRay r = rays[k];
    float po[3] = {0.0f, 0.0f, 0.0f};
    const PyrHit h = trace_scene<SKIPPING, true>(*scene, r.origin, r.direction, r.tmin, r.tmax, ray_mask, flags,
                                                  s_stk + threadIdx.x, levels, po);
    if (i < count && own_lane(per_wave)) store_extended(*scene, r.origin, r.direction, h, po, hits + i);
}

__global__ void __launch_bounds__(kTraceBlock) k_trace_dag(DagView g, const PyrRay* rays, PyrHit* hits,
                                                            uint32_t count, uint32_t flags, uint32_t per_wave) {
    const uint32_t i = shared_ray(per_wave);
    if (i >= count) return;
    const PyrRay r = rays[i];
    DagHitD h;
    bool f = walk<false>(g, r.origin, r.direction, r.tmin, r.tmax, (flags & PYR_TRACE_NO_ATTRIBUTE) == 0,
                  s_stk + threadIdx.x, &h);
    if (own_lane(per_wave)) hits[i] = to_hit(f, h, 0);
}

// cameraRay (render.zig:16-32) for pixel centre + jitter (render.zig:133-141)
__device__ __forceinline__ void camera_ray(const PyrCamera& c, uint32_t x, uint32_t y, float o[3], float d[3],
                                           float* tmin, float* tmax) {
    const float px = (float)x + 0.5f + c.jitter[0];
    const float py = (float)y + 0.5f + c.jitter[1];
    const float nx = 2.0f * px / (float)c.width - 1.0f;
    const float ny = 1.0f - 2.0f * py / (float)c.height;
    const float vx = (nx + c.shift[0]) * c.scale[0];
    const float vy = (ny + c.shift[1]) * c.scale[1];
    const bool ortho = c.projection == PYR_PROJECTION_ORTHOGRAPHIC;
    const float ov[3] = {ortho ? vx : 0.0f, ortho ? vy : 0.0f, 0.0f};
    const float dv[3] = {ortho ? 0.0f : vx, ortho ? 0.0f : vy, -1.0f};
    float dw[3];
    xform_vector(c.view_to_world, dv, dw);
    const float len = sqrtf(dw[0] * dw[0] + dw[1] * dw[1] + dw[2] * dw[2]);
    const float il = 1.0f / len;
    xform_point(c.view_to_world, ov, o);
    d[0] = dw[0] * il;
    d[1] = dw[1] * il;
    d[2] = dw[2] * il;
    *tmin = c.near_plane * len;
    *tmax = c.far_plane > 0 ? c.far_plane * len : PYR_FLT_MAX;
}

// pixel tiles (16 x 4 a wave in large frames) keep a wave's rays coherent
__global__ void __launch_bounds__(kTraceBlock) k_trace_camera(DagView g, PyrCamera cam, PyrHit* hits,
                                                               uint32_t flags, uint32_t tile) {
    uint32_t x, y;
    shared_pixel(tile, &x, &y);
    if (x >= cam.width || y >= cam.height) return;
    float o[3], d[3], tmin, tmax;
    camera_ray(cam, x, y, o, d, &tmin, &tmax);
    DagHitD h;
    bool f = walk<false>(g, o, d, tmin, tmax, (flags & PYR_TRACE_NO_ATTRIBUTE) == 0, s_stk + threadIdx.x, &h);
    if (own_lane(1u << ((tile & 0xFFu) + (tile >> 8)))) hits[(uint64_t)y * cam.width + x] = to_hit(f, h, 0);
}

__global__ void __launch_bounds__(kTraceBlock) k_camera_rays(PyrCamera cam, PyrRay* rays) {
    const uint32_t x = blockIdx.x * 16 + (threadIdx.x & 15), y = blockIdx.y * 8 + (threadIdx.x >> 4);
    if (x >= cam.width || y >= cam.height) return;
    PyrRay r;
    camera_ray(cam, x, y, r.origin, r.direction, &r.tmin, &r.tmax);
    rays[(uint64_t)y * cam.width + x] = r;
}

template <bool SKIPPING>
__global__ void __launch_bounds__(kTraceBlock) k_render_scene(const PyrScene* scene, PyrCamera cam, const float* w2v,
                                                               PyrHit* hits, float* depth, uint32_t ray_mask,
                                                               uint32_t flags, uint32_t levels, uint32_t tile) {
    uint32_t px, py;
    shared_pixel(tile, &px, &py);
    const uint32_t x = min(px, cam.width - 1), y = min(py, cam.height - 1);
    float o[3], d[3], tmin, tmax;
    camera_ray(cam, x, y, o, d, &tmin, &tmax);
    PyrHit h = trace_scene<SKIPPING>(*scene, o, d, tmin, tmax, ray_mask, flags, s_stk + threadIdx.x, levels);
    if (px >= cam.width || py >= cam.height || !own_lane(1u << ((tile & 0xFFu) + (tile >> 8)))) return;
    const uint64_t i = (uint64_t)y * cam.width + x;
    if (hits) hits[i] = h;
    if (depth) {
        float dp = PYR_FLT_MAX;
        if (h.instance != PYR_NO_HIT) {
            float p[3], q[3];
#pragma unroll
            for (int a = 0; a < 3; a++) p[a] = o[a] + d[a] * h.t;
            xform_point(w2v, p, q);
            dp = -q[2];
        }
        depth[i] = dp;
    }
}

// shadow ray per primary hit (shade.zig:626-629, 940): from the hit point
// moved 1e-3 voxel along the face normal toward the sun, any hit
__global__ void __launch_bounds__(kTraceBlock) k_trace_shadow(DagView g, const PyrRay* rays, const PyrHit* prim,
                                                               float sx, float sy, float sz, uint32_t* out,
                                                               uint32_t count, uint32_t per_wave) {
    const uint32_t i = shared_ray(per_wave);
    if (i >= count) return;
    const PyrHit h = prim[i];
    if (h.instance == PYR_NO_HIT) {
        if (own_lane(per_wave)) out[i] = 0xFFFFFFFFu;
        return;
    }
    const PyrRay r = rays[i];
    const uint32_t face = h.meta & PYR_HIT_FACE_MASK, axis = face >> 1;
    const float sign = (face & 1u) ? -1.0f : 1.0f;
    float o[3];
    const float d[3] = {sx, sy, sz};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float nrm = (uint32_t)a == axis ? sign : 0.0f;
        o[a] = r.origin[a] + r.direction[a] * h.t + nrm * 1e-3f;
    }
    DagHitD sh;
    const uint32_t dark = walk<false>(g, o, d, 0.0f, PYR_FLT_MAX, false, s_stk + threadIdx.x, &sh) ? 1u : 0u;
    if (own_lane(per_wave)) out[i] = dark;
}

// Rays of a wave: 64, halved while that makes at most `waves` waves of `count`
// rays.
uint32_t rays_per_wave(uint64_t count, uint32_t waves) {
    uint32_t p = kWave;
    while (p > 1 && count * 2 <= (uint64_t)waves * p) p /= 2;
    return p;
}
dim3 ray_grid(uint32_t count, uint32_t per_wave) {
    const uint32_t per_block = per_wave * (kTraceBlock / kWave);
    return dim3((uint32_t)(((uint64_t)count + per_block - 1) / per_block));
}
// tile of a frame's waves: 16 x 4 pixels, halved in turn down to one
uint32_t frame_tile(uint32_t width, uint32_t height, uint32_t waves) {
    const uint32_t p = rays_per_wave((uint64_t)width * height, waves);
    const uint32_t bits = (uint32_t)__builtin_ctz(p);
    const uint32_t ty = bits / 2 < 2 ? bits / 2 : 2;
    return (bits - ty) | (ty << 8);
}
dim3 frame_grid(uint32_t width, uint32_t height, uint32_t tile) {
    const uint32_t w = 1u << (tile & 0xFFu), h = (kTraceBlock / kWave) << (tile >> 8);
    return dim3((width + w - 1) / w, (height + h - 1) / h);
}

DagView view_of(const PyrhipDag& d) {
    DagView g;
    g.nodes = (Words)(uintptr_t)d.nodes;
    g.leaves = (Masks)(uintptr_t)d.leaves;
    g.attrs = (Words)(uintptr_t)d.attrs;
    g.palette = d.attrs ? (Words)(uintptr_t)d.palette : nullptr;
    g.root = d.root;
    g.log2_size = d.log2_size;
    g.default_attribute = d.default_attribute;
    g.attr_base = 0;
    return g;
}

PyrResult launch_trace_scene(const PyrScene* scene_dev, uint64_t rays, uint64_t hits, uint32_t count,
                             uint32_t ray_mask, uint32_t flags, uint32_t levels, uint32_t instances, bool skipping,
                             hipStream_t s) {
    if (count == 0) return PYR_OK;
    if (levels < 3 || levels > kMaxLevels) return fail(PYR_ERROR_INVALID_ARGUMENT, "scene levels %u", levels);
    const uint32_t per_wave = rays_per_wave(count, instances < kCullInstances ? kRayWaves : kSceneWaves);
    const dim3 grid = ray_grid(count, per_wave);
    if (flags & PYR_TRACE_EXTENDED) {
        if (skipping)
            hipLaunchKernelGGL(k_trace_scene_ex<true>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev,
                               (const PyrRay*)(uintptr_t)rays, (PyrHitEx*)(uintptr_t)hits, count, ray_mask, flags,
                               levels, per_wave);
        else
            hipLaunchKernelGGL(k_trace_scene_ex<false>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev,
                               (const PyrRay*)(uintptr_t)rays, (PyrHitEx*)(uintptr_t)hits, count, ray_mask, flags,
                               levels, per_wave);
    } else if (skipping)
        hipLaunchKernelGGL(k_trace_scene<true>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev,
                           (const PyrRay*)(uintptr_t)rays, (PyrHit*)(uintptr_t)hits, count, ray_mask, flags, levels, per_wave);
    else
        hipLaunchKernelGGL(k_trace_scene<false>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev,
                           (const PyrRay*)(uintptr_t)rays, (PyrHit*)(uintptr_t)hits, count, ray_mask, flags, levels, per_wave);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "trace launch: %s", hipGetErrorString(e));
}

PyrResult launch_render_scene(const PyrScene* scene_dev, const PyrCamera& cam, const float* w2v_dev, uint64_t hits,
                              uint64_t depth, uint32_t ray_mask, uint32_t flags, uint32_t levels, uint32_t instances,
                              bool skipping,
                              hipStream_t s) {
    if (levels < 3 || levels > kMaxLevels) return fail(PYR_ERROR_INVALID_ARGUMENT, "scene levels %u", levels);
    const uint32_t tile = frame_tile(cam.width, cam.height, instances < kCullInstances ? kRayWaves : kSceneWaves);
    const dim3 grid = frame_grid(cam.width, cam.height, tile);
    if (skipping)
        hipLaunchKernelGGL(k_render_scene<true>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev, cam,
                           w2v_dev, (PyrHit*)(uintptr_t)hits, (float*)(uintptr_t)depth, ray_mask, flags, levels, tile);
    else
        hipLaunchKernelGGL(k_render_scene<false>, grid, dim3(kTraceBlock), stack_bytes(levels), s, scene_dev, cam,
                           w2v_dev, (PyrHit*)(uintptr_t)hits, (float*)(uintptr_t)depth, ray_mask, flags, levels, tile);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "render launch: %s", hipGetErrorString(e));
}

}  // namespace pyr

using namespace pyr;

extern "C" {

PYR_API PyrResult pyrhip_trace_dag(const PyrhipDag* dag, uint64_t rays, uint64_t hits, uint32_t count,
                                   uint32_t flags, void* stream) {
    diag_clear();
    if (!dag || (count && (!rays || !hits))) return fail(PYR_ERROR_INVALID_ARGUMENT, "null argument");
    if (dag->log2_size < 3 || dag->log2_size > 20) return fail(PYR_ERROR_INVALID_ARGUMENT, "log2_size");
    if (count == 0) return PYR_OK;
    const uint32_t per_wave = rays_per_wave(count, kRayWaves);
    hipLaunchKernelGGL(k_trace_dag, ray_grid(count, per_wave), dim3(kTraceBlock),
                       stack_bytes(dag->log2_size), (hipStream_t)stream, view_of(*dag), (const PyrRay*)(uintptr_t)rays, (PyrHit*)(uintptr_t)hits,
                       count, flags, per_wave);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "trace launch: %s", hipGetErrorString(e));
}

PYR_API PyrResult pyrhip_trace_camera(const PyrhipDag* dag, const PyrCamera* camera, uint64_t hits, uint32_t flags,
                                      void* stream) {
    diag_clear();
    if (!dag || !camera || !hits) return fail(PYR_ERROR_INVALID_ARGUMENT, "null argument");
    if (dag->log2_size < 3 || dag->log2_size > 20) return fail(PYR_ERROR_INVALID_ARGUMENT, "log2_size");
    if (camera->width == 0 || camera->height == 0) return PYR_OK;
    const uint32_t tile = frame_tile(camera->width, camera->height, kRayWaves);
    hipLaunchKernelGGL(k_trace_camera, frame_grid(camera->width, camera->height, tile), dim3(kTraceBlock), stack_bytes(dag->log2_size), (hipStream_t)stream,
                       view_of(*dag), *camera,
                       (PyrHit*)(uintptr_t)hits, flags, tile);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "trace launch: %s", hipGetErrorString(e));
}

PYR_API PyrResult pyrhip_camera_rays(const PyrCamera* camera, uint64_t rays, void* stream) {
    diag_clear();
    if (!camera || !rays) return fail(PYR_ERROR_INVALID_ARGUMENT, "null argument");
    if (camera->width == 0 || camera->height == 0) return PYR_OK;
    dim3 grid((camera->width + 15) / 16, (camera->height + 7) / 8);
    hipLaunchKernelGGL(k_camera_rays, grid, dim3(kTraceBlock), 0, (hipStream_t)stream, *camera,
                       (PyrRay*)(uintptr_t)rays);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "camera rays: %s", hipGetErrorString(e));
}

PYR_API PyrResult pyrhip_trace_shadow(const PyrhipDag* dag, uint64_t rays, uint64_t hits, const float sun[3],
                                      uint64_t out, uint32_t count, void* stream) {
    diag_clear();
    if (!dag || !sun || (count && (!rays || !hits || !out))) return fail(PYR_ERROR_INVALID_ARGUMENT, "null argument");
    if (dag->log2_size < 3 || dag->log2_size > 20) return fail(PYR_ERROR_INVALID_ARGUMENT, "log2_size");
    if (count == 0) return PYR_OK;
    const uint32_t per_wave = rays_per_wave(count, kRayWaves);
    hipLaunchKernelGGL(k_trace_shadow, ray_grid(count, per_wave), dim3(kTraceBlock),
                       stack_bytes(dag->log2_size), (hipStream_t)stream, view_of(*dag), (const PyrRay*)(uintptr_t)rays,
                       (const PyrHit*)(uintptr_t)hits, sun[0], sun[1], sun[2], (uint32_t*)(uintptr_t)out, count,
                       per_wave);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PYR_OK : fail(PYR_ERROR_CUDA, "trace launch: %s", hipGetErrorString(e));
}

}  // extern "C"
