// dense.h - kernels of the dense build: single builds of small grids.
//
// A grid of edge up to 2^7 has few enough voxels that a table with a word for
// each of them, indexed by key, replaces the sort: one atomic max per record
// finds the last record of every key (the one that wins, as in the bucket
// finish), and a pass over the table in key order gives the unique voxels and
// the brick masks. The node levels work on dense arrays too: the children of
// cell c of a level are cells 8c .. 8c + 7 of the level below, so a parent
// gathers them without searching, and equal nodes have equal child references.
// Cell order is Morton order, so owners (smallest cell with a mask or a node)
// and positions come out as in the general build: same arrays, bit for bit.
//
// The general build of such a grid is bound by its 17 launches and the
// dependent steps inside them, not by its bytes; this one takes four
// (2^6 and below) or seven. Whole calls: 7179 voxels of a 2^5 model 267 -> 73 us,
// a 2^6 terrain chunk of 1.4e5 310 -> 74 us, 311 edits of a 2^7 chunk of 9.9e5
// 469 -> 112 us. The upper levels of every other build run on the same dense
// kernels (k_dense_spread lays a general level out by cell).
#pragma once
#include "common.h"
#include "dense_walk.h"

namespace pyr {

constexpr uint32_t kDenseTile = 64;          // bricks per workgroup round of k_dense_voxels
constexpr uint32_t kDenseTop = 4096;         // cells that k_dense_top takes (its LDS arrays)
constexpr uint32_t kDenseTopBlock = 1024;
constexpr uint32_t kDenseTopHash = 1024;     // slots for its at most kDenseTop / 8 nodes of a level
constexpr uint32_t kNoRef = 0xFFFFFFFFu;     // reference of an empty cell

// Zeroed before the build: counters, the look-back words, the voxel table and
// the hash tables (owners are kept as the largest complement of an index, so
// zero is "none" for them as well).
struct DenseArgs {
    const uint64_t* old_keys;
    const uint32_t* old_vals;
    uint32_t n_old;
    const int4* voxels;
    uint32_t n_new;
    uint32_t log2_size;
    uint32_t bricks;          // 8^(log2_size - 2)
    uint32_t* counters;
    uint64_t* status;         // look-back words of each scan launch in turn
    uint32_t* table;          // [64 * bricks] index + 1 of the last record of a voxel
    uint64_t* leaf_table;     // distinct masks
    uint32_t* leaf_owner;     // ~(smallest brick with that mask)
    uint32_t leaf_cap;        // power of two
    uint64_t* mask;           // [bricks]
    uint32_t* slot;           // [bricks] slot of the mask in leaf_table
    uint64_t* keys;           // outputs: unique voxels
    uint32_t* attrs;
    uint32_t n_cap;
};

// a level's cells: representative, reference of each representative, voxels
struct DenseLevel {
    uint32_t* rep;
    uint32_t* pos;
    uint32_t* count;
};

__global__ void __launch_bounds__(kBlock) k_dense_clear(uint4* p, uint64_t n) {
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// Records are taken last first: a record whose voxel already has a later one
// (the table is read before the atomic; a stale word is only smaller) does
// nothing, so many records of one voxel cost few atomics on its word.
constexpr int kDenseUnroll = 4;
__global__ void __launch_bounds__(kBlock) k_dense_scatter(DenseArgs a) {
    const uint32_t n = a.n_old + a.n_new, stride = gridDim.x * kBlock;
    const int32_t edge = 1 << a.log2_size;
    const uint64_t slots = (uint64_t)a.bricks * 64;
    for (DenseWalk w(blockIdx.x * kBlock + threadIdx.x, stride, n); w.more(); w.next(kDenseUnroll)) {
        uint64_t key[kDenseUnroll];
#pragma unroll
        for (int u = 0; u < kDenseUnroll; u++) {
            key[u] = ~0ull;
            if (!w.has(u)) continue;
            const uint32_t i = w.record(u);
            if (i < a.n_old) {
                key[u] = a.old_keys[i];
            } else {
                const int4 v = a.voxels[i - a.n_old];
                if (v.x >= 0 && v.y >= 0 && v.z >= 0 && v.x < edge && v.y < edge && v.z < edge)
                    key[u] = local_key((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z);
            }
        }
#pragma unroll
        for (int u = 0; u < kDenseUnroll; u++) {
            if (key[u] >= slots) continue;  // out of range, or past the last record
            const uint32_t i = w.record(u);
            if (a.table[key[u]] <= i) atomicMax(&a.table[key[u]], i + 1);
        }
    }
}

// One tile of kDenseTile bricks per round, a wave per 16 bricks, a lane per
// voxel: the winners' attributes, brick masks by ballot, the masks' slots in
// the leaf table, and one look-back for the tile's first unique position.
__global__ void __launch_bounds__(kBlock) k_dense_voxels(DenseArgs a, uint32_t* tile_ctr, uint32_t epoch, uint32_t c_err,
                                                          uint32_t c_unique) {
    constexpr uint32_t W = kBlock / kWave, G = kDenseTile / W;
    __shared__ uint32_t s_tile, s_wave[W];
    __shared__ uint64_t s_pre, s_mask[kDenseTile];
    const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
    const uint64_t lt = (1ull << lane) - 1;
    const uint32_t tiles = (a.bricks + kDenseTile - 1) / kDenseTile, hm = a.leaf_cap - 1;
    for (;;) {
        __syncthreads();  // the previous round's LDS use is over
        if (threadIdx.x == 0) s_tile = atomicAdd(tile_ctr, 1u);
        __syncthreads();
        const uint32_t tile = s_tile;
        if (tile >= tiles) break;
        const uint32_t b0 = tile * kDenseTile + wave * G;
        uint32_t idx[G], at[G];
#pragma unroll
        for (uint32_t q = 0; q < G; q++) idx[q] = b0 + q < a.bricks ? a.table[(uint64_t)(b0 + q) * 64 + lane] : 0u;
#pragma unroll
        for (uint32_t q = 0; q < G; q++) {
            at[q] = 0;
            if (idx[q]) {
                const uint32_t i = idx[q] - 1;
                at[q] = i < a.n_old ? a.old_vals[i] : (uint32_t)a.voxels[i - a.n_old].w;
            }
        }
        uint32_t kept = 0;  // of the wave
#pragma unroll
        for (uint32_t q = 0; q < G; q++) {
            const uint64_t m = __ballot(at[q] != 0);
            kept += (uint32_t)__popcll(m);
            if (lane == 0) s_mask[wave * G + q] = m;
        }
        if (lane == 0) s_wave[wave] = kept;
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t w = 0; w < W; w++) {
            before += w < wave ? s_wave[w] : 0u;
            total += s_wave[w];
        }
        if (wave == 0) {
            const uint64_t p = lookback_wave(a.status, tile, total, epoch, &a.counters[c_err]);
            if (lane == 0) s_pre = p;
        } else if (wave == 1) {
            // a lane per brick: the mask's slot; lanes with the first lane's
            // mask share its insert (solid regions hold one mask)
            const uint32_t b = tile * kDenseTile + lane;
            const uint64_t m = b < a.bricks ? s_mask[lane] : 0;
            if (b < a.bricks) a.mask[b] = m;
            if (m) {
                const uint64_t m0 = first_lane64(m);
                const uint32_t l0 = first_lane32(lane);
                uint32_t h = (uint32_t)mix64(m) & hm;
                if (m != m0 || lane == l0) {
                    for (uint32_t probes = 0;; h = (h + 1) & hm) {
                        uint64_t cur = load_agent(&a.leaf_table[h]);
                        if (cur == 0) cur = atomicCAS((unsigned long long*)&a.leaf_table[h], 0ull, (unsigned long long)m);
                        if (cur == 0 || cur == m) break;
                        if (++probes > a.leaf_cap) {
                            atomicOr(&a.counters[c_err], 4u);
                            break;
                        }
                    }
                    if (load_agent(&a.leaf_owner[h]) < ~b) atomicMax(&a.leaf_owner[h], ~b);
                }
                const uint32_t h0 = first_lane32(h);
                a.slot[b] = m == m0 ? h0 : h;
            }
        }
        __syncthreads();
        uint64_t pos = s_pre + before;
        if (s_pre + total > a.n_cap) {  // only after a failed look-back
            if (threadIdx.x == 0) atomicOr(&a.counters[c_err], 16u);
            continue;
        }
#pragma unroll
        for (uint32_t q = 0; q < G; q++) {
            const uint64_t m = s_mask[wave * G + q];
            if ((m >> lane) & 1) {
                const uint64_t at_pos = pos + __popcll(m & lt);
                a.keys[at_pos] = ((uint64_t)(b0 + q) << 6) | lane;
                a.attrs[at_pos] = at[q];
            }
            pos += __popcll(m);
        }
        if (tile == tiles - 1 && threadIdx.x == 0) a.counters[c_unique] = (uint32_t)(s_pre + total);
    }
}

// Owners' masks become leaves in brick order (grids of more than kDenseTop
// bricks; smaller ones leave this to k_dense_top).
constexpr int kDenseItems = 8;
__global__ void __launch_bounds__(kBlock) k_dense_leaves(DenseArgs a, DenseLevel lv, uint64_t* leaves_out,
                                                          uint64_t* status, uint32_t* tile_ctr, uint32_t epoch,
                                                          uint32_t c_err, uint32_t c_leaves) {
    constexpr uint32_t T = kBlock * kDenseItems;
    __shared__ uint32_t s_tile, s_wave[kBlock / kWave];
    __shared__ uint64_t s_pre;
    const uint32_t lane = lane_id(), wave = threadIdx.x / kWave, tiles = (a.bricks + T - 1) / T;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_tile = atomicAdd(tile_ctr, 1u);
        __syncthreads();
        const uint32_t tile = s_tile;
        if (tile >= tiles) break;
        uint32_t f[kDenseItems], e[kDenseItems], o[kDenseItems];
        uint64_t m[kDenseItems];
        auto brick = [&](int i) { return tile * T + wave * kWave * kDenseItems + (uint32_t)i * kWave + lane; };
#pragma unroll
        for (int i = 0; i < kDenseItems; i++) {
            const uint32_t b = brick(i);
            m[i] = b < a.bricks ? a.mask[b] : 0;
            o[i] = m[i] ? ~a.leaf_owner[a.slot[b]] : 0u;
            f[i] = m[i] && o[i] == b;
        }
        const uint32_t total = tile_scan<kDenseItems>(f, e, s_wave);
        if (wave == 0) {
            const uint64_t p = lookback_wave(status, tile, total, epoch, &a.counters[c_err]);
            if (lane == 0) s_pre = p;
        }
        __syncthreads();
        if (s_pre + total > a.bricks) {  // only after a failed look-back
            if (threadIdx.x == 0) atomicOr(&a.counters[c_err], 16u);
            continue;
        }
#pragma unroll
        for (int i = 0; i < kDenseItems; i++) {
            const uint32_t b = brick(i);
            if (b >= a.bricks) continue;
            lv.count[b] = (uint32_t)__popcll(m[i]);
            lv.rep[b] = o[i];
            if (f[i]) {
                leaves_out[s_pre + e[i]] = m[i];
                lv.pos[b] = (uint32_t)s_pre + e[i];
            }
        }
        if (tile == tiles - 1 && threadIdx.x == 0) a.counters[c_leaves] = (uint32_t)s_pre + total;
    }
}

// The eight child references of cell p of the level above lv, and their voxels.
__device__ __forceinline__ uint32_t dense_children(const DenseLevel& lv, uint32_t p, uint32_t (&ref)[8]) {
    uint32_t cnt[8], rep[8], total = 0;
    *(uint4*)&cnt[0] = ((const uint4*)lv.count)[p * 2];
    *(uint4*)&cnt[4] = ((const uint4*)lv.count)[p * 2 + 1];
    *(uint4*)&rep[0] = ((const uint4*)lv.rep)[p * 2];
    *(uint4*)&rep[4] = ((const uint4*)lv.rep)[p * 2 + 1];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        ref[q] = cnt[q] ? lv.pos[rep[q]] : kNoRef;
        total = sat_add(total, cnt[q]);
    }
    return total;
}

__device__ __forceinline__ uint64_t dense_hash(const uint32_t (&ref)[8]) {
    uint64_t h = 0;
#pragma unroll
    for (int q = 0; q < 8; q += 2) h = mix64(h ^ ((uint64_t)ref[q] << 32 | ref[q + 1]));
    return h;
}

// Chunks of a batch: cell c << 3 (log2_size - lv) is the first of chunk c on
// level lv. A chunk of edge 2^lv ends there: that cell is its root.
struct DenseChunks {
    const uint8_t* log2;      // per chunk, null: all of log2_size
    uint32_t* roots;          // null: a single build
    uint32_t count, log2_size;
};

// The elements of a general level (compact, by key) into cells whose counts
// are zero: their references, each representing itself.
__global__ void __launch_bounds__(kBlock) k_dense_spread(const uint32_t* counters, uint32_t count_slot, uint32_t cap,
                                                          const uint64_t* key, const uint32_t* rep, const uint32_t* pos,
                                                          const uint32_t* count, DenseLevel to, uint32_t cells,
                                                          uint32_t* err) {
    const uint32_t n = min(counters[count_slot], cap), stride = gridDim.x * kBlock;
    for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        const uint64_t c = key[i];
        if (c >= cells) {  // only after a failed look-back
            atomicOr(err, 16u);
            continue;
        }
        to.rep[c] = (uint32_t)c;
        to.pos[c] = pos[rep[i]];
        to.count[c] = count[i];
    }
}

// Parents of level lv's cells into the level's hash: equal child references
// are an equal node.
__global__ void __launch_bounds__(kBlock) k_dense_insert(DenseLevel ch, uint32_t lv, DenseChunks chunks, uint32_t parents,
                                                          uint32_t* table, uint32_t* owner, uint32_t cap, uint32_t* slot,
                                                          uint32_t* count, uint32_t* err) {
    const uint32_t hm = cap - 1, p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= parents) return;
    uint32_t ref[8];
    uint32_t total = dense_children(ch, p, ref);
    if (chunks.log2) {
        const uint32_t shift = 3 * (chunks.log2_size - lv - 1), c = p >> shift;
        const uint32_t edge = chunks.log2[c];
        if (edge <= lv) {
            if (edge == lv && p == c << shift && total) chunks.roots[c] = ref[0];
            total = 0;
        }
    }
    count[p] = total;
    if (!total) return;
    // (lanes with the first lane's node share its insert)
    const uint32_t p0 = first_lane32(p);
    bool same0 = true;
#pragma unroll
    for (int q = 0; q < 8; q++) same0 &= first_lane32(ref[q]) == ref[q];
    uint32_t h = (uint32_t)dense_hash(ref) & hm;
    if (!same0 || p == p0) {
        for (uint32_t probes = 0;; h = (h + 1) & hm) {
            uint32_t cur = load_agent(&table[h]);
            if (cur == 0) cur = atomicCAS(&table[h], 0u, p + 1);
            if (cur == 0 || cur == p + 1) break;
            uint32_t other[8];
            (void)dense_children(ch, cur - 1, other);
            bool same = true;
#pragma unroll
            for (int q = 0; q < 8; q++) same &= other[q] == ref[q];
            if (same) break;
            if (++probes > cap) {
                atomicOr(err, 8u);
                break;
            }
        }
        if (load_agent(&owner[h]) < ~p) atomicMax(&owner[h], ~p);
    }
    const uint32_t h0 = first_lane32(h);
    slot[p] = same0 ? h0 : h;
}

__device__ __forceinline__ uint32_t dense_words(const uint32_t (&ref)[8], uint32_t* mask) {
    uint32_t m = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) m |= ref[q] != kNoRef ? 1u << q : 0u;
    *mask = m;
    return 2 + (uint32_t)__popc(m);
}
__device__ __forceinline__ void dense_store(uint32_t* dst, const uint32_t (&ref)[8], uint32_t mask, uint32_t total) {
    dst[0] = mask;
    dst[1] = total;
    uint32_t k = 2;
#pragma unroll
    for (int q = 0; q < 8; q++)
        if (ref[q] != kNoRef) dst[k++] = ref[q];
}

// Owners' words at the level's cursor, in cell order.
__global__ void __launch_bounds__(kBlock) k_dense_compact(DenseLevel ch, DenseLevel par, uint32_t parents,
                                                           const uint32_t* owner, const uint32_t* slot,
                                                           uint32_t* nodes_out, uint64_t word_cap, uint64_t* status,
                                                           uint32_t* tile_ctr, uint32_t epoch, uint32_t* cursor,
                                                           uint32_t* err) {
    __shared__ uint32_t s_tile, s_wave[kBlock / kWave];
    __shared__ uint64_t s_pre;
    const uint32_t tiles = (parents + kBlock - 1) / kBlock, cur = cursor[0];
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_tile = atomicAdd(tile_ctr, 1u);
        __syncthreads();
        const uint32_t tile = s_tile;
        if (tile >= tiles) break;
        const uint32_t p = tile * kBlock + threadIdx.x;
        uint32_t f[1] = {0}, e[1], o = 0, ref[8], mask = 0, total = 0;
        if (p < parents && par.count[p]) {
            o = ~owner[slot[p]];
            if (o == p) {
                total = dense_children(ch, p, ref);
                f[0] = dense_words(ref, &mask);
            }
        }
        const uint32_t sum = tile_scan<1>(f, e, s_wave);
        if (threadIdx.x < kWave) {
            const uint64_t x = lookback_wave(status, tile, sum, epoch, err);
            if (threadIdx.x == 0) s_pre = x;
        }
        __syncthreads();
        const uint64_t at = cur + s_pre + e[0];
        if (p < parents) par.rep[p] = o;
        if (f[0]) {
            if (at + f[0] > word_cap) {  // only after a failed look-back
                atomicOr(err, 16u);
            } else {
                dense_store(nodes_out + at, ref, mask, total);
                par.pos[p] = (uint32_t)at;
            }
        }
        if (tile == tiles - 1 && threadIdx.x == 0) cursor[1] = cur + (uint32_t)(s_pre + sum);
    }
}

__device__ __forceinline__ uint32_t dense_block_scan(uint32_t v, uint32_t* s_wave, uint32_t* total) {
    constexpr uint32_t W = kDenseTopBlock / kWave;
    const uint32_t lane = lane_id(), wave = threadIdx.x / kWave, inc = wave_inclusive_scan(v);
    if (lane == kWave - 1) s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0, t = 0;
#pragma unroll
    for (uint32_t q = 0; q < W; q++) {
        const uint32_t x = s_wave[q];
        before += q < wave ? x : 0u;
        t += x;
    }
    __syncthreads();  // s_wave is written again by the next scan
    *total = t;
    return before + inc - v;
}

// The levels from at most kDenseTop cells up to the root in one workgroup, all
// of its arrays in LDS, and with `bricks` set (lv = 2) the leaves before them.
// Ends with the counters of the finished build.
__global__ void __launch_bounds__(kDenseTopBlock) k_dense_top(DenseArgs a, DenseLevel from, uint32_t lv, uint32_t bricks,
                                                               DenseChunks chunks, uint64_t* leaves_out, uint32_t* nodes_out,
                                                               uint64_t word_cap, const uint32_t* cursor, uint32_t c_err,
                                                               uint32_t c_unique, uint32_t c_leaves, uint32_t c_root,
                                                               uint32_t c_words, uint32_t counts, uint32_t* host) {
    __shared__ uint32_t s_ref[kDenseTop], s_cnt[kDenseTop];
    __shared__ uint32_t s_pos[kDenseTop];
    __shared__ uint32_t s_hash[kDenseTopHash], s_owner[kDenseTopHash];
    __shared__ uint32_t s_wave[kDenseTopBlock / kWave];
    const uint32_t tid = threadIdx.x;
    uint32_t cells = chunks.count << (3 * (a.log2_size - lv));
    uint32_t cur = 0;
    if (bricks) {
        uint32_t base = 0;
        for (uint32_t b0 = 0; b0 < cells; b0 += kDenseTopBlock) {
            const uint32_t b = b0 + tid;
            const uint64_t m = b < cells ? a.mask[b] : 0;
            const uint32_t o = m ? ~a.leaf_owner[a.slot[b]] : kNoRef;
            const uint32_t f = m && o == b;
            uint32_t total;
            const uint32_t e = dense_block_scan(f, s_wave, &total);
            if (b < cells) {
                s_ref[b] = o;
                s_cnt[b] = (uint32_t)__popcll(m);
                if (f) {
                    s_pos[b] = base + e;
                    leaves_out[base + e] = m;
                }
            }
            base += total;
        }
        if (tid == 0) a.counters[c_leaves] = base;
    } else {
        cur = *cursor;
        for (uint32_t b = tid; b < cells; b += kDenseTopBlock) {
            s_cnt[b] = from.count[b];
            s_ref[b] = from.count[b] ? from.rep[b] : kNoRef;
            s_pos[b] = from.pos[b];
        }
    }
    __syncthreads();
    // representatives to references
    for (uint32_t b = tid; b < cells; b += kDenseTopBlock) s_ref[b] = s_ref[b] != kNoRef ? s_pos[s_ref[b]] : kNoRef;
    for (; lv < a.log2_size; lv++) {
        __syncthreads();
        if (chunks.log2) {  // chunks that end on this level
            for (uint32_t c = tid; c < chunks.count; c += kDenseTopBlock) {
                const uint32_t first = c << (3 * (a.log2_size - lv));
                if (chunks.log2[c] == lv && s_cnt[first]) {
                    chunks.roots[c] = s_ref[first];
                    s_cnt[first] = 0;
                    s_ref[first] = kNoRef;
                }
            }
        }
        cells >>= 3;  // parents: at most kDenseTop / 8, one per thread
        for (uint32_t i = tid; i < kDenseTopHash; i += kDenseTopBlock) {
            s_hash[i] = 0;
            s_owner[i] = 0;
        }
        __syncthreads();
        uint32_t ref[8], total = 0, h = 0;
        const uint32_t p = tid;
        if (p < cells) {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                ref[q] = s_ref[p * 8 + q];
                total = sat_add(total, s_cnt[p * 8 + q]);
            }
            if (total) {
                // (at most 512 nodes in 1024 slots: a free one is always found)
                h = (uint32_t)dense_hash(ref) & (kDenseTopHash - 1);
                for (uint32_t probes = 0; probes < kDenseTopHash; probes++, h = (h + 1) & (kDenseTopHash - 1)) {
                    const uint32_t seen = atomicCAS(&s_hash[h], 0u, p + 1);
                    if (seen == 0) break;
                    bool same = true;
#pragma unroll
                    for (int q = 0; q < 8; q++) same &= s_ref[(seen - 1) * 8 + q] == ref[q];
                    if (same) break;
                }
                atomicMax(&s_owner[h], ~p);
            }
        }
        __syncthreads();
        uint32_t o = kNoRef, words = 0, mask = 0, sum;
        if (total) {
            o = ~s_owner[h];
            const uint32_t w = dense_words(ref, &mask);
            if (o == p) words = w;
        }
        const uint32_t e = dense_block_scan(words, s_wave, &sum);
        if (words) {
            if ((uint64_t)cur + e + words > word_cap) atomicOr(&a.counters[c_err], 16u);
            else dense_store(nodes_out + cur + e, ref, mask, total);
            s_pos[p] = cur + e;
        }
        __syncthreads();
        if (p < cells) {
            s_ref[p] = total ? s_pos[o] : kNoRef;
            s_cnt[p] = total;
        }
        cur += sum;
        __syncthreads();
    }
    // roots of the chunks of the largest edge; the build's own is the first of
    // them that is not empty
    __syncthreads();
    if (tid == 0) s_pos[0] = kNoRef;
    __syncthreads();
    for (uint32_t c = tid; c < chunks.count; c += kDenseTopBlock) {
        if (!s_cnt[c]) continue;
        if (chunks.roots) chunks.roots[c] = s_ref[c];
        atomicMin(&s_pos[0], c);
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t root = s_pos[0] != kNoRef ? s_ref[s_pos[0]] : 0;
        if (a.counters[c_unique] == 0 && cur + 2ull <= word_cap) {  // the empty geometry: a node without children
            nodes_out[cur] = 0;
            nodes_out[cur + 1] = 0;
            root = cur;
            cur += 2;
        }
        a.counters[c_root] = root;
        a.counters[c_words] = cur;
    }
    // counters, roots and first voxels into the caller's pinned words
    __syncthreads();
    for (uint32_t i = tid; i < counts; i += kDenseTopBlock) host[i] = a.counters[i];
    if (chunks.roots)
        for (uint32_t i = tid; i < 2 * chunks.count; i += kDenseTopBlock) host[counts + i] = chunks.roots[i];
}

}  // namespace pyr
