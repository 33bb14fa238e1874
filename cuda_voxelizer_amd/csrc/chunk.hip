// chunk.hip -- single-pass surface voxelization with LDS word merging.
//
// One workgroup takes a chunk of 256 consecutive triangles; the fewer chunks
// share a table word, the fewer atomics, so a mesh whose consecutive
// triangles lie close together voxelizes fastest (its chunks are compact
// patches; input order is kept as given).  Each lane loads and rasterizes
// its own triangle (ZX edges once per z slice, then per row the YZ edges
// and, at the x that passed ZX, the plane and XY edges) and ORs the passing
// bits into an LDS hash table keyed by table word, so bits that several
// triangles of the chunk set in one word are merged before memory is
// touched.  Triangles with a large voxel box (or one far larger than the rest
// of their wave's) are queued; afterwards the workgroup deals their rows over
// its lanes and ORs each row's interval (rows.h).  The table is then updated with
// one non-returning global atomicOr per distinct word; words that do not fit
// in the hash go straight to global atomics.  The table is zero-filled
// beforehand (unless accumulating), or the words go to a zeroed scratch table in
// blocked order, from which the table is then written.
//
// Blocked order: a memory atomic costs the same whatever it hits (26 G/s on
// scattered words, in 256 KB as in 1 GB; plain stores do 70 to 190 G/s), but
// neighbouring lanes with words of one 64-byte line are one request.  In a
// linear table such a line is 512 voxels of one row, of which a surface has one
// or two; a blocked line is a word of 4 x 4 rows (32 x 4 x 4 voxels), so a
// triangle's rows share two or three lines.
#include "jobs.h"
#include "raster.h"
#include "region.h"
#include "rows.h"
#include "scratch.h"
#include "vox_kernels.h"

#pragma clang fp contract(off)

namespace voxamd {

constexpr int kChunk = 256;  // triangles per workgroup (one per lane)
constexpr int kHashBits = 11;
constexpr int kHashCap = 1 << kHashBits;
constexpr uint32_t kEmpty = 0xFFFFFFFFu;
// Slots tried before a word goes straight to memory: a chunk of scattered
// triangles has more distinct words than slots, and probing a full table costs
// more than the atomic it would save.
constexpr int kProbes = 2;
constexpr int kBigVox = 256;    // voxel boxes above this (or wider than 32 in x) are queued
// ...and, with the built-in setting, boxes of more than kRowsFloor rows and
// more than kRowsRatio times the mean of their wave's boxes: one lane walking
// a box far larger than its neighbours' holds up the whole workgroup.  The
// Stanford bunny at 64^3 (5,110 triangles, 20 workgroups): the median
// workgroup's largest lane box has 40 rows against a mean of 7.4; queuing
// those 1.7 % of triangles halves it.  The icospheres, tori and displaced
// spheres of the benchmarks have no box above the floor, so their waves skip
// the rule after one ballot.
constexpr int kRowsFloor = 16;
constexpr int kRowsRatio = 3;
constexpr int kRecs = 20;       // queued triangles whose records are in LDS at once (26 KB of LDS in all: six
                                // workgroups per CU)

struct ChunkShared {
    uint32_t keys[kHashCap];
    uint32_t vals[kHashCap];
    uint32_t nbig[2][kChunk / 64];  // queued triangles per wave, of an even and an odd chunk
    union {
        BlockRows<kRecs, kChunk / 64> rows;  // queued triangles
        RegionFlushShared flush;             // last: grouping of the region algorithm's pairs
    };
};

// A word's bits into the table; kSpecFlagged: the flags that say which 256 bytes
// of the scratch table hold any come before it.
template <int SPEC>
__device__ __forceinline__ void memory_or(uint32_t* __restrict__ table, uint32_t key, uint32_t mask) {
    if (SPEC == kSpecFlagged) *((uint8_t*)table - 1 - (key >> 6)) = 1;
    atomicOr(table + key, mask);
}

// ident: the slot is the key modulo kHashCap.  Used when the whole table has
// at most kHashCap words (its slots are preset to their keys, so every word is
// found at its first probe) and for Morton keys (a chunk's words are a compact
// range of brick codes); linear keys repeat modulo the table size with the z
// stride, so they are hashed multiplicatively.
// REG (region algorithm): more slots are tried, and a word that finds none is
// staged as a fallback pair instead of going to the table.
// BLK (blocked keys): the 16 words of a key's line take the slots of one group of
// 16, in order, so that the flush finds them in neighbouring lanes; a word
// whose slot another line's word has moves on by whole groups.
template <bool REG, int SPEC>
__device__ __forceinline__ void word_or(ChunkShared& S, uint32_t* __restrict__ table, bool ident, uint32_t key,
                                        uint32_t mask, const RegionArgs& RA) {
    constexpr bool BLK = SPEC >= kSpecBlocked;
    uint32_t h = BLK     ? ((((key >> 4) * 2654435761u) >> (32 - (kHashBits - 4))) << 4) | (key & 15u)
                 : ident ? (key & (kHashCap - 1))
                         : (key * 2654435761u) >> (32 - kHashBits);
#pragma unroll 1
    for (int probe = 0; probe < (REG ? kRegionProbes : kProbes); probe++) {
        // one round trip: the CAS claims an empty slot or returns the key
        // already there (a read first, then a CAS on empty slots, took two for
        // every new word: 1024^3 linear torus 114 vs 108 us per call)
        const uint32_t k = atomicCAS(&S.keys[h], kEmpty, key);
        if (k == kEmpty || k == key) {
            atomicOr(&S.vals[h], mask);
            return;
        }
        h = (h + (BLK ? 16u : 1u)) & (kHashCap - 1);
    }
    if (REG)
        region_fallback(RA.P, RA.W, key, mask);
    else
        memory_or<SPEC>(table, key, mask);  // hash table crowded: go to memory directly
}

// Passing voxels of row (y, z) as a mask (bit k = voxel cx + k, cx a multiple
// of 32) -> hash, keyed by table word (REG, linear layout: by region row key).
// SPEC: what is known of every job at compile time (see ChunkSpec).
template <bool REG, int SPEC>
__device__ __forceinline__ void emit_mask(ChunkShared& S, uint32_t* __restrict__ table, bool ident,
                                          const vox_info& info, int layout, int cx, int y, int z, uint32_t mask,
                                          const RegionArgs& RA) {
    if (!mask) return;
    const uint32_t G = info.gridsize[0];
    if (SPEC == kSpecMorton || (SPEC == kSpecAny && layout == VOX_LAYOUT_MORTON)) {
        // codes of grids up to 1024 fit 30 bits: 32-bit spreads
        const uint64_t base = (SPEC == kSpecMorton || G <= 1024u) ? (uint64_t)(spread10((uint32_t)cx) | (spread10((uint32_t)y) << 1) |
                                                      (spread10((uint32_t)z) << 2))
                                         : morton3((uint32_t)cx, (uint32_t)y, (uint32_t)z);
        const uint32_t yz_low = ((uint32_t)(y & 1) << 1) | ((uint32_t)(z & 1) << 2) | ((uint32_t)((y >> 1) & 1) << 4);
        morton_chunk_words(base, yz_low, mask,
                           [&](uint64_t w, uint32_t bits) { word_or<REG, SPEC>(S, table, ident, (uint32_t)w, bits, RA); });
    } else if (REG) {
        word_or<REG, SPEC>(S, table, ident, region_row_key(RA.P, (uint32_t)cx >> 5, (uint32_t)y, (uint32_t)z),
                     __brev(mask), RA);
    } else if (SPEC >= kSpecBlocked) {
        word_or<REG, SPEC>(S, table, ident, blocked_word(G, (uint32_t)cx >> 5, (uint32_t)y, (uint32_t)z), __brev(mask),
                           RA);
    } else if (SPEC == kSpecLinear || (G & 31u) == 0) {
        // (z G + y) G/32 + cx/32 < G^3/32 < 2^32 (chunk_supported), so 32-bit arithmetic is exact
        const uint32_t w = ((uint32_t)z * G + (uint32_t)y) * (G >> 5) + ((uint32_t)cx >> 5);
        word_or<REG, SPEC>(S, table, ident, w, __brev(mask), RA);
    } else {
        // linear rows not aligned to words: per voxel
        const uint64_t row = (uint64_t)y * G + (uint64_t)z * G * G;
        uint32_t m = mask, cur = kEmpty, bits = 0;
        while (m) {
            const int k = __ffs(m) - 1;
            m &= m - 1;
            const uint64_t idx = row + (uint64_t)(cx + k);
            const uint32_t w = (uint32_t)(idx >> 5);
            if (w != cur) {
                if (bits) word_or<REG, SPEC>(S, table, ident, cur, bits, RA);
                cur = w;
                bits = 0;
            }
            bits |= bit_mask(idx);
        }
        if (bits) word_or<REG, SPEC>(S, table, ident, cur, bits, RA);
    }
}

// A lane's own box (x extent <= 32): the ZX edge tests depend on (z, x) only,
// so they are evaluated once per z slice into a mask over the box's x range;
// a row then tests the XY edges and the plane only at the x that passed ZX.
// Every test is the same binary32 expression as in vox_device.h, evaluated
// for a subset of the voxels: the resulting bits are unchanged.
// SPLIT: 2^lg lanes share the box; lane `sub` of them takes every 2^lg-th row.
template <bool REG, int SPEC, bool SPLIT>
__device__ __forceinline__ void lane_raster(ChunkShared& S, uint32_t* __restrict__ table, bool ident,
                                            const SurfTri& T, const vox_info& info, int layout,
                                            const RegionArgs& RA, int sub, int lg) {
    const float ux = info.unit[0], uy = info.unit[1], uz = info.unit[2];
    const int xa = T.lo[0], xb = T.hi[0];
    const int c0 = xa & ~31, sh = xa - c0;
    // Morton codes of grids up to 1024 fit 30 bits: the x, y and z spreads are
    // computed once per lane, row and slice instead of once per emitted mask
    const bool m32 = SPEC == kSpecMorton ||
                     (SPEC == kSpecAny && layout == VOX_LAYOUT_MORTON && info.gridsize[0] <= 1024u);
    const uint32_t sc0 = m32 ? spread10((uint32_t)c0) : 0u, sc1 = m32 ? spread10((uint32_t)c0 + 32u) : 0u;
    const auto put = [&](uint64_t w, uint32_t bits) { word_or<REG, SPEC>(S, table, ident, (uint32_t)w, bits, RA); };
    const int step = SPLIT ? 1 << lg : 1;
    int ynext = T.lo[1] + (SPLIT ? sub : 0);  // the lane's next row in y
    for (int z = T.lo[2]; z <= T.hi[2]; z++) {
        if (SPLIT && ynext > T.hi[1]) {  // no row of this slice is the lane's
            ynext -= T.hi[1] - T.lo[1] + 1;
            continue;
        }
        const int ybeg = ynext;
        if (SPLIT) ynext += ((T.hi[1] - ybeg) >> lg) * step + step - (T.hi[1] - T.lo[1] + 1);
        const float pz = (float)z * uz;
        float azx[3];
#pragma unroll
        for (int i = 0; i < 3; i++) azx[i] = T.zx.a[i] * pz;
        uint32_t zxm = 0;  // bit i: x = xa + i passes the ZX edges
        for (int x = xa; x <= xb; x++) {
            const float px = (float)x * ux;
            bool ok = true;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                float b = azx[i];
                b = b + T.zx.b[i] * px;
                b = b + T.zx.d[i];
                ok = ok && !(b < 0.0f);
            }
            if (ok) zxm |= 1u << (x - xa);
        }
        if (!zxm) continue;
        const float nzpz = T.n[2] * pz;
        for (int y = SPLIT ? ybeg : T.lo[1]; y <= T.hi[1]; y += step) {
            const float py = (float)y * uy;
            if (!edges_pass(T.yz, py, pz)) continue;
            const float nypy = T.n[1] * py;
            float bxy[3];
#pragma unroll
            for (int i = 0; i < 3; i++) bxy[i] = T.xy.b[i] * py;
            uint32_t m = 0, cand = zxm;
            while (cand) {
                const int k = __ffs(cand) - 1;
                cand &= cand - 1;
                const float px = (float)(xa + k) * ux;
                float t = T.n[0] * px;
                t = t + nypy;
                t = t + nzpz;
                const float r = (t + T.d1) * (t + T.d2);
                bool ok = !(r > 0.0f);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    float a = T.xy.a[i] * px;
                    a = a + bxy[i];
                    a = a + T.xy.d[i];
                    ok = ok && !(a < 0.0f);
                }
                if (ok) m |= 1u << k;
            }
            if (!m) continue;
            const uint64_t M = (uint64_t)m << sh;  // bit k = voxel c0 + k
            if (m32) {
                const uint32_t syz = (spread10((uint32_t)y) << 1) | (spread10((uint32_t)z) << 2);
                const uint32_t yz_low =
                    ((uint32_t)(y & 1) << 1) | ((uint32_t)(z & 1) << 2) | ((uint32_t)((y >> 1) & 1) << 4);
                if ((uint32_t)M) morton_chunk_words(sc0 | syz, yz_low, (uint32_t)M, put);
                if (M >> 32) morton_chunk_words(sc1 | syz, yz_low, (uint32_t)(M >> 32), put);
                continue;
            }
            emit_mask<REG, SPEC>(S, table, ident, info, layout, c0, y, z, (uint32_t)M, RA);
            if (M >> 32) emit_mask<REG, SPEC>(S, table, ident, info, layout, c0 + 32, y, z, (uint32_t)(M >> 32), RA);
        }
    }
}

// Work unit: `span` consecutive chunks of kChunk triangles of one job, merged
// in one LDS table and flushed once -- or one chunk of it.per triangles, each
// shared by 2^it.lg_split lanes (SPLIT; a job of a batch may have none).  With `parts` > 1 the row windows of
// a chunk's queued triangles are shared: the first units (part 0) take every
// parts-th window and the lane rasters, further units one part's windows each.
// MULTI: the job comes from the launch's job map; otherwise it is `one` (kernel
// arguments).
// LOOP: some job has span > 1 (otherwise the chunk loop is compiled out, which
// keeps the register count of the one-chunk form down).  REG: the merged
// words are staged as region pairs (RA) instead of ORed into the table.
// Workgroups per CU: the LDS allows six.  The bound holds the registers at
// five waves per SIMD, or six with WIDE and in a single job's specialised form
// (no spills there), or four for the chunk loop.  SPEC: the layout when it is
// known at compile time, so the other layout's word paths are compiled out (at
// six waves this removes the spills).
template <bool MULTI, bool LOOP, bool WIDE, bool REG, int SPEC = kSpecAny, bool SPLIT = false>
__global__ void __launch_bounds__(kChunk, LOOP ? 4 : (WIDE || (SPEC != kSpecAny && !MULTI) ? 6 : 5))
    surface_chunk_kernel(ItemDev one, ItemMap M, RegionArgs RA) {
    __shared__ ChunkShared S;
    __shared__ BlockJob J;
    uint32_t local = blockIdx.x;
    if (MULTI) {
        resolve_job(one, M, blockIdx.x, J);
        local = J.local;
        if (local == ~0u) return;
    }
    const ItemDev& it = MULTI ? J.it : one;
    const vox_info& info = it.info;
    uint32_t* __restrict__ table = SPEC >= kSpecBlocked ? it.scratch : it.table;
    const int layout = SPEC == kSpecLinear || SPEC >= kSpecBlocked ? (int)VOX_LAYOUT_LINEAR
                       : SPEC == kSpecMorton ? (int)VOX_LAYOUT_MORTON : it.layout;
    const uint64_t n = info.n_triangles;
    const uint32_t parts = it.parts > 1u ? it.parts : 1u;
    const uint32_t span = (!LOOP || parts > 1u) ? 1u : (it.span > 1u ? it.span : 1u);
    // lg: each triangle is shared by 2^lg lanes of a wave
    const int lg = SPLIT ? (int)it.lg_split : 0;
    const uint32_t per = (uint32_t)kChunk >> lg;
    uint32_t part = 0, unit = local;
    if (parts > 1u) {  // in the looping form too: its launch may hold jobs of either kind
        const uint32_t units = (uint32_t)((n + per - 1) >> (8 - lg));
        part = unit / units;
        unit -= part * units;
    }
    const uint64_t begin = (uint64_t)unit * span * per;
    if (begin >= n) return;
    const uint64_t end = n - begin > (uint64_t)span * per ? begin + (uint64_t)span * per : n;
    const uint32_t G = info.gridsize[0];
    const uint64_t words = ((uint64_t)G * G * G + 31) / 32;
    const bool dense = !REG && words <= (uint64_t)kHashCap;  // region keys are not table words
    const bool ident = dense || layout == VOX_LAYOUT_MORTON;
    const int wave = (int)(threadIdx.x >> 6);
    const uint32_t mine = threadIdx.x >> lg;  // the lane's triangle in the chunk
    const int sub = (int)(threadIdx.x & ((1u << lg) - 1u));
    const auto clear = [&]() {
        for (int i = threadIdx.x; i < kHashCap; i += kChunk) {
            S.keys[i] = dense && (uint64_t)i < words ? (uint32_t)i : kEmpty;
            S.vals[i] = 0u;
        }
    };
    if (LOOP || parts == 1u) clear();
    uint64_t first = begin;
    int odd = 0;
    do {
        const uint64_t left = end - first;
        const bool live = mine < left;
        // each lane loads its own triangle: the nine loads of a lane are in
        // flight together and a wave's 2304 bytes are contiguous, so they are
        // served by the cache after the first; staging the chunk through LDS
        // cost a barrier and 9 KB of LDS (512^3 Morton torus 51.2 vs 48.0 us)
        bool big = false;
        int rows = 0;  // rows of a lane-path box
        SurfTri T;
        float v[3][3];
        if (live) {
            load_tri(it.tris, first + mine, info, v);
            surface_box(v, info, T.lo, T.hi);
            const int nx = T.hi[0] - T.lo[0] + 1;
            const int ny = T.hi[1] - T.lo[1] + 1, nz = T.hi[2] - T.lo[2] + 1;
            const int64_t vol = (int64_t)nx * ny * nz;
            big = vol > (it.big ? (int64_t)it.big : (int64_t)kBigVox) || nx > 32;
            // the lane's rows; at most the queue threshold here (<= 2^15): no overflow
            rows = big ? 0 : (ny * nz + (1 << lg) - 1) >> lg;
        }
        if (!it.big && __ballot(rows > kRowsFloor)) {
            // sum over the wave (dead and queued lanes add 0); the mean is
            // taken over the lanes that hold a triangle
            int sum = rows;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
            const int nlive = (int)__popcll(__ballot(live));
            if (rows > kRowsFloor && rows * nlive > kRowsRatio * sum) big = true;
        }
        if (first == begin) {
            if (!LOOP && parts > 1u && !__syncthreads_or(big) && part) return;  // nothing to share
            if (!LOOP && parts > 1u) clear();
        }
        const bool queue = big && (!SPLIT || sub == 0);  // once, whatever lanes share it
        const unsigned long long queued = __ballot(queue);
        if (__lane_id() == 0) S.nbig[odd][wave] = (uint32_t)__popcll(queued);
        __syncthreads();  // every slot is set before any lane inserts into the table; the counts are there
        if (part == 0 && live && !big) {
            surface_setup_tests(v, info, T);  // the box is T's already
            if (SPLIT && (!MULTI || lg))  // nx <= 32 here
                lane_raster<REG, SPEC, SPLIT>(S, table, ident, T, info, layout, RA, sub, lg);
            else
                lane_raster<REG, SPEC, false>(S, table, ident, T, info, layout, RA, 0, 0);
        }
        const auto setup = [&](uint32_t thread, SurfTri& Q) {
            float p[3][3];
            load_tri(it.tris, first + (thread >> lg), info, p);
            surface_setup(p, info, Q);
        };
        block_rows(S.rows, S.nbig[odd], info, queue, part, parts, setup, [&](int xa, int xb, int y, int z) {
            for (int c = xa & ~31; c <= xb; c += 32) {
                uint32_t m = 0xFFFFFFFFu;
                if (c < xa) m &= 0xFFFFFFFFu << (xa - c);
                if (c + 31 > xb) m &= 0xFFFFFFFFu >> (31 - (xb - c));
                emit_mask<REG, SPEC>(S, table, ident, info, layout, c, y, z, m, RA);
            }
        });
        first += per;
        odd ^= 1;
    } while (LOOP && first < end);
    __syncthreads();
    // every slot read before the first atomic (one LDS wait, not one per slot)
    static_assert(kHashCap % kChunk == 0, "whole slots per thread");
    constexpr int kPer = kHashCap / kChunk;
    uint32_t kk[kPer], vv[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        kk[u] = S.keys[threadIdx.x + u * kChunk];
        vv[u] = S.vals[threadIdx.x + u * kChunk];
    }
    if (REG) {
        region_flush<kChunk, kPer>(S.flush, kk, vv, S.keys, S.vals, RA.P, RA.W);
    } else {
#pragma unroll
        for (int u = 0; u < kPer; u++)
            if (kk[u] != kEmpty && vv[u] != 0u) memory_or<SPEC>(table, kk[u], vv[u]);
    }
}

// Zero-fill with 16-byte stores (a kernel, so it can live inside a captured
// graph).  Work unit: kFillWords words of one job's table.
constexpr uint64_t kFillWords = 16384;

__global__ void __launch_bounds__(256) fill_zero_kernel(ItemDev one, ItemMap M) {
    __shared__ BlockJob J;
    resolve_job(one, M, blockIdx.x, J);
    if (J.local == ~0u) return;
    const uint32_t G = J.it.info.gridsize[0];
    const uint64_t words = ((uint64_t)G * G * G + 31) / 32;
    const uint64_t w0 = (uint64_t)J.local * kFillWords;
    const uint64_t w1 = w0 + kFillWords < words ? w0 + kFillWords : words;
    uint32_t* __restrict__ table = J.it.table;
    if ((((uintptr_t)table) & 15u) == 0) {
        uint4* t4 = (uint4*)table;
        const uint64_t a = (w0 + 3) / 4, b = w1 / 4;  // whole uint4 inside [w0, w1)
        for (uint64_t i = a + threadIdx.x; i < b; i += 256) t4[i] = make_uint4(0u, 0u, 0u, 0u);
        for (uint64_t i = w0 + threadIdx.x; i < w1 && i < 4 * a; i += 256) table[i] = 0u;
        for (uint64_t i = (b * 4 > w0 ? b * 4 : w0) + threadIdx.x; i < w1; i += 256) table[i] = 0u;
    } else {
        for (uint64_t i = w0 + threadIdx.x; i < w1; i += 256) table[i] = 0u;
    }
}

template <class Word>
__device__ __forceinline__ void table_or(Word* p, Word v) {
    if (v) atomicOr(p, v);
}

// Blocked scratch table -> rows of the linear table (G a multiple of 32); the
// scratch words that held bits return to zero.  A thread takes 4 words in x of
// the 4 rows in y of one z: four 16-byte loads, a transpose in registers, four
// 16-byte stores (VEC: rows of whole 16-byte groups, aligned tables), or else
// one word in x of those 4 rows.  Work unit: 256 threads.
// accumulate: bits are ORed into the table, only where there are any, and
// atomically: other calls, on other streams, may be adding to the table.
__device__ __forceinline__ void unblock_quad(const ItemDev& it, uint32_t t, bool vec) {
    const uint32_t G = it.info.gridsize[0], rw = G >> 5;
    uint4* __restrict__ s4 = (uint4*)it.scratch;
    const uint32_t zl = t & 3u;
    uint32_t r = t >> 2;
    if (vec) {
        const uint32_t wq = r % (rw >> 2);
        r /= rw >> 2;
        const uint32_t by = r % (G >> 2), bz = r / (G >> 2);
        if (bz >= G >> 2) return;
        const uint64_t base = ((uint64_t)(bz * (G >> 2) + by) * rw + 4u * wq) * 4u + zl;
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = s4[base + 4u * (uint32_t)u];
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (v[u].x | v[u].y | v[u].z | v[u].w) s4[base + 4u * (uint32_t)u] = make_uint4(0u, 0u, 0u, 0u);
        const uint4 o[4] = {make_uint4(v[0].x, v[1].x, v[2].x, v[3].x), make_uint4(v[0].y, v[1].y, v[2].y, v[3].y),
                            make_uint4(v[0].z, v[1].z, v[2].z, v[3].z), make_uint4(v[0].w, v[1].w, v[2].w, v[3].w)};
        uint4* __restrict__ d4 = (uint4*)it.table;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint64_t d = (((uint64_t)(4u * bz + zl) * G + 4u * by + (uint32_t)u) * rw >> 2) + wq;
            if (!it.accumulate) {
                d4[d] = o[u];
            } else {
                unsigned long long* p = (unsigned long long*)(d4 + d);
                table_or(p, (unsigned long long)o[u].y << 32 | o[u].x);
                table_or(p + 1, (unsigned long long)o[u].w << 32 | o[u].z);
            }
        }
        return;
    }
    const uint32_t w = r % rw;
    r /= rw;
    const uint32_t by = r % (G >> 2), bz = r / (G >> 2);
    if (bz >= G >> 2) return;
    const uint64_t i = ((uint64_t)(bz * (G >> 2) + by) * rw + w) * 4u + zl;
    const uint4 v = s4[i];
    if (v.x | v.y | v.z | v.w) s4[i] = make_uint4(0u, 0u, 0u, 0u);
    const uint32_t o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint64_t d = ((uint64_t)(4u * bz + zl) * G + 4u * by + (uint32_t)u) * rw + w;
        if (!it.accumulate)
            it.table[d] = o[u];
        else
            table_or(it.table + d, o[u]);
    }
}

// How rows are written: 16-byte groups, past the caches or not; words (a table at
// another address); words that are ORed into the table.
enum RowsForm : int { kRowsStreamed, kRowsCached, kRowsWords, kRowsAdded };
template <int FORM>
__device__ __forceinline__ void put_quad(uint4* d, const uint4& v) {
    if (FORM == kRowsStreamed)
        store_streaming(d, v);
    else
        *d = v;
}

// The same with flags: groups of 256 bytes whose flag is not set are zero and not
// read.  A workgroup takes a strip: K blocks in y of one 4-row slab in z, which lie
// together in the scratch table and are 4 runs of 4 K rows of the table.  One load
// by every wave has the strip's flags (at most 64).  What they name is turned in
// LDS, so that both sides are whole 16-byte groups of consecutive lanes whatever
// the row length (4-byte ones into tables at other addresses).  Lines without bits
// are written before the others have been read, whole ones: half a line at a time
// is what the stores must avoid (one at 2048^3 in two parts: 800 us a call, not
// 312).  Rows written per thread as in unblock_quad, 16 bytes of each of 4, lost up
// to half the time where rows are no powers of two (us a call, those and strips:
// 1,280 triangles at 1408^3 247 and 122, at 2016^3 693 and 310, at 992^3 73 and
// 62; torus of 400,000 at 1312^3 213 and 120; at 1024^3 69 and 68).
// From kStreamedGrid on the table and the scratch table are beyond the 256 MB of
// the last cache together, and the rows must not push the scratch words out of it
// (1,280 at 1152^3 88 -> 74 us, at 1408^3 170 -> 122, at 2048^3 402 -> 310; at
// 1056^3 69 either way).
constexpr uint32_t kStripQuads = 1024;
constexpr uint32_t kStripWords = 4u * kStripQuads + 4u * 80u;

__host__ __device__ inline uint32_t strip_blocks(uint32_t rw) {  // K: a multiple of 4, up to 16 KB a strip
    const uint32_t k = (kStripQuads / 4u / rw) & ~3u;
    return k < 4u ? 4u : k;
}

template <int FORM>
__global__ void __launch_bounds__(256) unblock_flagged_kernel(uint32_t* __restrict__ scratch,
                                                              uint32_t* __restrict__ out, uint32_t G) {
    __shared__ __align__(16) uint32_t lds[kStripWords];
    const uint32_t rw = G >> 5, nb = G >> 2, K = strip_blocks(rw), unit = blockIdx.x;
    const uint32_t strips = (nb + K - 1u) / K, bz = unit / strips, by = (unit - bz * strips) * K;
    const uint32_t kk = nb - by < K ? nb - by : K, run = kk * rw;  // run: 16-byte groups of one z
    const uint64_t q0 = (uint64_t)(bz * nb + by) * rw * 4u;
    uint4* __restrict__ s4 = (uint4*)scratch + q0;
    const uint32_t lane = (uint32_t)__lane_id();
    uint8_t* flag = (uint8_t*)scratch - 1 - (q0 >> 4) - lane;
    const bool set = lane < (run >> 2) && *flag != 0;
    const unsigned long long flags = __ballot(set);
    uint32_t* __restrict__ table = out + ((uint64_t)(4u * bz) * G + 4u * by) * rw;
    const uint64_t slab = (uint64_t)G * rw;        // words of one z
    const uint32_t inv = 65536u / rw + 1u;         // t / rw for t < 1024, rw <= 64
    const bool whole = (rw & 3u) == 0;             // the 16-byte groups of a row are each of one flag
    constexpr bool kQuads = FORM == kRowsStreamed || FORM == kRowsCached;
    // this thread's group of each z, if it has words of a flagged group
    bool hit = threadIdx.x < run && flags != 0;
    if (kQuads && hit && whole) {
        const uint32_t row = (4u * threadIdx.x * inv) >> 16;
        hit = (flags >> (((row >> 2) * rw + 4u * threadIdx.x - row * rw) >> 2)) & 1ull;
    }
    if (kQuads) hit = threadIdx.x < run && ((__ballot(hit) >> (lane & 56u)) & 255ull);  // whole 128-byte lines
    if (kQuads && threadIdx.x < run && !hit) {
#pragma unroll
        for (uint32_t z = 0; z < 4u; z++)
            put_quad<FORM>((uint4*)(table + z * slab) + threadIdx.x, make_uint4(0u, 0u, 0u, 0u));
    }
    if (!flags) {
        if (FORM == kRowsWords)
            for (uint32_t z = 0; z < 4u; z++)
                for (uint32_t i = threadIdx.x; i < 4u * run; i += 256u) table[z * slab + i] = 0u;
        return;
    }
    const uint32_t plane = ((4u * run + 63u) & ~63u) + 16u;  // spreads the 4 planes over the banks
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint32_t i = threadIdx.x + 256u * (uint32_t)u;
        v[u] = (flags >> (i >> 4)) & 1ull ? s4[i] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint32_t i = threadIdx.x + 256u * (uint32_t)u, t = i >> 2;
        if (v[u].x | v[u].y | v[u].z | v[u].w) s4[i] = make_uint4(0u, 0u, 0u, 0u);
        if (i >= 4u * run) continue;
        uint32_t* d = lds + (i & 3u) * plane + t + 3u * ((t * inv) >> 16) * rw;
        d[0] = v[u].x;
        d[rw] = v[u].y;
        d[2u * rw] = v[u].z;
        d[3u * rw] = v[u].w;
    }
    __syncthreads();
    if (set && threadIdx.x < 64u) *flag = 0;  // every wave has read it
#pragma unroll
    for (uint32_t z = 0; z < 4u; z++) {
        uint32_t* d = table + z * slab;
        if (kQuads) {
            if (hit) put_quad<FORM>((uint4*)d + threadIdx.x, *(const uint4*)(lds + z * plane + 4u * threadIdx.x));
        } else {
            for (uint32_t i = threadIdx.x; i < 4u * run; i += 256u) {
                const uint32_t o = lds[z * plane + i];
                if (FORM == kRowsAdded)
                    table_or(d + i, o);
                else
                    d[i] = o;
            }
        }
    }
}

// Rows that are no whole words (G not a multiple of 32; the scratch table's rows
// are padded to words): 32 rows are G words of the linear table, from a word
// boundary on, so a workgroup takes 32 rows into LDS, returns them to zero and
// packs its G words.  The lanes of a load hold 32 rows of one word, which an odd
// stride in LDS spreads over the banks (a stride of 32 words: torus of 400,000 at
// 1000^3 127 us a call, with 33 122, with flags and empty rows left out 88).
// FLAGS: as above, but a group's flag is read by the workgroups of its four z, so
// the caller clears the flags afterwards.
template <bool FLAGS>
__device__ __forceinline__ void unblock_ragged(uint32_t* __restrict__ scratch, uint32_t* __restrict__ table, uint32_t G,
                                               int accumulate, uint32_t unit, uint32_t* rows) {
    const uint32_t rw = (G + 31u) >> 5, stride = rw | 1u, r0 = unit * 32u, r = r0 + (threadIdx.x & 31u);
    const uint32_t y = r % G, z = r / G;  // four rows of a block are neighbours
    const int passes = (int)((rw + 7u) >> 3);
    bool any[4] = {false, false, false, false};
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (u >= passes) break;
        const uint32_t w = (threadIdx.x >> 5) + 8u * (uint32_t)u;
        any[u] = w < rw && z < G;
        if (FLAGS && any[u]) any[u] = *((const uint8_t*)scratch - 1 - (blocked_word(G, w, y, z) >> 6)) != 0;
    }
    if (FLAGS && !__syncthreads_or(any[0] || any[1] || any[2] || any[3])) {  // 32 empty rows
        const uint32_t total = (uint32_t)(((uint64_t)G * G * G + 31u) / 32u), w0 = unit * G;
        if (!accumulate)
            for (uint32_t k = threadIdx.x; k < G && w0 + k < total; k += 256u) table[w0 + k] = 0u;
        return;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (u >= passes) break;
        v[u] = any[u] ? scratch[blocked_word(G, (threadIdx.x >> 5) + 8u * (uint32_t)u, y, z)] : 0u;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (u >= passes) break;
        const uint32_t w = (threadIdx.x >> 5) + 8u * (uint32_t)u;
        if (v[u]) scratch[blocked_word(G, w, y, z)] = 0u;
        if (w < rw) rows[(threadIdx.x & 31u) * stride + w] = v[u];
    }
    __syncthreads();
    pack_rows(rows, stride, rw, G, r0, table, [&](uint32_t* d, uint32_t p) {
        if (!accumulate)
            *d = p;
        else
            table_or(d, p);
    });
}

__global__ void __launch_bounds__(256) unblock_ragged_kernel(uint32_t* __restrict__ scratch,
                                                             uint32_t* __restrict__ table, uint32_t G, int accumulate) {
    __shared__ uint32_t rows[kRaggedWords];
    unblock_ragged<true>(scratch, table, G, accumulate, blockIdx.x, rows);
}

__global__ void __launch_bounds__(256) clear_flags_kernel(uint4* __restrict__ flags, uint32_t quads) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < quads) flags[i] = make_uint4(0u, 0u, 0u, 0u);
}

__host__ __device__ inline bool unblock_vec(uint32_t G, const uint32_t* table) {
    return (G & 127u) == 0 && (((uintptr_t)table) & 15u) == 0;
}

__global__ void __launch_bounds__(256) unblock_kernel(ItemDev one, ItemMap M) {
    __shared__ BlockJob J;
    __shared__ uint32_t rows[kRaggedWords];
    if (M.items) {
        resolve_job(one, M, blockIdx.x, J);
        if (J.local == ~0u) return;
    }
    const ItemDev& it = M.items ? J.it : one;
    const uint32_t local = M.items ? J.local : blockIdx.x;
    if (it.info.gridsize[0] & 31u)
        unblock_ragged<false>(it.scratch, it.table, it.info.gridsize[0], it.accumulate, local, rows);
    else
        unblock_quad(it, local * 256u + threadIdx.x, unblock_vec(it.info.gridsize[0], it.table));
}

uint32_t unblock_units(uint32_t G, const uint32_t* table) {
    const uint64_t words = (uint64_t)G * G * G / 32u;
    if (G & 31u) return (G * G + 31u) / 32u;
    if (G <= kUnflaggedGrid) return (uint32_t)((words / (unblock_vec(G, table) ? 16u : 4u) + 255u) / 256u);
    const uint32_t nb = G >> 2, k = strip_blocks(G >> 5);
    return nb * ((nb + k - 1u) / k);
}

static void launch_unblock_flagged(const ItemDev& one, uint32_t units, hipStream_t stream) {
    const uint32_t G = one.info.gridsize[0];
    if (G & 31u) {
        unblock_ragged_kernel<<<units, 256, 0, stream>>>(one.scratch, one.table, G, one.accumulate);
        const uint32_t quads = (uint32_t)(blocked_flags(G) / 16u);
        clear_flags_kernel<<<(quads + 255u) / 256u, 256, 0, stream>>>((uint4*)one.scratch - quads, quads);
        return;
    }
    const bool quads = (((uintptr_t)one.table) & 15u) == 0;
    const auto kernel = one.accumulate ? unblock_flagged_kernel<kRowsAdded>
                        : !quads       ? unblock_flagged_kernel<kRowsWords>
                        : G >= kStreamedGrid ? unblock_flagged_kernel<kRowsStreamed> : unblock_flagged_kernel<kRowsCached>;
    kernel<<<units, 256, 0, stream>>>(one.scratch, one.table, G);
}

hipError_t launch_unblock_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, hipStream_t stream) {
    if (units == 0) return hipSuccess;
    if (!M.items && one.flagged)
        launch_unblock_flagged(one, units, stream);
    else
        unblock_kernel<<<units, 256, 0, stream>>>(one, M);
    return hipGetLastError();
}

// Where words go through a blocked scratch table: the linear layout, in tables
// beyond the dense LDS merge.  A call of few triangles at G <= 80 has too few
// atomics for it (displaced sphere of 1,280 at 64^3 12.3 us, 13.3 blocked; a soup
// of 100,003 at 64^3 76.6 and 27.9).  Measured with the rows of a linear table as
// keys -> blocked (us per call): soup of 300,003 at 128^3 160 -> 45, 100,003 at
// 256^3 88 -> 67; displaced sphere of 81,920 at 256^3 31 -> 21, at 512^3 65 -> 37,
// 327,680 at 512^3 92 -> 60; torus of 200,000 at 256^3 19 -> 14; with flags, 81,920
// at 1024^3 149 -> 86, at 2048^3 728 -> 300, torus of 1,048,576 at 1024^3 105 ->
// 76.  The flags save the row pass most of the scratch table from about 640^3 on;
// below, setting them costs more than that (327,680 at 256^3 41 without, 46 with;
// at 544^3 66 and 71).  Grids whose rows are no whole words: torus of 26,866 at
// 200^3 16.7 -> 14.2, soup of 100,000 at 201^3 89 -> 48, displaced sphere of 81,920
// at 200^3 32 -> 18, torus of 200,000 at 1000^3 105 -> 99.  No mesh of 1,280 to
// 1,310,720 triangles measured slower than with the rows of the table as keys at
// any grid of 200 to 2048.
//
// An accumulating call has no zero-fill to save, and its row pass adds to the table
// by atomics itself: few triangles go to the table directly (us, blocked and
// direct: 1,280 at 256^3 17.6 and 13.3, at 1024^3 97 and 82; soup of 3,000 at 128^3
// 16.0 and 12.7; displaced sphere of 20,480 at 128^3 15.9 and 12.7, at 200^3 18.2 and
// 21.6, of 81,920 at 128^3 16.2 and 20.0, at 512^3 46 and 60, at 1024^3 123 and 128).
bool chunk_blocked(int layout, uint32_t G, uint64_t n_triangles, bool accumulate) {
    const uint64_t words = (uint64_t)G * G * G / 32u;
    if (accumulate && n_triangles <= (G <= 160u ? 32768u : 4096u)) return false;
    return layout == VOX_LAYOUT_LINEAR && G <= ((G & 31u) ? kRaggedGrid : kBlockedGrid) &&
           words > (n_triangles < 16384u ? 16384u : (uint64_t)kHashCap);
}

bool chunk_supported(uint32_t G) { return (uint64_t)G * G * G / 32 < 0xFFFFFFFFull; }

uint32_t fill_units(uint32_t G) {
    const uint64_t words = ((uint64_t)G * G * G + 31) / 32;
    return (uint32_t)((words + kFillWords - 1) / kFillWords);
}

// Chunks per workgroup.  A table of at most kHashCap words is merged densely
// in LDS, and every workgroup that touches it flushes up to all its words to
// the same few addresses (16 of them a request): such jobs give each workgroup
// several chunks to cut those atomics, while keeping at least 512 workgroups of a
// lone call, or 128 of a batch's job.  With 64 a workgroup's chain of chunks was
// what the call lasted (us per call, 64 -> this): soup of 269,272 at 32^3 137 ->
// 28, torus of 100,000 at 32^3 29 -> 11; batches of 13 mixed meshes 190 -> 125
// (116 with 512), of 11 195 -> 163 (181 with 512), of 48 423 with any.
uint32_t chunk_span(uint32_t G, uint64_t n_triangles, bool lone) {
    const uint64_t words = ((uint64_t)G * G * G + 31) / 32;
    if (words > (uint64_t)kHashCap) return 1u;
    const uint64_t chunks = (n_triangles + kChunk - 1) / kChunk;
    const uint64_t s = chunks / (lone ? 512u : 128u);
    return s < 1 ? 1u : (s > 16 ? 16u : (uint32_t)s);
}

uint32_t chunk_units(uint64_t n_triangles, uint32_t span, uint32_t parts, uint32_t lg_split) {
    const uint64_t per = (uint32_t)kChunk >> lg_split;
    const uint64_t chunks = (n_triangles + per - 1) / per;
    if (parts > 1u) return (uint32_t)(chunks * parts);
    const uint64_t sp = span > 1u ? span : 1u;
    return (uint32_t)((chunks + sp - 1) / sp);
}

hipError_t launch_fill_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, hipStream_t stream) {
    if (units == 0) return hipSuccess;
    fill_zero_kernel<<<units, 256, 0, stream>>>(one, M);
    return hipGetLastError();
}

int chunk_spec(int layout, uint32_t G) {
    if (layout == VOX_LAYOUT_LINEAR && (G & 31u) == 0) return kSpecLinear;
    if (layout == VOX_LAYOUT_MORTON && G <= 1024u) return kSpecMorton;
    return kSpecAny;
}

template <bool MULTI, bool SPLIT>
static void launch_chunk_spec(int spec, uint32_t units, hipStream_t stream, const ItemDev& one, const ItemMap& M) {
    const RegionArgs none{};
    if (spec == kSpecLinear)
        surface_chunk_kernel<MULTI, false, false, false, kSpecLinear, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
    else if (spec == kSpecBlocked)
        surface_chunk_kernel<MULTI, false, false, false, kSpecBlocked, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
    else if (!MULTI && spec == kSpecFlagged)
        surface_chunk_kernel<false, false, false, false, kSpecFlagged, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
    else
        surface_chunk_kernel<MULTI, false, false, false, kSpecMorton, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
}

template <bool MULTI, bool SPLIT>
static void launch_chunk_any(bool wide, uint32_t units, hipStream_t stream, const ItemDev& one, const ItemMap& M) {
    const RegionArgs none{};
    if (wide)
        surface_chunk_kernel<MULTI, false, true, false, kSpecAny, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
    else
        surface_chunk_kernel<MULTI, false, false, false, kSpecAny, SPLIT><<<units, kChunk, 0, stream>>>(one, M, none);
}

template <bool MULTI>
static void launch_chunk_form(int spec, bool split, bool wide, uint32_t units, hipStream_t stream, const ItemDev& one,
                              const ItemMap& M) {
    if (spec == kSpecAny && split)
        launch_chunk_any<MULTI, true>(wide, units, stream, one, M);
    else if (spec == kSpecAny)
        launch_chunk_any<MULTI, false>(wide, units, stream, one, M);
    else if (split)
        launch_chunk_spec<MULTI, true>(spec, units, stream, one, M);
    else
        launch_chunk_spec<MULTI, false>(spec, units, stream, one, M);
}

// waves: 5 or 6 waves per SIMD for the layout-generic one-chunk form (0: 6 for a
// lone linear job without shared triangles, 5 otherwise); the layout-specialised
// ones need few enough registers to run at six (lone) or five whatever it is, and
// the chunk loop always runs at 4.  spec: the layout every job of M shares
// (chunk_spec of each, or kSpecAny); a single job's comes from `one`.  split: some
// job of M has lg_split.
hipError_t launch_chunk_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, bool loop, hipStream_t stream,
                             int waves, int spec, bool split) {
    if (units == 0) return hipSuccess;
    const RegionArgs none{};
    if (loop && M.items) {
        // its other jobs may be split
        surface_chunk_kernel<true, true, false, false, kSpecAny, true><<<units, kChunk, 0, stream>>>(one, M, none);
    } else if (loop) {
        surface_chunk_kernel<false, true, false, false><<<units, kChunk, 0, stream>>>(one, M, none);
    } else if (M.items) {
        launch_chunk_form<true>(spec, split, waves == 6, units, stream, one, M);
    } else {
        spec = one.scratch ? (int)(one.flagged ? kSpecFlagged : kSpecBlocked)
                           : chunk_spec(one.layout, one.info.gridsize[0]);
        const bool wide = waves == 6 || (waves == 0 && !one.lg_split && one.layout == VOX_LAYOUT_LINEAR);
        launch_chunk_form<false>(spec, one.lg_split != 0u, wide, units, stream, one, M);
    }
    return hipGetLastError();
}

static ItemDev single_job(const vox_info& info, const float* tris, uint32_t* table, int layout) {
    ItemDev one{};
    one.info = info;
    one.tris = tris;
    one.table = table;
    one.layout = layout;
    one.span = chunk_span(info.gridsize[0], info.n_triangles, true);
    one.parts = 1;
    return one;
}

// Voxel boxes above this are queued (0: the built-in rule): 16 voxels in a coarse
// mesh of few triangles, whose workgroups would wait for their largest boxes; 64
// in a coarser one of more (81,920 at 1024^3: 165 us at 256 voxels, 150 at 64; at
// 512^3 66 and 80).
static uint32_t chunk_big(uint32_t G, uint64_t n) {
    const uint64_t g2 = (uint64_t)G * G;
    if (n == 0 || !chunk_large(G, n)) return 0u;
    return n <= 32768u ? 16u : (8u * n < g2 ? 64u : 0u);
}

// The work shape of a lone call.  A mesh of few triangles must still give every
// CU several waves, so its triangles are shared by up to 16 lanes each, as long
// as the call has at most 1280 workgroups (five per CU) by that; more lanes
// only repeat the setup, and Morton chunks of under 32 triangles merge too few
// of their words.  A coarse mesh (about 2.5 voxels a triangle's edge and more)
// queues smaller boxes and shares its few workgroups' queued rows with further
// parts, the more the coarser it is.  A finer one of up to 262,144 triangles
// takes two parts, for the large triangles that it may have among them.  Where
// triangles are a voxel or less (16 G^2 and more) sharing them only repeats their
// setup: 81,920 at 64^3 Morton 16.6 us a call with four lanes a triangle, 15.5
// with two (14.4 with one, but a soup of as many 37 and 30).
// Measured (us per call, 256 triangles a workgroup and one part -> this rule; a
// loop of calls does not go below about 15): icosphere 5,120 at 64^3 21.7 ->
// 15, 1,280 at 256^3 277 -> 18; torus 26,896 at 200^3 32.7 -> 17, 5,000 at
// 128^3 76 -> 16; displaced sphere 20,480 at 256^3 90 -> 25, 81,920 at 256^3
// 39 -> 34; slivers of 150,000 at 512^3 Morton 39 -> 33; soups at 256^3 2,003
// 119 -> 20, 20,003 114 -> 40, 100,003 123 -> 90.
static void chunk_shape(ItemDev& one) {
    const uint64_t n = one.info.n_triangles, G = one.info.gridsize[0];
    if (one.span > 1u || n == 0) return;
    const bool fine = n >= 16u * G * G;  // triangles of a voxel or less
    const uint32_t top = fine ? 1u : (one.layout == VOX_LAYOUT_MORTON ? 3u : 4u);
    one.lg_split = 0;
    // (dense tables: fewer workgroups, each of which flushes the whole table)
    const uint64_t lanes = G * G * G / 32u <= (uint64_t)kHashCap ? 65536u : 327680u;
    while (one.lg_split < top && n << (one.lg_split + 1u) <= lanes) one.lg_split++;
    if (chunk_large((uint32_t)G, n)) {
        const uint64_t units = ((n << one.lg_split) + kChunk - 1) / kChunk;
        uint64_t p = 2048u / units;
        if (p > G * G / (2u * n)) p = G * G / (2u * n);
        one.parts = p < 1u ? 1u : (p > 16u ? 16u : (uint32_t)p);
        if (!one.big) one.big = chunk_big((uint32_t)G, n);
    } else {
        one.parts = one.lg_split <= 1u && n <= 262144u && !fine ? 2u : 1u;
    }
}

// The work shape of a batch's job.  A mesh of large triangles is a long chain of
// rounds to each of its few workgroups.  In a batch of few triangles they are shared
// as in a lone call, up to 16 lanes a triangle and 16 parts, for `share` workgroups:
// 1024 over all such jobs, 64 to 512 each.  In one of more, whose other jobs fill
// the device meanwhile (share 0), a coarse mesh (fewer than G^2/4 triangles) has up
// to 32 parts, for 256 workgroups.  Measured (us a launch, parts only and shared):
// displaced sphere of 1,280 at 64^3 93 and 20, of 20,480 at 256^3 94 and 37, six of
// them 104 and 78; mixed meshes, 13 of 0.3 million surface triangles 159 and 127,
// 38 of 0.7 million 182 and 150, 26 of 1.2 million 291 and 286, 17 of 0.1 million
// 118 and 121; 44 of 1.8 million 377 and 383.
void chunk_batch_shape(ItemDev& it, uint32_t share) {
    const uint64_t n = it.info.n_triangles, G = it.info.gridsize[0];
    it.parts = 1;
    if (!it.big) it.big = chunk_big((uint32_t)G, n);
    if (n == 0 || !(share ? chunk_large((uint32_t)G, n) : coarse_mesh(n, (uint32_t)G))) return;
    while (share && it.lg_split < 4u && n << (it.lg_split + 1u) <= 256u * share) it.lg_split++;
    const uint64_t units = ((n << it.lg_split) + kChunk - 1) / kChunk;
    uint64_t p = (share ? share : 256u) / units;
    if (share && p > G * G / (2u * n)) p = G * G / (2u * n);
    const uint64_t most = share ? 16u : 32u;
    it.parts = p < 1u ? 1u : (p > most ? (uint32_t)most : (uint32_t)p);
}

hipError_t launch_fill_zero(const vox_info& info, uint32_t* table, hipStream_t stream) {
    const ItemMap none{nullptr, nullptr, 1, 0};
    return launch_fill_jobs(single_job(info, nullptr, table, 0), none, fill_units(info.gridsize[0]), stream);
}

// Phase 1 of the region algorithm: one chunk of kChunk triangles per
// workgroup, its merged words staged as region pairs (no table writes).
hipError_t launch_surface_region_chunks(const vox_info& info, const float* tris, int layout, const RegionArgs& RA,
                                        hipStream_t stream, uint32_t big, int waves) {
    if (info.n_triangles == 0) return hipSuccess;
    const ItemMap none{nullptr, nullptr, 1, 0};
    ItemDev one = single_job(info, tris, nullptr, layout);
    one.span = 1;
    one.parts = 1;
    one.big = big;
    const uint32_t units = chunk_units(info.n_triangles, 1, 1);
    const bool wide = waves == 6;  // six waves per SIMD (knob); built-in: five
    if (wide)
        surface_chunk_kernel<false, false, true, true><<<units, kChunk, 0, stream>>>(one, none, RA);
    else
        surface_chunk_kernel<false, false, false, true><<<units, kChunk, 0, stream>>>(one, none, RA);
    return hipGetLastError();
}

hipError_t launch_surface_chunk(const vox_info& info, const float* tris, uint32_t* table, int layout, bool accumulate,
                                hipStream_t stream, uint32_t big, int waves, bool scratch) {
    const ItemMap none{nullptr, nullptr, 1, 0};
    ItemDev one = single_job(info, tris, table, layout);
    one.big = big;
    one.accumulate = accumulate ? 1 : 0;
    chunk_shape(one);
    const uint32_t G = info.gridsize[0];
    if (scratch && info.n_triangles && chunk_blocked(layout, G, info.n_triangles, accumulate)) {
        hipError_t e = hipSuccess;
        const uint64_t bytes = blocked_bytes(G);
        one.flagged = G > kUnflaggedGrid ? 1u : 0u;
        const uint64_t flags = one.flagged ? blocked_flags(G) : 0u;
        ScratchLease S(stream);
        if (uint32_t* words = S.table(bytes + flags)) {
            one.scratch = words + flags / 4u;
            e = launch_chunk_jobs(one, none, chunk_units(info.n_triangles, one.span, one.parts, one.lg_split), false,
                                  stream, waves);
            if (e == hipSuccess) e = launch_unblock_jobs(one, none, unblock_units(G, table), stream);
            if (e == hipSuccess) S.clean();
            return e;
        }
    }
    if (!accumulate) {
        const hipError_t e = launch_fill_zero(info, table, stream);
        if (e != hipSuccess) return e;
    }
    if (info.n_triangles == 0) return hipSuccess;
    return launch_chunk_jobs(one, none, chunk_units(info.n_triangles, one.span, one.parts, one.lg_split),
                             one.span > 1u && one.parts <= 1u, stream, waves);
}

}  // namespace voxamd
