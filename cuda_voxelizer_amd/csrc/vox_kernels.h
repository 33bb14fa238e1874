// vox_kernels.h -- internal launch functions shared by the C-ABI layer.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cuda_voxelizer_amd/vox_capi.h"
#include "region.h"
#include "slab.h"
#include "tile.h"

namespace voxamd {

hipError_t launch_surface_direct(const vox_info& info, const float* tris, uint32_t* table, int layout,
                                 hipStream_t stream);
hipError_t launch_solid_direct(const vox_info& info, const float* tris, uint32_t* table, int layout,
                               unsigned long long* offrow, hipStream_t stream);

uint32_t direct_units(uint64_t n_triangles);
hipError_t launch_direct_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, bool solid, hipStream_t stream);
bool make_plan(int G, int layout, bool solid, TilePlan& P, int scale = 0);
WorkspaceLayout workspace_layout(uint64_t tiles_cap, uint64_t n_cap, int max_tiles_per_tri);
hipError_t launch_tiled_jobs(const ItemDev& one, const ItemMap& M_bin, const ItemMap& M_tile, const ItemMap& M_tri,
                             uint32_t total_bin_blocks, uint32_t total_tiles, bool solid, uint32_t max_tile_words,
                             void* ws, const WorkspaceLayout& L, hipStream_t stream);
hipError_t launch_tiled(const vox_info& info, const float* tris, uint32_t* table, const TilePlan& P, bool solid,
                        int layout, bool accumulate, void* ws, const WorkspaceLayout& L,
                        unsigned long long* offrow, hipStream_t stream);

bool marker_supported(uint32_t G, int layout, bool accumulate);
bool marker_batch_supported(uint32_t G, int layout, bool accumulate);  // the in-place form
bool layout_convert_fast(uint32_t G);
hipError_t launch_layout_convert(const uint32_t* src, uint32_t* dst, uint32_t G, bool to_morton, hipStream_t stream);
uint64_t marker_ws_bytes();
uint32_t marker_block_units(ItemDev& it);  // sets the job's work shape
uint32_t marker_row_units(uint32_t G);
hipError_t launch_marker_jobs(const ItemMap& m_blocks, const ItemMap& m_rows, const ItemMap& m_tris,
                              uint32_t blocks, uint32_t row_units, void* mws, hipStream_t stream);
hipError_t launch_solid_marker(const vox_info& info, const float* tris, uint32_t* table, int layout,
                               bool accumulate, unsigned long long* offrow, hipStream_t stream, uint32_t big = 0,
                               bool scratch = true);
// The allocation-free solid form: its scratch is a static device array of
// static_scratch_bytes() bytes per GPU (address taken once per device).
size_t static_scratch_bytes();
hipError_t static_scratch_init(int device, void** out);
hipError_t launch_solid_marker_static(const vox_info& info, const float* tris, uint32_t* table,
                                      unsigned long long* offrow, hipStream_t stream);

bool make_slab_plan(uint32_t G, SlabPlan& P, int lg_ty = -1, int lg_tz = -1, int split_lg = -1, int wg = 0);
SlabLayout slab_layout(uint64_t tiles_cap, uint64_t n_cap);
bool slab_layout_fits(const SlabPlan& P, uint64_t n, const SlabLayout& L);
hipError_t launch_slab(const vox_info& info, const float* tris, uint32_t* table, const SlabPlan& P, bool solid,
                       bool accumulate, unsigned long long* offrow, void* mem, const SlabLayout& L,
                       hipStream_t stream);

// Region algorithm (region.hip): phase 1 stages (word, mask) pairs per output
// region (surface: chunk.hip, solid: marker.hip), the build pass writes each
// region once.  K: capacity overrides (flag bits), -1 fields are built-in.
bool make_region_plan(uint32_t G, int layout, bool solid, RegionPlan& P, const RegionKnobs& K);
bool region_supported(uint32_t G, int layout, bool solid);
// workgroups: phase-1 workgroups of the call (each stages into its own slice)
hipError_t region_workspace(const RegionPlan& P, uint64_t workgroups, hipStream_t stream, RegionWs& W);
hipError_t launch_region_build(const RegionPlan& P, const RegionWs& W, uint32_t* table, bool accumulate,
                               hipStream_t stream);
hipError_t launch_surface_region_chunks(const vox_info& info, const float* tris, int layout, const RegionArgs& RA,
                                        hipStream_t stream, uint32_t big, int waves);
hipError_t launch_surface_region(const vox_info& info, const float* tris, uint32_t* table, int layout,
                                 bool accumulate, hipStream_t stream, uint32_t big = 0, int waves = 0,
                                 const RegionKnobs& K = RegionKnobs{});
hipError_t launch_solid_region(const vox_info& info, const float* tris, uint32_t* table, int layout,
                               bool accumulate, unsigned long long* offrow, hipStream_t stream, uint32_t big = 0,
                               const RegionKnobs& K = RegionKnobs{});
// VOX_REGION_* bits of the flags
inline RegionKnobs region_knobs(unsigned flags) {
    RegionKnobs K;
    const unsigned w = (flags >> 8) & 15u, st = (flags >> 12) & 31u, d = (flags >> 17) & 15u;
    if (w) K.lg_words = (int)w + 9;
    if (st) K.lg_stage = (int)st - 1;
    if (d) K.lg_desc = (int)d - 1;
    return K;
}

bool chunk_supported(uint32_t G);
// A coarse mesh has few triangles for its grid, so each covers a large voxel
// box and many columns.  The defaults are chunk for surfaces and marker for
// solids at every size; both give a coarse mesh smaller workgroups that share
// its large triangles (chunk.hip, marker.hip: marker_shape).
inline bool coarse_mesh(uint64_t n_triangles, uint32_t G) {
    return n_triangles < (uint64_t)G * G / 4u;
}
// Solid default on small grids: a mesh of at least 4 G^2 triangles at G <= 64
// has boxes of a few columns each, and one lane per triangle with its
// atomics straight to the table beats the marker pass and its suffix (65,536
// triangles at 64^3: direct 0.0098 ms vs marker 0.0161 ms; 5,120 at 32^3:
// 0.0106 vs 0.0165 ms); at 128^3, or below 4 G^2, marker is faster (81,920 at
// 128^3: 0.0133 vs 0.0169 ms; the bunny's 5,110 at 64^3: 0.032 vs 0.046 ms).
inline bool prefer_direct_solid(uint64_t n_triangles, uint32_t G) {
    return G <= 64u && n_triangles >= 4ull * G * G;
}
// And where rows are no whole words, on grids up to 128^3 from G^2 triangles on:
// direct has a launch less (icosphere of 20,480 at 101^3 11.2 us, marker 13.3;
// torus of 5,000 at 40^3 11.0 and 14.1).  Larger or coarser ones are marker's:
// torus of 26,866 at 200^3 15.1 direct, 14.5 marker, 1,000 at 200^3 153 and 14,
// icosphere of 1,280 at 100^3 42 and 15, displaced sphere of 327,680 at 700^3 355
// and 72.
inline bool prefer_direct_ragged(uint64_t n_triangles, uint32_t G) {
    return (G & 31u) != 0 && G <= 128u && n_triangles >= (uint64_t)G * G;
}
// Coarse solids whose rows are no whole 16-byte groups work in the caller's table,
// which marker's row pass then reads and writes: on large grids that loses to the
// tiles (us, tile and marker: torus of 400,000 at 1312^3 264 and 272, at 1504^3 349
// and 442, at 2016^3 782 and 921; displaced sphere of 327,680 at 1504^3 477 and
// 524), but for few triangles of many columns each (81,920 at 1504^3 579 and 518,
// at 2016^3 1586 and 1085) and on smaller grids (327,680 at 1184^3 265 and 223,
// torus of 400,000 at 1056^3 167 and 158).
inline bool prefer_tile_solid(int layout, bool accumulate, uint64_t n_triangles, uint32_t G) {
    return layout == VOX_LAYOUT_LINEAR && !accumulate && (G & 31u) == 0 && (G & 127u) != 0 && G > 1184u &&
           24ull * n_triangles >= (uint64_t)G * G && coarse_mesh(n_triangles, G);
}
hipError_t launch_fill_zero(const vox_info& info, uint32_t* table, hipStream_t stream);
uint32_t fill_units(uint32_t G);
uint32_t chunk_span(uint32_t G, uint64_t n_triangles, bool lone);
void chunk_batch_shape(ItemDev& it, uint32_t share);
constexpr uint64_t kSharedBatch = 1600000;  // triangles of a batch's surfaces
// Triangles of about 2.5 voxels an edge and more.
inline bool chunk_large(uint32_t G, uint64_t n_triangles) { return 8u * n_triangles < 5ull * G * G; }
uint32_t chunk_units(uint64_t n_triangles, uint32_t span, uint32_t parts, uint32_t lg_split = 0);
hipError_t launch_fill_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, hipStream_t stream);
// What a chunk kernel instantiation knows of its jobs' layout: nothing, linear
// with G a multiple of 32 (whole words per row), Morton with G <= 1024
// (codes fit 30 bits), or blocked (ItemDev.scratch), without or with flags.
enum ChunkSpec : int { kSpecAny = 0, kSpecLinear = 1, kSpecMorton = 2, kSpecBlocked = 3, kSpecFlagged = 4 };
int chunk_spec(int layout, uint32_t G);
hipError_t launch_chunk_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, bool loop, hipStream_t stream,
                             int waves = 0, int spec = kSpecAny, bool split = false);
hipError_t launch_surface_chunk(const vox_info& info, const float* tris, uint32_t* table, int layout, bool accumulate,
                                hipStream_t stream, uint32_t big = 0, int waves = 0, bool scratch = true);
// Word w of row (y, z) in a blocked table: the 4 x 4 rows of a block lie together.
__device__ __forceinline__ uint32_t blocked_word(uint32_t G, uint32_t w, uint32_t y, uint32_t z) {
    return ((((z >> 2) * ((G + 3u) >> 2) + (y >> 2)) * ((G + 31u) >> 5) + w) << 4) | ((z & 3u) << 2) | (y & 3u);
}
inline uint64_t blocked_bytes(uint32_t G) {
    const uint64_t nb = (G + 3u) >> 2;
    return nb * nb * ((G + 31u) >> 5) * 64u;
}
// Bytes of flags before a flagged table: one for each 256 bytes of it.
inline uint64_t blocked_flags(uint32_t G) { return (blocked_bytes(G) / 256u + 256u) & ~255ull; }
// Grids whose rows are no whole words are packed from padded rows up to this one.
constexpr uint32_t kRaggedGrid = 1024;
constexpr uint32_t kRaggedWords = 32u * (kRaggedGrid / 32u + 1u);
// 32 rows of rw words in LDS, `stride` words apart, from row r0 on -> their words of
// the linear table (fewer at its end; bits from G on are zero in every row):
// put(word, value) for each.  A word has bits of at most two rows (G > 32).
template <class Put>
__device__ __forceinline__ void pack_rows(const uint32_t* rows, uint32_t stride, uint32_t rw, uint32_t G, uint32_t r0,
                                          uint32_t* __restrict__ table, Put&& put) {
    const uint32_t total = (uint32_t)(((uint64_t)G * G * G + 31u) / 32u), w0 = r0 / 32u * G;
    for (uint32_t k = threadIdx.x; k < G; k += blockDim.x) {
        if (w0 + k >= total) return;
        const uint32_t b = k * 32u, r = b / G, x = b - r * G;
        const uint32_t* p = rows + r * stride + (x >> 5);
        const uint32_t lo = p[0], hi = (x >> 5) + 1u < rw ? p[1] : 0u, s = x & 31u;
        uint32_t v = s ? (lo << s) | (hi >> (32u - s)) : lo;
        if (G - x < 32u && r < 31u) v |= rows[(r + 1u) * stride] >> (G - x);
        put(table + w0 + k, v);
    }
}
constexpr int kBlockedSpecs = kSpecBlocked + 1;  // what a batch's classes may be
constexpr uint32_t kBlockedGrid = 2048;
constexpr uint32_t kUnflaggedGrid = 608;  // (chunk.hip: chunk_blocked)
constexpr uint32_t kBatchBlockedGrid = 512;
constexpr uint32_t kStreamedGrid = 1152;  // (chunk.hip: unblock_flagged_kernel)
bool chunk_blocked(int layout, uint32_t G, uint64_t n_triangles, bool accumulate);
uint32_t unblock_units(uint32_t G, const uint32_t* table);
hipError_t launch_unblock_jobs(const ItemDev& one, const ItemMap& M, uint32_t units, hipStream_t stream);
// Tuning bits of the flags (VOX_TUNE_*): queue threshold, chunk waves per SIMD, tile size.
inline uint32_t tune_big(unsigned flags) {
    const unsigned lg = (flags >> 24) & 15u;
    return lg ? (1u << (lg - 1u)) : 0u;
}
inline int tune_waves(unsigned flags) {
    const unsigned w = (flags >> 28) & 3u;
    return w == 1u ? 5 : (w == 2u ? 6 : 0);
}
inline int tune_tile_scale(unsigned flags) {
    const unsigned t = (flags >> 30) & 3u;
    return t == 1u ? -1 : (t == 3u ? 1 : 0);
}

}  // namespace voxamd
