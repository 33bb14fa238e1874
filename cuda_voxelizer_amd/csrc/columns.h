// columns.h -- the columns of large solid triangles, dealt over a workgroup.
//
// A triangle's hit columns lie in a box of (y, z) columns.  One lane walking a
// large box holds up its workgroup, so the triangles with many columns are
// published to LDS, up to kColRecs at a time, and their columns are dealt to
// the waves in windows of 64, y fastest (rows of neighbouring y lie next to
// each other in the table).  Every column is decided by column_hit and
// column_xmax of vox_device.h.
#pragma once

#include "raster.h"
#include "vox_device.h"

#pragma clang fp contract(off)

namespace voxamd {

constexpr int kColRecs = 64;

struct __align__(16) ColRec {
    SolidTri S;
    int ylo, zlo, ny;
    float inv_ny;
    uint32_t cols;
    uint32_t pad;
};
static_assert(sizeof(ColRec) == 96, "whole 16-byte groups");

// A triangle's column box, clamped to the grid; empty: ny or nz below 1.
struct ColBox {
    int ylo, zlo, ny, nz;
};

__device__ __forceinline__ ColBox column_box(const SolidTri& S, int G) {
    ColBox B;
    B.ylo = (int)S.ymin < 0 ? 0 : (int)S.ymin;
    B.zlo = (int)S.zmin < 0 ? 0 : (int)S.zmin;
    // (float)y <= ymax for integer-valued ymax <=> y <= ymax
    const int yhi = S.ymax >= (float)(G - 1) ? G - 1 : (S.ymax >= 0.0f ? (int)S.ymax : -1);
    const int zhi = S.zmax >= (float)(G - 1) ? G - 1 : (S.zmax >= 0.0f ? (int)S.zmax : -1);
    B.ny = yhi - B.ylo + 1;
    B.nz = zhi - B.zlo + 1;
    return B;
}

// Records of one round: their columns together stay below 2^32.
__device__ __forceinline__ int column_recs(int G) { return G <= 4096 ? kColRecs : 8; }  // 64 * 2^24, 8 * 2^28

// Columns of the threads with `big`, whose triangle and box setup(S, B) gives.
// count[w]: the number of them in wave w (written by that wave before a
// barrier).  Of the windows this workgroup takes every `stride`-th of a wave's
// from `first` on.  hit(S, y, z, py, pz) is called for every hit column.  All
// threads of the workgroup call this.
template <int WAVES, class Setup, class Hit>
__device__ __forceinline__ void block_columns(ColRec* rec, const uint32_t* count, Setup&& setup, bool big,
                                              const vox_info& info, uint32_t first, uint32_t stride, Hit&& hit) {
    const int lane = __lane_id(), wave = (int)(threadIdx.x >> 6);
    int rank = 0, nq = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        rank += w < wave ? (int)count[w] : 0;
        nq += (int)count[w];
    }
    rank += (int)__popcll(__ballot(big) & ((1ull << lane) - 1ull));
    const int recs = column_recs((int)info.gridsize[0]);
    const float uy = info.unit[1], uz = info.unit[2];
    for (int r0 = 0; r0 < nq; r0 += recs) {
        const int nr = nq - r0 < recs ? nq - r0 : recs;
        __syncthreads();  // the previous round's records have been read
        if (big && rank >= r0 && rank < r0 + nr) {
            ColRec& R = rec[rank - r0];
            ColBox B;
            setup(R.S, B);
            R.ylo = B.ylo;
            R.zlo = B.zlo;
            R.ny = B.ny;
            R.inv_ny = 1.0f / (float)B.ny;
            R.cols = (uint32_t)B.ny * (uint32_t)B.nz;
        }
        __syncthreads();
        const uint32_t cols = lane < nr ? rec[lane].cols : 0u;
        uint32_t incl = cols;
#pragma unroll
        for (int d = 1; d < kColRecs; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d);
            if (lane >= d) incl += o;
        }
        const uint32_t total = __shfl(incl, kColRecs - 1);
        const uint32_t start = lane < nr ? incl - cols : 0xFFFFFFFFu;
        const uint32_t nwin = (total + 63u) >> 6;
        for (uint32_t w = first * WAVES + (uint32_t)wave; w < nwin; w += stride * WAVES) {
            const uint32_t j0 = w << 6, j = j0 + (uint32_t)lane;
            // the record of column j: the last that starts at or before it
            int o = (int)__popcll(__ballot(start <= j0)) - 1;
            const int last = (int)__popcll(__ballot(start <= j0 + 63u)) - 1;
            for (int k = o + 1; k <= last; k++) o += (uint32_t)__builtin_amdgcn_readlane((int)start, k) <= j ? 1 : 0;
            const uint32_t c = j - (uint32_t)__shfl((int)start, o);
            if (j < total) {
                const ColRec& R = rec[o];
                int zr = (int)((float)c * R.inv_ny);  // within one of c / ny
                int yr = (int)(c - (uint32_t)zr * (uint32_t)R.ny);
                if (yr < 0) {
                    zr--;
                    yr += R.ny;
                } else if (yr >= R.ny) {
                    zr++;
                    yr -= R.ny;
                }
                const int y = R.ylo + yr, z = R.zlo + zr;
                const float py = ((float)y + 0.5f) * uy, pz = ((float)z + 0.5f) * uz;
                if (column_hit(R.S, py, pz)) hit(R.S, y, z, py, pz);
            }
        }
    }
}

}  // namespace voxamd
