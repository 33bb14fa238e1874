// rows.h -- rasterization of large voxel boxes by a workgroup.
//
// The workgroup takes up to REC triangles at a time: one wave sets them up, a
// lane each, then their (y, z) rows are dealt to the waves in windows of 64
// and over a wave's lanes: the YZ edges are tested per row, the
// passing rows are compacted into a list, and every 64 of them are finished
// with all lanes busy.  What passes in a row is one x interval: each of the
// seven tests along x -- the plane and the three XY and ZX edges -- is a
// monotone function of x in binary32 (a product with a constant, then sums
// with constants), so each test passes on one interval.  Its ends are
// estimated from per-triangle slopes (one fused multiply-add per edge), with a
// bound on how far the binary32 tests of vox_device.h can be from the estimate.
// An end with no voxel within that bound is known; rows with such a voxel go
// to a second list, where the tests themselves decide.
#pragma once

#include "raster.h"

#pragma clang fp contract(off)

namespace voxamd {

// The bound, in units of 2^-24 times the magnitudes that a test sums.  A test
// (two or three products of two rounded factors, two or three sums) is within
// 7 units of the real value; its estimate (a reciprocal of 1 ulp, products,
// one or two fused operations, the sum with the bound) within 10.
constexpr float kRowUlp = 24.0f * 5.9604644775390625e-08f;

struct __align__(16) RowRec {
    float yz[9];                    // a[3], b[3], d[3] of the YZ edges
    int ya, za, ny;                 // first row, rows in y
    float pl0, ph0, py, pz;         // plane: x from pl0 + t to ph0 + t, t = py y + pz z (voxels)
    float pm, inv_ny;               // its bound
    int xa, xb;                     // x range
    float xyl[6], xyh[6];           // XY edges that bound x below / above: x = e[k] + e[2 + k] y +- e[4 + k]
    float zxl[6], zxh[6];           // ZX edges: x = e[k] + e[2 + k] z +- e[4 + k]
    int mono;                       // the tests along x are monotone (no overflow, no infinities)
    int nz;
    float n[3], d1, d2, xy[9], zx[9];  // the tests along x
    int pad[2];
};
static_assert(sizeof(RowRec) == 288, "whole 16-byte groups; 72 words spread the records over the LDS banks");

struct WaveLists {
    uint32_t list[128];  // passing rows: record << 26 | z << 13 | y (grids up to 8192)
    uint2 open[64];      // undecided rows: the same, and x0 | x1 << 15 | (end undecided) << 30
};

template <int REC, int WAVES>
struct BlockRows {
    RowRec rec[REC];
    WaveLists wave[WAVES];
    uint8_t queue[64 * WAVES];  // threads whose triangles are large
};

__device__ __forceinline__ bool row_finite(float f) { return fabsf(f) < 1e15f; }  // false for NaN

__device__ __forceinline__ void row_publish(RowRec& R, const SurfTri& T, const vox_info& info) {
    const float ux = info.unit[0], uy = info.unit[1], uz = info.unit[2];
    const float gx = (float)info.gridsize[0] * ux, gy = (float)info.gridsize[1] * uy, gz = (float)info.gridsize[2] * uz;
    bool fin = gx < 1e15f && gy < 1e15f && gz < 1e15f;
    const float inf = __builtin_inff();
#pragma unroll
    for (int k = 0; k < 2; k++) {
        R.xyl[k] = R.zxl[k] = -inf;
        R.xyh[k] = R.zxh[k] = inf;
        R.xyl[2 + k] = R.zxl[2 + k] = R.xyh[2 + k] = R.zxh[2 + k] = 0.0f;
        R.xyl[4 + k] = R.zxl[4 + k] = R.xyh[4 + k] = R.zxh[4 + k] = 0.0f;
    }
    // The edges of a projection bound x from below or above, at most two of the
    // three from one side (their slopes sum to zero, up to rounding).  One
    // whose bound is infinite -- a zero slope -- leaves every voxel open.
    const auto edges = [&](const float* slope, const float* cross, const float* d, float uc, float gc, float* lo,
                           float* hi) {
        int nl = 0, nh = 0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            fin = fin && row_finite(slope[i]) && row_finite(cross[i]) && row_finite(d[i]);
            const float q = __builtin_amdgcn_rcpf(slope[i] * ux);
            const float mi = (kRowUlp * (fabsf(slope[i]) * gx + fabsf(cross[i]) * gc + fabsf(d[i])) + 1e-30f) * fabsf(q);
            const bool weak = !(mi < 1e6f);
            const float e0 = weak ? 0.0f : -d[i] * q, e1 = weak ? 0.0f : -cross[i] * q * uc, em = weak ? inf : mi;
            if (slope[i] > 0.0f) {
                if (nl == 0) { lo[0] = e0; lo[2] = e1; lo[4] = em; }
                else { lo[1] = e0; lo[3] = e1; lo[5] = nl == 2 ? inf : em; }
                nl++;
            } else {
                if (nh == 0) { hi[0] = e0; hi[2] = e1; hi[4] = em; }
                else { hi[1] = e0; hi[3] = e1; hi[5] = nh == 2 ? inf : em; }
                nh++;
            }
        }
    };
    edges(T.xy.a, T.xy.b, T.xy.d, uy, gy, R.xyl, R.xyh);
    edges(T.zx.b, T.zx.a, T.zx.d, uz, gz, R.zxl, R.zxh);
#pragma unroll
    for (int i = 0; i < 3; i++) {
        R.yz[i] = T.yz.a[i]; R.yz[3 + i] = T.yz.b[i]; R.yz[6 + i] = T.yz.d[i];
        R.xy[i] = T.xy.a[i]; R.xy[3 + i] = T.xy.b[i]; R.xy[6 + i] = T.xy.d[i];
        R.zx[i] = T.zx.a[i]; R.zx[3 + i] = T.zx.b[i]; R.zx[6 + i] = T.zx.d[i];
        R.n[i] = T.n[i];
    }
    R.d1 = T.d1;
    R.d2 = T.d2;
    const bool nfin = row_finite(T.n[0]) && row_finite(T.n[1]) && row_finite(T.n[2]) && row_finite(T.d1) &&
                      row_finite(T.d2);
    // NaN in the normal or an offset (zero-area triangles): the plane test passes everywhere
    const bool nnan = T.n[0] != T.n[0] || T.n[1] != T.n[1] || T.n[2] != T.n[2] || T.d1 != T.d1 || T.d2 != T.d2;
    const float q = __builtin_amdgcn_rcpf(T.n[0] * ux);
    const float S = fabsf(T.n[0]) * gx + fabsf(T.n[1]) * gy + fabsf(T.n[2]) * gz + fabsf(T.d1) + fabsf(T.d2);
    // 3e-23: the product of two offsets below it rounds to zero, and the test passes
    const float mp = (kRowUlp * S + 3e-23f) * fabsf(q);
    R.pl0 = -inf;
    R.ph0 = inf;
    R.py = R.pz = R.pm = 0.0f;
    if (!nnan) {
        if (mp < 1e6f) {
            const float a = -T.d1 * q, b = -T.d2 * q;
            R.pl0 = a < b ? a : b;
            R.ph0 = a < b ? b : a;
            R.py = -T.n[1] * q * uy;
            R.pz = -T.n[2] * q * uz;
            R.pm = mp;
        } else {
            R.pl0 = R.ph0 = 0.0f;
            R.pm = inf;
        }
    }
    R.mono = fin && (nfin || nnan);
    R.xa = T.lo[0];
    R.xb = T.hi[0];
    R.ya = T.lo[1];
    R.za = T.lo[2];
    R.ny = T.hi[1] - T.lo[1] + 1;
    R.nz = T.hi[2] - T.lo[2] + 1;
    R.inv_ny = 1.0f / (float)R.ny;
}

// Row r of a record -> (y, z).
__device__ __forceinline__ void row_yz(const RowRec& R, uint32_t r, int& y, int& z) {
    int zr = (int)((float)r * R.inv_ny);  // within one of r / ny
    int yr = (int)r - __mul24(zr, R.ny);
    if (yr < 0) {
        zr--;
        yr += R.ny;
    } else if (yr >= R.ny) {
        zr++;
        yr -= R.ny;
    }
    y = R.ya + yr;
    z = R.za + zr;
}

// The interval [x0, x1] of a row outside of which no voxel passes (an empty
// one is x0 > x1).  Voxels in it may fail only at the ends named in the
// result: bit 0 from x0 on, bit 1 from x1 down.
__device__ __forceinline__ uint32_t row_estimate(const RowRec& R, int y, int z, int& x0, int& x1) {
    x0 = R.xa;
    x1 = R.xb;
    if (!R.mono) return 3u;
    const float fy = (float)y, fz = (float)z;
    const float t = __builtin_fmaf(R.py, fy, R.pz * fz);
    const float pl = R.pl0 + t, ph = R.ph0 + t;
    // outermost and innermost position of either end
    float lo0 = pl - R.pm, lo1 = pl + R.pm, hi0 = ph + R.pm, hi1 = ph - R.pm;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const float a = __builtin_fmaf(R.xyl[2 + k], fy, R.xyl[k]), b = __builtin_fmaf(R.zxl[2 + k], fz, R.zxl[k]);
        lo0 = fmaxf(lo0, fmaxf(a - R.xyl[4 + k], b - R.zxl[4 + k]));
        lo1 = fmaxf(lo1, fmaxf(a + R.xyl[4 + k], b + R.zxl[4 + k]));
        const float c = __builtin_fmaf(R.xyh[2 + k], fy, R.xyh[k]), d = __builtin_fmaf(R.zxh[2 + k], fz, R.zxh[k]);
        hi0 = fminf(hi0, fminf(c + R.xyh[4 + k], d + R.zxh[4 + k]));
        hi1 = fminf(hi1, fminf(c - R.xyh[4 + k], d - R.zxh[4 + k]));
    }
    const float fa = (float)x0, fb = (float)x1;
    const float a0 = fmaxf(ceilf(lo0), fa), a1 = fmaxf(ceilf(lo1), fa);
    const float b0 = fminf(floorf(hi0), fb), b1 = fminf(floorf(hi1), fb);
    if (a0 > b0) {
        x0 = 1;
        x1 = 0;
        return 0u;
    }
    x0 = (int)a0;
    x1 = (int)b0;
    return (a0 != a1 ? 1u : 0u) | (b0 != b1 ? 2u : 0u);
}

// The tests of vox_device.h decide the voxels x0 .. x1 of row (y, z), whose YZ
// edges pass, at the open ends; run(x0, x1, y, z) gets what passes.
template <class Run>
__device__ __forceinline__ void row_decide(const RowRec& R, const float* unit, int y, int z, int xa, int xb,
                                           uint32_t ends, Run&& run) {
    const float ux = unit[0], py = (float)y * unit[1], pz = (float)z * unit[2];
    const float n0 = R.n[0], nypy = R.n[1] * py, nzpz = R.n[2] * pz, d1 = R.d1, d2 = R.d2;
    float bxy[3], azx[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        bxy[i] = R.xy[3 + i] * py;
        azx[i] = R.zx[i] * pz;
    }
    // the tests that fail at x: bits 0..5 edges, 6 and 7 the plane (its side)
    const auto fails = [&](int x) -> uint32_t {
        const float px = (float)x * ux;
        float t = n0 * px;
        t = t + nypy;
        t = t + nzpz;
        const float A = t + d1;
        const float r = A * (t + d2);
        uint32_t f = r > 0.0f ? (A > 0.0f ? 64u : 128u) : 0u;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            float a = R.xy[i] * px;
            a = a + bxy[i];
            a = a + R.xy[6 + i];
            float b = azx[i];
            b = b + R.zx[3 + i] * px;
            b = b + R.zx[6 + i];
            f |= (a < 0.0f ? 1u << i : 0u) | (b < 0.0f ? 8u << i : 0u);
        }
        return f;
    };
    if (!R.mono) {
        for (int x = xa; x <= xb; x++)
            if (!fails(x)) run(x, x, y, z);
        return;
    }
    uint32_t fl = (ends & 1u) ? fails(xa) : 0u, fr = (ends & 2u) ? fails(xb) : 0u;
    if (fl & fr) return;  // one test fails at both ends, so it fails between them
    while (fl && xa < xb) fl = fails(++xa);
    if (fl) return;
    while (fr && xb > xa) fr = fails(--xb);
    if (!fr) run(xa, xb, y, z);
}

// The rows of nr <= REC published records (`rows`: lane i < nr holds record i's
// number of rows): of their windows of 64 this wave takes every `stride`-th
// from `first` on.  Uniform over the wave.
template <int REC, class Run>
__device__ __forceinline__ void row_round(const RowRec* rec, WaveLists& W, const float* unit, int nr, uint32_t rows,
                                          uint32_t first, uint32_t stride, Run&& run) {
    static_assert(REC <= 64, "a record per lane");
    const int lane = __lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    int held = 0, open = 0;  // rows in the two lists
    const auto decide = [&]() {
        wave_sync();
        if (lane < open) {
            const uint2 it = W.open[lane];
            row_decide(rec[it.x >> 26], unit, (int)(it.x & 0x1FFFu), (int)((it.x >> 13) & 0x1FFFu),
                       (int)(it.y & 0x7FFFu), (int)((it.y >> 15) & 0x7FFFu), it.y >> 30, run);
        }
        wave_sync();
        open = 0;
    };
    const auto finish = [&](int count) {
        uint32_t it = 0, ends = 0;
        int x0 = 0, x1 = 0;
        if (lane < count) {
            it = W.list[lane];
            const int y = (int)(it & 0x1FFFu), z = (int)((it >> 13) & 0x1FFFu);
            ends = row_estimate(rec[it >> 26], y, z, x0, x1);
            if (!ends && x0 <= x1) run(x0, x1, y, z);
        }
        const unsigned long long b = __ballot(ends != 0u);
        if (!b) return;
        const int k = (int)__popcll(b);
        if (open + k > 64) decide();
        if (ends)
            W.open[open + (int)__popcll(b & below)] =
                make_uint2(it, (uint32_t)x0 | ((uint32_t)x1 << 15) | (ends << 30));
        open += k;
    };
    uint32_t incl = rows;
#pragma unroll
    for (int d = 1; d < REC; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
    }
    const uint32_t total = __shfl(incl, REC - 1);
    const uint32_t start = lane < nr ? incl - rows : 0xFFFFFFFFu;
    for (uint32_t j0 = first * 64u; j0 < total; j0 += stride * 64u) {
        const uint32_t j = j0 + (uint32_t)lane;
        // the record of row j: the last that starts at or before it
        int o = (int)__popcll(__ballot(start <= j0)) - 1;
        const int last = (int)__popcll(__ballot(start <= j0 + 63u)) - 1;
        for (int k = o + 1; k <= last; k++) o += (uint32_t)__builtin_amdgcn_readlane((int)start, k) <= j ? 1 : 0;
        const uint32_t r = j - (uint32_t)__shfl((int)start, o);
        bool ok = false;
        int y = 0, z = 0;
        if (j < total) {
            const RowRec& R = rec[o];
            row_yz(R, r, y, z);
            ok = pass3(R.yz, (float)y * unit[1], (float)z * unit[2]);
        }
        const unsigned long long b = __ballot(ok);
        if (ok) W.list[held + (int)__popcll(b & below)] = ((uint32_t)o << 26) | ((uint32_t)z << 13) | (uint32_t)y;
        held += (int)__popcll(b);
        if (held >= 64) {
            wave_sync();
            finish(64);
            held -= 64;
            const uint32_t rest = W.list[64 + lane];
            wave_sync();
            if (lane < held) W.list[lane] = rest;
        }
    }
    wave_sync();
    if (held) finish(held);
    if (open) decide();
}

// Rasterizes the triangles of the threads with `big`, REC of them at a time.
// count[w] holds the number of them in wave w (written by that wave before a
// barrier); setup(i, T) gives thread i's triangle (box not empty).  Called by
// every thread of the workgroup.
//
// One wave sets up a round's records, so REC lanes of 64 do what took a wave
// to itself for every five of its own triangles before (24.5 -> 19.5 million
// instructions for a soup of 100,003 at 256^3), and all waves share the rows
// of whichever triangles are large.
template <int REC, int WAVES, class Setup, class Run>
__device__ __forceinline__ void block_rows(BlockRows<REC, WAVES>& W, const uint32_t* count, const vox_info& info,
                                           bool big, uint32_t first, uint32_t stride, Setup&& setup, Run&& run) {
    const int lane = __lane_id(), wave = (int)(threadIdx.x >> 6);
    int base = 0, nq = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        base += w < wave ? (int)count[w] : 0;
        nq += (int)count[w];
    }
    if (!nq) return;
    const unsigned long long mine = __ballot(big);
    if (big) W.queue[base + (int)__popcll(mine & ((1ull << lane) - 1ull))] = (uint8_t)threadIdx.x;
    const float unit[3] = {info.unit[0], info.unit[1], info.unit[2]};
    int turn = 0;
    for (int r0 = 0; r0 < nq; r0 += REC) {
        const int nr = nq - r0 < REC ? nq - r0 : REC;
        __syncthreads();  // the queue is written, the previous round's records have been read
        if (wave == turn && lane < nr) {
            SurfTri T;
            setup((uint32_t)W.queue[r0 + lane], T);
            row_publish(W.rec[lane], T, info);
        }
        turn = turn + 1 < WAVES ? turn + 1 : 0;
        __syncthreads();
        const uint32_t rows = lane < nr ? (uint32_t)W.rec[lane].ny * (uint32_t)W.rec[lane].nz : 0u;
        row_round<REC>(W.rec, W.wave[wave], unit, nr, rows, first * WAVES + (uint32_t)wave, stride * WAVES, run);
    }
}

}  // namespace voxamd
