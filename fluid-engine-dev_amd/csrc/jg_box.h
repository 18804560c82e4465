// jg_box.h -- the part of a system that a solve has to visit.
//
// A pressure system of a free surface is mostly empty: the rows of air and
// solid cells couple to nothing and their right-hand side is zero (60% fluid
// in the sphere pool, 35% in the torus pool, 20% in the dam break), yet
// every pass of a solve streams them.  Such a cell's solution is zero, and no
// other row reads it.  So a solve first finds the bounding box of the cells
// that take part, and where that is clearly smaller than the grid it copies
// the box's rows and right-hand side into dense arrays, runs on them, and
// scatters the solution.
//
// A cell takes part when its right-hand side is not zero, it couples to
// another cell (both ends then take part), or its centre is not a finite
// number of the working precision; a NaN compares unequal, so it takes part.
// Everything left out is exactly decoupled, whoever wrote the matrix.  The
// multigrid levels use the same box, aligned so that it halves with them: the
// coarse operators restricted to it are principal submatrices of the
// caller's, so the V-cycle stays symmetric and positive definite whatever
// they hold outside.
//
// The scan reads little but what is left out (about 50 us at 256^3 with 40%
// of the cells empty), the copy reads and writes the box once (0.1 ms there),
// against 13 V-cycles over the difference.  Whole steps (build, solve,
// gradient), before and after: sphere pool 256^3 mixed 12.9 -> 9.8 ms, torus
// pool 512^3 mixed 60.0 -> 35.6, dam break 192x160x144 FP64 6.34 -> 3.06,
// 2-D pool 2048x1536 FP64 14.4 -> 10.9.
#pragma once

#include "jg_device.h"

namespace jg {

// A box of cells of a grid d: origin o, size n.
struct Box {
    int o[3];
    Dims n;
};

__global__ void k_box_reset(BoxScan* box) {
    if (threadIdx.x < 3) {
        box->lo[threadIdx.x] = 0x7fffffff;
        box->hi[threadIdx.x] = -1;
    }
}

// One wave's row of 64 cells at (x0.., j, k), lane = x.  in: the lane's cell is
// inside the grid (one outside takes no part).
struct BoxCell {
    Row<double> row;
    double b;
};
__device__ __forceinline__ BoxCell box_load(const Row<double>* __restrict__ A, const double* __restrict__ b,
                                            const Dims& d, int x0, int j, int k, bool in) {
    BoxCell v{{1.0, 0.0, 0.0, 0.0}, 0.0};
    if (in) {
        const idx_t c = x0 + (int)(threadIdx.x & 63) + (idx_t)d.nx * (j + (idx_t)d.ny * k);
        v.row = A[c];
        v.b = b[c];
    }
    return v;
}
// Widens the running bounds by that row.
__device__ __forceinline__ void box_vote(const BoxCell& v, double most, int x0, int j, int k, int lo[3],
                                         int hi[3]) {
    const Row<double>& row = v.row;
    const double bv = v.b;
    const bool cr = row.r != 0.0, cu = row.u != 0.0, cf = row.f != 0.0;
    const unsigned long long on = __ballot(cr || cu || cf || bv != 0.0 || !(fabs(row.c) <= most));
    if (!on) return;
    const unsigned long long right = __ballot(cr);
    const int last = 63 - __clzll(on);
    lo[0] = min(lo[0], x0 + __ffsll(on) - 1);
    hi[0] = max(hi[0], x0 + (right ? max(last, 64 - __clzll(right)) : last));
    lo[1] = min(lo[1], j);
    hi[1] = max(hi[1], j + (__ballot(cu) ? 1 : 0));
    lo[2] = min(lo[2], k);
    hi[2] = max(hi[2], k + (__ballot(cf) ? 1 : 0));
}

__device__ __forceinline__ void box_widen(BoxScan* box, const int lo[3], const int hi[3]) {
    if ((threadIdx.x & 63) != 0 || hi[0] < 0) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (lo[a] < __hip_atomic_load(&box->lo[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&box->lo[a], lo[a]);
        if (hi[a] > __hip_atomic_load(&box->hi[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&box->hi[a], hi[a]);
    }
}

// Cells of a block: 64 in x, kBoxY rows, kBoxZ planes.
constexpr int kBoxY = 4, kBoxZ = 16;
constexpr int kBoxSamples = 2048;  // rows of 64 cells that the sample reads

// The scan, in two launches.  SAMPLE: whole grid rows spread over the system,
// an odd step apart (at every height), and the last one, for a first guess; a
// few waves read some 16 rows of 64 cells each, four at a time.  (With a row per
// wave the waves' first atomics on the bounds took 75 us at 256^3 and 185 us on
// a 2048 x 1536 plane; 512 grid rows whatever their length, one after the
// other, 26 us at 256^3, 82 on a 1000 x 1000 plane and 117 on 3000 x 2000; so
// 28, 27 and 28.)
// Otherwise a block looks at its cells only where they reach beyond the box
// found so far: a dense system is hardly read, and of a free-surface one what
// is read is the part that every pass of the solve then leaves out.
template <bool SAMPLE>
__global__ __launch_bounds__(64 * kBoxY) void k_box_scan(const Row<double>* __restrict__ A,
                                                         const double* __restrict__ b, Dims d, double most,
                                                         BoxScan* __restrict__ box) {
    const int x0 = blockIdx.x * 64;
    const bool in = x0 + (int)(threadIdx.x & 63) < d.nx;
    const int w = threadIdx.x >> 6;
    int lo[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, hi[3] = {-1, -1, -1};
    if (SAMPLE) {
        const idx_t rows = (idx_t)d.ny * d.nz, step = rows * gridDim.x / kBoxSamples | 1;
        const idx_t next = (idx_t)gridDim.y * kBoxY * step;
        auto load = [&](idx_t r) { return box_load(A, b, d, x0, (int)(r % d.ny), (int)(r / d.ny), in && r < rows); };
        auto vote = [&](const BoxCell& v, idx_t r) { box_vote(v, most, x0, (int)(r % d.ny), (int)(r / d.ny), lo, hi); };
        for (idx_t r = (blockIdx.y * kBoxY + w) * step; r < rows; r += 4 * next) {
            BoxCell v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = load(r + q * next);
#pragma unroll
            for (int q = 0; q < 4; ++q) vote(v[q], r + q * next);
        }
        if (blockIdx.y == 0 && w == 0) vote(load(rows - 1), rows - 1);
    } else {
        const int y0 = blockIdx.y * kBoxY, k0 = blockIdx.z * kBoxZ;
        const int x1 = min(x0 + 63, d.nx - 1), y1 = min(y0 + kBoxY, d.ny) - 1, k1 = min(k0 + kBoxZ, d.nz) - 1;
        int cl[3], ch[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            cl[a] = __hip_atomic_load(&box->lo[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ch[a] = __hip_atomic_load(&box->hi[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // (a cell on the box's upper faces may couple beyond it: inside means
        // below them, or at the grid's end)
        const bool inside = x0 >= cl[0] && y0 >= cl[1] && k0 >= cl[2] && (x1 < ch[0] || ch[0] == d.nx - 1) &&
                            (y1 < ch[1] || ch[1] == d.ny - 1) && (k1 < ch[2] || ch[2] == d.nz - 1);
        if (inside) return;
        const int j = y0 + w;
        if (j < d.ny) {
            for (int k = k0; k <= k1; k += 4) {
                BoxCell v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = box_load(A, b, d, x0, j, k + q, in && k + q <= k1);
#pragma unroll
                for (int q = 0; q < 4; ++q) box_vote(v[q], most, x0, j, k + q, lo, hi);
            }
        }
    }
    box_widen(box, lo, hi);
}

// Rows of the box, dense: to64 and / or to32.  ALL: over the whole level,
// checking that what lies outside the box is finite too (*odd is set if not:
// a solve of the whole grid would have met it).
template <bool ALL>
__global__ __launch_bounds__(256) void k_box_rows(const Row<double>* __restrict__ A, Dims d, Box box,
                                                  double most, Row<double>* __restrict__ to64,
                                                  Row<float>* __restrict__ to32, int* __restrict__ odd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    const Dims over = ALL ? d : box.n;
    if (i >= over.nx || j >= over.ny) return;
    const int bi = ALL ? i - box.o[0] : i, bj = ALL ? j - box.o[1] : j, bk = ALL ? k - box.o[2] : k;
    const Row<double> r =
        A[bi + box.o[0] + (idx_t)d.nx * (bj + box.o[1] + (idx_t)d.ny * (bk + box.o[2]))];
    if (!ALL || ((unsigned)bi < (unsigned)box.n.nx && (unsigned)bj < (unsigned)box.n.ny &&
                 (unsigned)bk < (unsigned)box.n.nz)) {
        const idx_t c = bi + (idx_t)box.n.nx * (bj + (idx_t)box.n.ny * bk);
        if (to64) to64[c] = r;
        if (to32) to32[c] = Row<float>{(float)r.c, (float)r.r, (float)r.u, (float)r.f};
    } else if (!(fabs(r.c) <= most && fabs(r.r) <= most && fabs(r.u) <= most && fabs(r.f) <= most)) {
        *odd = 1;
    }
}

__global__ __launch_bounds__(256) void k_box_gather(const double* __restrict__ v, Dims d, Box box,
                                                    double* __restrict__ to) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= box.n.nx || j >= box.n.ny) return;
    to[i + (idx_t)box.n.nx * (j + (idx_t)box.n.ny * k)] =
        v[i + box.o[0] + (idx_t)d.nx * (j + box.o[1] + (idx_t)d.ny * (k + box.o[2]))];
}

// The whole grid's vector from the box's: zero outside.
__global__ __launch_bounds__(256) void k_box_scatter(const double* __restrict__ v, Dims d, Box box,
                                                     double* __restrict__ to) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= d.nx || j >= d.ny) return;
    const int bi = i - box.o[0], bj = j - box.o[1], bk = k - box.o[2];
    const bool in = (unsigned)bi < (unsigned)box.n.nx && (unsigned)bj < (unsigned)box.n.ny &&
                    (unsigned)bk < (unsigned)box.n.nz;
    to[i + (idx_t)d.nx * (j + (idx_t)d.ny * k)] =
        in ? v[bi + (idx_t)box.n.nx * (bj + (idx_t)box.n.ny * bk)] : 0.0;
}

}  // namespace jg
