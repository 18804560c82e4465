// jg_boundary.h -- the velocity boundary conditions Jet applies after the
// pressure projection: GridFractionalBoundaryConditionSolver3::
// constrainVelocity (src/jet/grid_fractional_boundary_condition_solver3.cpp:
// 26-232) and the blocked solver's extra pass (src/jet/grid_blocked_boundary_
// condition_solver3.cpp:23-69), for a rigid-body collider.
//
// A face whose SDF samples can only see positive cells lies outside the
// collider: it is valid, keeps its velocity and is read by others only.  So
// the stages run over lists of the other faces (one list per axis), and a
// call's traffic is one read of the SDF plus the collider's surroundings:
//   bits       one bit per cell, sdf > 0 (one read of the SDF);
//   dilate     one bit per cell, every cell of its 3^3 neighbourhood positive;
//   list       the faces with a cell whose bit is not set, per axis;
//   init       marker of the face (1 where any part of it is outside the
//              collider), collider velocity on fully covered faces;
//   extrapolate one pass of extrapolateToRegion (include/jet/detail/
//              array_utils-inl.h:172-241) -- a pass writes only faces that were
//              invalid and reads only faces that were valid at its start, so
//              its faces are independent; validity ping-pongs between two
//              byte arrays, which hold 1 outside the lists at all times;
//   project    no-flux projection with friction inside the collider, into a
//              scratch copy (it samples all three extrapolated components);
//   finish     copy back, zeroing the closed domain walls; in the blocked
//              solver, faces between a collider cell and a fluid cell take the
//              collider velocity.
// FP64 with contraction off, in Jet's operand order: the result is bitwise
// Jet's, and does not depend on the order of a list.
//
// On 256 x 224 x 240 cells with eight spheres the kernels take 172 us, 33 of
// them the read of the SDF (3.3 TB/s) and 48 five extrapolation passes, each
// of which is a chain of dependent misses (list, masks and neighbours,
// store); every stage over every face took 2.08 ms (990 us in the
// projection, 530 in the markers, 330 in the extrapolation).
#pragma once

#include "jg_device.h"

namespace jg {

// Cells nx*ny*nz, spacing and origin of the face-centred grid.
struct BcGrid {
    Dims d;
    double h[3], o[3];
};

// RigidBodyCollider3 (velocities, surface translation) and Collider3's friction.
struct BcCollider {
    double lin[3], ang[3], tr[3], friction;
};

// Face grid of axis A: sizes and data origin o + h/2 off the axis
// (src/jet/face_centered_grid3.cpp:216-238, 437-447).
template <int A>
__device__ __forceinline__ void bc_face_dims(const Dims& d, int s[3]) {
    s[0] = d.nx + (A == 0);
    s[1] = d.ny + (A == 1);
    s[2] = d.nz + (A == 2);
}
template <int A>
__device__ __forceinline__ void bc_face_origin(const BcGrid& g, double fo[3]) {
#pragma clang fp contract(off)
    for (int b = 0; b < 3; ++b) fo[b] = g.o[b] + 0.5 * (b == A ? 0.0 : g.h[b]);
}
__device__ __forceinline__ void bc_pos(const double fo[3], const double h[3], int i, int j, int k,
                                       double p[3]) {
#pragma clang fp contract(off)
    p[0] = fo[0] + h[0] * (double)i;
    p[1] = fo[1] + h[1] * (double)j;
    p[2] = fo[2] + h[2] * (double)k;
}

// RigidBodyCollider3::velocityAt (src/jet/rigid_body_collider3.cpp:25-28) with
// Vector3::cross (include/jet/detail/vector3-inl.h:125-127).
__device__ __forceinline__ void bc_collider_velocity(const BcCollider& c, const double p[3],
                                                     double out[3]) {
#pragma clang fp contract(off)
    const double r0 = p[0] - c.tr[0], r1 = p[1] - c.tr[1], r2 = p[2] - c.tr[2];
    out[0] = c.lin[0] + (c.ang[1] * r2 - r1 * c.ang[2]);
    out[1] = c.lin[1] + (c.ang[2] * r0 - r2 * c.ang[0]);
    out[2] = c.lin[2] + (c.ang[0] * r1 - r0 * c.ang[1]);
}

// getBarycentric (include/jet/detail/math_utils-inl.h:147-175), iLow = 0.
__device__ __forceinline__ void bc_barycentric(double x, int ihigh, int& i, double& f) {
#pragma clang fp contract(off)
    const double s = floor(x);
    i = (int)s;
    if (ihigh == 0) {
        i = 0;
        f = 0;
    } else if (i < 0) {
        i = 0;
        f = 0;
    } else if (i > ihigh - 1) {
        i = ihigh - 1;
        f = 1;
    } else {
        f = x - s;
    }
}

__device__ __forceinline__ double bc_lerp(double a, double b, double f) {
#pragma clang fp contract(off)
    return (1 - f) * a + f * b;  // include/jet/detail/math_utils-inl.h:177-180
}

// LinearArraySampler3::operator() (include/jet/detail/array_samplers3-inl.h:
// 116-156): data of size s at data origin dorg, spacing h.
__device__ double bc_sample(const double* __restrict__ data, const int s[3], const double h[3],
                            const double dorg[3], const double p[3]) {
#pragma clang fp contract(off)
    int i, j, k;
    double fx, fy, fz;
    bc_barycentric((p[0] - dorg[0]) / h[0], s[0] - 1, i, fx);
    bc_barycentric((p[1] - dorg[1]) / h[1], s[1] - 1, j, fy);
    bc_barycentric((p[2] - dorg[2]) / h[2], s[2] - 1, k, fz);
    const int ip1 = min(i + 1, s[0] - 1), jp1 = min(j + 1, s[1] - 1), kp1 = min(k + 1, s[2] - 1);
    auto D = [&](int a, int b, int c) { return data[a + (idx_t)s[0] * (b + (idx_t)s[1] * c)]; };
    const double b0 = bc_lerp(bc_lerp(D(i, j, k), D(ip1, j, k), fx),
                              bc_lerp(D(i, jp1, k), D(ip1, jp1, k), fx), fy);
    const double b1 = bc_lerp(bc_lerp(D(i, j, kp1), D(ip1, j, kp1), fx),
                              bc_lerp(D(i, jp1, kp1), D(ip1, jp1, kp1), fx), fy);
    return bc_lerp(b0, b1, fz);
}

// The collider SDF (cell-centred, data origin o + h/2) at p.
__device__ __forceinline__ double bc_sdf(const double* __restrict__ sdf, const BcGrid& g,
                                         const double p[3]) {
#pragma clang fp contract(off)
    const int s[3] = {g.d.nx, g.d.ny, g.d.nz};
    const double dorg[3] = {g.o[0] + 0.5 * g.h[0], g.o[1] + 0.5 * g.h[1], g.o[2] + 0.5 * g.h[2]};
    return bc_sample(sdf, s, g.h, dorg, p);
}

// ScalarGrid3::gradient (src/jet/scalar_grid3.cpp:89-102): the weights of
// getCoordinatesAndWeights (include/jet/detail/array_samplers3-inl.h:152-194,
// which scales by 1/h) on gradient3 at the 8 data points (src/jet/fdm_utils.cpp:49-67).
__device__ void bc_sdf_gradient(const double* __restrict__ sdf, const BcGrid& g, const double p[3],
                                double out[3]) {
#pragma clang fp contract(off)
    const int s[3] = {g.d.nx, g.d.ny, g.d.nz};
    int lo[3], hi[3];
    double f[3];
    for (int a = 0; a < 3; ++a) {
        const double dorg = g.o[a] + 0.5 * g.h[a];
        const double inv = 1.0 / g.h[a];
        bc_barycentric((p[a] - dorg) * inv, s[a] - 1, lo[a], f[a]);
        hi[a] = min(lo[a] + 1, s[a] - 1);
    }
    const double fx = f[0], fy = f[1], fz = f[2];
    const double wt[8] = {(1 - fx) * (1 - fy) * (1 - fz), fx * (1 - fy) * (1 - fz),
                          (1 - fx) * fy * (1 - fz),       fx * fy * (1 - fz),
                          (1 - fx) * (1 - fy) * fz,       fx * (1 - fy) * fz,
                          (1 - fx) * fy * fz,             fx * fy * fz};
    auto D = [&](int a, int b, int c) { return sdf[a + (idx_t)s[0] * (b + (idx_t)s[1] * c)]; };
    out[0] = out[1] = out[2] = 0.0;
    for (int q = 0; q < 8; ++q) {
        const int i = (q & 1) ? hi[0] : lo[0];
        const int j = (q & 2) ? hi[1] : lo[1];
        const int k = (q & 4) ? hi[2] : lo[2];
        const double left = D(i > 0 ? i - 1 : i, j, k), right = D(i + 1 < s[0] ? i + 1 : i, j, k);
        const double down = D(i, j > 0 ? j - 1 : j, k), up = D(i, j + 1 < s[1] ? j + 1 : j, k);
        const double back = D(i, j, k > 0 ? k - 1 : k), front = D(i, j, k + 1 < s[2] ? k + 1 : k);
        out[0] += wt[q] * (0.5 * (right - left) / g.h[0]);
        out[1] += wt[q] * (0.5 * (up - down) / g.h[1]);
        out[2] += wt[q] * (0.5 * (front - back) / g.h[2]);
    }
}

// projectAndApplyFriction (src/jet/physics_helpers.h:34-45).
__device__ __forceinline__ void bc_friction(const double vel[3], const double n[3], double friction,
                                            double out[3]) {
#pragma clang fp contract(off)
    const double dn = vel[0] * n[0] + vel[1] * n[1] + vel[2] * n[2];
    out[0] = vel[0] - n[0] * dn;
    out[1] = vel[1] - n[1] * dn;
    out[2] = vel[2] - n[2] * dn;
    if (out[0] * out[0] + out[1] * out[1] + out[2] * out[2] > 0) {
        const double nd = -(vel[0] * n[0] + vel[1] * n[1] + vel[2] * n[2]);
        const double veln = nd < 0.0 ? 0.0 : nd;
        double sc = 1.0 - friction * veln / sqrt(out[0] * out[0] + out[1] * out[1] + out[2] * out[2]);
        sc = sc < 0.0 ? 0.0 : sc;
        out[0] *= sc;
        out[1] *= sc;
        out[2] *= sc;
    }
}

// fractionInsideSdf (include/jet/detail/level_set_utils-inl.h:51-62).
__device__ __forceinline__ double bc_fraction_inside_sdf(double phi0, double phi1) {
#pragma clang fp contract(off)
    if (phi0 < 0 && phi1 < 0) return 1;
    if (phi0 < 0 && !(phi1 < 0)) return phi0 / (phi0 - phi1);
    if (!(phi0 < 0) && phi1 < 0) return phi1 / (phi1 - phi0);
    return 0;
}

// ------------------------------------------------------------ face lists

// Words of 64 cells per x row, and of 64 faces (the u row has nx + 1).
__host__ __device__ inline int bc_cell_words(const Dims& d) { return (d.nx + 63) / 64; }
__host__ __device__ inline int bc_face_words(const Dims& d) { return d.nx / 64 + 1; }

// The faces that need work, per axis: index lists and their lengths.
struct BcLists {
    unsigned* f[3];
    unsigned* count;
};

// Every face valid: the masks' state between calls.
__global__ __launch_bounds__(256) void k_bc_valid(int8_t* __restrict__ v, idx_t n) {
    for (idx_t f = blockIdx.x * (idx_t)256 + threadIdx.x; f < n; f += (idx_t)gridDim.x * 256) v[f] = 1;
}

// Bit x of word w of a row: sdf > 0 at cell 64 w + x (set past the row's end;
// a NaN is not positive).  all != 0: no cell counts as positive, so that
// every face is listed.  Each wave reads eight words at a time.  Also zeroes
// the list lengths.
__global__ __launch_bounds__(256) void k_bc_bits(const double* __restrict__ sdf, Dims d, int all,
                                                 unsigned long long* __restrict__ bits,
                                                 unsigned* __restrict__ count) {
    if (blockIdx.x == 0 && threadIdx.x < 3) count[threadIdx.x] = 0;
    const int lane = threadIdx.x & 63, W = bc_cell_words(d);
    const idx_t words = (idx_t)W * d.ny * d.nz;
    const idx_t wave = blockIdx.x * (idx_t)4 + (threadIdx.x >> 6), waves = (idx_t)gridDim.x * 4;
    for (idx_t w0 = wave * 8; w0 < words; w0 += waves * 8) {
        bool pos[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const idx_t w = w0 + q, row = w / W;
            const int x = (int)(w - row * W) * 64 + lane;
            pos[q] = true;
            if (w < words && x < d.nx) pos[q] = !all && sdf[row * d.nx + x] > 0;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const unsigned long long m = __ballot(pos[q]);
            if (lane == 0 && w0 + q < words) bits[w0 + q] = m;
        }
    }
}

// Bit of a cell: every cell of its 3^3 neighbourhood inside the grid is
// positive.  A sample at a cell centre reads within that neighbourhood
// whichever way its coordinate rounds.
__global__ __launch_bounds__(256) void k_bc_dilate(const unsigned long long* __restrict__ bits, Dims d,
                                                   unsigned long long* __restrict__ out) {
    const int W = bc_cell_words(d);
    const idx_t words = (idx_t)W * d.ny * d.nz;
    const idx_t w = blockIdx.x * (idx_t)256 + threadIdx.x;
    if (w >= words) return;
    const int x = (int)(w % W), j = (int)((w / W) % d.ny), k = (int)(w / ((idx_t)W * d.ny));
    unsigned long long m = ~0ull;
#pragma unroll
    for (int b = -1; b <= 1; ++b)
#pragma unroll
        for (int a = -1; a <= 1; ++a) {
            const int jj = min(max(j + a, 0), d.ny - 1), kk = min(max(k + b, 0), d.nz - 1);
            const unsigned long long* row = bits + (idx_t)W * (jj + (idx_t)d.ny * kk);
            const unsigned long long c = row[x];
            const unsigned long long l = x > 0 ? row[x - 1] >> 63 : 1ull;
            const unsigned long long r = x + 1 < W ? row[x + 1] << 63 : 1ull << 63;
            m &= c & (c << 1 | l) & (c >> 1 | r);
        }
    out[w] = m;
}

// The lists: a face is left out when both its cells' bits are set (a cell
// beyond the domain counts as set: its sample is clamped to the other's
// neighbourhood).  One thread per word of faces.  Room is reserved by one
// atomic per axis and block of 1024 words: per wave, the same-address
// atomics of all XCDs took 37 us of a 256 x 224 x 240 call.
constexpr int kBcListThreads = 1024;
__global__ __launch_bounds__(kBcListThreads) void k_bc_list(const unsigned long long* __restrict__ open,
                                                            Dims d, BcLists lists) {
    constexpr int NW = kBcListThreads / 64;
    __shared__ unsigned wsum[3][NW], wbase[3][NW];
    const int W = bc_cell_words(d), F = bc_face_words(d), lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const idx_t w = blockIdx.x * (idx_t)kBcListThreads + threadIdx.x;
    const idx_t plane = (idx_t)F * (d.ny + 1);
    const int x = (int)(w % F), j = (int)((w / F) % (d.ny + 1)), k = (int)min((idx_t)d.nz + 1, w / plane);
    auto at = [&](int a, int b, int c) -> unsigned long long {
        if (a < 0 || a >= W || b < 0 || b >= d.ny || c < 0 || c >= d.nz) return ~0ull;
        return open[a + (idx_t)W * (b + (idx_t)d.ny * c)];
    };
    // bits of the word that are faces of a row of n faces
    auto row = [&](int n) -> unsigned long long {
        const int left = n - 64 * x;
        return left >= 64 ? ~0ull : (left > 0 ? (1ull << left) - 1 : 0ull);
    };
    unsigned long long m[3] = {0, 0, 0};
    if (k <= d.nz) {
        const unsigned long long c = at(x, j, k);
        if (j < d.ny && k < d.nz) m[0] = ~(c & (c << 1 | at(x - 1, j, k) >> 63)) & row(d.nx + 1);
        if (k < d.nz) m[1] = ~(c & at(x, j - 1, k)) & row(d.nx);
        if (j < d.ny) m[2] = ~(c & at(x, j, k - 1)) & row(d.nx);
    }
    unsigned before[3];  // faces of the wave's earlier words
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const unsigned n = (unsigned)__popcll(m[a]);
        unsigned sum = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned t = __shfl_up(sum, o, 64);
            if (lane >= o) sum += t;
        }
        if (lane == 63) wsum[a][wv] = sum;
        before[a] = sum - n;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        unsigned total = 0;
        for (int q = 0; q < NW; ++q) total += wsum[threadIdx.x][q];
        unsigned base = total > 0 ? atomicAdd(&lists.count[threadIdx.x], total) : 0;
        for (int q = 0; q < NW; ++q) {
            wbase[threadIdx.x][q] = base;
            base += wsum[threadIdx.x][q];
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const unsigned base = wbase[a][wv] + before[a];
        const unsigned f0 = (unsigned)(64 * x + (idx_t)(d.nx + (a == 0)) * (j + (idx_t)(d.ny + (a == 1)) * k));
        // word by word, a lane per bit: a word's entries are written side by side
        for (unsigned long long todo = __ballot(m[a] != 0); todo; todo &= todo - 1) {
            const int src = __ffsll(todo) - 1;
            const unsigned long long bits =
                (unsigned long long)(unsigned)__shfl((int)(unsigned)(m[a] >> 32), src, 64) << 32 |
                (unsigned)__shfl((int)(unsigned)m[a], src, 64);
            const unsigned to = __shfl(base, src, 64), from = __shfl(f0, src, 64);
            if (bits >> lane & 1)
                lists.f[a][to + __popcll(bits & ((1ull << lane) - 1))] = from + lane;
        }
    }
}

// Loop over the listed faces of axis A: e numbers the entry, f the face.
#define JG_BC_LISTED(A, g, lists, s, e, f)                                           \
    int s[3];                                                                        \
    bc_face_dims<A>((g).d, s);                                                       \
    const unsigned listed = (lists).count[A];                                        \
    for (unsigned e = blockIdx.x * blockDim.x + threadIdx.x, f = 0;                  \
         e < listed && (f = (lists).f[A][e], true); e += gridDim.x * blockDim.x)

// (i, j, k) of face f of a grid of faces of size s.
__device__ __forceinline__ void bc_face_ijk(unsigned f, const int s[3], int& i, int& j, int& k) {
    const unsigned r = f / (unsigned)s[0];
    i = (int)(f - r * (unsigned)s[0]);
    k = (int)(r / (unsigned)s[1]);
    j = (int)(r - (unsigned)k * (unsigned)s[1]);
}

// What the stages share: the faces, the scratch and the lists; the grid's y
// index of a launch is the axis.
struct BcArgs {
    BcGrid g;
    BcCollider c;
    const double* sdf;
    double* comp[3];
    double* tmp[3];  // per list entry
    int8_t* valid[2][3];
    BcLists lists;
};

// Stage 1 (grid_fractional_boundary_condition_solver3.cpp:54-102): the face
// is valid (1) unless its whole extent lies in the collider; there it takes
// the collider velocity.
template <int A>
__device__ __forceinline__ void bc_init(const BcArgs& p) {
#pragma clang fp contract(off)
    const BcGrid& g = p.g;
    double fo[3];
    bc_face_origin<A>(g, fo);
    JG_BC_LISTED(A, g, p.lists, s, e, f) {
        int i, j, k;
        bc_face_ijk(f, s, i, j, k);
        double x[3], q0[3], q1[3];
        bc_pos(fo, g.h, i, j, k, x);
        for (int b = 0; b < 3; ++b) {
            const double off = b == A ? 0.5 * g.h[A] : 0.0;
            q0[b] = x[b] - off;
            q1[b] = x[b] + off;
        }
        double frac = bc_fraction_inside_sdf(bc_sdf(p.sdf, g, q0), bc_sdf(p.sdf, g, q1));
        frac = 1.0 - (frac < 0.0 ? 0.0 : (frac > 1.0 ? 1.0 : frac));  // clamp(frac, 0, 1)
        if (frac > 0.0) {
            p.valid[0][A][f] = 1;
        } else {
            double cv[3];
            bc_collider_velocity(p.c, x, cv);
            p.comp[A][f] = cv[A];
            p.valid[0][A][f] = 0;
        }
    }
}
__global__ __launch_bounds__(256) void k_bc_init(BcArgs p) {
    if (blockIdx.y == 0) bc_init<0>(p);
    else if (blockIdx.y == 1) bc_init<1>(p);
    else bc_init<2>(p);
}

// Stage 2: one pass of extrapolateToRegion, neighbour order +x, -x, +y, -y,
// +z, -z as Jet's.
template <int A>
__device__ __forceinline__ void bc_extrapolate(const BcArgs& p, int in) {
#pragma clang fp contract(off)
    double* comp = p.comp[A];
    const int8_t* v0 = p.valid[in][A];
    int8_t* v1 = p.valid[1 - in][A];
    // Every load a face may need is issued at once: taken one condition at a
    // time, a pass over a short list costs its chain of dependent misses.
    JG_BC_LISTED(A, p.g, p.lists, s, e, f) {
        int i, j, k;
        bc_face_ijk(f, s, i, j, k);
        const idx_t sy = s[0], sz = (idx_t)s[0] * s[1], c = f;
        const bool in6[6] = {i + 1 < s[0], i > 0, j + 1 < s[1], j > 0, k + 1 < s[2], k > 0};
        const idx_t off[6] = {1, -1, sy, -sy, sz, -sz};
        int8_t ok[6];
        double val[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const idx_t n = in6[q] ? c + off[q] : c;
            ok[q] = v0[n];
            val[q] = comp[n];
        }
        if (v0[c]) {
            v1[c] = 1;
            continue;
        }
        double sum = 0.0;
        unsigned count = 0;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (in6[q] && ok[q]) {
                sum += val[q];
                ++count;
            }
        if (count > 0) {
            comp[c] = sum / (double)count;
            v1[c] = 1;
        } else {
            v1[c] = 0;
        }
    }
}
__global__ __launch_bounds__(256) void k_bc_extrapolate(BcArgs p, int in) {
    if (blockIdx.y == 0) bc_extrapolate<0>(p, in);
    else if (blockIdx.y == 1) bc_extrapolate<1>(p, in);
    else bc_extrapolate<2>(p, in);
}

// Stage 3 (:104-176): inside the collider, the velocity relative to the
// collider loses its normal component and friction scales the tangential
// one; elsewhere the value is kept.  Reads u, v, w; writes tmp.
template <int A>
__device__ __forceinline__ void bc_project(const BcArgs& p) {
#pragma clang fp contract(off)
    const BcGrid& g = p.g;
    double fo[3];
    bc_face_origin<A>(g, fo);
    JG_BC_LISTED(A, g, p.lists, s, e, f) {
        int i, j, k;
        bc_face_ijk(f, s, i, j, k);
        double x[3];
        bc_pos(fo, g.h, i, j, k, x);
        if (!(bc_sdf(p.sdf, g, x) < 0)) {
            p.tmp[A][e] = p.comp[A][f];
            continue;
        }
        double cv[3], vel[3], gr[3];
        bc_collider_velocity(p.c, x, cv);
        {
            int su[3], sv[3], sw[3];
            double ou[3], ov[3], ow[3];
            bc_face_dims<0>(g.d, su);
            bc_face_dims<1>(g.d, sv);
            bc_face_dims<2>(g.d, sw);
            bc_face_origin<0>(g, ou);
            bc_face_origin<1>(g, ov);
            bc_face_origin<2>(g, ow);
            vel[0] = bc_sample(p.comp[0], su, g.h, ou, x);  // FaceCenteredGrid3::sample
            vel[1] = bc_sample(p.comp[1], sv, g.h, ov, x);
            vel[2] = bc_sample(p.comp[2], sw, g.h, ow, x);
        }
        bc_sdf_gradient(p.sdf, g, x, gr);
        if (gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2] > 0.0) {
            const double l = sqrt(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2]);
            const double nrm[3] = {gr[0] / l, gr[1] / l, gr[2] / l};
            const double velr[3] = {vel[0] - cv[0], vel[1] - cv[1], vel[2] - cv[2]};
            double velt[3];
            bc_friction(velr, nrm, p.c.friction, velt);
            p.tmp[A][e] = velt[A] + cv[A];
        } else {
            p.tmp[A][e] = cv[A];
        }
    }
}
__global__ __launch_bounds__(256) void k_bc_project(BcArgs p) {
    if (blockIdx.y == 0) bc_project<0>(p);
    else if (blockIdx.y == 1) bc_project<1>(p);
    else bc_project<2>(p);
}

// Stage 4 (:178-232): the projected values back into the component, zero on
// closed domain walls (closed: Jet's kDirection* bits, include/jet/
// constants.h:312-335); blocked: the blocked solver's pass (src/jet/
// grid_blocked_boundary_condition_solver3.cpp:39-66, marker :86-94), where an
// interior face whose two cells are one collider (SDF < 0 at the centre) and
// one fluid takes the collider velocity.  Such a face is always listed.  The
// listed faces' validity goes back to 1.
template <int A>
__device__ __forceinline__ void bc_finish(const BcArgs& p, int closed, int blocked) {
#pragma clang fp contract(off)
    const BcGrid& g = p.g;
    const int lo = A == 0 ? 1 : (A == 1 ? 4 : 16), hi = 2 * lo;
    double fo[3];
    bc_face_origin<A>(g, fo);
    JG_BC_LISTED(A, g, p.lists, s, e, f) {
        p.valid[0][A][f] = 1;
        p.valid[1][A][f] = 1;
        int i, j, k;
        bc_face_ijk(f, s, i, j, k);
        const int a = A == 0 ? i : (A == 1 ? j : k);
        double val = p.tmp[A][e];
        if (((closed & lo) && a == 0) || ((closed & hi) && a == s[A] - 1)) val = 0.0;
        if (blocked && a > 0 && a < s[A] - 1) {
            const idx_t up = i + (idx_t)g.d.nx * (j + (idx_t)g.d.ny * k);  // the cell at +A
            const idx_t down = up - (A == 0 ? 1 : (A == 1 ? (idx_t)g.d.nx : (idx_t)g.d.nx * g.d.ny));
            if ((p.sdf[up] < 0) != (p.sdf[down] < 0)) {
                double x[3], cv[3];
                bc_pos(fo, g.h, i, j, k, x);
                bc_collider_velocity(p.c, x, cv);
                val = cv[A];
            }
        }
        p.comp[A][f] = val;
    }
}
// The unlisted faces of a closed wall (a listed one gets the same zero twice).
template <int A>
__device__ __forceinline__ void bc_walls(const BcArgs& p, int closed) {
    const int lo = A == 0 ? 1 : (A == 1 ? 4 : 16), hi = 2 * lo;
    int s[3];
    bc_face_dims<A>(p.g.d, s);
    const int P = A == 0 ? 1 : 0, Q = A == 2 ? 1 : 2;  // the wall's axes
    const idx_t n = (idx_t)s[P] * s[Q];
    const idx_t st[3] = {1, s[0], (idx_t)s[0] * s[1]};
    for (idx_t e = blockIdx.x * (idx_t)blockDim.x + threadIdx.x; e < n;
         e += (idx_t)gridDim.x * blockDim.x) {
        const idx_t q = e / s[P], c = (e - q * s[P]) * st[P] + q * st[Q];
        if (closed & lo) p.comp[A][c] = 0.0;
        if (closed & hi) p.comp[A][c + (s[A] - 1) * st[A]] = 0.0;
    }
}
__global__ __launch_bounds__(256) void k_bc_finish(BcArgs p, int closed, int blocked) {
    switch (blockIdx.y) {
        case 0: bc_finish<0>(p, closed, blocked); break;
        case 1: bc_finish<1>(p, closed, blocked); break;
        case 2: bc_finish<2>(p, closed, blocked); break;
        case 3: bc_walls<0>(p, closed); break;
        case 4: bc_walls<1>(p, closed); break;
        default: bc_walls<2>(p, closed);
    }
}

#undef JG_BC_LISTED

}  // namespace jg
