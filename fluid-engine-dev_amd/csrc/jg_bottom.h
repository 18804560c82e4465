// jg_bottom.h -- the bottom of the V-cycle in one workgroup.
//
// Below a few thousand cells a level's kernels are pure launch and memory
// latency (a fused sweep over a 16^3 level costs as much as one over 64^3).
// k_bottom runs the whole lower part of the V-cycle -- every level from the
// first one with at most BotCfg<T>::MaxCells cells down to the coarsest -- as one
// 1024-thread workgroup: vectors of every level in LDS, the stencil of the
// top level (BotCfg<T>::MC cells per thread) and of the coarsest level (one
// cell per thread) in registers, the rows of the levels between staged in
// LDS with precomputed cell coordinates, __syncthreads between phases.
// Zero-centre rows are set to zero by the smoother, as in k_rb_sweep.
// The sequence is exactly the multi-kernel V-cycle's: `pre` forward (red,
// black) sweeps from zero, residual, Jet's restriction, recursion, Jet's
// prolongation-correction, `post` backward (black, red) sweeps; on the
// coarsest level `cfwd` forward then `cfwd` backward sweeps.  Restriction and
// prolongation are FdmMgUtils3::restrict / correct
// (src/jet/fdm_mg_linear_system3.cpp:43-179); the smoother is Jet's
// relaxRedBlack update (src/jet/fdm_gauss_seidel_solver3.cpp:163-190).
// What bounds it is one CU's instruction rate on the top level and the chain
// LDS read - six products - LDS write of the coarsest level's sweeps.  FP64:
// 8^3 over 4^3 12.4 us, 14x8x18 over 7x4x9 20.4 us (14.3 and 26.6 us with
// neighbour offsets formed at each use, divisions for the coordinates and a
// block barrier between the coarsest half-sweeps of one wave).
#pragma once

#include "jg_device.h"
#include "jg_sweep.h"

namespace jg {

constexpr int kBotThreads = 1024;
constexpr int kBotMaxLevels = 6;  // 4096 -> 512 -> 64 -> 8 -> 1 (+1 spare)

// Cells per thread on the top level: 4 in FP32; 2 in FP64, where four
// cells' stencils no longer fit in the 128 VGPRs of a 1024-thread block.
template <typename T>
struct BotCfg {
    static constexpr int MC = sizeof(T) == 4 ? 4 : 2;
    static constexpr int MaxCells = MC * kBotThreads;
    static constexpr int Pool = MaxCells + MaxCells / 7 + 8;  // >= sum of the level sizes
    static constexpr int Rows = MaxCells / 7 + 8;             // >= sizes below the top
};

template <typename T>
struct BotLevels {
    int L;  // levels in this bottom solve (>= 1); level 0 is the top, each halves exactly
    Dims d[1];
    const Row<T>* A[kBotMaxLevels];
};

// Cell coordinates packed 10 bits each (every level below a top level that
// has a coarser level has dimensions <= 1024).
__device__ __forceinline__ int bot_pack(int i, int j, int k) { return i | (j << 10) | (k << 20); }
__device__ __forceinline__ void bot_unpack(int v, int& i, int& j, int& k) {
    i = v & 1023;
    j = (v >> 10) & 1023;
    k = v >> 20;
}

// c / n and c % n for 0 <= c < 2^16 and 1 <= n < 2^16, by one multiplication:
// with m = ceil(2^32 / n) the product c * m exceeds c * 2^32 / n by less than
// c < 2^32 / n, so its high word is the quotient.  (The compiler's division by
// a value it does not know is some 30 instructions; a wave of this block's
// sixteen went through it twenty times.)
struct BotDiv {
    unsigned m;
    int n;
    __device__ __forceinline__ explicit BotDiv(int n_) : m(0xFFFFFFFFu / (unsigned)n_ + 1u), n(n_) {}
    __device__ __forceinline__ int div(int c) const { return n == 1 ? c : (int)__umulhi((unsigned)c, m); }
    __device__ __forceinline__ void split(int c, int& q, int& r) const {
        q = div(c);
        r = c - q * n;
    }
};
// Coordinates of a level's cells.
struct BotCoords {
    BotDiv dx, dy;
    __device__ __forceinline__ explicit BotCoords(const Dims& d) : dx(d.nx), dy(d.ny) {}
    __device__ __forceinline__ void at(int c, int& i, int& j, int& k) const {
        int q;
        dx.split(c, q, i);
        dy.split(q, k, j);
    }
};

// Stencil of MC cells per thread, held in registers: omega / center, the six
// couplings (zero where the neighbour is outside the grid) and the byte
// offsets of the cell and its six neighbours in a pool of level vectors (the
// cell's own where there is none), two to a register.  One CU runs all of
// this, so a sweep costs its instructions: unpacking an offset is one, where
// forming it from flags and strides was five.  With an even nx the cells are
// taken in x-adjacent pairs (2p, 2p + 1), p = tid + kBotThreads * h, which
// always have opposite colours; slot 2h holds the pair's red cell and slot
// 2h + 1 its black cell, so every lane updates exactly one cell of each pair
// per half-sweep.  Otherwise slot m of a thread is cell tid + kBotThreads * m.
template <typename T, int MC, bool PAIRS>
struct BotRegs {
    static_assert(!PAIRS || MC % 2 == 0, "pairs need an even cell count");
    T wc[MC], xp[MC], xm[MC], yp[MC], ym[MC], zp[MC], zm[MC];
    // own | -x << 16, +x | -y << 16, +y | -z << 16, +z | flags << 16
    // (flags: bit 0 the cell exists, bit 1 its parity)
    unsigned o[MC][4];

    // `off`: where the level starts in the pool.  `q` (or null) receives the
    // packed coordinates of the level's cells, `cen` (or null) their centres.
    __device__ __forceinline__ void load(const Row<T>* __restrict__ A, const Dims& d, T omega,
                                         int off, int* q, T* cen) {
        const int n = d.nx * d.ny * d.nz, nx = d.nx, nxy = d.nx * d.ny;
        const BotCoords co(d);
#pragma unroll
        for (int m = 0; m < MC; ++m) {
            int i, j, k, cc;
            bool ok;
            if (PAIRS) {
                const int c0 = 2 * ((int)threadIdx.x + kBotThreads * (m >> 1));
                ok = c0 < n;
                cc = ok ? c0 : 0;
                co.at(cc, i, j, k);
                const int dx = (m ^ (i + j + k)) & 1;  // cell 2p is black: the red one is 2p + 1
                i += dx;
                cc += dx;
            } else {
                const int c0 = (int)threadIdx.x + kBotThreads * m;
                ok = c0 < n;
                cc = ok ? c0 : 0;
                co.at(cc, i, j, k);
            }
            const bool hxm = i > 0, hxp = i + 1 < d.nx, hym = j > 0, hyp = j + 1 < d.ny,
                       hzm = k > 0, hzp = k + 1 < d.nz;
            const Row<T> row = A[cc];
            const int cxm = hxm ? cc - 1 : cc, cym = hym ? cc - nx : cc, czm = hzm ? cc - nxy : cc;
            const int cxp = hxp ? cc + 1 : cc, cyp = hyp ? cc + nx : cc, czp = hzp ? cc + nxy : cc;
            const T lx = A[cxm].r, ly = A[cym].u, lz = A[czm].f;
            auto at = [&](int c) { return (unsigned)(c + off) * (unsigned)sizeof(T); };
            o[m][0] = at(cc) | (at(cxm) << 16);
            o[m][1] = at(cxp) | (at(cym) << 16);
            o[m][2] = at(cyp) | (at(czm) << 16);
            o[m][3] = at(czp) | ((ok ? 1u : 0u) << 16) | (((unsigned)(i + j + k) & 1u) << 17);
            wc[m] = (ok && row.c != T(0)) ? omega / row.c : T(0);  // 0: zero-centre row
            xp[m] = (ok && hxp) ? row.r : T(0);
            yp[m] = (ok && hyp) ? row.u : T(0);
            zp[m] = (ok && hzp) ? row.f : T(0);
            xm[m] = (ok && hxm) ? lx : T(0);
            ym[m] = (ok && hym) ? ly : T(0);
            zm[m] = (ok && hzm) ? lz : T(0);
            if (ok && q) q[cc] = bot_pack(i, j, k);
            if (ok && cen) cen[cc] = row.c;
        }
    }
    __device__ static __forceinline__ T get(const T* V, unsigned o) {
        return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(V) + o);
    }
    __device__ static __forceinline__ void put(T* V, unsigned o, T v) {
        *reinterpret_cast<T*>(reinterpret_cast<char*>(V) + o) = v;
    }
    // The offsets of slot m, unpacked where they are used: an empty asm keeps
    // the compiler from holding them unpacked through the kernel's loops (it
    // spilled to scratch).
    struct At {
        unsigned c, xm, xp, ym, yp, zm, zp;
    };
    template <bool HOLD = false>
    __device__ __forceinline__ At at(int m) const {
        unsigned a = o[m][0], b = o[m][1], c = o[m][2], d = o[m][3];
        if (!HOLD) asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
        return {a & 0xFFFFu, a >> 16, b & 0xFFFFu, b >> 16, c & 0xFFFFu, c >> 16, d & 0xFFFFu};
    }
    __device__ __forceinline__ bool exists(int m) const { return o[m][3] & (1u << 16); }
    __device__ __forceinline__ int parity(int m) const { return (o[m][3] >> 17) & 1; }
    __device__ __forceinline__ T offdiag(int m, const T* X, const At& a) const {
#pragma clang fp contract(off)
        T s = xm[m] * get(X, a.xm);
        s += xp[m] * get(X, a.xp);
        s += ym[m] * get(X, a.ym);
        s += yp[m] * get(X, a.yp);
        s += zm[m] * get(X, a.zm);
        s += zp[m] * get(X, a.zp);
        return s;
    }
    // (1 - w) x + (w / c)(b - s): the relaxRedBlack update with w / c
    // precomputed (one rounding apart from Jet's w (b - s) / c).
    __device__ __forceinline__ T update(int m, const T* X, const T* B, const At& a, T omega) const {
#pragma clang fp contract(off)
        const T v = (T(1) - omega) * get(X, a.c) + wc[m] * (get(B, a.c) - offdiag(m, X, a));
        return wc[m] == T(0) ? T(0) : v;
    }
    // X, B, R: the pools.  A half-sweep reads only the other colour, so all
    // loads are issued before any store.  Callers pass a constant colour.
    __device__ __forceinline__ void relax(T* X, const T* B, int colour, T omega) const {
        if (PAIRS) {
            constexpr int H = PAIRS ? MC / 2 : 1;
            T nv[H];
#pragma unroll
            for (int h = 0; h < H; ++h) nv[h] = update(2 * h + colour, X, B, at(2 * h + colour), omega);
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (exists(2 * h + colour)) put(X, o[2 * h + colour][0] & 0xFFFFu, nv[h]);
        } else {
#pragma unroll
            for (int m = 0; m < MC; ++m) {
                if (!exists(m) || parity(m) != colour) continue;
                const At a = at(m);
                put(X, a.c, update(m, X, B, a, omega));
            }
        }
    }
    // `off` and `cen` as in load
    __device__ __forceinline__ void residual(const T* cen, const T* X, const T* B, T* R, int off) const {
#pragma clang fp contract(off)
#pragma unroll
        for (int m = 0; m < MC; ++m) {
            if (!exists(m)) continue;
            const At a = at(m);
            const T c = get(cen - off, a.c);
            put(R, a.c, get(B, a.c) - (c * get(X, a.c) + offdiag(m, X, a)));
        }
    }
    // The coarsest level's sweeps (one cell per thread): `n` times red, black,
    // then `n` times black, red.  What the half-sweeps share stays in
    // registers; a level of one wave needs no barrier between them, as a
    // wave's LDS operations complete in order.
    template <bool WAVE>
    __device__ __forceinline__ void coarsest(T* X, const T* B, int n, T omega) const {
#pragma clang fp contract(off)
        const At a = at<true>(0);
        const bool ok = exists(0);
        const T bv = get(B, a.c), keep = T(1) - omega;
        const int par = parity(0);
        T x = get(X, a.c);
        auto half = [&](int colour) __attribute__((always_inline)) {
            if (ok && par == colour) {
                const T v = keep * x + wc[0] * (bv - offdiag(0, X, a));
                x = wc[0] == T(0) ? T(0) : v;
                put(X, a.c, x);
            }
            if (WAVE) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            } else {
                __syncthreads();
            }
        };
#pragma unroll 1
        for (int s = 0; s < n; ++s) {
            half(0);
            half(1);
        }
#pragma unroll 1
        for (int s = 0; s < n; ++s) {
            half(1);
            half(0);
        }
    }
};

template <typename T>
__device__ __forceinline__ void bot_relax_lds(const Row<T>* R, const int* Q, T* X, const T* B,
                                              const Dims& d, int colour, T omega) {
#pragma clang fp contract(off)
    const int n = d.nx * d.ny * d.nz;
    for (int c = threadIdx.x; c < n; c += kBotThreads) {
        int i, j, k;
        bot_unpack(Q[c], i, j, k);
        if (((i + j + k) & 1) != colour) continue;
        const Row<T> row = R[c];
        const T s = offdiag<T, T, T>(R, X, row, c, i, j, k, d);
        X[c] = row.c == T(0) ? T(0) : (T(1) - omega) * X[c] + omega * (B[c] - s) / row.c;
    }
}

template <typename T>
__device__ __forceinline__ void bot_residual_lds(const Row<T>* R, const int* Q, const T* X,
                                                 const T* B, T* Rs, const Dims& d) {
#pragma clang fp contract(off)
    const int n = d.nx * d.ny * d.nz;
    for (int c = threadIdx.x; c < n; c += kBotThreads) {
        int i, j, k;
        bot_unpack(Q[c], i, j, k);
        const Row<T> row = R[c];
        Rs[c] = B[c] - (row.c * X[c] + offdiag<T, T, T>(R, X, row, c, i, j, k, d));
    }
}

// coarse = restriction of fine (Jet's 4x4x4 kernel, clamped), cd = coarse dims.
// Tap t of coarse index i is fine index 2i - 1 + t, clamped to 2i at the low
// edge and to 2i + 1 at the high edge; weights 1/8, 3/8, 3/8, 1/8.  One z tap
// per loop iteration keeps 16 loads in flight, not 64.
template <typename T>
__device__ __forceinline__ void bot_restrict(const T* fine, T* coarse, const int* Qc,
                                             const Dims& cd) {
#pragma clang fp contract(off)
    const int n = cd.nx * cd.ny * cd.nz;
    const int fnx = 2 * cd.nx, fny = 2 * cd.ny;
    auto tap = [](int i, int t, int cn) {
        const int f = 2 * i - 1 + t;
        return (t == 0 && i == 0) ? 2 * i : ((t == 3 && i + 1 == cn) ? 2 * i + 1 : f);
    };
    auto wt = [](int t) { return (t == 0 || t == 3) ? T(0.125) : T(0.375); };
    for (int c = threadIdx.x; c < n; c += kBotThreads) {
        int i, j, k;
        bot_unpack(Qc[c], i, j, k);
        T sum = 0;
#pragma unroll 1
        for (int z = 0; z < 4; ++z) {
            const int kz = tap(k, z, cd.nz);
            const T wz = wt(z);
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const T* row = fine + fnx * (tap(j, y, cd.ny) + fny * kz);
#pragma unroll
                for (int x = 0; x < 4; ++x) sum += wt(x) * wt(y) * wz * row[tap(i, x, cd.nx)];
            }
        }
        coarse[c] = sum;
    }
}

// fine += prolongation of coarse: prolong_at's taps and order, with 32-bit
// indices.
template <typename T>
__device__ __forceinline__ void bot_correct(const T* coarse, T* fine, const int* Qf,
                                            const Dims& fd) {
#pragma clang fp contract(off)
    const int n = fd.nx * fd.ny * fd.nz;
    const int cnx = fd.nx / 2, cnxy = cnx * (fd.ny / 2), kclamp = fd.kclamp();
    for (int c = threadIdx.x; c < n; c += kBotThreads) {
        int i, j, k;
        bot_unpack(Qf[c], i, j, k);
        const int io = i & 1, jo = j & 1, ko = k & 1;
        const int ci = i >> 1, cj = j >> 1, ck = k >> 1;
        const int i0 = (!io && i > 1) ? ci - 1 : ci, i1 = (io && i + 1 < fd.nx) ? ci + 1 : ci;
        const int j0 = (!jo && j > 1) ? cj - 1 : cj, j1 = (jo && j + 1 < fd.ny) ? cj + 1 : cj;
        const int k0 = (!ko && k > 1) ? ck - 1 : ck, k1 = (ko && k + 1 < kclamp) ? ck + 1 : ck;
        const T wi[2] = {io ? T(0.75) : T(0.25), io ? T(0.25) : T(0.75)};
        const T wj[2] = {jo ? T(0.75) : T(0.25), jo ? T(0.25) : T(0.75)};
        const T wk[2] = {ko ? T(0.75) : T(0.25), ko ? T(0.25) : T(0.75)};
        const int yz[4] = {cnx * j0 + cnxy * k0, cnx * j1 + cnxy * k0, cnx * j0 + cnxy * k1,
                           cnx * j1 + cnxy * k1};
        T v = 0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            v += wi[0] * wj[p & 1] * wk[p >> 1] * coarse[yz[p] + i0];
            v += wi[1] * wj[p & 1] * wk[p >> 1] * coarse[yz[p] + i1];
        }
        fine[c] += v;
    }
}

// x0 = bottom V-cycle applied to b0 (level 0 of `bl`).  post0: post-sweeps
// on the top level, post: on the levels below it.  PAIRS: the top level's nx
// is even (pair-slotted registers, see BotRegs).
template <typename T, bool PAIRS>
__global__ __launch_bounds__(kBotThreads) void k_bottom(BotLevels<T> bl, const T* __restrict__ b0,
                                                        T* __restrict__ x0, int pre, int post0,
                                                        int post, int cfwd, T omega,
                                                        const Ctl* __restrict__ ctl) {
#pragma clang fp contract(off)
    // one workgroup per system of a batch group; AL(l): its rows of level l
    const int sys = blockIdx.x;
    if (sys > 0) {
        b0 += sys * bl.d[0].n();
        x0 += sys * bl.d[0].n();
        if (ctl) ctl += sys * kSysCtl;
    }
    auto AL = [&](int l) { return bl.A[l] + sys * (bl.d[0].n() >> (3 * l)); };
    if (ctl && ctl->done) return;
    __shared__ T sv[3][BotCfg<T>::Pool];    // x, b, residual of every level
    __shared__ int sq[BotCfg<T>::Pool];     // packed cell coordinates (L >= 2)
    __shared__ Row<T> sA[BotCfg<T>::Rows];  // rows of the levels below the top
    __shared__ T sc[BotCfg<T>::MaxCells];   // centres of the top level (L >= 2)
    const int L = bl.L;
    // Levels halve exactly, so level l has n0 >> 3l cells; the vectors of
    // level l start at the sum of the sizes above it.
    const int n0 = bl.d[0].nx * bl.d[0].ny * bl.d[0].nz;
    auto off = [&](int l) {
        int o = 0;
        for (int m = 0; m < l; ++m) o += n0 >> (3 * m);
        return o;
    };
    auto D = [&](int l) { return Dims{bl.d[0].nx >> l, bl.d[0].ny >> l, bl.d[0].nz >> l, bl.d[0].box}; };
    auto X = [&](int l) { return &sv[0][off(l)]; };
    auto B = [&](int l) { return &sv[1][off(l)]; };
    auto Rv = [&](int l) { return &sv[2][off(l)]; };
    auto Q = [&](int l) { return &sq[off(l)]; };
    auto RA = [&](int l) { return &sA[off(l) - n0]; };  // rows of level l >= 1

    // Prologue: every global load is issued before the LDS is filled, so
    // their latencies overlap.
    constexpr int MC = BotCfg<T>::MC;
    const int tid = threadIdx.x;
    T bv[MC];
#pragma unroll
    for (int m = 0; m < MC; ++m) {
        const int c = tid + kBotThreads * m;
        bv[m] = c < n0 ? b0[c] : T(0);
    }
    BotRegs<T, MC, PAIRS> top;
    top.load(AL(0), bl.d[0], omega, 0, L >= 2 ? sq : nullptr, L >= 2 ? sc : nullptr);
    BotRegs<T, 1, false> bot;  // coarsest level when it is not the top
    if (L >= 2) bot.load(AL(L - 1), D(L - 1), omega, off(L - 1), nullptr, nullptr);

    for (int c = tid; c < off(L); c += kBotThreads) sv[0][c] = T(0);
#pragma unroll
    for (int m = 0; m < MC; ++m) {
        const int c = tid + kBotThreads * m;
        if (c < n0) sv[1][c] = bv[m];
    }
    for (int l = 1; l < L; ++l) {  // at most 512 cells each
        const Dims d = D(l);
        int i, j, k;
        if (tid < d.nx * d.ny * d.nz) {
            BotCoords(d).at(tid, i, j, k);
            Q(l)[tid] = bot_pack(i, j, k);
        }
    }
    for (int l = 1; l + 1 < L; ++l)  // rows of the levels between (<= 512 cells each)
        if (tid < (n0 >> (3 * l))) RA(l)[tid] = AL(l)[tid];
    __syncthreads();

    auto relax = [&](int l, int colour) __attribute__((always_inline)) {
        if (l == 0) top.relax(sv[0], sv[1], colour, omega);
        else bot_relax_lds<T>(RA(l), Q(l), X(l), B(l), D(l), colour, omega);
        __syncthreads();
    };
    // down
    for (int l = 0; l + 1 < L; ++l) {
        for (int s = 0; s < pre; ++s) {
            relax(l, 0);
            relax(l, 1);
        }
        if (l == 0) top.residual(sc, sv[0], sv[1], sv[2], 0);
        else bot_residual_lds<T>(RA(l), Q(l), X(l), B(l), Rv(l), D(l));
        __syncthreads();
        bot_restrict<T>(Rv(l), B(l + 1), Q(l + 1), D(l + 1));
        __syncthreads();
    }
    // coarsest
    if (L == 1) {
        for (int s = 0; s < cfwd; ++s) {
            relax(0, 0);
            relax(0, 1);
        }
        for (int s = 0; s < cfwd; ++s) {
            relax(0, 1);
            relax(0, 0);
        }
    } else if (n0 >> (3 * (L - 1)) <= kWave) {
        if (tid < kWave) bot.template coarsest<true>(sv[0], sv[1], cfwd, omega);
        __syncthreads();
    } else {
        bot.template coarsest<false>(sv[0], sv[1], cfwd, omega);
    }
    // up
    for (int l = L - 2; l >= 0; --l) {
        bot_correct<T>(X(l + 1), X(l), Q(l), D(l));
        __syncthreads();
        const int np = l == 0 ? post0 : post;
        for (int s = 0; s < np; ++s) {
            relax(l, 1);
            relax(l, 0);
        }
    }
#pragma unroll
    for (int m = 0; m < MC; ++m) {
        const int c = tid + kBotThreads * m;
        if (c < n0) x0[c] = sv[0][c];
    }
}

}  // namespace jg
