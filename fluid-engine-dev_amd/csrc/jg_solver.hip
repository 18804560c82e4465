// jg_solver.hip -- solver objects, CG / MGPCG drivers and the C ABI.
//
// Host code only launches kernels; every scalar of the Krylov loop (alpha,
// beta, sigma, the stop test) lives in device memory (jg::Ctl) and is
// computed by one-block finalize kernels, so iterations run back to back on
// one stream and the host only polls the stop flag.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>
#include <vector>

#include "jg_internal.h"
#include "jg_kernels.h"
#include "jg_sweep.h"
#include "jg_sweep2.h"
#include "jg_plane2.h"
#include "jg_brick.h"
#include "jg_bottom.h"
#include "jg_transfer.h"
#include "jg_csr.h"
#include "jg_cggrid.h"
#include "jg_box.h"

#include <cstdlib>

using namespace jg;

// ------------------------------------------- scratch of the no-allocation entry
//
// jg_relax_red_black_noalloc keeps the copy of x that its sweep reads in this
// array instead of a hipMalloc'd temporary.  Every GPU holds its own copy of
// the array (16 MiB) from module load until the process ends.  Host code
// never passes the array's name to a kernel or a copy: that name is a host-side
// stand-in.  The device address comes from hipGetSymbolAddress, resolved once
// per device by jg_solver_create with that device current.
constexpr size_t kNoAllocMaxCells = size_t(1) << 21;
static __device__ __align__(256) double scratch[kNoAllocMaxCells];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kScratchDevices] = {};
hipError_t g_scratch_err[kScratchDevices] = {};
bool g_scratch_done[kScratchDevices] = {};

// Resolves the address of `scratch` on `device` (which must be current) the
// first time it is asked for that device.
hipError_t scratch_init(int device) {
    if (device < 0 || device >= kScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_done[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        g_scratch_err[device] = e;
        g_scratch_ptr[device] = e == hipSuccess ? static_cast<double*>(p) : nullptr;
        g_scratch_done[device] = true;
    }
    return g_scratch_err[device];
}

hipError_t scratch_address(int device, double** out) {
    if (device < 0 || device >= kScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_done[device]) return hipErrorNotInitialized;
    *out = g_scratch_ptr[device];
    return g_scratch_err[device];
}

// ------------------------------------------------------- level kernels

// A z-marching launch of `tiles` columns (over all systems) on nz planes: the
// planes per block zc that make it cheapest, and that cost, in plane steps of
// a block that has its CU to itself.
struct March {
    int zc;
    double cost;
};
// A block's pipeline and halo cost `halo` plane steps, and the CUs run `cus`
// blocks at once, or (pair > 0) twice as many, when a step of two blocks on one
// CU takes `pair` times the step of one.  A launch costs its rounds of blocks,
// each zc + halo steps: whole rounds where the blocks wait on their own chains
// (a last round that is nearly empty costs like a full one), the blocks' share
// of the chip where they wait for memory; `whole` weighs the two.  Against
// timing every chunk of {2, 4, 8, ... 64} on 76 level shapes from 2 x 2 x 32768
// over 24^3 and 512 x 512 x 2 to 512^3, this picks within 1% of the fastest on
// average, at worst 8%, and it is free to take a chunk between them:
// 256 x 160 x 256 cells run 245 two-sweep blocks of 38 planes instead of 210
// of 48.
March march(int nz, long tiles, long cus, double halo, double pair, double whole) {
    March best{nz, 1e300};
    for (long chunks = 1; chunks <= nz;) {
        const int zc = std::min<long>(nz, (((nz + chunks - 1) / chunks) + 1) & ~1l);  // even
        if (zc <= 64 || tiles <= cus / 4) {  // longer only to cut the halo of few columns
            const double share = (double)(tiles * ((nz + zc - 1) / zc)) / cus;
            double rounds = std::ceil(share), work = share;
            if (pair > 0.0) {
                const double two = std::floor(share / 2), rest = share - 2 * two;
                rounds = two * pair + (rest > 1 ? pair : (rest > 0 ? 1.0 : 0.0));
                work = share * pair / 2;
            }
            const double c = (whole * rounds + (1.0 - whole) * work) * (zc + halo);
            if (c < best.cost) best = March{zc, c};
        }
        if (zc <= 2) break;
        chunks = (nz + zc - 3) / (zc - 2);  // the fewest of a smaller zc
    }
    return best;
}

// How k_rb_sweep runs on shape d: tile rows per thread, planes per block, and
// the cost in plane steps of one-row blocks.  FP32: one row, two blocks per CU.
// FP64: one row and one block per CU, or (without a correction) two rows and
// two blocks, whose step alone costs 1.2 times as much, and 1.5 times where it
// sums b.x and b.b (that kernel spills).  Two rows are the better where they
// make two rounds of blocks one or many; one / two, us: 512 x 512 x 2 cells
// plain 18 / 14, from zero 17 / 14, with the sums 21 / 18; 192 x 160 x 144 75 /
// 63, 67 / 58, 78 / 80; 256 x 160 x 256 175 / 165, 149 / 149, 187 / 206; 96^3
// 20 / 23, 16 / 17, 22 / 27.  Over 22 such shapes the rule is 0.3% above the
// faster of the two on average in plain sweeps, 1.3% from zero (at worst 12%, 250^3)
// and 0.2% with the sums.
struct SweepShape {
    int rows, zc;
    double cost;
};
template <typename T>
SweepShape sweep_shape(const jg_solver* s, const Dims& d, bool zero, bool correct, bool sums) {
    const long tiles = (long)((d.nx + kSwIX - 1) / kSwIX) * ((d.ny + kSwIY - 1) / kSwIY) * s->nsys;
    if (sizeof(T) == 4) {
        const March m = march(d.nz, tiles, s->cus, 2, 1.8, 0.85);
        return {1, m.zc, m.cost};
    }
    const March one = march(d.nz, tiles, s->cus, 3, 0.0, 0.5);
    if (!correct) {
        const March two = march(d.nz, tiles, s->cus, 3, 1.5, 0.5);
        const double cost = two.cost * (1.2 + (sums ? 0.3 * two.zc / (two.zc + 3) : 0.0));
        // from zero nothing is loaded for the planes before the first
        if (cost < one.cost)
            return {2, zero ? march(d.nz, tiles, s->cus, 1, 1.5, 0.5).zc : two.zc, cost};
    }
    return {1, one.zc, one.cost};
}
// k_rb_sweep2 on tiles of ix x iy cells: one block per CU; a chunk adds 8
// planes of halo, some of them cheap.
March sweep2_march(const jg_solver* s, const Dims& d, int ix, int iy) {
    const long tiles = (long)((d.nx + ix - 1) / ix) * ((d.ny + iy - 1) / iy) * s->nsys;
    return march(d.nz, tiles, s->cus, 6, 0.0, 0.5);
}

// Grids of a launch over every system of s (one, or a batch group): the
// stencil kernels repeat their z extent, the elementwise kernels take the
// system from the grid's y index, the one-block kernels one block each.
inline dim3 grid_sys(dim3 g, const jg_solver* s) {
    g.z *= (unsigned)s->nsys;
    return g;
}
inline dim3 grid_1d(int nb, const jg_solver* s) { return dim3((unsigned)nb, (unsigned)s->nsys, 1); }

// One fused red-black sweep (see jg_sweep.h).  first: colour updated first
// (0 = red, forward; 1 = black, backward).  xin == nullptr: x starts at zero.
// coarse != nullptr: add the prolongation of coarse to x on load.
// p_bx/p_bb != nullptr: emit b.x and b.b partials.  Returns the number of
// b.x / b.b partials written (the block count; 0 without partials, or when
// the grid has more blocks than a slot holds -- the caller then reduces with
// k_dot).
template <typename T>
int launch_sweep(jg_solver* s, const Row<T>* A, const T* b, const T* xin, T* xout, const Dims& d,
                 int first, const T* coarse, double* p_bx, double* p_bb, T omega, const Ctl* ctl) {
    const SweepShape shape = sweep_shape<T>(s, d, !xin && !coarse, coarse != nullptr, p_bx != nullptr);
    int zc = shape.zc;
    const long cols = (long)((d.nx + kSwIX - 1) / kSwIX) * ((d.ny + kSwIY - 1) / kSwIY);
    // one b.x / b.b partial per block: keep the block count within a slot
    while (p_bx && zc < d.nz && cols * ((d.nz + zc - 1) / zc) > kMaxPartials) ++zc;
    dim3 grid((d.nx + kSwIX - 1) / kSwIX, (d.ny + kSwIY - 1) / kSwIY, (d.nz + zc - 1) / zc);
    if ((long)grid.x * grid.y * grid.z > kMaxPartials) p_bx = p_bb = nullptr;  // caller uses k_dot
    const int nb = (int)(grid.x * grid.y * grid.z);  // per system
    grid = grid_sys(grid, s);
    const int code = (first ? 8 : 0) | (xin ? 0 : 4) | (coarse ? 2 : 0) | (p_bx ? 1 : 0);
    const dim3 block(kSwLX, kSwLY / shape.rows, 1);
#define JG_SWEEP_CASE(C, F, Z, K, D)                                                              \
    case C: {                                                                                     \
        constexpr int R2 = sizeof(T) == 8 && !K ? 2 : 1;                                          \
        if (shape.rows == 2)                                                                      \
            k_rb_sweep<T, F, Z, K, D, R2><<<grid, block, 0, s->stream>>>(                         \
                A, b, xin, xout, d, zc, omega, coarse, p_bx, p_bb, ctl);                          \
        else                                                                                      \
            k_rb_sweep<T, F, Z, K, D, 1><<<grid, block, 0, s->stream>>>(                         \
                A, b, xin, xout, d, zc, omega, coarse, p_bx, p_bb, ctl);                          \
        break;                                                                                    \
    }
    switch (code) {
        JG_SWEEP_CASE(0, 0, false, false, false)
        JG_SWEEP_CASE(1, 0, false, false, true)
        JG_SWEEP_CASE(2, 0, false, true, false)
        JG_SWEEP_CASE(3, 0, false, true, true)
        JG_SWEEP_CASE(4, 0, true, false, false)
        JG_SWEEP_CASE(5, 0, true, false, true)
        JG_SWEEP_CASE(6, 0, true, true, false)
        JG_SWEEP_CASE(7, 0, true, true, true)
        JG_SWEEP_CASE(8, 1, false, false, false)
        JG_SWEEP_CASE(9, 1, false, false, true)
        JG_SWEEP_CASE(10, 1, false, true, false)
        JG_SWEEP_CASE(11, 1, false, true, true)
        JG_SWEEP_CASE(12, 1, true, false, false)
        JG_SWEEP_CASE(13, 1, true, false, true)
        JG_SWEEP_CASE(14, 1, true, true, false)
        JG_SWEEP_CASE(15, 1, true, true, true)
    }
#undef JG_SWEEP_CASE
    return p_bx ? nb : 0;
}

// Two sweeps in one launch (jg_sweep2.h, FP32 only).  res != nullptr: also
// write the residual b - A x of the result there (not with a coarse
// correction).  Returns JG_OK, or JG_ERR_UNSUPPORTED for FP64 or for res with
// a coarse correction.
template <typename T>
int launch_sweep2(jg_solver* s, const Row<T>* A, const T* b, const T* xin, T* xout, const Dims& d,
                  int first, const T* coarse, T* res, T omega, const Ctl* ctl) {
    if constexpr (sizeof(T) != 4) {
        return JG_ERR_UNSUPPORTED;
    } else {
        if (res && coarse) return JG_ERR_UNSUPPORTED;
        // the tile of a zero-start launch without a correction has a one cell
        // narrower halo (jg_sweep2.h)
        const bool z = !xin && !coarse;
        const int ix = res ? (z ? S2Tile<true, true>::IX : S2Tile<true>::IX)
                           : (z ? S2Tile<false, true>::IX : S2Tile<false>::IX);
        const int iy = res ? (z ? S2Tile<true, true>::IY : S2Tile<true>::IY)
                           : (z ? S2Tile<false, true>::IY : S2Tile<false>::IY);
        const int zc = sweep2_march(s, d, ix, iy).zc;
        const dim3 grid = grid_sys(dim3((d.nx + ix - 1) / ix, (d.ny + iy - 1) / iy, (d.nz + zc - 1) / zc), s);
        const dim3 block(kS2LX, kS2TY, 1);
        const int code = (first ? 8 : 0) | (xin ? 0 : 4) | (coarse ? 2 : 0) | (res ? 1 : 0);
#define JG_SWEEP2_CASE(C, F, Z, K, R)                                                     \
    case C:                                                                               \
        k_rb_sweep2<T, F, Z, K, R><<<grid, block, 0, s->stream>>>(A, b, xin, xout, d, zc, \
                                                                  omega, coarse, res,     \
                                                                  ctl);                   \
        break;
        switch (code) {
            JG_SWEEP2_CASE(0, 0, false, false, false)
            JG_SWEEP2_CASE(1, 0, false, false, true)
            JG_SWEEP2_CASE(2, 0, false, true, false)
            JG_SWEEP2_CASE(4, 0, true, false, false)
            JG_SWEEP2_CASE(5, 0, true, false, true)
            JG_SWEEP2_CASE(6, 0, true, true, false)
            JG_SWEEP2_CASE(8, 1, false, false, false)
            JG_SWEEP2_CASE(9, 1, false, false, true)
            JG_SWEEP2_CASE(10, 1, false, true, false)
            JG_SWEEP2_CASE(12, 1, true, false, false)
            JG_SWEEP2_CASE(13, 1, true, false, true)
            JG_SWEEP2_CASE(14, 1, true, true, false)
        }
#undef JG_SWEEP2_CASE
        return JG_OK;
    }
}

// Two sweeps of a small level in one launch by 8^3 bricks (jg_brick.h).
template <typename T>
void launch_brick2(jg_solver* s, const Row<T>* A, const T* b, const T* xin, T* xout, const Dims& d,
                   int first, const T* coarse, T omega, const Ctl* ctl) {
    const dim3 grid = grid_sys(
        dim3((d.nx + kBkB - 1) / kBkB, (d.ny + kBkB - 1) / kBkB, (d.nz + kBkB - 1) / kBkB), s);
    const int code = (first ? 4 : 0) | (xin ? 0 : 2) | (coarse ? 1 : 0);
#define JG_BRICK_CASE(C, F, Z, K)                                                               \
    case C:                                                                                     \
        k_brick_sweep2<T, F, Z, K><<<grid, kBkThreads, 0, s->stream>>>(A, b, xin, xout, d, omega, \
                                                                       coarse, ctl);            \
        break;
    switch (code) {
        JG_BRICK_CASE(0, 0, false, false)
        JG_BRICK_CASE(1, 0, false, true)
        JG_BRICK_CASE(2, 0, true, false)
        JG_BRICK_CASE(3, 0, true, true)
        JG_BRICK_CASE(4, 1, false, false)
        JG_BRICK_CASE(5, 1, false, true)
        JG_BRICK_CASE(6, 1, true, false)
        JG_BRICK_CASE(7, 1, true, true)
    }
#undef JG_BRICK_CASE
}

// Levels up to this size may use the brick kernel (it reloads a 16^3 region
// per 8^3 brick, which only pays where launches are latency-bound).
constexpr idx_t kBrickMaxCells = idx_t(1) << 21;

// Sweeps of one smoothing step, grouped into launches: 1 = one sweep,
// kLaunchMarch / kLaunchBrick = two sweeps in one launch of k_rb_sweep2 /
// k_brick_sweep2.  A brick launch costs by its bricks (FP32 16.5 ns, FP64
// 34 ns each once the chip is full, less where a brick reaches out of the
// grid), the marching ones a chain of plane steps (two-sweep FP32 1.55 us
// each, single FP64 1.62 us) that a small grid does not shorten, and that a
// narrow one pays for columns it does not have.  Measured, the mean of the
// pre- and the post-smoothing pair, us, as two launches / march / bricks:
//   FP32  64^3 (512 bricks) - / 22 / 10       96x80x72 (1080) - / 22 / 21
//         128x48x128 (1536) - / 23 / 27       128^3 (4096) - / 35 / 63
//         16x16x4096 (2048) - / 43 / 30       4x4x16384 (2048) - / 125 / 23
//   FP64  64^3 (512) 30 / - / 18              80x48x80 (600) 30 / - / 30
//         96x80x72 (1080) 31 / - / 42         128^3 (4096) 87 / - / 132
//         16x16x4096 (2048) 122 / - / 67      8x8x8192 (1024) 105 / - / 28
// So: bricks where these costs say so, else march in FP32 (a single system or
// a group) and single sweeps in FP64.  With the bricks' number alone deciding
// (768; FP32: 1536) a V-cycle of 4x4x16384 cells takes 1270 us in FP64 and 920
// in FP32, so 370 and 185.
// pairs > 0 forces two-sweep launches wherever two sweeps follow (FP32:
// bricks up to 2^18 cells, else the z-marching kernel; FP64: bricks up to
// kBrickMaxCells cells), pairs < 0 forbids them.
constexpr int kLaunchSingle = 1, kLaunchMarch = 2, kLaunchBrick = 3;
template <typename T>
std::vector<int> sweep_plan(const jg_solver* s, const Dims& d, unsigned n, int pairs) {
    const long bricks_z = (long)((d.nz + kBkB - 1) / kBkB) * s->nsys;
    const long bricks = (long)((d.nx + kBkB - 1) / kBkB) * ((d.ny + kBkB - 1) / kBkB) * bricks_z;
    int two;
    if (pairs > 0)  // FP32: bricks up to 64^3 cells, the z-marching kernel above
        two = sizeof(T) == 4 ? (d.n() <= (idx_t(1) << 18) ? kLaunchBrick : kLaunchMarch)
                             : (d.n() <= kBrickMaxCells ? kLaunchBrick : kLaunchSingle);
    else if (sizeof(T) == 4) {
        const double m = sweep2_march(s, d, S2Tile<false>::IX, S2Tile<false>::IY).cost;
        two = bricks_z < 65536 && 3 + 0.0165 * bricks < 6.5 + 1.55 * (m + 2) ? kLaunchBrick : kLaunchMarch;
    } else {
        const double m = sweep_shape<T>(s, d, false, false, false).cost;
        two = bricks_z < 65536 && 3 + 0.034 * bricks < 2 * (4.3 + 1.62 * m) ? kLaunchBrick : kLaunchSingle;
    }
    if (pairs < 0 || s->twod || d.n() <= BotCfg<T>::MaxCells) two = kLaunchSingle;
    std::vector<int> v;
    for (unsigned k = 0; k < n;) {
        const int mode = n - k < 2 ? kLaunchSingle : two;
        v.push_back(mode);
        k += mode == kLaunchSingle ? 1 : 2;
    }
    return v;
}

// Coarse planes per block of the fused residual-restriction: about `blocks`
// blocks, to fill the chip; each block recomputes one fine plane per chunk.
int rr_zc(const Dims& cd, long blocks = 1024) {
    const long tiles = (long)((cd.nx + kRrCX - 1) / kRrCX) * ((cd.ny + kRrCY - 1) / kRrCY);
    long zc = (long)cd.nz * tiles / blocks;
    zc = std::max<long>(2, std::min<long>(32, zc));
    return (int)std::min<long>(zc, cd.nz);
}

// Whether the stencil kernels take the tiled z-march on shape d: rows of at
// least 48 cells (a 64-lane row would idle too many lanes below that).  On
// small grids its chunks shorten to keep the chip busy (tm_grid), which
// measured as fast or faster than the per-cell z-march down to 64^3 (64^3
// CG 15.5 -> 11.9 ms, 128^3 MGPCG and the 64-system batch level or better).
inline bool use_tm(const Dims& d) { return d.nx >= 48; }

// r = b - A x on shape d (nsys systems back to back) stored as TR, with
// k_residual's DOT / GATED options; returns the partial count per system.
// Rows of at least 48 cells take the tiled z-march (k_residual_tile),
// narrower grids the per-cell one (k_residual).
template <typename T, typename TR, bool DOT, bool GATED>
int launch_residual(jg_solver* s, const Row<T>* A, const T* x, const T* b, TR* r, const Dims& d,
                    double* partial, const Ctl* ctl) {
    if (use_tm(d)) {
        dim3 grid;
        int zc;
        tm_grid(d, grid, zc);
        k_residual_tile<T, TR, DOT, GATED><<<grid_sys(grid, s), dim3(kTmX, kTmY, 1), 0, s->stream>>>(
            A, x, b, r, d, zc, partial, ctl);
        return (int)(grid.x * grid.y * grid.z);
    }
    const Geo g = geo_stencil(d);
    k_residual<T, T, TR, DOT, false, GATED><<<grid_sys(g.grid, s), g.block, 0, s->stream>>>(
        A, x, b, r, d, g.zc, partial, ctl);
    return nblocks(g);
}

// PCG's true residual on the iterations that ask for it, over a bounded
// number of blocks; RR: partials of r.r, whose count per system is returned.
template <typename T, bool RR>
int launch_refresh(jg_solver* s, const Row<T>* A, const T* x, const T* b, T* r, const Dims& d,
                   double* partial, const Ctl* ctl) {
    if (d.nz == 1 && s->nsys == 1) {
        const int nb = std::min(nblocks_1d(d.n()), 1024);
        k_residual_plane_refresh<T, RR><<<nb, NT, 0, s->stream>>>(A, x, b, r, d, partial, ctl);
        return nb;
    }
    if (use_tm(d)) {
        dim3 grid;
        int zc;
        tm_grid(d, grid, zc);
        const int tiles = (int)(grid.x * grid.y * grid.z), nb = std::min(tiles, 1024);
        k_refresh_tile<T, RR><<<dim3((unsigned)nb, (unsigned)s->nsys, 1), dim3(kTmX, kTmY, 1), 0,
                                s->stream>>>(A, x, b, r, d, zc, tiles, partial, ctl);
        return nb;
    }
    const Geo g = geo_stencil(d);
    k_residual<T, T, T, RR, true><<<grid_sys(g.grid, s), g.block, 0, s->stream>>>(A, x, b, r, d, g.zc,
                                                                                  partial, ctl);
    return nblocks(g);
}

// One (weighted) Jacobi sweep of a single system: the tiled z-march where the
// grid is large and deep enough for it, else the per-cell kernel.  Whole calls
// of jg_relax_jacobi, us, per cell / tiled: 150x122x106 41 + 14 / 22 + 14;
// 48^3 (110 592 cells) 14.9 / 15.9, 1000x500x1 17.5 / 18.3.
constexpr idx_t kJacobiTileCells = idx_t(1) << 17;
template <typename T, bool ZC>
void launch_jacobi(jg_solver* s, const Row<T>* A, const T* b, const T* x, T* xo, const Dims& d, T omega,
                   const Ctl* ctl) {
    if (use_tm(d) && d.nz > 1 && d.n() >= kJacobiTileCells) {
        dim3 grid;
        int zc;
        tm_grid(d, grid, zc);
        k_jacobi_tile<T, ZC><<<grid, dim3(kTmX, kTmY, 1), 0, s->stream>>>(A, b, x, xo, d, zc, omega, ctl);
        return;
    }
    const Geo g = geo_stencil(d);
    k_jacobi<T, T, ZC><<<g.grid, g.block, 0, s->stream>>>(A, b, x, xo, d, g.zc, omega, ctl);
}

template <typename T>
struct MgCfg {
    unsigned pre, post0, post, coarsest;
    T omega;
    int pairs = 0;         // jg_gpu_options.sweep_pairs
    bool jacobi = false;   // weighted-Jacobi smoothing (JG_SMOOTH_JACOBI)
};

// The V-cycle with weighted Jacobi smoothing (JG_SMOOTH_JACOBI): zero initial
// guess, `pre` sweeps x += omega ((b - s) / c - x) (FdmJacobiSolver3::relax,
// src/jet/fdm_jacobi_solver3.cpp:95-112, weighted), the residual and Jet's
// restriction, recursion, Jet's correction, `post` sweeps; `coarsest` sweeps
// on the coarsest level.  Every level keeps its current iterate in x and
// sweeps out of place into y, copying back after an odd count; 2-D
// hierarchies take FdmMgUtils2's transfers and the one-plane residual.
template <typename T>
int vcycle_jacobi(jg_solver* s, const T* r0, T* z0, const MgCfg<T>& c, const Ctl* ctl) {
    const size_t L = s->lv.size();
    auto B = [&](size_t l) -> const T* { return l == 0 ? r0 : Prec<T>::b(s->lv[l]); };
    auto X = [&](size_t l) -> T* { return l == 0 ? z0 : Prec<T>::x(s->lv[l]); };
    // `count` sweeps of level l's x (through y; the result ends in x)
    auto sweeps = [&](size_t l, unsigned count) {
        Level& lv = s->lv[l];
        const Dims& d = lv.d;
        T* x = X(l);
        T* y = Prec<T>::y(lv);
        const T* in = x;
        for (unsigned k = 0; k < count; ++k) {
            T* out = in == x ? y : x;
            launch_jacobi<T, true>(s, Prec<T>::A(lv), B(l), in, out, d, c.omega, ctl);
            in = out;
        }
        if (in != x) k_convert<T, T><<<nblocks_1d(d.n()), NT, 0, s->stream>>>(in, x, d.n());
    };
    for (size_t l = 0; l < L; ++l) {
        Level& lv = s->lv[l];
        const Dims& d = lv.d;
        k_fill<T><<<nblocks_1d(d.n()), NT, 0, s->stream>>>(X(l), T(0), d.n());
        if (l + 1 == L) {
            sweeps(l, c.coarsest);
            break;
        }
        sweeps(l, c.pre);
        const Dims& cd = s->lv[l + 1].d;
        const Geo gc = geo_planes(cd);
        if (s->twod) {
            const Geo gf = geo_planes(d);
            k_residual_plane<T><<<gf.grid, gf.block, 0, s->stream>>>(Prec<T>::A(lv), X(l), B(l),
                                                                    Prec<T>::t(lv), d, ctl);
            k_restrict2<T><<<gc.grid, gc.block, 0, s->stream>>>(Prec<T>::t(lv),
                                                                Prec<T>::b(s->lv[l + 1]), cd, ctl);
        } else {
            const Geo gf = geo_stencil(d);
            k_residual<T, T, T, false, false, true><<<gf.grid, gf.block, 0, s->stream>>>(
                Prec<T>::A(lv), X(l), B(l), Prec<T>::t(lv), d, gf.zc, nullptr, ctl);
            k_restrict<T><<<gc.grid, gc.block, 0, s->stream>>>(Prec<T>::t(lv),
                                                               Prec<T>::b(s->lv[l + 1]), cd, ctl);
        }
        JG_TRY(check_launch(s, "jacobi vcycle down"));
    }
    for (size_t l = L - 1; l-- > 0;) {
        const Dims& d = s->lv[l].d;
        const Geo gf = geo_planes(d);
        if (s->twod)
            k_correct2<T><<<gf.grid, gf.block, 0, s->stream>>>(X(l + 1), X(l), d, ctl);
        else
            k_correct<T><<<gf.grid, gf.block, 0, s->stream>>>(X(l + 1), X(l), d, ctl);
        sweeps(l, l == 0 ? c.post0 : c.post);
        JG_TRY(check_launch(s, "jacobi vcycle up"));
    }
    return JG_OK;
}

// Two sweeps of a one-plane level in one launch (k_rb_sweep2_plane): xin
// nullptr starts from zero, coarse adds its prolongation to the start, res
// receives the residual of the result.  The residual is fused only into
// first-colour-0 (pre-smoothing) pairs and the correction only into
// first-colour-1 (post-smoothing) pairs, never both; dot (post-smoothing
// only) writes the b.x / b.b partials to slots 0 and 1 and returns their
// count (else 0).
template <typename T>
int launch_plane2(jg_solver* s, const Row<T>* A, const T* b, const T* xin, const T* coarse,
                  T* xout, T* res, const Dims& d, int first, T omega, const Ctl* ctl,
                  bool dot = false) {
    const int H = p2_halo(res != nullptr);
    const int IX = kP2X - 2 * H, IY = P2Cfg<T>::TY - 2 * H;
    const dim3 grid((d.nx + IX - 1) / IX, (d.ny + IY - 1) / IY, 1);
    const dim3 block(kP2Lanes, P2Cfg<T>::NW, 1);
    hipStream_t st = s->stream;
    double *p0 = s->slot(0), *p1 = s->slot(1);
#define JG_P2(F, XI, RE, CO, DO)                                                                \
    k_rb_sweep2_plane<T, F, XI, RE, CO, DO><<<grid, block, 0, st>>>(A, b, xin, coarse, xout, res, \
                                                                    d, omega, ctl, p0, p1)
    if (first == 0) {
        if (xin) {
            if (res) JG_P2(0, true, true, false, false);
            else JG_P2(0, true, false, false, false);
        } else {
            if (res) JG_P2(0, false, true, false, false);
            else JG_P2(0, false, false, false, false);
        }
        return 0;
    }
    if (dot) {
        if (xin) {
            if (coarse) JG_P2(1, true, false, true, true);
            else JG_P2(1, true, false, false, true);
        } else {
            if (coarse) JG_P2(1, false, false, true, true);
            else JG_P2(1, false, false, false, true);
        }
        return (int)(grid.x * grid.y);
    }
    if (xin) {
        if (coarse) JG_P2(1, true, false, true, false);
        else JG_P2(1, true, false, false, false);
    } else {
        if (coarse) JG_P2(1, false, false, true, false);
        else JG_P2(1, false, false, false, false);
    }
#undef JG_P2
    return 0;
}

// The V-cycle on a 2-D hierarchy (FdmMgLinearSystem2): the same symmetric
// cycle as vcycle() below, with FdmMgUtils2's transfers and Jet's 2-D relax.
// Consecutive sweeps of a level run two per launch (k_rb_sweep2_plane): the
// last pre-smoothing pair also writes the residual the restriction reads,
// and the first post-smoothing pair adds the prolonged correction as it
// loads x.  Leftover single sweeps (odd counts, or pairs < 0) take
// k_rb_sweep_plane, with separate k_residual_plane / k_correct2 launches
// where nothing fuses them; a coarsest level of at most kCoarseMaxCells
// cells runs all its sweeps in one workgroup (k_coarsest_plane).  The
// result is bit-identical either way.
template <typename T>
int vcycle2d(jg_solver* s, const T* r0, T* z0, const MgCfg<T>& c, const Ctl* ctl, int* dot_blocks) {
    const size_t L = s->lv.size();
    auto B = [&](size_t l) -> const T* { return l == 0 ? r0 : Prec<T>::b(s->lv[l]); };
    auto X = [&](size_t l) -> T* { return l == 0 ? z0 : Prec<T>::x(s->lv[l]); };
    const unsigned fwd = std::max(1u, (c.coarsest + 1) / 2);
    // one sweep of a one-plane level: k_rb_sweep_plane, 60 x 12 interiors
    auto sweep = [&](size_t l, const T* in, T* out, int first) {
        Level& lv = s->lv[l];
        const Dims& d = lv.d;
        const dim3 grid((d.nx + kSwIX - 1) / kSwIX, (d.ny + kSwIY - 1) / kSwIY, 1);
        const dim3 block(kSwLX, kSwLY, 1);
        const Row<T>* A = Prec<T>::A(lv);
        if (first == 0) {
            if (in)
                k_rb_sweep_plane<T, 0, false><<<grid, block, 0, s->stream>>>(A, B(l), in, out, d, c.omega, ctl);
            else
                k_rb_sweep_plane<T, 0, true><<<grid, block, 0, s->stream>>>(A, B(l), in, out, d, c.omega, ctl);
        } else {
            if (in)
                k_rb_sweep_plane<T, 1, false><<<grid, block, 0, s->stream>>>(A, B(l), in, out, d, c.omega, ctl);
            else
                k_rb_sweep_plane<T, 1, true><<<grid, block, 0, s->stream>>>(A, B(l), in, out, d, c.omega, ctl);
        }
    };
    // n sweeps of one colour order as launches of 2 and 1 sweeps: a leftover
    // single first (lead = true: the pre-smoothing, whose last pair carries
    // the residual) or last (the post-smoothing, whose first pair carries the
    // correction)
    auto plan = [&](unsigned n, bool lead) {
        std::vector<int> p;
        if (c.pairs < 0) return std::vector<int>(n, 1);
        if (lead && n % 2) p.push_back(1);
        for (unsigned k = 0; k + 1 < n; k += 2) p.push_back(2);
        if (!lead && n % 2) p.push_back(1);
        return p;
    };
    // Launch m of a level's M launches writes ((M-1-m) even ? x : y), so the
    // last lands in x; an unfused correction is added in place to the buffer
    // the pre-smoothing left (zeroed first when there is none).
    std::vector<const T*> pre_out(L, nullptr);
    for (size_t l = 0; l < L; ++l) {
        Level& lv = s->lv[l];
        const Dims& d = lv.d;
        const Row<T>* A = Prec<T>::A(lv);
        T* Y = Prec<T>::y(lv);
        if (l + 1 == L && c.pairs >= 0 && d.n() <= (idx_t)kCoarseMaxCells) {
            // every coarsest sweep in one workgroup
            k_coarsest_plane<T><<<1, kCoarseThreads, 0, s->stream>>>(A, B(l), X(l), d, (int)fwd,
                                                                     c.omega, ctl);
            JG_TRY(check_launch(s, "coarsest 2-D"));
            break;
        }
        if (l + 1 == L) {
            const std::vector<int> fw = plan(fwd, true), bw = plan(fwd, false);
            const size_t M = fw.size() + bw.size();
            const T* in = nullptr;
            for (size_t m = 0; m < M; ++m) {
                T* out = ((M - 1 - m) % 2 == 0) ? X(l) : Y;
                const bool f = m < fw.size();
                const int n = f ? fw[m] : bw[m - fw.size()];
                if (n == 2)
                    launch_plane2<T>(s, A, B(l), in, nullptr, out, nullptr, d, f ? 0 : 1, c.omega, ctl);
                else
                    sweep(l, in, out, f ? 0 : 1);
                in = out;
            }
            JG_TRY(check_launch(s, "coarsest 2-D"));
            break;
        }
        const unsigned post = l == 0 ? c.post0 : c.post;
        const std::vector<int> pre = plan(c.pre, true);
        const size_t M = pre.size() + plan(post, false).size();
        const T* in = nullptr;
        bool res_done = false;
        for (size_t m = 0; m < pre.size(); ++m) {
            T* out = ((M - 1 - m) % 2 == 0) ? X(l) : Y;
            res_done = pre[m] == 2 && m + 1 == pre.size();
            if (pre[m] == 2)
                launch_plane2<T>(s, A, B(l), in, nullptr, out, res_done ? Prec<T>::t(lv) : nullptr, d,
                                 0, c.omega, ctl);
            else
                sweep(l, in, out, 0);
            in = out;
        }
        pre_out[l] = in;
        const Dims& cd = s->lv[l + 1].d;
        const Geo gc = geo_planes(cd);
        if (in) {
            if (!res_done) {
                const Geo gf = geo_planes(d);
                k_residual_plane<T><<<gf.grid, gf.block, 0, s->stream>>>(A, in, B(l), Prec<T>::t(lv),
                                                                        d, ctl);
            }
            k_restrict2<T><<<gc.grid, gc.block, 0, s->stream>>>(Prec<T>::t(lv),
                                                                Prec<T>::b(s->lv[l + 1]), cd, ctl);
        } else {
            k_restrict2<T><<<gc.grid, gc.block, 0, s->stream>>>(B(l), Prec<T>::b(s->lv[l + 1]), cd,
                                                                ctl);
        }
        JG_TRY(check_launch(s, "vcycle 2-D down"));
    }
    for (size_t l = L - 1; l-- > 0;) {
        Level& lv = s->lv[l];
        const Dims& d = lv.d;
        const Row<T>* A = Prec<T>::A(lv);
        T* Y = Prec<T>::y(lv);
        const unsigned post_n = l == 0 ? c.post0 : c.post;
        const size_t P = plan(c.pre, true).size();
        const std::vector<int> post = plan(post_n, false);
        const size_t M = P + post.size();
        const T* in = pre_out[l];
        const bool fused = !post.empty() && post[0] == 2;
        if (!fused) {
            T* cur = const_cast<T*>(in);
            if (!cur) {
                cur = (M % 2 == 0) ? X(l) : Y;
                k_fill<T><<<nblocks_1d(d.n()), NT, 0, s->stream>>>(cur, T(0), d.n());
            }
            const Geo gf = geo_planes(d);
            k_correct2<T><<<gf.grid, gf.block, 0, s->stream>>>(X(l + 1), cur, d, ctl);
            in = cur;
        }
        for (size_t q = 0; q < post.size(); ++q) {
            T* out = ((M - 1 - (P + q)) % 2 == 0) ? X(l) : Y;
            // the last level-0 launch also forms PCG's r.z and r.r partials
            const bool dot = l == 0 && q + 1 == post.size();
            if (post[q] == 2)
                *dot_blocks = launch_plane2<T>(s, A, B(l), in, q == 0 ? X(l + 1) : nullptr, out,
                                               nullptr, d, 1, c.omega, ctl, dot);
            else
                sweep(l, in, out, 1);
            in = out;
        }
        JG_TRY(check_launch(s, "vcycle 2-D up"));
    }
    return JG_OK;
}

// z = M r: one symmetric V-cycle with zero initial guess.  Level 0 reads
// its right-hand side from r0 and writes its result to z0.  Each level runs
// `pre` forward sweeps (red then black) from x = 0, restricts the residual,
// recurses, then `post` backward sweeps (black then red), the first of which
// adds the prolonged coarse correction as it loads x.  Sweeps ping-pong
// between the level's x and y vectors so that the last one lands in x.
// Returns the number of b.x / b.b partials the last level-0 sweep wrote to
// slots 0 and 1 (0 if it wrote none).
template <typename T>
int vcycle(jg_solver* s, const T* r0, T* z0, const MgCfg<T>& c, const Ctl* ctl, int* dot_blocks) {
    const size_t L = s->lv.size();
    *dot_blocks = 0;
    if ((c.jacobi || s->twod) && s->nsys > 1) return JG_ERR_UNSUPPORTED;  // batches are 3-D red-black
    if (c.jacobi) return vcycle_jacobi<T>(s, r0, z0, c, ctl);
    if (s->twod) return vcycle2d<T>(s, r0, z0, c, ctl, dot_blocks);
    auto B = [&](size_t l) -> const T* { return l == 0 ? r0 : Prec<T>::b(s->lv[l]); };
    auto X = [&](size_t l) -> T* { return l == 0 ? z0 : Prec<T>::x(s->lv[l]); };
    std::vector<const T*> pre_out(L, nullptr);
    // Levels from `bot` down run in one workgroup (k_bottom).
    size_t bot = L;
    for (size_t l = 0; l < L; ++l)
        if (s->lv[l].d.n() <= BotCfg<T>::MaxCells) {
            bot = l;
            break;
        }
    const int fwd = (int)std::max(1u, (c.coarsest + 1) / 2);
    size_t top = L;  // first level of the upward pass
    for (size_t l = 0; l < L; ++l) {
        Level& lv = s->lv[l];
        const Row<T>* A = Prec<T>::A(lv);
        const Dims& d = lv.d;
        T* Y = Prec<T>::y(lv);
        if (l == bot) {
            if (L - l > (size_t)kBotMaxLevels) return JG_ERR_UNSUPPORTED;
            BotLevels<T> bl;
            bl.L = (int)(L - l);
            bl.d[0] = d;
            for (size_t m = l; m < L; ++m) bl.A[m - l] = Prec<T>::A(s->lv[m]);
            const int post_top = (int)(l == 0 ? c.post0 : c.post);
            if (d.nx % 2 == 0)
                k_bottom<T, true><<<s->nsys, kBotThreads, 0, s->stream>>>(bl, B(l), X(l), (int)c.pre,
                                                                    post_top, (int)c.post, fwd,
                                                                    c.omega, ctl);
            else
                k_bottom<T, false><<<s->nsys, kBotThreads, 0, s->stream>>>(bl, B(l), X(l), (int)c.pre,
                                                                     post_top, (int)c.post, fwd,
                                                                     c.omega, ctl);
            JG_TRY(check_launch(s, "bottom"));
            top = l;
            break;
        }
        if (l + 1 == L) {
            // coarsest level too large for one workgroup: symmetric fused
            // sweeps, fwd forward and fwd backward ones
            const std::vector<int> plan = sweep_plan<T>(s, d, (unsigned)fwd, c.pairs);
            const size_t half = plan.size(), M = 2 * half;
            const T* in = nullptr;
            for (size_t m = 0; m < M; ++m) {
                T* out = ((M - 1 - m) % 2 == 0) ? X(l) : Y;
                const int first = m < half ? 0 : 1, mode = plan[m < half ? m : m - half];
                if (mode == kLaunchBrick)
                    launch_brick2<T>(s, A, B(l), in, out, d, first, nullptr, c.omega, ctl);
                else if (mode == kLaunchMarch)
                    JG_TRY(launch_sweep2<T>(s, A, B(l), in, out, d, first, nullptr, nullptr, c.omega, ctl));
                else
                    launch_sweep<T>(s, A, B(l), in, out, d, first, nullptr, nullptr, nullptr, c.omega, ctl);
                in = out;
            }
            JG_TRY(check_launch(s, "coarsest"));
            top = l;
            break;
        }
        const unsigned post = l == 0 ? c.post0 : c.post;
        // launches of the level ping-pong between x and y so the last lands in x
        const std::vector<int> pre_plan = sweep_plan<T>(s, d, c.pre, c.pairs);
        const size_t M = pre_plan.size() + sweep_plan<T>(s, d, post, c.pairs).size();
        auto buf = [&](size_t m) -> T* { return ((M - 1 - m) % 2 == 0) ? X(l) : Y; };
        const T* in = nullptr;
        for (size_t m = 0; m < pre_plan.size(); ++m) {
            if (pre_plan[m] == kLaunchBrick)
                launch_brick2<T>(s, A, B(l), in, buf(m), d, 0, nullptr, c.omega, ctl);
            else if (pre_plan[m] == kLaunchMarch) {
                const bool res = m + 1 == pre_plan.size();
                JG_TRY(launch_sweep2<T>(s, A, B(l), in, buf(m), d, 0, nullptr,
                                        res ? Prec<T>::t(lv) : nullptr, c.omega, ctl));
            }
            else
                launch_sweep<T>(s, A, B(l), in, buf(m), d, 0, nullptr, nullptr, nullptr, c.omega, ctl);
            in = buf(m);
        }
        pre_out[l] = in;  // nullptr: x is still zero
        const Dims& cd = s->lv[l + 1].d;
        Geo gc = geo_planes(cd);
        const bool from_t = in && sizeof(T) == 4 && pre_plan.back() == kLaunchMarch;  // t holds the residual
        if (in && !from_t && d.n() * s->nsys <= kRbMaxCells) {
            const dim3 grid = grid_sys(dim3((cd.nx + kRbX - 1) / kRbX, (cd.ny + kRbY - 1) / kRbY,
                                            (cd.nz + kRbZ - 1) / kRbZ), s);
            k_residual_restrict_brick<T><<<grid, kRbThreads, 0, s->stream>>>(
                A, in, B(l), Prec<T>::b(s->lv[l + 1]), d, cd, ctl);
        } else if (in && sizeof(T) == 8) {
            // FP64: residual into t, then restriction (the fused kernel's
            // register footprint halves its occupancy in FP64, and the pair
            // measures faster)
            launch_residual<T, T, false, true>(s, A, in, B(l), Prec<T>::t(lv), d, nullptr, ctl);
            k_restrict<T><<<grid_sys(gc.grid, s), gc.block, 0, s->stream>>>(Prec<T>::t(lv), Prec<T>::b(s->lv[l + 1]),
                                                               cd, ctl);
        } else if (in) {
            // restricting a stored residual is one load per cell: twice the
            // blocks (shorter chunks) keep more loads in flight
            const int zc = from_t ? rr_zc(cd, 2048) : rr_zc(cd);
            const dim3 grid = grid_sys(
                dim3((cd.nx + kRrCX - 1) / kRrCX, (cd.ny + kRrCY - 1) / kRrCY, (cd.nz + zc - 1) / zc), s);
            if (from_t)
                k_residual_restrict<T, true><<<grid, dim3(kRrLX, kRrTY, 1), 0, s->stream>>>(
                    nullptr, nullptr, Prec<T>::t(lv), Prec<T>::b(s->lv[l + 1]), d, cd, zc, ctl);
            else
                k_residual_restrict<T><<<grid, dim3(kRrLX, kRrTY, 1), 0, s->stream>>>(
                    A, in, B(l), Prec<T>::b(s->lv[l + 1]), d, cd, zc, ctl);
        } else {
            k_restrict<T><<<grid_sys(gc.grid, s), gc.block, 0, s->stream>>>(B(l), Prec<T>::b(s->lv[l + 1]), cd,
                                                               ctl);
        }
        JG_TRY(check_launch(s, "vcycle down"));
    }
    for (size_t l = top; l-- > 0;) {
        Level& lv = s->lv[l];
        const Row<T>* A = Prec<T>::A(lv);
        const Dims& d = lv.d;
        T* Y = Prec<T>::y(lv);
        const unsigned post = l == 0 ? c.post0 : c.post;
        const size_t P0 = sweep_plan<T>(s, d, c.pre, c.pairs).size();
        const std::vector<int> post_plan = sweep_plan<T>(s, d, post, c.pairs);
        const size_t M = P0 + post_plan.size();
        auto buf = [&](size_t m) -> T* { return ((M - 1 - m) % 2 == 0) ? X(l) : Y; };
        const T* coarse = X(l + 1);
        if (post == 0) {
            // No post-smoothing: x = pre-smoothed x (already in X) + P e.
            if (!pre_out[l]) k_fill<T><<<grid_1d(nblocks_1d(d.n()), s), NT, 0, s->stream>>>(X(l), T(0), d.n());
            Geo gf = geo_planes(d);
            k_correct<T><<<grid_sys(gf.grid, s), gf.block, 0, s->stream>>>(coarse, X(l), d, ctl);
        } else {
            const T* in = pre_out[l];
            for (size_t q = 0; q < post_plan.size(); ++q) {
                const size_t m = P0 + q;
                const bool last0 = (l == 0 && m + 1 == M);
                const T* cor = q == 0 ? coarse : nullptr;
                // the two-sweep kernel leaves r.z / r.r to one fused dot kernel
                // (accumulating them in it costs more than that pass)
                const bool dot = last0 && post_plan[q] == kLaunchSingle;
                double* pbx = dot ? s->slot(0) : nullptr;
                double* pbb = dot ? s->slot(1) : nullptr;
                int nb = 0;
                if (post_plan[q] == kLaunchBrick)
                    launch_brick2<T>(s, A, B(l), in, buf(m), d, 1, cor, c.omega, ctl);
                else if (post_plan[q] == kLaunchMarch)
                    JG_TRY(launch_sweep2<T>(s, A, B(l), in, buf(m), d, 1, cor, nullptr, c.omega, ctl));
                else
                    nb = launch_sweep<T>(s, A, B(l), in, buf(m), d, 1, cor, pbx, pbb, c.omega, ctl);
                if (dot) *dot_blocks = nb;
                in = buf(m);
            }
        }
        JG_TRY(check_launch(s, "vcycle up"));
    }
    return JG_OK;
}

// --------------------------------------------------------------- PCG

// Vectors and control block of one PCG solve.
template <typename T>
struct Pcg {
    const Row<T>* A;
    const T* b;
    T *x, *r, *z, *dA, *dB, *q;
    Dims d;
    Ctl* ctl;
    const MgCfg<T>* mg;  // nullptr: no preconditioner (z aliases r)
    const CsrDev* csr = nullptr;  // compressed system (FP64, no preconditioner): A unused, d = {rows, 1, 1}
    const EllDev* ell = nullptr;  // its ELL copy, when it has one
};

// z = M r and the r.z / r.r partials in slots 0 / 1 (from the V-cycle's last
// sweep when it provides them, else from dot kernels); returns the partial
// count, or minus a status.
// The fused direction update and SpMV of a PCG iteration on level-0 shape d
// (nsys systems back to back), its d.q partials in `partial`; returns their
// count per system.  One plane: k_dir_spmv_plane; rows of at least 48
// cells: the tiled z-march k_dir_spmv_tile; narrower grids keep the
// per-cell z-march k_dir_spmv (a 64-lane row would idle too many lanes).
template <typename T>
int launch_dir_spmv(jg_solver* s, const Row<T>* A, const T* z, const T* dold, T* dnew, T* q,
                    const Dims& d, double* partial, const Ctl* ctl) {
    if (d.nz == 1 && s->nsys == 1) {
        const dim3 grid((d.nx + kP2X - 1) / kP2X, (d.ny + SpCfg<T>::TY - 1) / SpCfg<T>::TY, 1);
        k_dir_spmv_plane<T><<<grid, dim3(kP2Lanes, SpCfg<T>::NW, 1), 0, s->stream>>>(
            A, z, dold, dnew, q, d, partial, ctl);
        return (int)(grid.x * grid.y);
    }
    if (use_tm(d)) {
        dim3 grid;
        int zc;
        tm_grid(d, grid, zc);
        k_dir_spmv_tile<T><<<grid_sys(grid, s), dim3(kTmX, kTmY, 1), 0, s->stream>>>(
            A, z, dold, dnew, q, d, zc, partial, ctl);
        return (int)(grid.x * grid.y * grid.z);
    }
    const Geo g = geo_stencil(d);
    k_dir_spmv<T, T><<<grid_sys(g.grid, s), g.block, 0, s->stream>>>(A, z, dold, dnew, q, d, g.zc,
                                                                     partial, ctl);
    return nblocks(g);
}

template <typename T>
int pcg_precondition(jg_solver* s, const Pcg<T>& v, const Ctl* c) {
    const idx_t n = v.d.n();
    const int nb1 = nblocks_1d(n);
    int nb = 0;
    const int st = vcycle<T>(s, v.r, v.z, *v.mg, c, &nb);
    if (st != JG_OK) return -st;
    if (nb == 0) {
        k_dot_rz_rr<T><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.r, v.z, n, s->slot(0), s->slot(1), c);
        nb = nb1;
    }
    return nb;
}

// Start of Jet's pcg (include/jet/detail/cg-inl.h:15-50): r = b - A x, d = 0,
// z = M r, sigma = r.z.  Launches only; the control block says whether to go on.
template <typename T>
int pcg_init(jg_solver* s, const Pcg<T>& v) {
    const idx_t n = v.d.n();
    const int nb1 = nblocks_1d(n);
    // r = b - A x with x = 0 (every caller zeroes x first, as Jet's solvers
    // do): b - A 0 is b bit for bit, so a copy
    k_convert<T, T><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.b, v.r, n);
    k_fill<T><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.dA, T(0), n);
    k_fill<T><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.dB, T(0), n);
    // (a batch group gates the preconditioner by the control blocks, which
    // say which members take part; a single system's is not set up yet)
    int nb = nb1;
    if (v.mg)
        nb = pcg_precondition<T>(s, v, s->nsys > 1 ? v.ctl : nullptr);
    else  // z = r
        k_dot<T, T><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.r, v.r, n, s->slot(0), nullptr);
    if (nb < 0) return -nb;
    k_fin_init<<<s->nsys, kFinThreads, 0, s->stream>>>(
        v.ctl, s->slot(0), v.mg ? s->slot(1) : s->slot(0), nb, s->nsys > 1 ? nullptr : s->ctl_host);
    return check_launch(s, "pcg init");
}

// One iteration of Jet's pcg loop (include/jet/detail/cg-inl.h:52-91) on the
// device; every kernel is gated by the control block, so iterations can be
// launched (or replayed from a graph) past convergence.  odd: the two
// direction buffers swap roles every iteration.  host: where the host polls
// the control block (nullptr: nowhere).
template <typename T>
int pcg_iteration(jg_solver* s, const Pcg<T>& v, bool odd, Ctl* host) {
    const idx_t n = v.d.n();
    const int nb1 = nblocks_1d(n);
    T* dold = odd ? v.dB : v.dA;
    T* dnew = odd ? v.dA : v.dB;
    if constexpr (sizeof(T) == 8) {
        // (no stencil geometry here: geo_stencil of a {rows, 1, 1} shape
        // never meets its partial-count bound once rows > 64 * kMaxPartials)
        if (v.csr) {
            if (v.ell) {
                // d first, then q = A d gathering d alone: 477.8 ms for the 256^3
                // scene's compressed CG against 493.9 with d formed per entry
                k_ell_dir<<<nb1, NT, 0, s->stream>>>(v.z, dold, dnew, n, v.ctl);
                k_ell_spmv_dot<<<nb1, NT, 0, s->stream>>>(*v.ell, dnew, v.q, s->slot(2), v.ctl);
            } else
                k_csr_dir_spmv<<<nb1, NT, 0, s->stream>>>(*v.csr, v.z, dold, dnew, v.q, n,
                                                          s->slot(2), v.ctl);
            k_fin_alpha<<<1, kFinThreads, 0, s->stream>>>(v.ctl, s->slot(2), nb1, host);
            k_update_xr<T, true><<<nb1, NT, 0, s->stream>>>(v.x, v.r, dnew, v.q, n, s->slot(0), v.ctl);
            if (v.ell)
                k_ell_residual<true, true><<<nb1, NT, 0, s->stream>>>(*v.ell, v.x, v.b, v.r, s->slot(0),
                                                                      v.ctl);
            else
                k_csr_residual<true, true><<<nb1, NT, 0, s->stream>>>(*v.csr, v.x, v.b, v.r, n,
                                                                      s->slot(0), v.ctl);
            k_fin_sigma<<<1, kFinThreads, 0, s->stream>>>(v.ctl, s->slot(0), s->slot(0), nb1, nb1, host);
            return check_launch(s, "csr pcg iteration");
        }
    }
    const int nsp = launch_dir_spmv<T>(s, v.A, v.z, dold, dnew, v.q, v.d, s->slot(2), v.ctl);
    k_fin_alpha<<<s->nsys, kFinThreads, 0, s->stream>>>(v.ctl, s->slot(2), nsp, host);
    if (!v.mg) {  // z = r: sigma is r.r
        k_update_xr<T, true><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.x, v.r, dnew, v.q, n, s->slot(0),
                                                                    v.ctl);
        const int nr = launch_refresh<T, true>(s, v.A, v.x, v.b, v.r, v.d, s->slot(0), v.ctl);
        k_fin_sigma<<<s->nsys, kFinThreads, 0, s->stream>>>(v.ctl, s->slot(0), s->slot(0), nb1, nr, host);
        return check_launch(s, "cg iteration");
    }
    k_update_xr<T, false><<<grid_1d(nb1, s), NT, 0, s->stream>>>(v.x, v.r, dnew, v.q, n, nullptr, v.ctl);
    launch_refresh<T, false>(s, v.A, v.x, v.b, v.r, v.d, nullptr, v.ctl);
    const int nb = pcg_precondition<T>(s, v, v.ctl);
    if (nb < 0) return -nb;
    k_fin_sigma<<<s->nsys, kFinThreads, 0, s->stream>>>(v.ctl, s->slot(0), s->slot(1), nb, nb, host);
    return check_launch(s, "pcg iteration");
}

// Rows per thread when the CG of v (FP64, no preconditioner) runs as one
// launch (k_cg_grid), 0 when it does not: every row of the system has to fit
// the registers of one block per CU, with at most kCgW entries.  One row per thread as far as that goes: at 64^3 256 blocks of
// one take 8.2 us an iteration, 128 blocks of two 10.4, though their sums
// cost less.
int cg_grid_rows(jg_solver* s, const Pcg<double>& v) {
    const idx_t n = v.d.n(), per = (idx_t)std::min(s->cus, kCgMaxBlocks) * kCgThreads;
    if (v.mg || s->nsys > 1 || !s->cg_grid_ok || s->cg_polls <= 0 || n > 2 * per) return 0;
    if (v.csr && (!v.ell || s->csr.ell_w > kCgW)) return 0;
    return n > per ? 2 : 1;
}

// dalloc of something that a solve can do without: no room is no error.
template <typename T>
bool dalloc_spare(jg_solver* s, T** p, size_t count) {
    const std::string before = s->err;
    if (dalloc(s, p, count) == JG_OK) return true;
    (void)hipGetLastError();
    s->err = before;
    return false;
}

// pcg_device through k_cg_grid; the state after pcg_init in, x and the
// control block out.  *ran is false where that launch is not to be had (no
// room for its slots, refused, or a block did not arrive in time): the caller
// starts again without it, and so does every later solve of s.
int cg_grid(jg_solver* s, const Pcg<double>& v, int C, bool* ran) {
    *ran = false;
    if (!s->cg_slots && !dalloc_spare(s, &s->cg_slots, 3 * kCgSumWords)) {
        s->cg_grid_ok = false;
        return JG_OK;
    }
    const idx_t n = v.d.n();
    CgGridArgs a{v.A, v.ell ? *v.ell : EllDev{}, v.d, v.b, v.x, v.r, v.dA, v.ctl, s->cg_slots, s->cg_polls};
    const dim3 grid((unsigned)((n + (idx_t)C * kCgThreads - 1) / ((idx_t)C * kCgThreads)));
    auto* const f = v.ell ? (C == 1 ? k_cg_grid<1, true> : k_cg_grid<2, true>)
                          : (C == 1 ? k_cg_grid<1, false> : k_cg_grid<2, false>);
    // two of these launches at once could each hold the CUs the other waits for
    static std::mutex busy[16];
    std::lock_guard<std::mutex> lock(busy[s->device % 16]);
    do {
        k_fill<unsigned long long><<<nblocks_1d(3 * kCgSumWords), NT, 0, s->stream>>>(s->cg_slots, 0ull,
                                                                                  3 * kCgSumWords);
        JG_TRY(check_launch(s, "cg grid"));
        f<<<grid, kCgThreads, 0, s->stream>>>(a);
        const bool refused = hipGetLastError() != hipSuccess;
        JG_HIP(hipMemcpyAsync(s->ctl_host, v.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, s->stream));
        JG_TRY(sync(s));
        if (refused || s->ctl_host->pad) {
            s->cg_grid_ok = false;
            return JG_OK;
        }
    } while (!s->ctl_host->done);
    *ran = true;
    return JG_OK;
}

int upload_ctl(jg_solver* s, Ctl* dev, const Ctl& h) {
    JG_HIP(hipMemcpyAsync(dev, &h, sizeof(Ctl), hipMemcpyHostToDevice, s->stream));
    return JG_OK;
}

// Jet's pcg control flow (include/jet/detail/cg-inl.h:15-94) on the device.
// Vectors of type T; the matrix of level 0 is A; M is either the identity
// (z aliases r) or the V-cycle.  x must be zero on entry (Jet zeroes it).
// The host only polls the stop flag, every check_every iterations.
template <typename T>
int pcg_device(jg_solver* s, const Pcg<T>& v, unsigned check_every) {
    JG_TRY(pcg_init<T>(s, v));
    if constexpr (sizeof(T) == 8) {
        const int rows = cg_grid_rows(s, v);
        if (rows) {
            bool ran = false;
            JG_TRY(cg_grid(s, v, rows, &ran));
            if (ran) return JG_OK;
            JG_TRY(sync(s));
            const Ctl c = *s->ctl_host;
            Ctl h;
            std::memset(&h, 0, sizeof(Ctl));
            h.max_iter = c.max_iter;
            h.tol2 = c.tol2;
            h.stop_rule = c.stop_rule;
            h.rel2 = c.rel2;
            JG_TRY(upload_ctl(s, v.ctl, h));
            k_fill<T><<<nblocks_1d(v.d.n()), NT, 0, s->stream>>>(v.x, T(0), v.d.n());
            JG_TRY(pcg_init<T>(s, v));
        }
    }
    JG_TRY(sync(s));
    if (s->ctl_host->done) return JG_OK;
    const unsigned max_iter = s->ctl_host->max_iter;
    // One iteration of lookahead: iteration k+1 is enqueued before the host
    // waits for the stop flag iteration k left (every kernel of an iteration
    // returns at once once the control block says the solve has stopped), so
    // the device does not idle while the host polls.  When the last two
    // polled iterations predict (by their ratio) that the iteration in flight
    // meets the stop test, the host waits first instead: a speculative
    // iteration after the last one still costs its launches.
    auto metric = [](const Ctl& c) { return c.stop_rule == 1 ? c.rr : c.sigma; };
    const Ctl c0 = *s->ctl_host;
    const double lim = c0.stop_rule == 1 ? c0.rel2 * c0.bb : c0.tol2;
    double m_prev = -1.0, m_last = metric(c0);
    // Iteration k (from 1) belongs to the poll after its check_every, and every
    // iteration of a poll writes the poll's slot: the poll finds there the last
    // iteration that ran, its own or the one that stopped the solve, and the
    // iteration of look-ahead in flight by then writes the other slot.
    auto slot_of = [&](unsigned k) { return (int)(((k - 1) / check_every + 1) & 1); };
    unsigned launched = 0;
    auto iterate = [&]() -> int {
        const int st = pcg_iteration<T>(s, v, (launched & 1) != 0, s->ctl_host + slot_of(launched + 1));
        ++launched;
        return st;
    };
    int slot = 0;  // of the iteration polled
    JG_TRY(iterate());
    while (true) {
        const bool poll = launched % check_every == 0 || launched >= max_iter;
        if (poll) {
            slot = slot_of(launched);
            JG_HIP(hipEventRecord(s->evp[slot], s->stream));
        }
        bool more = launched <= max_iter;  // the device stops by itself at max_iter
        const bool likely_last = poll && m_prev > 0.0 && m_last > 0.0 && m_last < m_prev &&
                                 m_last * (m_last / m_prev) <= lim;
        if (more && !likely_last) {
            JG_TRY(iterate());
            more = false;  // already launched this pass
        }
        if (poll) {
            JG_HIP(hipEventSynchronize(s->evp[slot]));
            const Ctl& c = s->ctl_host[slot];
            if (c.done) {
                // final state in slot 0 for the callers (the look-ahead
                // iteration is a no-op and writes nothing)
                if (slot != 0) s->ctl_host[0] = c;
                return JG_OK;
            }
            m_prev = m_last;
            m_last = metric(c);
        }
        if (more) {  // the prediction was wrong: go on
            JG_TRY(iterate());
        } else if (launched > max_iter) {
            break;
        }
    }
    JG_HIP(hipMemcpyAsync(s->ctl_host, v.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, s->stream));
    return sync(s);
}

void init_ctl(Ctl* h, unsigned max_iter, double tol, int stop_rule, double rel_tol) {
    std::memset(h, 0, sizeof(Ctl));
    h->max_iter = max_iter;
    h->tol2 = tol * tol;
    h->stop_rule = stop_rule;
    h->rel2 = rel_tol * rel_tol;
}

int ensure_f32(jg_solver* s) {
    if (s->f32_valid) return JG_OK;
    for (auto& l : s->lv)
        k_rows_to_f32<<<grid_1d(nblocks_1d(l.d.n()), s), NT, 0, s->stream>>>(l.A64, l.A32, l.d.n());
    JG_TRY(check_launch(s, "rows_to_f32"));
    s->f32_valid = true;
    return JG_OK;
}

// r = b - A x of the FP64 finest level, stored as TR, with the partials of
// r.r written to `partial`; returns their count.  One-plane levels take the
// plane kernel (the z-marching one would spend its pipeline on one plane).
template <typename TR>
int residual_dot64(jg_solver* s, const Level& l0, TR* r, double* partial) {
    if (l0.d.nz == 1) {
        const int nb = nblocks_1d(l0.d.n());
        k_residual_plane_dot<TR><<<nb, NT, 0, s->stream>>>(l0.A64, s->x, s->b, r, l0.d, partial);
        return nb;
    }
    return launch_residual<double, TR, true, false>(s, l0.A64, s->x, s->b, r, l0.d, partial,
                                                          nullptr);
}

// FP64 ||b - A x|| / ||b|| of the finest level (reporting).
int true_rel_residual(jg_solver* s, double* out) {
    Level& l0 = s->lv[0];
    const int nb1 = nblocks_1d(l0.d.n());
    const int nr = residual_dot64<double>(s, l0, s->r, s->slot(0));
    k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(0), nr, s->scal + 0);
    k_dot<double, double><<<nb1, NT, 0, s->stream>>>(s->b, s->b, l0.d.n(), s->slot(1), nullptr);
    k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(1), nb1, s->scal + 1);
    JG_TRY(check_launch(s, "true residual"));
    double h[2];
    JG_HIP(hipMemcpyAsync(h, s->scal, sizeof(h), hipMemcpyDeviceToHost, s->stream));
    JG_TRY(sync(s));
    *out = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
    return JG_OK;
}

bool valid_dims(size_t nx, size_t ny, size_t nz) {
    const size_t lim = (size_t)1 << 30;
    return nx > 0 && ny > 0 && nz > 0 && nx < 65536 && ny < 65536 && nz < 65536 &&
           nx * ny * nz < lim * 2;
}

}  // namespace

namespace {

// Options of an MGPCG solve or V-cycle.  Every level of the caller's
// hierarchy is used, as Jet's mgVCycle recurses over A.levels.size()
// (include/jet/detail/mg-inl.h:26); max_levels only tells callers how deep to
// build it.  Relaxation factor of the red-black smoother: the GPU option if
// given, else the caller's Jet sorFactor (FdmMgSolver3's, default 1.5).  Any
// 0 < omega < 2 keeps the symmetric V-cycle positive definite.  Weight of the
// Jacobi smoother: the GPU option if given, else 6/7 (the weight that damps
// the high-frequency half of the 7-point Laplacian's spectrum best); it must
// lie in (0, 1], where 2 D / omega - A stays positive definite on diagonally
// dominant rows (plain Jacobi, omega = 1, barely smooths the checkerboard
// mode).
int mg_options(jg_solver* s, const jg_mg_params* p, const jg_gpu_options* o, jg_gpu_options* opt,
               double* omega) {
    if (o)
        *opt = *o;
    else
        jg_gpu_options_default(opt);
    if (opt->check_every == 0) opt->check_every = 1;
    if (opt->smoother == JG_SMOOTH_JACOBI) {
        *omega = opt->omega > 0 ? opt->omega : 6.0 / 7.0;
        if (!(*omega > 0.0 && *omega <= 1.0)) {
            s->err = "Jacobi smoother weight must lie in (0, 1]";
            return JG_ERR_INVALID_ARG;
        }
        return JG_OK;
    }
    if (opt->smoother != JG_SMOOTH_RBGS) {
        s->err = "unsupported smoother";
        return JG_ERR_UNSUPPORTED;
    }
    *omega = opt->omega > 0 ? opt->omega : p->sor;
    if (!(*omega > 0.0 && *omega < 2.0)) {
        s->err = "smoother relaxation factor must lie in (0, 2)";
        return JG_ERR_INVALID_ARG;
    }
    return JG_OK;
}

}  // namespace

// ====================================================================== C ABI

// The ELL copy of the resident compressed system when its rows are short
// enough (the longest row is found on the device); otherwise ell_w = 0 and
// the CG runs the CSR kernels.
static int csr_prepare_ell(jg_solver* s) {
    jg_solver::Csr& c = s->csr;
    if (c.ell_valid) return JG_OK;
    c.ell_w = 0;
    const int w = c.max_row;
    if (c.rows == 0 || w <= 0 || w > kEllMaxW) {
        c.ell_valid = true;  // the CSR kernels run
        return JG_OK;
    }
    const size_t cells = (size_t)w * c.rows;
    if (cells > c.ell_cap) {
        JG_TRY(dalloc(s, &c.ell_val, cells));
        JG_TRY(dalloc(s, &c.ell_ci, cells));
        c.ell_cap = cells;
    }
    if (c.rows > c.ell_rows_cap) {
        JG_TRY(dalloc(s, &c.ell_len, c.rows));
        c.ell_rows_cap = c.rows;
    }
    k_csr_to_ell<<<nblocks_1d((idx_t)c.rows), NT, 0, s->stream>>>(
        CsrDev{c.rp, c.ci, c.val, (int)c.nnz}, (idx_t)c.rows, c.ell_val, c.ell_ci, c.ell_len, w);
    JG_TRY(check_launch(s, "csr to ell"));
    c.ell_w = w;
    c.ell_valid = true;
    return JG_OK;
}

// FdmCgSolver3::solveCompressed on the solver's resident compressed system
// (A, b; x is overwritten): Jet's cg through pcg_device with the CSR kernels.
static int csr_solve(jg_solver* s, unsigned max_iter, double tol, jg_solve_info* info) {
    jg_solver::Csr& c = s->csr;
    JG_TRY(csr_prepare_ell(s));
    const CsrDev m{c.rp, c.ci, c.val, (int)c.nnz};
    const idx_t n = (idx_t)c.rows;
    const int nb1 = nblocks_1d(n);
    Ctl h;
    init_ctl(&h, max_iter, tol, 0, 0.0);
    JG_TRY(upload_ctl(s, s->ctl, h));
    k_fill<double><<<nb1, NT, 0, s->stream>>>(c.x, 0.0, n);  // Jet zeroes x (fdm_cg_solver3.cpp:62)
    JG_HIP(hipEventRecord(s->ev0, s->stream));
    Pcg<double> v{nullptr, c.b, c.x, c.r, c.r, c.dA, c.dB, c.q, Dims{(int)c.rows, 1, 1}, s->ctl, nullptr};
    v.csr = &m;
    const EllDev e{c.ell_val, c.ell_ci, c.ell_len, (idx_t)c.rows};
    if (c.ell_w > 0) v.ell = &e;
    JG_TRY(pcg_device<double>(s, v, 1));
    JG_HIP(hipEventRecord(s->ev1, s->stream));
    JG_TRY(sync(s));
    const Ctl ch = *s->ctl_host;
    if (info) {
        std::memset(info, 0, sizeof(*info));
        float ms = 0.f;
        JG_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
        info->solve_ms = ms;
        info->iterations = ch.iter;
        info->last_residual = std::sqrt(std::fabs(ch.sigma));
        // FdmCgSolver3::solveCompressed's return (src/jet/fdm_cg_solver3.cpp:72-73)
        info->converged = (info->last_residual <= tol) || (ch.iter < max_iter);
        // ||b - A x|| / ||b|| in FP64 (reporting)
        k_csr_residual<true, false><<<nb1, NT, 0, s->stream>>>(m, c.x, c.b, c.r, n, s->slot(0), nullptr);
        k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(0), nb1, s->scal + 0);
        k_dot<double, double><<<nb1, NT, 0, s->stream>>>(c.b, c.b, n, s->slot(1), nullptr);
        k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(1), nb1, s->scal + 1);
        JG_TRY(check_launch(s, "csr true residual"));
        double sc[2];
        JG_HIP(hipMemcpyAsync(sc, s->scal, sizeof(sc), hipMemcpyDeviceToHost, s->stream));
        JG_TRY(sync(s));
        info->rel_residual = sc[1] > 0 ? std::sqrt(sc[0] / sc[1]) : std::sqrt(sc[0]);
    }
    if (ch.nonfinite) {
        s->err = "non-finite value in CG reduction";
        return JG_ERR_NONFINITE;
    }
    return JG_OK;
}

// Room for a compressed system of rows x nnz and its CG vectors (grown when
// needed: the old arrays stay owned by the solver until it is released), and
// the reduction slots / control block if the solver has no hierarchy yet.
int csr_reserve(jg_solver* s, size_t rows, size_t nnz) {
    jg_solver::Csr& c = s->csr;
    if (rows > c.cap_rows || nnz > c.cap_nnz) {
        c.val = nullptr;
        JG_TRY(dalloc(s, &c.val, nnz));
        JG_TRY(dalloc(s, &c.rp, rows + 1));
        JG_TRY(dalloc(s, &c.ci, nnz));
        for (double** p : {&c.b, &c.x, &c.r, &c.dA, &c.dB, &c.q}) JG_TRY(dalloc(s, p, rows));
        c.cap_rows = rows;
        c.cap_nnz = nnz;
    }
    if (!s->part) {
        JG_TRY(dalloc(s, &s->part, (size_t)jg_solver::kSlots * kMaxPartials));
        JG_TRY(dalloc(s, &s->scal, 16));
        JG_TRY(dalloc(s, &s->ctl, 2));
    }
    c.rows = rows;
    c.nnz = nnz;
    return JG_OK;
}

// Validates a host MatrixCsr (32-bit sizes, row pointers from 0 to nnz and
// non-decreasing, columns inside the square matrix) and uploads it to the
// solver's compressed-system arrays, growing them when needed; the CG
// vectors and reduction slots come with it.  Synchronous on return.
static int csr_upload(jg_solver* s, size_t rows, size_t nnz, const double* values, const size_t* row_ptr,
               const size_t* col_idx) {
    if (rows == 0 || !row_ptr || (nnz > 0 && (!values || !col_idx))) return JG_ERR_INVALID_ARG;
    if (rows >= (size_t(1) << 31) || nnz >= (size_t(1) << 31) || row_ptr[0] != 0 ||
        row_ptr[rows] != nnz) {
        s->err = "compressed matrix: row pointers must run from 0 to nnz (< 2^31)";
        return JG_ERR_INVALID_ARG;
    }
    std::vector<int> rp(rows + 1), ci(nnz);
    int max_row = 0;
    for (size_t i = 0; i <= rows; ++i) {
        if (i > 0 && row_ptr[i] < row_ptr[i - 1]) {
            s->err = "compressed matrix: row pointers decrease";
            return JG_ERR_INVALID_ARG;
        }
        rp[i] = (int)row_ptr[i];
        if (i > 0) max_row = std::max(max_row, rp[i] - rp[i - 1]);
    }
    for (size_t k = 0; k < nnz; ++k) {
        if (col_idx[k] >= rows) {
            s->err = "compressed matrix: column index outside the square matrix";
            return JG_ERR_INVALID_ARG;
        }
        ci[k] = (int)col_idx[k];
    }
    JG_HIP(hipSetDevice(s->device));
    JG_TRY(csr_reserve(s, rows, nnz));
    jg_solver::Csr& c = s->csr;
    c.from_grid = false;
    c.max_row = max_row;
    c.ell_valid = false;
    JG_HIP(hipMemcpyAsync(c.rp, rp.data(), (rows + 1) * sizeof(int), hipMemcpyHostToDevice, s->stream));
    if (nnz > 0) {
        JG_HIP(hipMemcpyAsync(c.ci, ci.data(), nnz * sizeof(int), hipMemcpyHostToDevice, s->stream));
        JG_HIP(hipMemcpyAsync(c.val, values, nnz * sizeof(double), hipMemcpyHostToDevice, s->stream));
    }
    return sync(s);  // the staging vectors go out of scope
}

namespace {

// Allocates the hierarchy (levels halving as checked by the caller) for
// nsys systems held back to back (jg_device.h, kSys*).
int levels_alloc(jg_solver* s, size_t nlev, const size_t* nx, const size_t* ny, const size_t* nz,
                 int nsys) {
    JG_HIP(hipSetDevice(s->device));
    JG_HIP(hipStreamSynchronize(s->stream));
    s->release();
    s->nsys = nsys;
    s->twod = nlev > 1 && nz[0] == 1;
    s->lv.resize(nlev);
    const size_t m = (size_t)nsys;
    for (size_t l = 0; l < nlev; ++l) {
        Level& lv = s->lv[l];
        lv.d = Dims{(int)nx[l], (int)ny[l], (int)nz[l]};
        const size_t n = lv.d.n() * m;
        JG_TRY(dalloc(s, &lv.A64, n));
        JG_TRY(dalloc(s, &lv.A32, n));
        JG_TRY(dalloc(s, &lv.t64, n));
        JG_TRY(dalloc(s, &lv.t32, n));
        JG_TRY(dalloc(s, &lv.markers, n));
        JG_TRY(dalloc(s, &lv.y64, n));
        JG_TRY(dalloc(s, &lv.y32, n));
        JG_TRY(dalloc(s, &lv.x64, n));
        JG_TRY(dalloc(s, &lv.x32, n));
        if (l > 0) {
            JG_TRY(dalloc(s, &lv.b64, n));
            JG_TRY(dalloc(s, &lv.b32, n));
        }
    }
    const size_t n0 = s->lv[0].d.n() * m;
    for (double** p : {&s->b, &s->x, &s->r, &s->z, &s->dA, &s->dB, &s->q}) JG_TRY(dalloc(s, p, n0));
    for (float** p : {&s->rhs32, &s->r32, &s->z32, &s->d32A, &s->d32B, &s->q32, &s->e32})
        JG_TRY(dalloc(s, p, n0));
    JG_TRY(dalloc(s, &s->part, (size_t)kSysPart * m));
    JG_TRY(dalloc(s, &s->scal, (size_t)kSysScal * m));
    JG_TRY(dalloc(s, &s->ctl, (size_t)kSysCtl * m));
    return JG_OK;
}

// Makes v a view of member i of group g: g's hierarchy, every
// pointer offset to member i's part of g's arrays, g's stream.
void make_view(jg_solver* g, int i, jg_solver* v) {
    v->view = true;
    v->nsys = 1;
    v->twod = g->twod;
    v->lv = g->lv;
    for (Level& l : v->lv) {
        const idx_t n = l.d.n() * i;
        l.A64 += n;
        l.A32 += n;
        l.t64 += n;
        l.t32 += n;
        l.markers += n;
        l.y64 += n;
        l.y32 += n;
        l.x64 += n;
        l.x32 += n;
        if (l.b64) l.b64 += n;
        if (l.b32) l.b32 += n;
    }
    const idx_t n0 = g->lv[0].d.n() * i;
    v->b = g->b + n0;
    v->x = g->x + n0;
    v->r = g->r + n0;
    v->z = g->z + n0;
    v->dA = g->dA + n0;
    v->dB = g->dB + n0;
    v->q = g->q + n0;
    v->rhs32 = g->rhs32 + n0;
    v->r32 = g->r32 + n0;
    v->z32 = g->z32 + n0;
    v->d32A = g->d32A + n0;
    v->d32B = g->d32B + n0;
    v->q32 = g->q32 + n0;
    v->e32 = g->e32 + n0;
    v->part = g->part + kSysPart * i;
    v->scal = g->scal + kSysScal * i;
    v->ctl = g->ctl + kSysCtl * i;
    if (v->stream) (void)hipStreamDestroy(v->stream);
    v->stream = g->stream;
}

}  // namespace

namespace {

// jg_solver_cg on s's arrays (the grid's, or a box's); ev0 is recorded.
int cg_run(jg_solver* s, unsigned max_iter, double tol, jg_solve_info* info,
           const std::function<int()>& finish) {
    Level& l0 = s->lv[0];
    Ctl h;
    init_ctl(&h, max_iter, tol, 0, 0.0);
    JG_TRY(upload_ctl(s, s->ctl, h));
    k_fill<double><<<nblocks_1d(l0.d.n()), NT, 0, s->stream>>>(s->x, 0.0, l0.d.n());
    JG_TRY(pcg_device<double>(s, Pcg<double>{l0.A64, s->b, s->x, s->r, s->r, s->dA, s->dB, s->q, l0.d,
                                              s->ctl, nullptr},
                              1));
    JG_TRY(finish());
    JG_HIP(hipEventRecord(s->ev1, s->stream));
    JG_TRY(sync(s));
    const Ctl& c = *s->ctl_host;
    const bool nonfinite = c.nonfinite != 0;
    if (info) {
        std::memset(info, 0, sizeof(*info));
        float ms = 0.f;
        JG_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
        info->solve_ms = ms;
        info->iterations = c.iter;
        info->last_residual = std::sqrt(std::fabs(c.sigma));
        // FdmCgSolver3::solve's return (src/jet/fdm_cg_solver3.cpp:45-46)
        info->converged = (info->last_residual <= tol) || (c.iter < max_iter);
        JG_TRY(true_rel_residual(s, &info->rel_residual));
    }
    if (nonfinite) {
        s->err = "non-finite value in CG reduction";
        return JG_ERR_NONFINITE;
    }
    return JG_OK;
}

// jg_solver_mgpcg on s's arrays (the grid's, or a box's); ev0 is recorded.
int mgpcg_run(jg_solver* s, unsigned max_iter, const jg_mg_params* p, const jg_gpu_options& opt,
              double omega, jg_solve_info* info, const std::function<int()>& finish) {
    Level& l0 = s->lv[0];
    const idx_t n = l0.d.n();
    int status = JG_OK;
    unsigned iters = 0, refinements = 0;
    double last_res = 0.0;
    double bnorm = 0.0;  // mixed: ||b||, for the relative residual of the final x
    double mixed_goal = -1.0;  // mixed: the FP64 residual norm the refinement had to reach
    Ctl* ctl = s->ctl;
    if (opt.precision == JG_MIXED) JG_TRY(ensure_f32(s));
    k_fill<double><<<nblocks_1d(n), NT, 0, s->stream>>>(s->x, 0.0, n);
    if (opt.precision != JG_MIXED) {
        MgCfg<double> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter, omega};
        mg.pairs = opt.sweep_pairs;
        mg.jacobi = opt.smoother == JG_SMOOTH_JACOBI;
        Ctl h;
        init_ctl(&h, max_iter, p->max_tol, opt.stop_rule == JG_STOP_RELATIVE ? 1 : 0, opt.rel_tol);
        JG_TRY(upload_ctl(s, ctl, h));
        JG_TRY(pcg_device<double>(s, Pcg<double>{l0.A64, s->b, s->x, s->r, s->z, s->dA, s->dB, s->q,
                                                  l0.d, ctl, &mg},
                                  opt.check_every));
        iters = s->ctl_host->iter;
        last_res = std::sqrt(std::fabs(s->ctl_host->sigma));
        if (s->ctl_host->nonfinite) status = JG_ERR_NONFINITE;
    } else {
        // Iterative refinement: FP64 residual and correction, FP32 MGPCG
        // (FP32 stencil, smoother and V-cycle; FP64 dot accumulation).
        MgCfg<float> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter,
                        (float)omega};
        mg.pairs = opt.sweep_pairs;
        mg.jacobi = opt.smoother == JG_SMOOTH_JACOBI;
        const int nb1 = nblocks_1d(n);
        k_dot<double, double><<<nb1, NT, 0, s->stream>>>(s->b, s->b, n, s->slot(3), nullptr);
        k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(3), nb1, s->scal + 2);
        double bb = 0.0;
        JG_HIP(hipMemcpyAsync(&bb, s->scal + 2, sizeof(double), hipMemcpyDeviceToHost, s->stream));
        JG_TRY(sync(s));
        bnorm = std::sqrt(bb);
        const double goal = opt.stop_rule == JG_STOP_RELATIVE ? opt.rel_tol * bnorm : p->max_tol;
        Ctl* ictl = s->ctl + 1;
        for (unsigned outer = 0;; ++outer) {
            double rr = 0.0;
            if (outer == 0) {
                // x = 0: b - A x is b itself (bit for bit), and its norm is known
                k_convert<double, float><<<nb1, NT, 0, s->stream>>>(s->b, s->rhs32, n);
                rr = bb;
            } else {
                const int nr = residual_dot64<float>(s, l0, s->rhs32, s->slot(3));
                k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(3), nr, s->scal + 3);
                JG_HIP(hipMemcpyAsync(&rr, s->scal + 3, sizeof(double), hipMemcpyDeviceToHost,
                                      s->stream));
                JG_TRY(sync(s));
            }
            last_res = std::sqrt(rr);
            if (!std::isfinite(rr)) {
                status = JG_ERR_NONFINITE;
                break;
            }
            if (last_res <= goal || outer >= opt.max_refine || iters >= max_iter) break;
            Ctl h;
            // The last refinement only needs to close the remaining gap to
            // the goal (with a factor 2 margin for the FP32 inner residual).
            const double inner = std::max(opt.inner_rel_tol, std::min(0.5, 0.5 * goal / last_res));
            init_ctl(&h, max_iter - iters, 0.0, 1, inner);
            JG_TRY(upload_ctl(s, ictl, h));
            k_fill<float><<<nb1, NT, 0, s->stream>>>(s->e32, 0.f, n);
            JG_TRY(pcg_device<float>(s, Pcg<float>{l0.A32, s->rhs32, s->e32, s->r32, s->z32, s->d32A,
                                                   s->d32B, s->q32, l0.d, ictl, &mg},
                                     opt.check_every));
            iters += s->ctl_host->iter;
            if (s->ctl_host->nonfinite) {
                // a value beyond FP32 range (or a NaN) in the inner solve: the
                // correction is meaningless, and x keeps the last finite one
                status = JG_ERR_NONFINITE;
                break;
            }
            k_add_correction<<<nb1, NT, 0, s->stream>>>(s->x, s->e32, n, nullptr);
            JG_TRY(check_launch(s, "refinement"));
            ++refinements;
        }
        mixed_goal = goal;
    }
    JG_TRY(finish());
    JG_HIP(hipEventRecord(s->ev1, s->stream));
    JG_TRY(sync(s));
    if (info) {
        std::memset(info, 0, sizeof(*info));
        float ms = 0.f;
        JG_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
        info->solve_ms = ms;
        info->iterations = iters;
        info->refinements = refinements;
        info->last_residual = last_res;
        // FP64: Jet's rule (cg-inl.h:93 and fdm_mgpcg_solver3.cpp:78). Mixed: the
        // outer loop stops on the true residual, so converged means it reached
        // the goal; running out of refinements or iterations above it is not.
        info->converged = opt.precision == JG_MIXED ? last_res <= mixed_goal
                                                    : (last_res <= p->max_tol) || (iters < max_iter);
        if (status != JG_OK) info->converged = 0;
        if (opt.precision == JG_MIXED && bnorm > 0.0)
            info->rel_residual = last_res / bnorm;  // the FP64 b - A x of the final x
        else
            JG_TRY(true_rel_residual(s, &info->rel_residual));
        if (opt.stop_rule == JG_STOP_RELATIVE && status == JG_OK)
            info->converged = info->rel_residual <= opt.rel_tol;
    }
    if (status == JG_ERR_NONFINITE) s->err = "non-finite value in MGPCG reduction";
    return status;
}

// ------------------------------------------------ solves in a box (jg_box.h)

// Grids above which a solve looks for its box: up to there, the scan's launches
// and its wait (about 40 us) outweigh the cells it could leave out.  Whole
// solves of a pool, time whole / in its box, FP64 and mixed: 64^3 (2^18 cells)
// with 30% fluid 1.30 and 1.11, 60% 0.98 and 1.02, 75% 0.90 and 0.93; 512^2
// 1.04 and 0.99, 1.00 and 0.97, 0.93 and 0.95.
constexpr idx_t kBoxMgCells = idx_t(1) << 18, kBoxCgCells = idx_t(1) << 16;
// A box of more than this share of the grid is not worth its copy.
constexpr double kBoxShare = 0.85;

// The box of the cells that take part in a solve of s's resident system,
// aligned to the coarsest of L levels; share of the grid's cells in *share.
int find_box(jg_solver* s, size_t L, double most, Box* box, double* share) {
    const Level& l0 = s->lv[0];
    const Dims& d = l0.d;
    k_box_reset<<<1, 64, 0, s->stream>>>(s->box_scan);
    const unsigned gx = (d.nx + 63) / 64;
    // at most 128 waves in all up to 2048 columns
    k_box_scan<true><<<dim3(gx, std::max(1u, 32u / gx), 1), 64 * kBoxY, 0, s->stream>>>(
        l0.A64, s->b, d, most, s->box_scan);
    const dim3 grid(gx, (d.ny + kBoxY - 1) / kBoxY, (d.nz + kBoxZ - 1) / kBoxZ);
    k_box_scan<false><<<grid, 64 * kBoxY, 0, s->stream>>>(l0.A64, s->b, d, most, s->box_scan);
    JG_TRY(check_launch(s, "box scan"));
    JG_HIP(hipMemcpyAsync(s->box_host, s->box_scan, sizeof(BoxScan), hipMemcpyDeviceToHost, s->stream));
    JG_TRY(sync(s));
    const BoxScan r = *s->box_host;
    const int dims[3] = {d.nx, d.ny, d.nz};
    int n[3];
    for (int a = 0; a < 3; ++a) {
        const int g = a == 2 && s->twod ? 1 : 1 << (L - 1);
        const int lo = std::max(0, std::min(r.lo[a], dims[a])), hi = std::max(0, std::min(r.hi[a] + 1, dims[a]));
        box->o[a] = lo / g * g;
        n[a] = std::max(0, (hi + g - 1) / g * g - box->o[a]);
    }
    box->n = Dims{n[0], n[1], n[2]};
    *share = (double)box->n.n() / (double)d.n();
    return JG_OK;
}

// The arrays of box solves: rows of every level, b and x, for boxes of up to
// kBoxShare of the grid; one allocation, so that there is all or nothing, kept
// until the hierarchy changes.  false: no room.
bool box_reserve(jg_solver* s, size_t L) {
    if (s->box_cells > 0 || s->box_failed) return !s->box_failed;
    auto room = [&](size_t l) { return ((size_t)(kBoxShare * (double)s->lv[l].d.n()) / 32 + 1) * 32; };
    size_t cells = 0;
    for (size_t l = 0; l < L; ++l) cells += room(l);
    double* all = nullptr;
    if (!dalloc_spare(s, &all, 4 * cells + 2 * room(0))) {
        s->box_failed = true;
        return false;
    }
    s->box_rows = (Row<double>*)all;
    s->box_b = all + 4 * cells;
    s->box_x = s->box_b + room(0);
    s->box_cells = cells;
    return true;
}

// Runs a solve (run(solver, finish), finish called when the solution is
// there and before the closing event) on s, or on a solver whose dense
// arrays hold the box of s that takes part.  That solver is a view: its
// work vectors and control blocks are s's own, which are larger; A32 too, so
// s's FP32 copy has to be made anew afterwards.
template <typename Run>
int solve_in_box(jg_solver* s, size_t L, idx_t above, double most, bool mixed, Run&& run) {
    auto whole = [&]() { return run(s, [] { return (int)JG_OK; }); };
    Level& l0 = s->lv[0];
    if (l0.d.n() <= above || s->nsys > 1) return whole();
    if (!s->box_scan && !dalloc_spare(s, &s->box_scan, 2)) return whole();
    Box box;
    double share = 1.0;
    JG_TRY(find_box(s, L, most, &box, &share));
    if (share == 0.0 || share > kBoxShare || !box_reserve(s, s->lv.size())) return whole();
    int* const odd = (int*)(s->box_scan + 1);
    k_fill<int><<<1, NT, 0, s->stream>>>(odd, 0, 1);
    jg_solver v;
    v.device = s->device;
    v.cus = s->cus;
    v.cg_grid_ok = s->cg_grid_ok;
    v.cg_polls = s->cg_polls;
    v.view = true;
    v.stream = s->stream;
    v.ev0 = s->ev0;
    v.ev1 = s->ev1;
    v.evp[0] = s->evp[0];
    v.evp[1] = s->evp[1];
    v.ctl_host = s->ctl_host;
    v.twod = s->twod;
    v.r = s->r;
    v.z = s->z;
    v.dA = s->dA;
    v.dB = s->dB;
    v.q = s->q;
    v.rhs32 = s->rhs32;
    v.r32 = s->r32;
    v.z32 = s->z32;
    v.d32A = s->d32A;
    v.d32B = s->d32B;
    v.q32 = s->q32;
    v.e32 = s->e32;
    v.part = s->part;
    v.scal = s->scal;
    v.ctl = s->ctl;
    v.cg_slots = s->cg_slots;
    v.b = s->box_b;
    v.x = s->box_x;
    v.lv.assign(s->lv.begin(), s->lv.begin() + L);
    Row<double>* rows = s->box_rows;
    for (size_t l = 0; l < L; ++l) {
        Level& lv = v.lv[l];
        const Dims full = lv.d;
        Box bl = box;
        for (int a = 0; a < 3; ++a) bl.o[a] >>= (a == 2 && s->twod) ? 0 : l;
        bl.n = Dims{box.n.nx >> l, box.n.ny >> l, s->twod ? 1 : box.n.nz >> l, true};
        lv.d = bl.n;
        const Geo g = geo_planes(l == 0 ? bl.n : full);
        Row<double>* const to64 = !mixed || l == 0 ? rows : nullptr;
        Row<float>* const to32 = mixed ? lv.A32 : nullptr;
        if (l == 0)
            k_box_rows<false><<<g.grid, g.block, 0, s->stream>>>(lv.A64, full, bl, most, to64, to32, odd);
        else
            k_box_rows<true><<<g.grid, g.block, 0, s->stream>>>(lv.A64, full, bl, most, to64, to32, odd);
        lv.A64 = rows;
        rows += bl.n.n();
    }
    const Geo gb = geo_planes(box.n), gf = geo_planes(l0.d);
    k_box_gather<<<gb.grid, gb.block, 0, s->stream>>>(s->b, l0.d, box, v.b);
    v.f32_valid = mixed;
    if (mixed) s->f32_valid = false;
    int bad = 0;
    int st = check_launch(s, "box");
    if (st == JG_OK)
        st = run(&v, [&]() -> int {
            k_box_scatter<<<gf.grid, gf.block, 0, s->stream>>>(v.x, l0.d, box, s->x);
            JG_HIP(hipMemcpyAsync(&s->box_host->lo[0], odd, sizeof(int), hipMemcpyDeviceToHost, s->stream));
            return check_launch(s, "box scatter");
        });
    // the solver's own parts stay with s
    bad = s->box_host->lo[0];
    s->cg_slots = v.cg_slots;
    s->cg_grid_ok = v.cg_grid_ok;
    s->allocs.insert(s->allocs.end(), v.allocs.begin(), v.allocs.end());
    v.allocs.clear();
    if (!v.err.empty()) s->err = v.err;
    v.ctl_host = nullptr;
    v.ev0 = v.ev1 = v.evp[0] = v.evp[1] = nullptr;
    if ((st == JG_OK || st == JG_ERR_NONFINITE) && bad) return whole();
    return st;
}

}  // namespace

extern "C" {

void jg_mg_params_default(jg_mg_params* p) {
    // MgParameters defaults (include/jet/mg.h:58-86) and FdmMgSolver3's
    // sorFactor / ordering defaults (include/jet/fdm_mg_solver3.h:24-30).
    p->max_levels = 1;
    p->restrict_iter = 5;
    p->correct_iter = 5;
    p->coarsest_iter = 20;
    p->final_iter = 20;
    p->max_tol = 1e-9;
    p->sor = 1.5;
    p->red_black = 0;
}

void jg_gpu_options_default(jg_gpu_options* o) {
    std::memset(o, 0, sizeof(*o));
    o->precision = JG_FP64;
    o->stop_rule = JG_STOP_JET;
    o->rel_tol = 1e-8;
    o->smoother = JG_SMOOTH_RBGS;
    o->omega = 0.0;
    o->max_refine = 8;
    o->inner_rel_tol = 1e-4;
    o->check_every = 1;
}

int jg_solver_create(int device, jg_solver** out) {
    if (!out) return JG_ERR_INVALID_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= device || device < 0)
        return JG_ERR_NO_DEVICE;
    jg_solver* s = new jg_solver();
    s->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&s->stream) != hipSuccess ||
        hipEventCreate(&s->ev0) != hipSuccess || hipEventCreate(&s->ev1) != hipSuccess ||
        hipEventCreateWithFlags(&s->evp[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s->evp[1], hipEventDisableTiming) != hipSuccess ||
        hipHostMalloc((void**)&s->ctl_host, 2 * sizeof(Ctl), hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void**)&s->box_host, sizeof(BoxScan), hipHostMallocDefault) != hipSuccess) {
        delete s;
        return JG_ERR_HIP;
    }
    if (hipDeviceGetAttribute(&s->cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
        delete s;
        return JG_ERR_HIP;
    }
    // this device's address of the no-allocation scratch array (a failure is
    // reported by jg_relax_red_black_noalloc, the only user)
    (void)scratch_init(device);
    *out = s;
    return JG_OK;
}

void jg_solver_destroy(jg_solver* s) {
    if (!s) return;
    (void)hipSetDevice(s->device);
    (void)hipStreamSynchronize(s->stream);
    delete s;
}

const char* jg_last_error(const jg_solver* s) { return s ? s->err.c_str() : "null solver"; }

void* jg_solver_stream(jg_solver* s) { return s ? (void*)s->stream : nullptr; }

int jg_solver_set_levels(jg_solver* s, size_t nlev, const size_t* nx, const size_t* ny,
                         const size_t* nz) {
    if (!s || nlev == 0 || nlev > 16 || !nx || !ny || !nz) return JG_ERR_INVALID_ARG;
    for (size_t l = 0; l < nlev; ++l) {
        if (!valid_dims(nx[l], ny[l], nz[l])) {
            s->err = "invalid level size";
            return JG_ERR_INVALID_ARG;
        }
        // a finest level one plane thick with coarser levels is a 2-D
        // hierarchy (a 3-D one cannot halve an odd nz): every level one plane
        const bool twod = nlev > 1 && nz[0] == 1;
        if (l > 0 && (nx[l - 1] != 2 * nx[l] || ny[l - 1] != 2 * ny[l] ||
                      (twod ? nz[l] != 1 : nz[l - 1] != 2 * nz[l]))) {
            s->err = "level sizes must halve exactly (in x and y only for one-plane levels)";
            return JG_ERR_INVALID_ARG;
        }
        // one reduction partial per stencil tile of a plane at least
        const Geo g = geo_stencil(Dims{(int)nx[l], (int)ny[l], (int)nz[l]});
        if ((long)g.grid.x * g.grid.y * g.grid.z > kMaxPartials) {
            s->err = "level plane too large for the reduction partials (more than 65536 tiles of 64 x 4 cells)";
            return JG_ERR_UNSUPPORTED;
        }
    }
    bool same = s->lv.size() == nlev;
    for (size_t l = 0; same && l < nlev; ++l)
        same = s->lv[l].d.nx == (int)nx[l] && s->lv[l].d.ny == (int)ny[l] && s->lv[l].d.nz == (int)nz[l];
    if (same) return JG_OK;
    if (s->view) {
        s->err = "a batch member keeps the hierarchy its batch was created with";
        return JG_ERR_INVALID_ARG;
    }
    return levels_alloc(s, nlev, nx, ny, nz, 1);
}

double* jg_solver_matrix(jg_solver* s, size_t level) {
    if (!s || level >= s->lv.size()) return nullptr;
    return (double*)s->lv[level].A64;
}

double* jg_solver_rhs(jg_solver* s) { return s ? s->b : nullptr; }

double* jg_solver_solution(jg_solver* s) { return s ? s->x : nullptr; }

int jg_solver_upload(jg_solver* s, size_t level, const double* rows, const double* b) {
    if (!s || level >= s->lv.size() || !rows) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    const size_t n = s->lv[level].d.n();
    JG_HIP(hipMemcpyAsync(s->lv[level].A64, rows, n * sizeof(Row<double>), hipMemcpyHostToDevice,
                          s->stream));
    if (b && level == 0)
        JG_HIP(hipMemcpyAsync(s->b, b, n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    s->f32_valid = false;
    return sync(s);
}

int jg_solver_download_x(jg_solver* s, double* x) {
    if (!s || s->lv.empty() || !x) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    JG_HIP(hipMemcpyAsync(x, s->x, s->lv[0].d.n() * sizeof(double), hipMemcpyDeviceToHost,
                          s->stream));
    return sync(s);
}

int jg_solver_matrices_changed(jg_solver* s) {
    if (!s) return JG_ERR_INVALID_ARG;
    s->f32_valid = false;
    return JG_OK;
}

int jg_solver_cg(jg_solver* s, unsigned max_iter, double tol, jg_solve_info* info) {
    if (!s || s->lv.empty()) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    JG_HIP(hipEventRecord(s->ev0, s->stream));
    return solve_in_box(s, 1, kBoxCgCells, DBL_MAX, false,
                        [&](jg_solver* v, const std::function<int()>& finish) {
                            return cg_run(v, max_iter, tol, info, finish);
                        });
}

int jg_solver_cg_polls(jg_solver* s, unsigned polls) {
    if (!s) return JG_ERR_INVALID_ARG;
    s->cg_polls = (int)std::min(polls, 1u << 30);
    return JG_OK;
}

int jg_mg_vcycle(jg_solver* s, const jg_mg_params* p, const jg_gpu_options* o, const double* r,
                 double* z) {
    if (!s || s->lv.empty() || !p || !r || !z || r == z) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    jg_gpu_options opt;
    double omega = 0.0;
    JG_TRY(mg_options(s, p, o, &opt, &omega));
    const idx_t n = s->lv[0].d.n();
    const int nb1 = nblocks_1d(n);
    int nb = 0;
    if (opt.precision == JG_MIXED) {
        JG_TRY(ensure_f32(s));
        MgCfg<float> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter,
                        (float)omega};
        mg.pairs = opt.sweep_pairs;
        mg.jacobi = opt.smoother == JG_SMOOTH_JACOBI;
        k_convert<double, float><<<nb1, NT, 0, s->stream>>>(r, s->r32, n);
        JG_TRY(vcycle<float>(s, s->r32, s->z32, mg, nullptr, &nb));
        k_convert<float, double><<<nb1, NT, 0, s->stream>>>(s->z32, z, n);
    } else {
        MgCfg<double> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter, omega};
        mg.pairs = opt.sweep_pairs;
        mg.jacobi = opt.smoother == JG_SMOOTH_JACOBI;
        JG_TRY(vcycle<double>(s, r, z, mg, nullptr, &nb));
    }
    JG_TRY(check_launch(s, "vcycle"));
    return sync(s);
}

// FdmMgSolver3::solve(FdmMgLinearSystem3*) (src/jet/fdm_mg_solver3.cpp:69-74):
// one V-cycle from the resident x.  For the linear V-cycle this is
// x += M (b - A x) with M the zero-start cycle of jg_mg_vcycle; Jet's result
// is lastResidualNorm < maxTolerance, the norm of b - A x afterwards
// (include/jet/detail/mg-inl.h:62-66).
int jg_solver_mg(jg_solver* s, const jg_mg_params* p, const jg_gpu_options* o, jg_solve_info* info) {
    if (!s || s->lv.empty() || !p) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Level& l0 = s->lv[0];
    const idx_t n = l0.d.n();
    const int nb1 = nblocks_1d(n);
    JG_HIP(hipEventRecord(s->ev0, s->stream));
    launch_residual<double, double, false, false>(s, l0.A64, s->x, s->b, s->r, l0.d, nullptr,
                                                         nullptr);
    JG_TRY(check_launch(s, "mg residual"));
    JG_TRY(jg_mg_vcycle(s, p, o, s->r, s->z));
    k_axpy<double><<<nb1, NT, 0, s->stream>>>(1.0, s->z, s->x, s->x, n);
    const int nr = launch_residual<double, double, true, false>(s, l0.A64, s->x, s->b, s->r,
                                                                       l0.d, s->slot(0), nullptr);
    k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(0), nr, s->scal + 0);
    k_dot<double, double><<<nb1, NT, 0, s->stream>>>(s->b, s->b, n, s->slot(1), nullptr);
    k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(1), nb1, s->scal + 1);
    JG_HIP(hipEventRecord(s->ev1, s->stream));
    JG_TRY(check_launch(s, "mg solve"));
    double h[2];
    JG_HIP(hipMemcpyAsync(h, s->scal, sizeof(h), hipMemcpyDeviceToHost, s->stream));
    JG_TRY(sync(s));
    if (!std::isfinite(h[0])) {
        s->err = "non-finite value in the V-cycle";
        if (info) info->converged = 0;
        return JG_ERR_NONFINITE;
    }
    if (info) {
        std::memset(info, 0, sizeof(*info));
        float ms = 0.f;
        JG_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
        info->solve_ms = ms;
        info->iterations = 1;
        info->last_residual = std::sqrt(h[0]);
        info->rel_residual = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
        info->converged = info->last_residual < p->max_tol;
    }
    return JG_OK;
}

int jg_solver_mgpcg(jg_solver* s, unsigned max_iter, const jg_mg_params* p,
                    const jg_gpu_options* o, jg_solve_info* info) {
    if (!s || s->lv.empty() || !p) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    jg_gpu_options opt;
    double omega = 0.0;
    JG_TRY(mg_options(s, p, o, &opt, &omega));
    const bool mixed = opt.precision == JG_MIXED;
    JG_HIP(hipEventRecord(s->ev0, s->stream));
    return solve_in_box(s, s->lv.size(), kBoxMgCells, mixed ? FLT_MAX : DBL_MAX, mixed,
                        [&](jg_solver* v, const std::function<int()>& finish) {
                            return mgpcg_run(v, max_iter, p, opt, omega, info, finish);
                        });
}

int jg_cg_solve_host(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                     const double* b, double* x, unsigned max_iter, double tol,
                     jg_solve_info* info) {
    if (!s || !rows || !b || !x) return JG_ERR_INVALID_ARG;
    size_t sx[1] = {nx}, sy[1] = {ny}, sz[1] = {nz};
    JG_TRY(jg_solver_set_levels(s, 1, sx, sy, sz));
    JG_TRY(jg_solver_upload(s, 0, rows, b));
    JG_TRY(jg_solver_cg(s, max_iter, tol, info));
    return jg_solver_download_x(s, x);
}

int jg_csr_cg_solve_host(jg_solver* s, size_t rows, size_t nnz, const double* values,
                         const size_t* row_ptr, const size_t* col_idx, const double* b, double* x,
                         unsigned max_iter, double tol, jg_solve_info* info) {
    if (!s || !b || !x) return JG_ERR_INVALID_ARG;
    JG_TRY(csr_upload(s, rows, nnz, values, row_ptr, col_idx));
    jg_solver::Csr& c = s->csr;
    JG_HIP(hipMemcpyAsync(c.b, b, rows * sizeof(double), hipMemcpyHostToDevice, s->stream));
    const int st = csr_solve(s, max_iter, tol, info);
    if (st != JG_OK && st != JG_ERR_NONFINITE) return st;
    JG_HIP(hipMemcpyAsync(x, c.x, rows * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    JG_TRY(sync(s));
    return st;
}

int jg_solver_csr_cg(jg_solver* s, unsigned max_iter, double tol, jg_solve_info* info) {
    if (!s || s->csr.rows == 0 || !s->csr.rp) {
        if (s) s->err = "jg_solver_csr_cg before a compressed system was built or uploaded";
        return JG_ERR_INVALID_ARG;
    }
    JG_HIP(hipSetDevice(s->device));
    return csr_solve(s, max_iter, tol, info);
}

int jg_csr_mvm_host(jg_solver* s, size_t rows, size_t nnz, const double* values,
                    const size_t* row_ptr, const size_t* col_idx, const double* v, double* result) {
    if (!s || !v || !result) return JG_ERR_INVALID_ARG;
    JG_TRY(csr_upload(s, rows, nnz, values, row_ptr, col_idx));
    jg_solver::Csr& c = s->csr;
    JG_HIP(hipMemcpyAsync(c.x, v, rows * sizeof(double), hipMemcpyHostToDevice, s->stream));
    k_csr_mvm<<<nblocks_1d((idx_t)rows), NT, 0, s->stream>>>(CsrDev{c.rp, c.ci, c.val, (int)c.nnz}, c.x, c.q,
                                                             (idx_t)rows);
    JG_TRY(check_launch(s, "csr mvm"));
    JG_HIP(hipMemcpyAsync(result, c.q, rows * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    return sync(s);
}

int jg_csr_residual_host(jg_solver* s, size_t rows, size_t nnz, const double* values,
                         const size_t* row_ptr, const size_t* col_idx, const double* x,
                         const double* b, double* result) {
    if (!s || !x || !b || !result) return JG_ERR_INVALID_ARG;
    JG_TRY(csr_upload(s, rows, nnz, values, row_ptr, col_idx));
    jg_solver::Csr& c = s->csr;
    JG_HIP(hipMemcpyAsync(c.x, x, rows * sizeof(double), hipMemcpyHostToDevice, s->stream));
    JG_HIP(hipMemcpyAsync(c.b, b, rows * sizeof(double), hipMemcpyHostToDevice, s->stream));
    k_csr_residual<false, false><<<nblocks_1d((idx_t)rows), NT, 0, s->stream>>>(
        CsrDev{c.rp, c.ci, c.val, (int)c.nnz}, c.x, c.b, c.r, (idx_t)rows, nullptr, nullptr);
    JG_TRY(check_launch(s, "csr residual"));
    JG_HIP(hipMemcpyAsync(result, c.r, rows * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    return sync(s);
}

int jg_mgpcg_solve_host(jg_solver* s, size_t nlev, const size_t* nx, const size_t* ny,
                        const size_t* nz, const double* const* rows, const double* b, double* x,
                        unsigned max_iter, const jg_mg_params* p, const jg_gpu_options* o,
                        jg_solve_info* info) {
    if (!s || !rows || !b || !x || !p) return JG_ERR_INVALID_ARG;
    JG_TRY(jg_solver_set_levels(s, nlev, nx, ny, nz));
    for (size_t l = 0; l < nlev; ++l) JG_TRY(jg_solver_upload(s, l, rows[l], l == 0 ? b : nullptr));
    JG_TRY(jg_solver_mgpcg(s, max_iter, p, o, info));
    return jg_solver_download_x(s, x);
}

int jg_mg_solve_host(jg_solver* s, size_t nlev, const size_t* nx, const size_t* ny, const size_t* nz,
                     const double* const* rows, const double* b, double* x, const jg_mg_params* p,
                     const jg_gpu_options* o, jg_solve_info* info) {
    if (!s || !rows || !b || !x || !p) return JG_ERR_INVALID_ARG;
    JG_TRY(jg_solver_set_levels(s, nlev, nx, ny, nz));
    for (size_t l = 0; l < nlev; ++l) JG_TRY(jg_solver_upload(s, l, rows[l], l == 0 ? b : nullptr));
    // the V-cycle starts from the caller's x, as Jet's does
    JG_HIP(hipMemcpyAsync(s->x, x, s->lv[0].d.n() * sizeof(double), hipMemcpyHostToDevice, s->stream));
    JG_TRY(jg_solver_mg(s, p, o, info));
    return jg_solver_download_x(s, x);
}

int jg_solver_coarsen(jg_solver* s) {
    if (!s || s->lv.empty()) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    for (size_t l = 1; l < s->lv.size(); ++l) {
        const Dims cd = s->lv[l].d;
        const Geo g = geo_planes(cd);
        if (s->twod)
            k_mg_coarsen<1><<<g.grid, g.block, 0, s->stream>>>(s->lv[l - 1].A64, s->lv[l].A64, cd);
        else
            k_mg_coarsen<2><<<g.grid, g.block, 0, s->stream>>>(s->lv[l - 1].A64, s->lv[l].A64, cd);
    }
    JG_TRY(check_launch(s, "mg_coarsen"));
    s->f32_valid = false;
    return sync(s);
}

int jg_mgpcg_flat_solve_host(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                             const double* b, double* x, unsigned max_iter, const jg_mg_params* p,
                             const jg_gpu_options* o, jg_solve_info* info) {
    if (!s || !rows || !b || !x || !p) return JG_ERR_INVALID_ARG;
    // FdmMgUtils3::resizeArrayWithFinest (include/jet/detail/fdm_mg_linear_system3-inl.h:
    // 35-50): halve while every extent is even, up to max_levels; one-plane
    // systems halve in x and y (FdmMgUtils2's rule)
    size_t lx[16] = {nx}, ly[16] = {ny}, lz[16] = {nz};
    const bool plane = nz == 1;
    const size_t cap = std::min<size_t>(std::max<size_t>(p->max_levels, 1), 16);
    size_t nlev = 1;
    while (nlev < cap && lx[nlev - 1] % 2 == 0 && ly[nlev - 1] % 2 == 0 &&
           (plane || lz[nlev - 1] % 2 == 0)) {
        lx[nlev] = lx[nlev - 1] / 2;
        ly[nlev] = ly[nlev - 1] / 2;
        lz[nlev] = plane ? 1 : lz[nlev - 1] / 2;
        ++nlev;
    }
    JG_TRY(jg_solver_set_levels(s, nlev, lx, ly, lz));
    JG_TRY(jg_solver_upload(s, 0, rows, b));
    JG_TRY(jg_solver_coarsen(s));
    JG_TRY(jg_solver_mgpcg(s, max_iter, p, o, info));
    return jg_solver_download_x(s, x);
}

}  // extern "C"

// ------------------------------------------------------ kernel timing

namespace {

template <typename T>
struct Vecs {
    T *x, *b, *r, *z, *dA, *dB, *q;
};

Vecs<double> vecs64(jg_solver* s) { return {s->x, s->b, s->r, s->z, s->dA, s->dB, s->q}; }
Vecs<float> vecs32(jg_solver* s) { return {s->e32, s->rhs32, s->r32, s->z32, s->d32A, s->d32B, s->q32}; }

// The first level-0 launch of the pre-smoothing (post = false) or of the
// post-smoothing (post = true) of a V(2,2) cycle, exactly as vcycle() issues
// it: the sweep plan of the solve, b = r, the result in z (pre:
// x starts at zero and, for a two-sweep launch, the residual is written for
// the restriction; post: the coarse correction of level 1 is added as x is
// loaded).
template <typename T>
int level0_plan(jg_solver* s) {
    return sweep_plan<T>(s, s->lv[0].d, 2, 0).front();
}

template <typename T>
void level0_launch(jg_solver* s, const Vecs<T>& v, bool post, T omega) {
    Level& l0 = s->lv[0];
    const Row<T>* A = Prec<T>::A(l0);
    const int mode = level0_plan<T>(s);
    const T* xin = post ? Prec<T>::y(l0) : nullptr;
    const T* coarse = post && s->lv.size() > 1 ? Prec<T>::x(s->lv[1]) : nullptr;
    if (mode == kLaunchBrick)
        launch_brick2<T>(s, A, v.r, xin, v.z, l0.d, post ? 1 : 0, coarse, omega, s->ctl);
    else if (mode == kLaunchMarch)
        launch_sweep2<T>(s, A, v.r, xin, v.z, l0.d, post ? 1 : 0, coarse,
                         post ? nullptr : Prec<T>::t(l0), omega, s->ctl);
    else
        launch_sweep<T>(s, A, v.r, xin, v.z, l0.d, post ? 1 : 0, coarse, nullptr, nullptr, omega,
                        s->ctl);
}

// Algorithmic bytes per cell of that launch under the 4-coefficient model:
// a sweep reads A, b and x and writes x; the residual written by a pre-
// smoothing two-sweep launch reads A, x and b (4 coefficients, 2 vectors)
// and writes r; the prolongation-correction reads the coarse vector (1/8)
// and reads and writes x.
template <typename T>
double level0_launch_bytes(jg_solver* s, bool post) {
    const double sa = sizeof(Row<T>), sv = sizeof(T);
    const int mode = level0_plan<T>(s);
    const double sweeps = mode == kLaunchSingle ? 1.0 : 2.0;
    double b = sweeps * (sa + 3 * sv);
    if (post && s->lv.size() > 1) b += 2 * sv + sv / 8;
    if (!post && mode == kLaunchMarch) b += sa + 3 * sv;
    return b;
}

template <typename T>
int time_kernel_t(jg_solver* s, const Vecs<T>& v, int kernel, unsigned reps, double* avg_ms,
                  double* bytes) {
    Level& l0 = s->lv[0];
    const Dims d = l0.d;
    const idx_t n = d.n();
    const int nb1 = nblocks_1d(n);
    Geo g = geo_stencil(d);
    const Row<T>* A = Prec<T>::A(l0);
    Ctl h;
    init_ctl(&h, 1u << 30, 0.0, 0, 0.0);
    h.alpha = 1e-3;
    h.beta = 0.5;
    h.sigma = 1.0;
    JG_TRY(upload_ctl(s, s->ctl, h));
    // the kernels that read a right-hand side take level 0's y, a V-cycle
    // scratch vector, so the system's b survives the measurement
    T* const bt = Prec<T>::y(l0);
    for (T* p : {v.x, bt, v.r, v.z, v.dA, v.dB, v.q})
        k_fill<T><<<nb1, NT, 0, s->stream>>>(p, T(1), n);
    const double sa = sizeof(Row<T>), sv = sizeof(T);
    auto launch = [&]() {
        switch (kernel) {
            case JG_KERNEL_RBGS:
                k_rbgs<T, T, false><<<g.grid, g.block, 0, s->stream>>>(A, bt, v.x, d, g.zc, 1, T(1),
                                                                       s->ctl);
                break;
            case JG_KERNEL_DIR_SPMV:
                launch_dir_spmv<T>(s, A, v.z, v.dA, v.dB, v.q, d, s->slot(2), s->ctl);
                break;
            case JG_KERNEL_RESIDUAL:
                launch_residual<T, T, false, false>(s, A, v.x, bt, v.r, d, nullptr, nullptr);
                break;
            case JG_KERNEL_UPDATE_XR:
                k_update_xr<T, false><<<nb1, NT, 0, s->stream>>>(v.x, v.r, v.dA, v.q, n, nullptr, s->ctl);
                break;
            case JG_KERNEL_DOT:
                k_dot<T, T><<<nb1, NT, 0, s->stream>>>(v.r, v.z, n, s->slot(0), s->ctl);
                break;
            case JG_KERNEL_SWEEP:
                launch_sweep<T>(s, A, bt, v.r, v.x, d, 1, nullptr, nullptr, nullptr, T(1), s->ctl);
                break;
            case JG_KERNEL_SWEEP2:
                launch_sweep2<T>(s, A, bt, v.r, v.x, d, 1, nullptr, nullptr, T(1), s->ctl);
                break;
            case JG_KERNEL_PRE0:
            case JG_KERNEL_POST0:
                level0_launch<T>(s, v, kernel == JG_KERNEL_POST0, T(1.3));
                break;
            default:
                k_convert<T, T><<<nb1, NT, 0, s->stream>>>(v.r, v.q, n);
                break;
        }
    };
    // Compulsory bytes per launch under Jet's 4-coefficient data model.
    double per_cell;
    switch (kernel) {
        case JG_KERNEL_RBGS: per_cell = sa + 2 * sv; break;      // A (own + neighbour couplings), x, b/2, x/2 written
        case JG_KERNEL_DIR_SPMV: per_cell = sa + 4 * sv; break;  // A, z, d_old -> d_new, q
        case JG_KERNEL_RESIDUAL: per_cell = sa + 3 * sv; break;  // A, x, b -> r
        case JG_KERNEL_UPDATE_XR: per_cell = 6 * sv; break;      // x, d, r, q -> x, r
        case JG_KERNEL_DOT: per_cell = 2 * sv; break;
        case JG_KERNEL_SWEEP: per_cell = sa + 3 * sv; break;     // A, b, x -> x (both colours)
        case JG_KERNEL_SWEEP2: per_cell = 2 * (sa + 3 * sv); break;  // two sweeps, each as above
        case JG_KERNEL_PRE0:
        case JG_KERNEL_POST0: per_cell = level0_launch_bytes<T>(s, kernel == JG_KERNEL_POST0); break;
        default: per_cell = 2 * sv; break;
    }
    launch();  // warm
    JG_TRY(check_launch(s, "time_kernel"));
    JG_HIP(hipEventRecord(s->ev0, s->stream));
    for (unsigned i = 0; i < reps; ++i) launch();
    JG_HIP(hipEventRecord(s->ev1, s->stream));
    JG_TRY(sync(s));
    float ms = 0.f;
    JG_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
    *avg_ms = (double)ms / reps;
    *bytes = per_cell * (double)n;
    return JG_OK;
}

}  // namespace

extern "C" int jg_solver_time_kernel(jg_solver* s, int kernel, int precision, unsigned reps,
                                     double* avg_ms, double* bytes) {
    if (!s || s->lv.empty() || !avg_ms || !bytes || reps == 0 || kernel < 0 ||
        kernel > JG_KERNEL_POST0)
        return JG_ERR_INVALID_ARG;
    if (kernel == JG_KERNEL_SWEEP2 && precision != JG_MIXED) {
        s->err = "the two-sweep kernel is FP32 only";
        return JG_ERR_UNSUPPORTED;
    }
    JG_HIP(hipSetDevice(s->device));
    if (precision == JG_MIXED) {
        JG_TRY(ensure_f32(s));
        return time_kernel_t<float>(s, vecs32(s), kernel, reps, avg_ms, bytes);
    }
    return time_kernel_t<double>(s, vecs64(s), kernel, reps, avg_ms, bytes);
}

extern "C" {

// --------------------------------------------------------- BLAS entries

int jg_blas_mvm(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                const double* x, double* y) {
    if (!s || !valid_dims(nx, ny, nz) || !rows || !x || !y) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims d{(int)nx, (int)ny, (int)nz};
    Geo g = geo_stencil(d);
    k_spmv<double, double, false><<<g.grid, g.block, 0, s->stream>>>(
        (const Row<double>*)rows, x, y, d, g.zc, nullptr, nullptr);
    JG_TRY(check_launch(s, "mvm"));
    return sync(s);
}

int jg_blas_residual(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                     const double* x, const double* b, double* r) {
    if (!s || !valid_dims(nx, ny, nz) || !rows || !x || !b || !r) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims d{(int)nx, (int)ny, (int)nz};
    launch_residual<double, double, false, false>(s, (const Row<double>*)rows, x, b, r, d,
                                                         nullptr, nullptr);
    JG_TRY(check_launch(s, "residual"));
    return sync(s);
}

int jg_blas_dot(jg_solver* s, size_t n, const double* a, const double* b, double* result) {
    if (!s || !a || !b || !result) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    if (!s->part) {
        JG_TRY(dalloc(s, &s->part, (size_t)jg_solver::kSlots * kMaxPartials));
        JG_TRY(dalloc(s, &s->scal, 16));
    }
    const int nb = nblocks_1d((idx_t)n);
    k_dot<double, double><<<nb, NT, 0, s->stream>>>(a, b, (idx_t)n, s->slot(0), nullptr);
    k_fin_sum<<<1, kFinThreads, 0, s->stream>>>(s->slot(0), nb, s->scal + 4);
    JG_TRY(check_launch(s, "dot"));
    JG_HIP(hipMemcpyAsync(result, s->scal + 4, sizeof(double), hipMemcpyDeviceToHost, s->stream));
    return sync(s);
}

int jg_blas_axpy(jg_solver* s, size_t n, double a, const double* x, const double* y, double* out) {
    if (!s || !x || !y || !out) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    k_axpy<double><<<nblocks_1d((idx_t)n), NT, 0, s->stream>>>(a, x, y, out, (idx_t)n);
    JG_TRY(check_launch(s, "axpy"));
    return sync(s);
}

int jg_relax_red_black(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                       const double* b, double sor, double* x) {
    if (!s || !valid_dims(nx, ny, nz) || !rows || !b || !x) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims d{(int)nx, (int)ny, (int)nz};
    // One fused forward sweep (red then black) reading a copy of x (the sweep
    // is out of place because its tiles overlap), in a buffer that the solver
    // keeps and grows; its allocation per call cost a third of a 2M-cell
    // sweep's time.
    const size_t n = (size_t)d.n();
    if (n > s->relax_cap) {
        double* grown = nullptr;
        JG_HIP(hipMalloc(&grown, n * sizeof(double)));
        (void)hipFree(s->relax_tmp);  // (no call is in flight: each ends synchronised)
        s->relax_tmp = grown;
        s->relax_cap = n;
    }
    k_convert<double, double><<<nblocks_1d((idx_t)n), NT, 0, s->stream>>>(x, s->relax_tmp, (idx_t)n);
    launch_sweep<double>(s, (const Row<double>*)rows, b, s->relax_tmp, x, d, 0, nullptr, nullptr, nullptr,
                         sor, nullptr);
    JG_TRY(check_launch(s, "relax_red_black"));
    return sync(s);
}

int jg_relax_red_black_noalloc(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                               const double* b, double sor, double* x) {
    if (!s || !valid_dims(nx, ny, nz) || !rows || !b || !x) return JG_ERR_INVALID_ARG;
    const size_t n = nx * ny * nz;
    if (n > kNoAllocMaxCells) {
        s->err = "relax_red_black_noalloc: " + std::to_string(n) + " cells exceed the " +
                 std::to_string(kNoAllocMaxCells) + "-cell scratch array";
        return JG_ERR_INVALID_ARG;
    }
    JG_HIP(hipSetDevice(s->device));
    double* tmp = nullptr;
    const hipError_t se = scratch_address(s->device, &tmp);
    if (se != hipSuccess) {
        s->err = std::string("relax_red_black_noalloc: no scratch address: ") + hipGetErrorString(se);
        return JG_ERR_HIP;
    }
    Dims d{(int)nx, (int)ny, (int)nz};
    // the copy of x that the out-of-place sweep reads, then the sweep itself:
    // the kernels of jg_relax_red_black, with its temporary replaced by scratch
    k_convert<double, double><<<nblocks_1d((idx_t)n), NT, 0, s->stream>>>(x, tmp, (idx_t)n);
    launch_sweep<double>(s, (const Row<double>*)rows, b, tmp, x, d, 0, nullptr, nullptr, nullptr, sor,
                         nullptr);
    JG_TRY(check_launch(s, "relax_red_black_noalloc"));
    return sync(s);
}

int jg_relax_jacobi(jg_solver* s, size_t nx, size_t ny, size_t nz, const double* rows,
                    const double* b, const double* x, double* xtemp) {
    if (!s || !valid_dims(nx, ny, nz) || !rows || !b || !x || !xtemp || x == xtemp)
        return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims d{(int)nx, (int)ny, (int)nz};
    launch_jacobi<double, false>(s, (const Row<double>*)rows, b, x, xtemp, d, 1.0, nullptr);
    JG_TRY(check_launch(s, "relax_jacobi"));
    return sync(s);
}

int jg_mg_restrict(jg_solver* s, size_t cnx, size_t cny, size_t cnz, const double* fine,
                   double* coarse) {
    if (!s || !valid_dims(cnx, cny, cnz) || !fine || !coarse) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims cd{(int)cnx, (int)cny, (int)cnz};
    Geo g = geo_planes(cd);
    k_restrict<double><<<g.grid, g.block, 0, s->stream>>>(fine, coarse, cd, nullptr);
    JG_TRY(check_launch(s, "restrict"));
    return sync(s);
}

int jg_mg_correct(jg_solver* s, size_t fnx, size_t fny, size_t fnz, const double* coarse,
                  double* fine) {
    if (!s || !valid_dims(fnx, fny, fnz) || !coarse || !fine || (fnx | fny | fnz) & 1)
        return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims fd{(int)fnx, (int)fny, (int)fnz};
    Geo g = geo_planes(fd);
    k_correct<double><<<g.grid, g.block, 0, s->stream>>>(coarse, fine, fd, nullptr);
    JG_TRY(check_launch(s, "correct"));
    return sync(s);
}

int jg_mg_restrict2(jg_solver* s, size_t cnx, size_t cny, const double* fine, double* coarse) {
    if (!s || !valid_dims(cnx, cny, 1) || !fine || !coarse) return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims cd{(int)cnx, (int)cny, 1};
    Geo g = geo_planes(cd);
    k_restrict2<double><<<g.grid, g.block, 0, s->stream>>>(fine, coarse, cd, nullptr);
    JG_TRY(check_launch(s, "restrict2"));
    return sync(s);
}

int jg_mg_correct2(jg_solver* s, size_t fnx, size_t fny, const double* coarse, double* fine) {
    if (!s || !valid_dims(fnx, fny, 1) || !coarse || !fine || (fnx | fny) & 1)
        return JG_ERR_INVALID_ARG;
    JG_HIP(hipSetDevice(s->device));
    Dims fd{(int)fnx, (int)fny, 1};
    Geo g = geo_planes(fd);
    k_correct2<double><<<g.grid, g.block, 0, s->stream>>>(coarse, fine, fd, nullptr);
    JG_TRY(check_launch(s, "correct2"));
    return sync(s);
}

}  // extern "C"

// ============================================================ batched solves
//
// Many independent systems of uneven sizes.  Systems with the same hierarchy
// form a group: one jg_solver holds all of them back to back (nsys > 1), and
// every V-cycle and PCG launch covers the whole group, each block taking its
// system from its grid index and exiting at once when that system's control
// block says it has stopped -- the per-system convergence mask.  A member is
// a view into its group (its own handle for building, uploading and reading
// its system).  The PCG iterations of all groups are captured once into one
// hipGraph (a fork from the batch stream, one branch per group, K
// iterations on that group's stream, a join); the host replays it and
// gathers every member's stop flag with one kernel and one copy per replay.

namespace {

constexpr int kBatchIters = 4;  // PCG iterations per graph replay (even: direction buffers realign)

// done flag and iteration count of every system's control block
__global__ void k_gather_ctl(Ctl* const* ctls, int n, int* out) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        out[2 * i] = ctls[i]->done | ctls[i]->nonfinite << 1;
        out[2 * i + 1] = (int)ctls[i]->iter;
    }
}

__global__ void k_gather_scal(double* const* scal, int idx, int n, double* out) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = scal[i][idx];
}

__global__ void k_gather_sigma(Ctl* const* ctls, int n, double* out) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = ctls[i]->sigma;
}

}  // namespace

struct jg_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t fork = nullptr, ev0 = nullptr, ev1 = nullptr;
    std::vector<jg_solver*> sys;     // member views, in the caller's order
    std::vector<jg_solver*> groups;  // one solver per distinct hierarchy, owning the arrays
    std::vector<std::vector<int>> members;  // per group: its members in group order
    std::vector<hipEvent_t> join;    // per group
    Ctl** dctl = nullptr;       // per member: ctl (FP64 solve), then ctl + 1 (mixed inner solve)
    double** dscal = nullptr;   // per member: scal
    int* dflags = nullptr;      // gathered (flags, iteration) pairs
    double* dvals = nullptr;    // gathered scalars
    int* hflags = nullptr;      // pinned
    double* hvals = nullptr;    // pinned
    struct Graph {
        int precision;
        unsigned pre, post0, post, coarsest;
        double omega;
        int pairs;
        hipGraph_t graph;
        hipGraphExec_t exec;
    };
    std::vector<Graph> graphs;
    std::string err;

    ~jg_batch() {
        for (auto& g : graphs) {
            (void)hipGraphExecDestroy(g.exec);
            (void)hipGraphDestroy(g.graph);
        }
        for (auto* s : sys) jg_solver_destroy(s);  // views first: they use the groups' streams
        for (auto* g : groups) jg_solver_destroy(g);
        for (auto e : join) (void)hipEventDestroy(e);
        for (void* p : {(void*)dctl, (void*)dscal, (void*)dflags, (void*)dvals}) (void)hipFree(p);
        if (hflags) (void)hipHostFree(hflags);
        if (hvals) (void)hipHostFree(hvals);
        for (auto e : {fork, ev0, ev1})
            if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

#define JG_HIPB(call)                                                    \
    do {                                                                 \
        hipError_t e_ = (call);                                          \
        if (e_ != hipSuccess) {                                          \
            B->err = std::string(#call) + ": " + hipGetErrorString(e_);  \
            return JG_ERR_HIP;                                           \
        }                                                                \
    } while (0)

namespace {

// The batch stream waits for the work queued so far on every group stream.
int batch_join(jg_batch* B) {
    for (size_t g = 0; g < B->groups.size(); ++g) {
        JG_HIPB(hipEventRecord(B->join[g], B->groups[g]->stream));
        JG_HIPB(hipStreamWaitEvent(B->stream, B->join[g], 0));
    }
    return JG_OK;
}

// Every group stream waits for the work queued so far on the batch stream.
int batch_fork(jg_batch* B) {
    JG_HIPB(hipEventRecord(B->fork, B->stream));
    for (auto* g : B->groups) JG_HIPB(hipStreamWaitEvent(g->stream, B->fork, 0));
    return JG_OK;
}

// Gathers (flags, iteration) of control block `which` (0: FP64, 1: inner) of
// every member into hflags; synchronises.
int batch_poll(jg_batch* B, int which) {
    const int S = (int)B->sys.size();
    k_gather_ctl<<<1, 256, 0, B->stream>>>(B->dctl + which * S, S, B->dflags);
    JG_HIPB(hipGetLastError());
    JG_HIPB(hipMemcpyAsync(B->hflags, B->dflags, 2 * S * sizeof(int), hipMemcpyDeviceToHost,
                           B->stream));
    JG_HIPB(hipStreamSynchronize(B->stream));
    return JG_OK;
}

int batch_scal(jg_batch* B, int idx) {
    const int S = (int)B->sys.size();
    k_gather_scal<<<1, 256, 0, B->stream>>>(B->dscal, idx, S, B->dvals);
    JG_HIPB(hipGetLastError());
    JG_HIPB(hipMemcpyAsync(B->hvals, B->dvals, S * sizeof(double), hipMemcpyDeviceToHost, B->stream));
    JG_HIPB(hipStreamSynchronize(B->stream));
    return JG_OK;
}

// The control blocks of a group's members, both of each, in one copy.
int batch_upload_ctl(jg_batch* B, jg_solver* g, const std::vector<Ctl>& h) {
    JG_HIPB(hipMemcpyAsync(g->ctl, h.data(), h.size() * sizeof(Ctl), hipMemcpyHostToDevice, g->stream));
    return JG_OK;
}

// ||b||^2 (into scal + at) and, with x, ||b - A x||^2 (into scal + at + 1,
// the residual itself into r) of every member of a group, in FP64; one launch
// covers the group.
void group_bb(jg_solver* g, int at) {
    const int nb1 = nblocks_1d(g->lv[0].d.n());
    k_dot<double, double><<<grid_1d(nb1, g), NT, 0, g->stream>>>(g->b, g->b, g->lv[0].d.n(), g->slot(3),
                                                                nullptr);
    k_fin_sum<<<g->nsys, kFinThreads, 0, g->stream>>>(g->slot(3), nb1, g->scal + at);
}
template <typename TR>
void group_residual(jg_solver* g, TR* r, int at) {
    Level& l0 = g->lv[0];
    const int nr = launch_residual<double, TR, true, false>(g, l0.A64, g->x, g->b, r, l0.d, g->slot(3),
                                                            nullptr);
    k_fin_sum<<<g->nsys, kFinThreads, 0, g->stream>>>(g->slot(3), nr, g->scal + at);
}

// Precision-specific views of a solver's level-0 PCG buffers (a group's:
// its first member's pointers, which every launch extends to all members).
Pcg<double> pcg64(jg_solver* s, const MgCfg<double>* mg) {
    Level& l0 = s->lv[0];
    return Pcg<double>{l0.A64, s->b, s->x, s->r, s->z, s->dA, s->dB, s->q, l0.d, s->ctl, mg};
}
Pcg<float> pcg32(jg_solver* s, const MgCfg<float>* mg) {
    Level& l0 = s->lv[0];
    return Pcg<float>{l0.A32, s->rhs32, s->e32, s->r32, s->z32, s->d32A, s->d32B, s->q32, l0.d,
                      s->ctl + 1, mg};
}

// Captures kBatchIters PCG iterations of every group into one graph (or
// returns the cached one for the same precision and V-cycle parameters).
template <typename T>
int batch_graph(jg_batch* B, int precision, const MgCfg<T>& mg, hipGraphExec_t* out) {
    for (auto& g : B->graphs)
        if (g.precision == precision && g.pre == mg.pre && g.post0 == mg.post0 && g.post == mg.post &&
            g.coarsest == mg.coarsest && g.omega == (double)mg.omega && g.pairs == mg.pairs) {
            *out = g.exec;
            return JG_OK;
        }
    JG_HIPB(hipStreamBeginCapture(B->stream, hipStreamCaptureModeRelaxed));
    int st = JG_OK;
    if (hipEventRecord(B->fork, B->stream) != hipSuccess) st = JG_ERR_HIP;
    for (size_t gi = 0; gi < B->groups.size() && st == JG_OK; ++gi) {
        jg_solver* g = B->groups[gi];
        if (hipStreamWaitEvent(g->stream, B->fork, 0) != hipSuccess) {
            st = JG_ERR_HIP;
            break;
        }
        for (int k = 0; k < kBatchIters && st == JG_OK; ++k) {
            if constexpr (sizeof(T) == 8)
                st = pcg_iteration<double>(g, pcg64(g, &mg), (k & 1) != 0, nullptr);
            else
                st = pcg_iteration<float>(g, pcg32(g, &mg), (k & 1) != 0, nullptr);
        }
        if (st == JG_OK && (hipEventRecord(B->join[gi], g->stream) != hipSuccess ||
                            hipStreamWaitEvent(B->stream, B->join[gi], 0) != hipSuccess))
            st = JG_ERR_HIP;
    }
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(B->stream, &graph);
    if (st != JG_OK || e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        B->err = "graph capture failed";
        return st != JG_OK ? st : JG_ERR_HIP;
    }
    hipGraphExec_t exec = nullptr;
    JG_HIPB(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    B->graphs.push_back(
        {precision, mg.pre, mg.post0, mg.post, mg.coarsest, (double)mg.omega, mg.pairs, graph, exec});
    *out = exec;
    return JG_OK;
}

// Replays the iteration graph until every member's control block `which`
// is done (or the iteration budget is spent).
int batch_replay(jg_batch* B, hipGraphExec_t exec, int which, unsigned max_iter) {
    const size_t S = B->sys.size();
    for (unsigned launched = 0;; launched += kBatchIters) {
        JG_TRY(batch_poll(B, which));
        bool all = true;
        for (size_t i = 0; i < S; ++i) all = all && (B->hflags[2 * i] & 1);
        if (all || launched > max_iter + kBatchIters) break;
        JG_HIPB(hipGraphLaunch(exec, B->stream));
    }
    return JG_OK;
}

// The FP32 copies of every group whose members' matrices changed.
int batch_f32(jg_batch* B) {
    for (size_t gi = 0; gi < B->groups.size(); ++gi) {
        jg_solver* g = B->groups[gi];
        for (int m : B->members[gi])
            if (!B->sys[m]->f32_valid) g->f32_valid = false;
        const int st = ensure_f32(g);
        if (st != JG_OK) {
            B->err = g->err;
            return st;
        }
        for (int m : B->members[gi]) B->sys[m]->f32_valid = true;
    }
    return JG_OK;
}

}  // namespace

extern "C" {

int jg_batch_create(int device, size_t nsys, const size_t* nx, const size_t* ny, const size_t* nz,
                    const size_t* nlev, jg_batch** out) {
    if (!out || nsys == 0 || nsys > 4096 || !nx || !ny || !nz || !nlev) return JG_ERR_INVALID_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= device || device < 0)
        return JG_ERR_NO_DEVICE;
    jg_batch* B = new jg_batch();
    B->device = device;
    auto fail = [&](int st) {
        delete B;
        return st;
    };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&B->stream) != hipSuccess ||
        hipEventCreateWithFlags(&B->fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreate(&B->ev0) != hipSuccess || hipEventCreate(&B->ev1) != hipSuccess)
        return fail(JG_ERR_HIP);
    // group the systems by hierarchy (finest size and level count)
    std::vector<int> group_of(nsys, -1), index_in(nsys, 0);
    std::vector<size_t> rep;  // a member of each group
    for (size_t i = 0; i < nsys; ++i) {
        if (nlev[i] == 0 || nlev[i] > 16) return fail(JG_ERR_INVALID_ARG);
        for (size_t g = 0; g < rep.size() && group_of[i] < 0; ++g) {
            const size_t r = rep[g];
            if (nx[r] == nx[i] && ny[r] == ny[i] && nz[r] == nz[i] && nlev[r] == nlev[i])
                group_of[i] = (int)g;
        }
        if (group_of[i] < 0) {
            group_of[i] = (int)rep.size();
            rep.push_back(i);
            B->members.emplace_back();
        }
        index_in[i] = (int)B->members[group_of[i]].size();
        B->members[group_of[i]].push_back((int)i);
    }
    for (size_t g = 0; g < rep.size(); ++g) {
        const size_t r = rep[g];
        std::vector<size_t> lx(nlev[r]), ly(nlev[r]), lz(nlev[r]);
        for (size_t l = 0; l < nlev[r]; ++l) {
            lx[l] = nx[r] >> l;
            ly[l] = ny[r] >> l;
            lz[l] = nz[r] >> l;
        }
        jg_solver* s = nullptr;
        int st = jg_solver_create(device, &s);
        if (st != JG_OK) return fail(st);
        B->groups.push_back(s);
        // the checks of a single hierarchy, then the arrays of every member
        st = jg_solver_set_levels(s, nlev[r], lx.data(), ly.data(), lz.data());
        if (st == JG_OK && (s->twod || lz[0] == 1)) st = JG_ERR_UNSUPPORTED;  // batches are 3-D
        if (st == JG_OK)
            st = levels_alloc(s, nlev[r], lx.data(), ly.data(), lz.data(),
                              (int)B->members[g].size());
        if (st != JG_OK) return fail(st);
        hipEvent_t e = nullptr;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return fail(JG_ERR_HIP);
        B->join.push_back(e);
    }
    for (size_t i = 0; i < nsys; ++i) {
        jg_solver* v = nullptr;
        const int st = jg_solver_create(device, &v);
        if (st != JG_OK) return fail(st);
        make_view(B->groups[group_of[i]], index_in[i], v);
        B->sys.push_back(v);
    }
    std::vector<Ctl*> ctls(2 * nsys);
    std::vector<double*> scals(nsys);
    for (size_t i = 0; i < nsys; ++i) {
        ctls[i] = B->sys[i]->ctl;
        ctls[nsys + i] = B->sys[i]->ctl + 1;
        scals[i] = B->sys[i]->scal;
    }
    if (hipMalloc((void**)&B->dctl, 2 * nsys * sizeof(Ctl*)) != hipSuccess ||
        hipMalloc((void**)&B->dscal, nsys * sizeof(double*)) != hipSuccess ||
        hipMalloc((void**)&B->dflags, 2 * nsys * sizeof(int)) != hipSuccess ||
        hipMalloc((void**)&B->dvals, nsys * sizeof(double)) != hipSuccess ||
        hipHostMalloc((void**)&B->hflags, 2 * nsys * sizeof(int), hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void**)&B->hvals, nsys * sizeof(double), hipHostMallocDefault) != hipSuccess ||
        hipMemcpy(B->dctl, ctls.data(), 2 * nsys * sizeof(Ctl*), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(B->dscal, scals.data(), nsys * sizeof(double*), hipMemcpyHostToDevice) != hipSuccess)
        return fail(JG_ERR_OUT_OF_MEMORY);
    *out = B;
    return JG_OK;
}

void jg_batch_destroy(jg_batch* B) {
    if (!B) return;
    (void)hipSetDevice(B->device);
    (void)hipStreamSynchronize(B->stream);
    for (auto* g : B->groups) (void)hipStreamSynchronize(g->stream);
    delete B;
}

const char* jg_batch_last_error(const jg_batch* B) { return B ? B->err.c_str() : "null batch"; }

size_t jg_batch_size(const jg_batch* B) { return B ? B->sys.size() : 0; }

jg_solver* jg_batch_system(jg_batch* B, size_t i) {
    return (B && i < B->sys.size()) ? B->sys[i] : nullptr;
}

int jg_batch_mgpcg(jg_batch* B, unsigned max_iter, const jg_mg_params* p, const jg_gpu_options* o,
                   jg_solve_info* infos, double* total_ms) {
    if (!B || !p) return JG_ERR_INVALID_ARG;
    JG_HIPB(hipSetDevice(B->device));
    const size_t S = B->sys.size();
    jg_gpu_options opt;
    double omega = 0.0;
    {
        const int st = mg_options(B->sys[0], p, o, &opt, &omega);
        if (st != JG_OK) {
            B->err = B->sys[0]->err;
            return st;
        }
    }
    if (opt.smoother == JG_SMOOTH_JACOBI) {
        B->err = "batched solves use the red-black smoother";
        return JG_ERR_UNSUPPORTED;
    }
    const bool mixed = opt.precision == JG_MIXED;
    if (mixed) JG_TRY(batch_f32(B));
    for (auto* g : B->groups) JG_TRY(sync(g));
    std::vector<unsigned> iters(S, 0), refinements(S, 0);
    std::vector<double> last(S, 0.0), bnorm(S, 0.0);
    std::vector<int> status(S, JG_OK);
    JG_TRY(batch_join(B));
    JG_HIPB(hipEventRecord(B->ev0, B->stream));
    JG_TRY(batch_fork(B));
    if (!mixed) {
        MgCfg<double> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter, omega};
        mg.pairs = opt.sweep_pairs;
        hipGraphExec_t exec = nullptr;
        JG_TRY(batch_graph<double>(B, JG_FP64, mg, &exec));
        JG_TRY(batch_fork(B));
        for (size_t gi = 0; gi < B->groups.size(); ++gi) {
            jg_solver* g = B->groups[gi];
            const Dims& d0 = g->lv[0].d;
            k_fill<double><<<grid_1d(nblocks_1d(d0.n()), g), NT, 0, g->stream>>>(g->x, 0.0, d0.n());
            std::vector<Ctl> h(kSysCtl * (size_t)g->nsys);
            for (int q = 0; q < g->nsys; ++q)
                init_ctl(&h[kSysCtl * q], max_iter, p->max_tol, opt.stop_rule == JG_STOP_RELATIVE ? 1 : 0,
                         opt.rel_tol);
            JG_TRY(batch_upload_ctl(B, g, h));
            JG_TRY(pcg_init<double>(g, pcg64(g, &mg)));
        }
        JG_TRY(batch_join(B));
        JG_TRY(batch_replay(B, exec, 0, max_iter));
        JG_TRY(batch_poll(B, 0));
        for (size_t i = 0; i < S; ++i) {
            iters[i] = (unsigned)B->hflags[2 * i + 1];
            if (B->hflags[2 * i] & 2) status[i] = JG_ERR_NONFINITE;
        }
    } else {
        MgCfg<float> mg{p->restrict_iter, p->final_iter, p->correct_iter, p->coarsest_iter, (float)omega};
        mg.pairs = opt.sweep_pairs;
        hipGraphExec_t exec = nullptr;
        JG_TRY(batch_graph<float>(B, JG_MIXED, mg, &exec));
        JG_TRY(batch_fork(B));
        // x = 0, ||b|| and the FP32 right-hand side of every member (b - A x is b)
        for (auto* g : B->groups) {
            const Dims& d0 = g->lv[0].d;
            const int nb1 = nblocks_1d(d0.n());
            k_fill<double><<<grid_1d(nb1, g), NT, 0, g->stream>>>(g->x, 0.0, d0.n());
            k_convert<double, float><<<grid_1d(nb1, g), NT, 0, g->stream>>>(g->b, g->rhs32, d0.n());
            group_bb(g, 2);
        }
        JG_TRY(batch_join(B));
        JG_TRY(batch_scal(B, 2));
        std::vector<double> goal(S);
        for (size_t i = 0; i < S; ++i) {
            bnorm[i] = std::sqrt(B->hvals[i]);
            goal[i] = opt.stop_rule == JG_STOP_RELATIVE ? opt.rel_tol * bnorm[i] : p->max_tol;
        }
        std::vector<char> done(S, 0);
        for (unsigned outer = 0;; ++outer) {
            if (outer > 0) {
                // FP64 residual r = b - A x into the FP32 right-hand side (of
                // a finished member too: its x, and so its norm, is unchanged)
                JG_TRY(batch_fork(B));
                for (auto* g : B->groups) group_residual<float>(g, g->rhs32, 3);
                JG_TRY(batch_join(B));
                JG_TRY(batch_scal(B, 3));
            }
            bool any = false;
            for (size_t i = 0; i < S; ++i) {
                if (done[i]) continue;
                const double rr = B->hvals[i];
                last[i] = std::sqrt(rr);
                if (!std::isfinite(rr)) {
                    status[i] = JG_ERR_NONFINITE;
                    done[i] = 1;
                } else if (last[i] <= goal[i] || outer >= opt.max_refine || iters[i] >= max_iter) {
                    done[i] = 1;
                }
                any = any || !done[i];
            }
            if (!any) break;
            JG_TRY(batch_fork(B));
            for (size_t gi = 0; gi < B->groups.size(); ++gi) {
                jg_solver* g = B->groups[gi];
                // each member's inner control block: a finished member's
                // blocks exit at once
                std::vector<Ctl> h(kSysCtl * (size_t)g->nsys);
                for (int q = 0; q < g->nsys; ++q) {
                    const int m = B->members[gi][q];
                    Ctl& c = h[kSysCtl * q + 1];
                    if (done[m]) {
                        init_ctl(&c, 0, 0.0, 1, 0.0);
                        c.done = 1;
                    } else {
                        const double inner =
                            std::max(opt.inner_rel_tol, std::min(0.5, 0.5 * goal[m] / last[m]));
                        init_ctl(&c, max_iter - iters[m], 0.0, 1, inner);
                    }
                }
                JG_TRY(batch_upload_ctl(B, g, h));
                const Dims& d0 = g->lv[0].d;
                k_fill<float><<<grid_1d(nblocks_1d(d0.n()), g), NT, 0, g->stream>>>(g->e32, 0.f, d0.n());
                JG_TRY(pcg_init<float>(g, pcg32(g, &mg)));
            }
            JG_TRY(batch_join(B));
            JG_TRY(batch_replay(B, exec, 1, max_iter));
            JG_TRY(batch_poll(B, 1));
            JG_TRY(batch_fork(B));
            for (size_t i = 0; i < S; ++i) {
                if (done[i]) continue;
                iters[i] += (unsigned)B->hflags[2 * i + 1];
                if (B->hflags[2 * i] & 2) {  // the inner FP32 solve met a non-finite value
                    status[i] = JG_ERR_NONFINITE;
                    done[i] = 1;
                    continue;
                }
                ++refinements[i];
            }
            // (a finished member's e32 is zero)
            for (auto* g : B->groups)
                k_add_correction<<<grid_1d(nblocks_1d(g->lv[0].d.n()), g), NT, 0, g->stream>>>(
                    g->x, g->e32, g->lv[0].d.n(), g->ctl + 1);
        }
    }
    JG_TRY(batch_join(B));
    JG_HIPB(hipEventRecord(B->ev1, B->stream));
    JG_HIPB(hipStreamSynchronize(B->stream));
    float ms = 0.f;
    JG_HIPB(hipEventElapsedTime(&ms, B->ev0, B->ev1));
    if (total_ms) *total_ms = ms;
    std::vector<double> rel(S, 0.0);
    if (infos) {
        // mixed: last is the FP64 norm of the final x's residual already
        JG_TRY(batch_fork(B));
        if (!mixed)
            for (auto* g : B->groups) {
                group_bb(g, 0);
                group_residual<double>(g, g->r, 1);
            }
        JG_TRY(batch_join(B));
        if (!mixed) {
            JG_TRY(batch_scal(B, 0));
            for (size_t i = 0; i < S; ++i) bnorm[i] = std::sqrt(B->hvals[i]);
            JG_TRY(batch_scal(B, 1));
            for (size_t i = 0; i < S; ++i) rel[i] = std::sqrt(B->hvals[i]);
            k_gather_sigma<<<1, 256, 0, B->stream>>>(B->dctl, (int)S, B->dvals);
            JG_HIPB(hipGetLastError());
            JG_HIPB(hipMemcpyAsync(B->hvals, B->dvals, S * sizeof(double), hipMemcpyDeviceToHost, B->stream));
            JG_HIPB(hipStreamSynchronize(B->stream));
            for (size_t i = 0; i < S; ++i) last[i] = std::sqrt(std::fabs(B->hvals[i]));
        }
        for (size_t i = 0; i < S; ++i) {
            if (mixed) rel[i] = last[i];
            if (bnorm[i] > 0) rel[i] /= bnorm[i];
        }
    }
    int worst = JG_OK;
    for (size_t i = 0; i < S; ++i) {
        if (status[i] != JG_OK) worst = status[i];
        if (!infos) continue;
        jg_solve_info& info = infos[i];
        std::memset(&info, 0, sizeof(info));
        info.iterations = iters[i];
        info.refinements = refinements[i];
        info.solve_ms = ms;
        info.rel_residual = rel[i];
        info.last_residual = last[i];
        if (status[i] != JG_OK)
            info.converged = 0;
        else if (opt.stop_rule == JG_STOP_RELATIVE)
            info.converged = info.rel_residual <= opt.rel_tol;
        else if (mixed)
            info.converged = last[i] <= p->max_tol;  // the outer loop's goal
        else
            info.converged = last[i] <= p->max_tol || iters[i] < max_iter;
    }
    if (worst == JG_ERR_NONFINITE) B->err = "non-finite value in a batched solve";
    return worst;
}

}  // extern "C"
