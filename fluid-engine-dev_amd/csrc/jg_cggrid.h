// jg_cggrid.h -- Jet's plain CG (include/jet/detail/cg-inl.h:15-94) on a
// system that fits the chip: one launch runs the iterations, and
// matrix and vectors stay in registers.
//
// A CG iteration of a small grid is bound by its kernel boundaries: at 64^3
// the product, the update, the dot, two one-block sums, the skipped refresh
// and the host's poll took 30 us for 31 MB of traffic.  Here a thread owns C
// rows (C * 1024 consecutive rows per block, one block per CU): their
// entries, x, r and d.  The d of the block's own rows is in LDS; a neighbour
// row of another block is read as that block's published r, and its d kept
// by the same recurrence d = r + beta d (the same expression on the same
// operands, so the same value).  So an iteration has two grid-wide points,
// the sums d.q and r.r, and each of them is also the barrier.
//
// A grid sum is an all-gather: every block publishes its partial, cut in two
// words that carry the iteration's number, into its own slot, and waits until
// every slot holds this number; then it adds the partials in slot order.
// There is no atomic read-modify-write and no separate flag, every block
// gets the same bits, and a run is deterministic.  What crosses blocks (r,
// on refresh iterations x, the slots) is written and read by agent-scope
// atomics, which go through the XCDs' private L2s; a block waits for its
// stores before its slot is written.  The waits end because all blocks become
// resident: there are at most as many as CUs, a block fits a free CU, other
// work on the device ends without waiting for this kernel, and one process
// runs one such launch on a device at a time (cg_grid).  Where that fails (a
// device shared with another program that waits the same way, fewer CUs than
// reported), a wait that does not end within CgGridArgs::polls makes every
// block leave, and the solve starts again as the loop of one launch per step
// (so does one whose launch is refused).
// (hipLaunchCooperativeKernel, which guarantees residency, makes the runtime
// add a queue of its own kind, and from then on graphs with many branches run
// at half their rate for the rest of the process: a batch of 16 hierarchies 6
// -> 16 ms.)
//
// At 64^3 an iteration takes 7.9 us: 2.7 and 3.2 (with the wait for the
// published r) in the two sums, the rest the loads of the neighbours' r
// (0.7) and two FP64 divisions.  cg-64 went from 12.4 to 3.5 ms and a
// compressed system of 368 000 rows, two rows per thread, from 38 to 11.7 us
// an iteration.
//
// Per-row values are those of k_dir_spmv_tile / k_ell_spmv_dot and
// k_update_xr; the sums run in another order.
#pragma once

#include "jg_device.h"
#include "jg_csr.h"

namespace jg {

constexpr int kCgThreads = 1024;
constexpr int kCgMaxBlocks = 256;   // one slot per thread that polls
constexpr int kCgCopies = 8;        // copies of the slots
constexpr int kCgCopyWords = kCgMaxBlocks * 4;
constexpr int kCgSumWords = kCgCopies * kCgCopyWords;  // of one kind of grid sum
constexpr int kCgW = 7;             // entries of a row
constexpr int kCgChunk = 2048;      // iterations per launch

struct CgGridArgs {
    const Row<double>* A;  // the grid's rows (nullptr: ell)
    EllDev ell;
    Dims d;                // grid (ELL: {rows, 1, 1})
    const double* b;
    double *x, *r, *dir;   // state in and out: iterate, residual, last direction
    Ctl* ctl;
    unsigned long long* slots;  // [3][kCgSumWords], zero at launch
    int polls;                  // bound of a wait for the other blocks
};

__device__ __forceinline__ void agent_store(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long agent_load(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(double* p, double v) {
    agent_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v));
}
__device__ __forceinline__ double agent_load(const double* p) {
    return __builtin_bit_cast(double, agent_load(reinterpret_cast<const unsigned long long*>(p)));
}
// Element o of p: a uniform base and a 32-bit offset (the rows of a chip-sized
// system fill a few MB).
__device__ __forceinline__ double* at32(double* p, int o) {
    return reinterpret_cast<double*>(reinterpret_cast<char*>(p) + (unsigned)o * 8u);
}

struct CgShared {
    double part[kCgThreads / kWave];
    double tot[kCgMaxBlocks / kWave];
    int bad[kCgMaxBlocks / kWave];
    Ctl ctl;  // the block's copy of the control block; thread 0 writes it
};

// The sum of v over the grid, in every thread, and a barrier: what any block
// published before it is visible to all after it.  Adds lanes, waves and
// blocks in a fixed order.  false: a block did not arrive.
//
// The slots exist kCgCopies times and a block reads one copy, so that the
// polls of all blocks spread over the memory channels; slots of 32 B up to
// 128 blocks, packed ones above.  Measured alone: 1.5 us with 32 blocks,
// 1.6 with 64, 1.9 with 128, 2.6 with 256 (one packed copy and shuffles: 2.9,
// 3.2, 4.1, 4.5).
__device__ __forceinline__ bool grid_sum(double v, unsigned long long* slots, unsigned epoch,
                                         int polls, CgShared& sh, double& sum) {
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    const int G = gridDim.x, step = G <= 128 ? 4 : 2;
    v = wave_sum(v);
    if (lane == kWave - 1) sh.part[wave] = v;
    // the wave's published values have been performed before the block's slot is
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (wave == 0) {
        static_assert(kCgThreads / kWave == 16, "one row of lanes adds the waves");
        const double s = lane_value(row_sum(sh.part[lane & 15]), 15);
        if (t < kCgCopies) {
            const unsigned long long u = __builtin_bit_cast(unsigned long long, s);
            const unsigned long long e = (unsigned long long)epoch << 32;
            unsigned long long* p = slots + t * kCgCopyWords + step * blockIdx.x;
            agent_store(p, e | (u & 0xffffffffull));
            agent_store(p + 1, e | (u >> 32));
        }
    }
    if (wave < kCgMaxBlocks / kWave) {
        double p = 0.0;
        int bad = 0;
        if (t < G) {
            const unsigned long long* from = slots + (blockIdx.x % kCgCopies) * kCgCopyWords + step * t;
            unsigned long long lo, hi;
            int polled = 0;
            do {
                lo = agent_load(from);
                hi = agent_load(from + 1);
                bad = ++polled > polls;
            } while (!bad && ((unsigned)(lo >> 32) != epoch || (unsigned)(hi >> 32) != epoch));
            p = __builtin_bit_cast(double, hi << 32 | (lo & 0xffffffffull));
        }
        p = wave_sum(p);
        const int any = __ballot(bad) != 0;
        if (lane == kWave - 1) {
            sh.tot[wave] = p;
            sh.bad[wave] = any;
        }
    }
    __syncthreads();
    sum = sh.tot[0];
    int bad = sh.bad[0];
#pragma unroll
    for (int w = 1; w < kCgMaxBlocks / kWave; ++w) {
        sum += sh.tot[w];
        bad |= sh.bad[w];
    }
    return !bad;
}

template <int C, bool ELL>
__global__ __launch_bounds__(kCgThreads) void k_cg_grid(CgGridArgs a) {
#pragma clang fp contract(off)
    constexpr int kOwn = C * kCgThreads;
    // d of the block's rows, then of its entries in other blocks' rows: entry
    // e of the thread's row q at kOwn + (q * kCgW + e) * kCgThreads + t
    __shared__ double dl[kOwn + C * kCgW * kCgThreads];
    static_assert(kOwn + C * kCgW * kCgThreads <= 65536, "16-bit places in dl");
    __shared__ CgShared sh;
    if (a.ctl->done) return;
    // (opaque in the loop: addresses formed from it where they are used cost
    // fewer registers than addresses kept across it)
    int t = threadIdx.x;
    const int n = (int)a.d.n();
    const int base = blockIdx.x * kOwn;
    const int sy = a.d.nx, sz = a.d.nx * a.d.ny;
    double val[C][kCgW], x[C], r[C], d[C];
    // places in dl of a row's entries, two to a word; an entry that does not
    // exist has value 0 and the row's own place
    unsigned place[C][(kCgW + 1) / 2];
    int ecol[C][ELL ? kCgW : 1];  // columns (the grid's follow from the cell)
    auto at = [&](int q, int e) __attribute__((always_inline)) -> int {
        return (int)(place[q][e / 2] >> (16 * (e & 1)) & 0xffffu);
    };
    // Jet's mvm order: centre, -x, +x, -y, +y, -z, +z
    auto col = [&](int q, int e) __attribute__((always_inline)) -> int {
        if constexpr (ELL) return ecol[q][e];
        const int off = e == 0 ? 0 : (e <= 2 ? 1 : (e <= 4 ? sy : sz));
        return base + q * kCgThreads + t + (e & 1 ? -off : off);
    };
#pragma unroll
    for (int q = 0; q < C; ++q) {
        const int c = base + q * kCgThreads + t;
        x[q] = r[q] = d[q] = 0.0;
        bool has[kCgW] = {};
#pragma unroll
        for (int e = 0; e < kCgW; ++e) val[q][e] = 0.0;
#pragma unroll
        for (int e = 0; e < (ELL ? kCgW : 1); ++e) ecol[q][e] = 0;
        if (c < n) {
            x[q] = a.x[c];
            r[q] = a.r[c];
            d[q] = a.dir[c];
            if constexpr (ELL) {
                const int len = a.ell.len[c];
#pragma unroll
                for (int e = 0; e < kCgW; ++e)
                    if (e < len) {
                        has[e] = true;
                        ecol[q][e] = a.ell.ci[e * a.ell.rows + c];
                        val[q][e] = a.ell.val[e * a.ell.rows + c];
                    }
            } else {
                const int i = c % sy, j = (c / sy) % a.d.ny, k = c / sz;
                const Row<double> row = a.A[c];
                has[0] = true;
                has[1] = i > 0;
                has[2] = i + 1 < a.d.nx;
                has[3] = j > 0;
                has[4] = j + 1 < a.d.ny;
                has[5] = k > 0;
                has[6] = k + 1 < a.d.nz;
                val[q][0] = row.c;
                if (has[1]) val[q][1] = a.A[c - 1].r;
                if (has[2]) val[q][2] = row.r;
                if (has[3]) val[q][3] = a.A[c - sy].u;
                if (has[4]) val[q][4] = row.u;
                if (has[5]) val[q][5] = a.A[c - sz].f;
                if (has[6]) val[q][6] = row.f;
            }
        }
#pragma unroll
        for (int e = 0; e < (kCgW + 1) / 2; ++e) place[q][e] = 0;
#pragma unroll
        for (int e = 0; e < kCgW; ++e) {
            unsigned l = q * kCgThreads + t;
            if (has[e]) {
                const int cc = col(q, e);
                l = (unsigned)(cc - base);
                if (l >= (unsigned)kOwn) {
                    l = kOwn + (q * kCgW + e) * kCgThreads + t;
                    dl[l] = a.dir[cc];
                }
            }
            place[q][e / 2] |= l << (16 * (e & 1));
        }
    }
    // the scalars of the control block: the same bits in every block, in
    // scalar registers
    double sigma = lane_value(a.ctl->sigma, 0), beta = lane_value(a.ctl->beta, 0);
    const double tol2 = a.ctl->tol2, lim = a.ctl->rel2 * a.ctl->bb;
    const bool relative = a.ctl->stop_rule == 1;
    const unsigned max_iter = a.ctl->max_iter;
    unsigned iter = __builtin_amdgcn_readfirstlane(a.ctl->iter);
    int trigger = __builtin_amdgcn_readfirstlane(a.ctl->trigger);
    double dq = 0.0, alpha = 0.0, sigma_old = sigma;
    bool refresh = false, nonfinite = false, done = false;
    unsigned long long* const slot_dq = a.slots;
    unsigned long long* const slot_rr = a.slots + kCgSumWords;
    unsigned long long* const slot_x = a.slots + 2 * kCgSumWords;
    bool ok = true;
    // forgets what the compiler derived from the thread index, columns and places
    auto opaque = [&]() __attribute__((always_inline)) {
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int q = 0; q < C; ++q) {
#pragma unroll
            for (int e = 0; e < (kCgW + 1) / 2; ++e) asm volatile("" : "+v"(place[q][e]));
#pragma unroll
            for (int e = 0; e < (ELL ? kCgW : 1); ++e) asm volatile("" : "+v"(ecol[q][e]));
        }
    };
    for (unsigned epoch = 1; epoch <= kCgChunk; ++epoch) {
        opaque();
        // d = r + beta d, here and at the other blocks' rows
        double rx[C][kCgW];
#pragma unroll
        for (int q = 0; q < C; ++q)
#pragma unroll
            for (int e = 0; e < kCgW; ++e)
                if (at(q, e) >= kOwn) rx[q][e] = agent_load(at32(a.r, col(q, e)));
#pragma unroll
        for (int q = 0; q < C; ++q) {
            d[q] = r[q] + beta * d[q];
            dl[q * kCgThreads + t] = d[q];
        }
#pragma unroll
        for (int q = 0; q < C; ++q)
#pragma unroll
            for (int e = 0; e < kCgW; ++e)
                if (at(q, e) >= kOwn) dl[at(q, e)] = rx[q][e] + beta * dl[at(q, e)];
        opaque();
        __syncthreads();
        double s[C], acc = 0.0;
#pragma unroll
        for (int q = 0; q < C; ++q) {
            s[q] = 0.0;
#pragma unroll
            for (int e = 0; e < kCgW; ++e) s[q] += val[q][e] * dl[at(q, e)];
            acc += d[q] * s[q];
        }
        ok = grid_sum(acc, slot_dq, epoch, a.polls, sh, dq);
        if (!ok) break;
        // k_fin_alpha
        dq = lane_value(dq, 0);
        alpha = lane_value(sigma / dq, 0);
        refresh = trigger || (iter % 50 == 0 && iter > 0);
        trigger = 0;
        if (!isfinite(alpha)) {
            nonfinite = done = true;
            break;
        }
        // k_update_xr
#pragma unroll
        for (int q = 0; q < C; ++q) x[q] += alpha * d[q];
        if (!refresh) {
#pragma unroll
            for (int q = 0; q < C; ++q) r[q] -= alpha * s[q];
        } else {
            // the true residual b - A x (k_residual / k_ell_residual)
#pragma unroll
            for (int q = 0; q < C; ++q) {
                const int c = base + q * kCgThreads + t;
                if (c < n) agent_store(at32(a.x, c), x[q]);
            }
            double none;
            ok = grid_sum(0.0, slot_x, epoch, a.polls, sh, none);
            if (!ok) break;
#pragma unroll
            for (int q = 0; q < C; ++q) {
                const int c = base + q * kCgThreads + t;
                if (c >= n) continue;
                double xv[kCgW];
#pragma unroll
                for (int e = 0; e < kCgW; ++e)  // (a missing entry reads the row itself)
                    xv[e] = agent_load(at32(a.x, at(q, e) < kOwn ? base + at(q, e) : col(q, e)));
                const double bv = a.b[c];
                double rv = ELL ? 0.0 : bv;
#pragma unroll
                for (int e = 0; e < kCgW; ++e) {
                    const double p = val[q][e] * xv[e];
                    rv = ELL ? rv + p : rv - p;
                }
                r[q] = ELL ? bv - rv : rv;
            }
        }
        acc = 0.0;
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int c = base + q * kCgThreads + t;
            acc += r[q] * r[q];
            if (c < n) agent_store(at32(a.r, c), r[q]);
        }
        double rz;
        ok = grid_sum(acc, slot_rr, epoch, a.polls, sh, rz);
        if (!ok) break;
        // k_fin_sigma (z = r)
        rz = lane_value(rz, 0);
        beta = lane_value(rz / sigma, 0);
        trigger = rz > sigma;
        sigma_old = sigma;
        sigma = rz;
        ++iter;
        const bool go = rz > (relative ? lim : tol2);
        nonfinite = !isfinite(rz);
        done = !(go && iter < max_iter) || nonfinite;
        if (done) break;
    }
#pragma unroll
    for (int q = 0; q < C; ++q) {
        const int c = base + q * kCgThreads + t;
        if (c < n) {
            a.x[c] = x[q];
            a.dir[c] = d[q];
        }
    }
    if (blockIdx.x == 0 && t == 0) {
        Ctl c = *a.ctl;
        c.dq = dq;
        c.alpha = alpha;
        c.refresh = refresh;
        c.sigma_old = sigma_old;
        c.sigma = sigma;
        if (iter > c.iter) c.rr = sigma;
        c.beta = beta;
        c.iter = iter;
        c.trigger = trigger;
        c.nonfinite |= nonfinite;
        c.done = done || !ok;
        c.pad = !ok;
        *a.ctl = c;
    }
}

}  // namespace jg
