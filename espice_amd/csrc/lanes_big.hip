// Lanes whose working set is beyond a workgroup's LDS (the 64 x 64 RC mesh:
// 4,099 unknowns and about 137,000 factor slots, 1.1 MB per lane): one
// workgroup of kT wavefronts per lane (kTeam, or 1 where the elimination is
// too narrow to feed more: big_team), with the lane's factor slots and
// vectors in HBM (one contiguous region per lane) and LDS as the staging
// area of each phase:
// - assembly: the stamp cells of kT chunks of 64 instances, one chunk a
//   wavefront; each reduce task adds its cells into its target in HBM;
// - refactor: the tape's replay cut into blocks of as many slots as the lane's
//   LDS holds; a block gathers its slots into LDS, runs its rows (64 kT
//   independent updates per step, each slot's updates in the order of the
//   column replay, lane_kernels.zig:49-118) and scatters what it wrote;
// - solves: the solve vector in LDS, the factor entries read from their
//   slots ahead of use (lane_kernels.zig:123-143).
// A team has the whole LDS of a CU: the mesh is 35 blocks and 9,600 rows of
// 512, each an LDS round trip and a barrier (about 530 cycles with its share
// of the gathers; the refactor is 5.1 M of an iteration's 6.1 M cycles). On
// one wavefront with a quarter of the LDS (four lanes a CU) its blocks hold a
// few columns at a time, whose dependency chains leave half of 64 threads idle
// over 91,400 rows. Measured,
// 64 x 64 mesh, an operating point and two steps: 355 ms on one wavefront with
// the solves in column chunks, 226 ms with the solves as rows, 47 ms on
// eight (64 lanes; 1,662 and 844 ms for 4,096). A line of 3,000 nodes: 76,
// 47 and 74 ms (64 lanes; 316, 229 and 1,173 ms for 4,096).
// The reference's lanes keep these arrays in global memory too, one thread
// per lane walking the tape serially (lane_kernels.zig:7-8). Every value is
// bitwise the wavefront kernels' and the oracle's: the same sums in the same
// order, compiled without contraction.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "esl_device.h"
#include "esl_eval.h"
#include "esl_internal.h"
#include "eslmath.h"

namespace esl {

// Pointers with their address space explicit (gptr/lptr): global for the
// lane's HBM arrays and the tape, LDS for the staging area.
typedef __attribute__((address_space(1))) double gdbl;
typedef __attribute__((address_space(1))) const double gcdbl;
typedef __attribute__((address_space(1))) const uint32_t gcu32;
typedef __attribute__((address_space(3))) double ldbl;

// The lane's arrays in HBM and its LDS area (the kernel's dynamic LDS,
// passed down so that no function looks its address up).
struct BigLane {
    gdbl *tv, *rhs, *x, *xold, *sdiag, *q, *cq;
    ldbl *sm;
    ldbl *scratch;   // team_scratch doubles: the team's reductions
};

// The team's reductions: the largest of every thread's v (as bit patterns),
// and whether any thread's p holds; uniform. They are barriers.
template <uint32_t kT>
__device__ inline uint64_t team_max_u64(uint64_t v, ldbl *scratch)
{
    if (kT == 1) return wave_max_u64(v);
    auto *s = (__attribute__((address_space(3))) uint64_t *)scratch;
    const uint64_t w = wave_max_u64(v);
    if (threadIdx.x % kWave == 0) s[threadIdx.x / kWave] = w;
    __syncthreads();
    uint64_t m = s[0];
#pragma unroll
    for (uint32_t k = 1; k < kT; k++) m = s[k] > m ? s[k] : m;
    __syncthreads();
    return uni(m);
}
template <uint32_t kT>
__device__ inline bool team_any(bool p, ldbl *scratch)
{
    return kT == 1 ? wave_any(p) : team_max_u64<kT>(p ? 1u : 0u, scratch) != 0;
}

template <uint32_t kT>
__device__ inline BigLane big_lane(const BigArgs &b, uint32_t g, ldbl *sm)
{
    const uint32_t n = b.ta.op.dp.n;
    BigLane L;
    L.tv = gptr(b.ws) + (size_t)g * b.ws_stride;
    L.rhs = L.tv + b.tv_cap;
    L.x = L.rhs + n;
    L.xold = L.x + n;
    L.sdiag = L.xold + n;
    L.q = L.sdiag + n;
    L.cq = L.q + n;
    L.sm = sm;
    L.scratch = sm + (b.lds - team_scratch(kT));
    return L;
}

// Assembly with the deck's reduce tasks, one target per thread: Jacobian
// entries into M[amap[slot]] (amap null: M[slot], pattern order). tran: the
// charges too (row charges into q, charge-Jacobian cells into cq), then the
// ground pin and the companion A = G + ag0 C, F += ag0 (q - q1) - ag1 i_prev
// (assemble_tran's arithmetic); otherwise capacitors and charge targets are
// skipped and only the ground pin follows (assemble_pattern's). A round
// stages the stamp cells of kTeam chunks in LDS, one chunk a wavefront, and
// adds each target's cells in instance order.
template <uint32_t kT>
__device__ void big_assemble(const BigArgs &b, const uint32_t *amap_, uint32_t n_slots, const double *live,
                             gdbl *x, double *lim, gdbl *M, const BigLane &L, bool tran, double t, double ag0,
                             double ag1, gcdbl *q1, gcdbl *ip, uint32_t tid)
{
    const DeckProg &dp = b.ta.op.dp;
    const uint32_t n = dp.n;
    ldbl *st = L.sm;
    gcu32 *amap = amap_ ? gptr(amap_) : nullptr;
    gcu32 *rt_target = gptr(b.rt_target), *rt_cell = gptr(b.rt_cell), *rt_round = gptr(b.rt_round);
    const __attribute__((address_space(1))) uint16_t *cells = gptr(b.rt_cells);
    const uint32_t wv = uni(tid / kWave), wt = tid % kWave;
    for (uint32_t i = tid; i < n_slots; i += kT * kWave) M[i] = 0.0;
    for (uint32_t i = tid; i < n; i += kT * kWave) {
        L.rhs[i] = 0.0;
        if (tran) L.q[i] = 0.0;
    }
    if (tran)
        for (uint32_t k = tid; k < dp.n_cslot; k += kT * kWave) L.cq[k] = 0.0;
    __syncthreads();
    for (uint32_t r = 0; r < b.n_rounds; r++) {
        const uint32_t c = r * kT + wv;
        if (c < dp.n_chunks) {
            const Chunk ch = dp.chunks[c];
            if (tran || ch.kind != kC)   // capacitors have no static stamps
                eval_chunk(dp, ch, live, x, lim, dp.n_mos, st + wv * kStageDoubles, wt, t, tran);
        }
        __syncthreads();
        const uint32_t t1 = rt_round[r + 1];
        for (uint32_t k = rt_round[r] + tid; k < t1; k += kT * kWave) {
            const uint32_t tgt = rt_target[k];
            const uint32_t idx = tgt & kTargetMask;
            gdbl *d;
            if (tgt & kRhsBit) {
                d = &L.rhs[idx];
            } else if (tgt & (kCBit | kQBit)) {
                if (!tran) continue;
                d = (tgt & kQBit) ? &L.q[idx] : &L.cq[idx];
            } else {
                d = &M[amap ? amap[tgt] : tgt];
            }
            double acc = *d;
            const uint32_t cc1 = rt_cell[k + 1];
            for (uint32_t cc = rt_cell[k]; cc < cc1; cc++) acc = acc + st[cells[cc]];
            *d = acc;
        }
        __syncthreads();
    }
    if (tid == 0) {
        const uint32_t d0 = amap ? amap[dp.diag0_slot] : dp.diag0_slot;
        M[d0] = M[d0] + 1.0;
        L.rhs[0] = L.rhs[0] + x[0];
    }
    __syncthreads();
    if (!tran) return;
    gcu32 *cslot_pat = gptr(dp.cslot_pat);
    for (uint32_t k = tid; k < dp.n_cslot; k += kT * kWave) {
        const uint32_t sl = amap ? amap[cslot_pat[k]] : cslot_pat[k];
        M[sl] = M[sl] + ag0 * L.cq[k];
    }
    for (uint32_t i = tid; i < n; i += kT * kWave) {
        const double d = ag0 * (L.q[i] - q1[i]);
        const double base = L.rhs[i] + d;
        L.rhs[i] = base - ag1 * ip[i];
    }
    __syncthreads();
}

// Batched moves between HBM and LDS: each thread issues kBatch independent
// loads before it uses any, so a wavefront has up to 8 x 64 loads in flight
// (a wavefront alone 16 x 64) instead of waiting on each.
template <uint32_t kT>
constexpr uint32_t kBatch = kT == 1 ? 16 : 8;

// dst[j] = src[idx[j]] for j < count (LDS from HBM through an index list).
// Pipelined: the next batch's indices load while this batch's values do, so
// a batch costs one memory latency, not two.
template <uint32_t kT>
__device__ inline void gather(ldbl *dst, gcdbl *src, gcu32 *idx, uint32_t count, uint32_t tid)
{
    uint32_t id[kBatch<kT>];
#pragma unroll
    for (uint32_t u = 0; u < kBatch<kT>; u++) {
        const uint32_t j = u * kT * kWave + tid;
        id[u] = idx[j < count ? j : 0];
    }
    for (uint32_t j0 = 0; j0 < count; j0 += kBatch<kT> * kT * kWave) {
        double v[kBatch<kT>];
#pragma unroll
        for (uint32_t u = 0; u < kBatch<kT>; u++) v[u] = src[id[u]];
        const uint32_t j1 = j0 + kBatch<kT> * kT * kWave;
#pragma unroll
        for (uint32_t u = 0; u < kBatch<kT>; u++) {
            const uint32_t j = j1 + u * kT * kWave + tid;
            id[u] = idx[j < count ? j : 0];
        }
#pragma unroll
        for (uint32_t u = 0; u < kBatch<kT>; u++) {
            const uint32_t j = j0 + u * kT * kWave + tid;
            if (j < count) dst[j] = v[u];
        }
    }
}

// dst[idx[j]] = src[j] for j < count (HBM from LDS through an index list).
template <uint32_t kT>
__device__ inline void scatter(gdbl *dst, gcu32 *idx, const ldbl *src, uint32_t count, uint32_t tid)
{
    for (uint32_t j0 = 0; j0 < count; j0 += kBatch<kT> * kT * kWave) {
        uint32_t id[kBatch<kT>];
#pragma unroll
        for (uint32_t u = 0; u < kBatch<kT>; u++) {
            const uint32_t j = j0 + u * kT * kWave + tid;
            id[u] = idx[j < count ? j : 0];
        }
#pragma unroll
        for (uint32_t u = 0; u < kBatch<kT>; u++) {
            const uint32_t j = j0 + u * kT * kWave + tid;
            if (j < count) dst[id[u]] = src[j];
        }
    }
}

// Between two rows: the team's LDS writes are done and seen.
__device__ inline void row_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// run_rows for a team: rows of kT * kWave words, a barrier between rows
// (a row reads what other wavefronts wrote in earlier rows).
template <uint32_t kT, typename WP>
__device__ void run_rows_team(WP words, uint32_t rows, ldbl *M, double growth, LuFlags &f, uint32_t tid)
{
    const uint32_t base = (uint32_t)(uintptr_t)M;
    WP w = words + tid;
    uint2_t q[kRing];
#pragma unroll
    for (int k = 0; k < kRing; k++) {
        q[k] = uint2_t{w[k * kT * kWave].x, w[k * kT * kWave].y};
        __builtin_amdgcn_sched_barrier(0);
    }
    RowOp o = row_decode<double, false, false>(q[0], base);
    for (uint32_t row = 0; row < rows; row += kRing) {
        w += kRing * kT * kWave;
#pragma unroll
        for (int k = 0; k < kRing; k++) {
            const double v = *(ldbl *)(uintptr_t)o.d, A = *(ldbl *)(uintptr_t)o.b, B = *(ldbl *)(uintptr_t)o.c;
            const RowOp cur = o;
            __builtin_amdgcn_sched_barrier(0);
            q[k] = uint2_t{w[k * kT * kWave].x, w[k * kT * kWave].y};
            o = row_decode<double, false, false>(q[(k + 1) % kRing], base);
            __builtin_amdgcn_sched_barrier(0);
            row_finish<double, false, false>(cur, v, A, B, growth, f);
            row_sync();
        }
    }
}

// The replay on the lane's slots in HBM: void pivots set to 1, the blocks
// (gather into LDS, rows, scatter), then the peel tests of refactor(). True
// when the lane must re-pivot.
template <uint32_t kT>
__device__ bool big_refactor(const TapeProg &T, uint32_t n, gdbl *tv, const BigLane &L, uint32_t tid)
{
    ldbl *M = L.sm;
    gcu32 *flags = gptr(T.flags), *amap = gptr(T.amap), *void_slots = gptr(T.void_slots);
    LuFlags f{false, 0, 0};
    for (uint32_t v = tid; v < T.n_void; v += kT * kWave) f.bad |= tv[amap[void_slots[v]]] != 0.0;
    // a void column's own diagonal is among the void slots: every wavefront
    // has read it before any sets it
    if (T.n_void) __syncthreads();
    for (uint32_t k = tid; k < n; k += kT * kWave)
        if (flags[k] & kVoidBit) tv[T.n_u + k] = 1.0;
    __syncthreads();
    const __attribute__((address_space(1))) BigBlock *blk = gptr(T.blk);
    for (uint32_t b = 0; b < T.n_blk; b++) {
        const uint32_t m = uni(blk[b].m), w = uni(blk[b].w), rows = uni(blk[b].rows), row0 = uni(blk[b].row0);
        gcu32 *sl = gptr(T.blk_slots) + uni(blk[b].slot_off);
        gather<kT>(M, tv, sl, m, tid);
        __syncthreads();
        const auto words = gptr(T.blk_words) + (size_t)row0 * kT * kWave;
        if constexpr (kT == 1) {
            run_rows<double>(words, rows, M, T.growth, f, tid, 0u);
            wsync();
        } else {
            run_rows_team<kT>(words, rows, M, T.growth, f, tid);
        }
        scatter<kT>(tv, sl, M, w, tid);
        __syncthreads();
    }
    for (uint32_t p = tid; p < T.n_u; p += kT * kWave) {
        const double u = tv[p];
        f.nonfinite |= dbits(u - u);
    }
    for (uint32_t k = tid; k < n; k += kT * kWave) {
        if (flags[k] & kVoidBit) continue;
        const double d = tv[T.n_u + k];
        f.bad |= d == 0.0 || !(fabs(d) < __builtin_inf());
    }
    const uint64_t worst = team_max_u64<kT>(f.worst, L.scratch);
    const bool fail = f.bad || f.nonfinite != 0 || !(bitsd(worst) <= T.wide);
    return team_any<kT>(fail, L.scratch);
}

// dx = -A^-1 rhs into y (LDS, pivot order; row i's dx is y[qinv[i]]): the
// tape's solve program. A word and, kAhead rows later, the factor entry it
// names are read ahead of their row, so a row costs its LDS round trip on
// the solve vector and a barrier (every row's terms in the order of
// lane_kernels.zig:123-143, with its zero skip).
template <uint32_t kT>
__device__ void big_solve(const TapeProg &T, uint32_t n, gcdbl *tv, gcdbl *rhs, ldbl *y, uint32_t tid)
{
    constexpr int kAhead = kRing / 2;
    gcu32 *pinv = gptr(T.pinv);
    for (uint32_t r = tid; r < n; r += kT * kWave) y[pinv[r]] = -rhs[r];
    y[n + tid] = 0.0;   // the pads
    const __attribute__((address_space(1))) uint2_t *w = gptr(T.sol_w) + tid;
    uint2_t q[kRing];
    double a[kAhead];
#pragma unroll
    for (int k = 0; k < kRing; k++) {
        q[k] = uint2_t{w[k * kT * kWave].x, w[k * kT * kWave].y};
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int k = 0; k < kAhead; k++) a[k] = tv[q[k].y & ~kSolDiv];
    __syncthreads();
    for (uint32_t row = 0; row < T.sol_rows; row += kRing) {
        w += kRing * kT * kWave;
#pragma unroll
        for (int k = 0; k < kRing; k++) {
            const uint32_t x = q[k].x, kind = uni(q[k].y) & kSolDiv;
            const uint32_t d = x & 0xffffu;
            const double v = y[d], B = y[x >> 16], A = a[k % kAhead];
            __builtin_amdgcn_sched_barrier(0);
            // row + k + kAhead's entry, row + k + kRing's word
            a[k % kAhead] = tv[q[(k + kAhead) % kRing].y & ~kSolDiv];
            q[k] = uint2_t{w[k * kT * kWave].x, w[k * kT * kWave].y};
            __builtin_amdgcn_sched_barrier(0);
            const double m = A * B;
            double r = B != 0.0 ? v - m : v;
            if (kind) {
                double piv = A;
                pin(piv);   // a branch: every row would pay for a speculated division
                r = v / piv;
            }
            y[d] = r;
            // (a wavefront's own LDS accesses complete in issue order)
            if constexpr (kT > 1) row_sync();
            else __builtin_amdgcn_wave_barrier();
        }
    }
}

// The plausible limit of a Newton run's first iterate (converger.zig:377-384).
template <uint32_t kT>
__device__ inline double big_limit_at(const TapeProg &T, uint32_t n, const BigLane &L, uint32_t tid)
{
    gcu32 *diag_tv = gptr(T.diag_tv);
    gcdbl *tv = L.tv, *x = L.x, *rhs = L.rhs;
    double gm = 1.0;
    uint64_t xm = 0, fm = 0;
    for (uint32_t i = tid; i < n; i += kT * kWave) {
        gm = fmax(gm, fabs(tv[diag_tv[i]]));
        const uint64_t xb = dbits(fabs(x[i])), fb = dbits(fabs(rhs[i]));
        xm = xb > xm ? xb : xm;
        fm = fb > fm ? fb : fm;
    }
    // gm >= 1: fmax drops a NaN, and non-negative doubles order as their bits
    gm = bitsd(team_max_u64<kT>(dbits(gm), L.scratch));
    xm = team_max_u64<kT>(xm, L.scratch);
    fm = team_max_u64<kT>(fm, L.scratch);
    const double scale = fmin(fmax(bitsd(xm), bitsd(fm) * gm), 1e18);
    return !(1e3 * scale > 1e9) ? 1e9 : 1e3 * scale;
}

// x += dx (dx = y[qinv[i]]), x_old kept; returns the largest scaled update
// (converger.zig:794-819).
template <uint32_t kT>
__device__ inline double big_update(const OpArgs &a, const TapeProg &T, const BigLane &L, uint32_t tid)
{
    const DeckProg &dp = a.dp;
    const ldbl *y = L.sm;
    gcu32 *qinv = gptr(T.qinv);
    const __attribute__((address_space(1))) uint8_t *current_row = gptr(dp.current_row);
    uint64_t worst = 0;
    for (uint32_t i = tid; i < dp.n; i += kT * kWave) {
        const double xo = L.x[i];
        const double d = y[qinv[i]];
        const double xn = xo + d;
        L.xold[i] = xo;
        L.x[i] = xn;
        const double tl = a.reltol * fmax(fabs(xn), fabs(xo)) + (current_row[i] ? a.abstol : a.vntol);
        const bool finite = fabs(xn) < __builtin_inf() && fabs(d) < __builtin_inf();
        const double qq = fabs(d) / tl;
        const double score = !finite ? __builtin_inf() : (qq == qq ? qq : 0.0);
        const uint64_t sb = dbits(score);
        worst = sb > worst ? sb : worst;
    }
    return bitsd(team_max_u64<kT>(worst, L.scratch));
}

// Limiting after an update (MOS1, diodes, BJTs): true when any limited.
template <uint32_t kT>
__device__ __forceinline__ bool big_limit(const DeckProg &dp, const double *live, const BigLane &L, double *lim,
                                          uint32_t tid)
{
    return team_any<kT>(limit_pass<kT * kWave>(dp, live, (gcdbl *)L.x, lim, tid), L.scratch);
}

// One lane's operating point (op_lane's FP64 path: cold, given or resumed
// start; dump: the Jacobian and residual at the start or saved iterate into
// row g of a_out and f_out).
template <uint32_t kT>
__device__ __forceinline__ void big_op_lane(const BigArgs &b, uint32_t g, uint32_t lane, ldbl *sm)
{
    const OpArgs &a = b.ta.op;
    const uint32_t tid = threadIdx.x;
    const DeckProg &dp = a.dp;
    const uint32_t n = dp.n;
    const BigLane L = big_lane<kT>(b, g, sm);
    const double *live = a.live + (size_t)lane * dp.n_live;
    double *lim = a.lim + (size_t)lane * lim_width(dp);
    gdbl *xg = gptr(a.x) + (size_t)lane * n;
    lane_init<kT * kWave>(a, lane, live, (double *)L.x, lim, tid);
    __syncthreads();
    if (a.dump) {
        big_assemble<kT>(b, nullptr, dp.nnz, live, L.x, lim, gptr(a.a_out) + (size_t)g * dp.nnz, L, false, 0.0, 0.0,
                     0.0, nullptr, nullptr, tid);
        gdbl *f = gptr(a.f_out) + (size_t)g * n;
        for (uint32_t i = tid; i < n; i += kT * kWave) f[i] = L.rhs[i];
        return;
    }
    const LaneResume rs = a.resume[lane];
    const TapeProg T = a.tapes[rs.tape];
    uint32_t iter0 = 0, k0 = 0;
    bool init_fix = a.mode == 0;
    double limit = 1e9;
    if (a.mode == 2) {
        iter0 = rs.iter;
        init_fix = rs.init_fix != 0;
        limit = rs.limit;
        k0 = rs.k0;
    }
    uint32_t status = kNoConvergence, iters = a.max_iter;
    unsigned long long pc[kProfPhases] = {};
    unsigned long long tc = clock64();
    auto lap = [&](int ph) {
        if (a.prof) {
            const unsigned long long now = clock64();
            pc[ph] += now - tc;
            tc = now;
        }
    };
    uint32_t iter = iter0;
    for (; iter - k0 < a.max_iter; iter++) {
        lap(3);
        big_assemble<kT>(b, T.amap, T.n_tv, live, L.x, lim, L.tv, L, false, 0.0, 0.0, 0.0, nullptr, nullptr, tid);
        if (iter == k0) limit = big_limit_at<kT>(T, n, L, tid);
        for (uint32_t i = tid; i < n; i += kT * kWave) L.sdiag[i] = L.tv[T.diag_tv[i]];
        __syncthreads();
        lap(0);
        const bool repivot = big_refactor<kT>(T, n, L.tv, L, tid);
        lap(1);
        if (repivot) {
            for (uint32_t i = tid; i < n; i += kT * kWave) xg[i] = L.x[i];
            if (tid == 0) {
                LaneResume o{};
                o.iter = iter;
                o.init_fix = init_fix ? 1u : 0u;
                o.tape = rs.tape;
                o.limit = limit;
                o.k0 = k0;
                a.resume[lane] = o;
            }
            if (a.a_out) {
                // the Jacobian at this iterate (pattern order) for the host's
                // re-pivot: the same sums as the failed assembly
                __syncthreads();
                big_assemble<kT>(b, nullptr, dp.nnz, live, L.x, lim, gptr(a.a_out) + (size_t)lane * dp.nnz, L, false,
                             0.0, 0.0, 0.0, nullptr, nullptr, tid);
            }
            status = kRepivot;
            iters = iter;
            break;
        }
        big_solve<kT>(T, n, L.tv, L.rhs, L.sm, tid);
        __syncthreads();
        lap(2);
        const double scaled = big_update<kT>(a, T, L, tid);
        __syncthreads();
        const bool limited = big_limit<kT>(dp, live, L, lim, tid);
        bool ok = !limited && iter != k0 && scaled < 1.0;
        if (ok) {
            bool miss = false;
            for (uint32_t i = tid; i < n; i += kT * kWave) {
                const double xi = L.x[i];
                miss |= !(fabs(xi) <= limit);
                const double s0 = fabs(L.sdiag[i]);
                const double s = s0 == 0.0 ? 1.0 : s0;
                const double rt = fmax(a.residual_tol, 10.0 * s * (a.reltol * fabs(xi) + a.vntol));
                miss |= !(fabs(L.rhs[i]) <= rt);
            }
            ok = !team_any<kT>(miss, L.scratch);
        }
        if (ok && init_fix) {
            init_fix = false;
        } else if (ok) {
            for (uint32_t i = tid; i < n; i += kT * kWave) L.x[i] = L.xold[i];
            status = kConverged;
            iters = iter + 1;
            break;
        }
        __syncthreads();
    }
    if (status == kNoConvergence) iters = iter;
    __syncthreads();
    if (status != kRepivot)
        for (uint32_t i = tid; i < n; i += kT * kWave) xg[i] = L.x[i];
    lap(3);
    if (tid == 0) {
        a.status[lane] = status;
        a.iterations[lane] = iters;
        if (a.prof)
            for (int p = 0; p < kProfPhases; p++) a.prof[(size_t)lane * kProfPhases + p] += pc[p];
    }
}

// Transient steps [s0, s1) of one lane (tran_lane's FP64 path: companion,
// Newton with the transient gates, acceptance, probes and predictor; a lane
// whose replay fails leaves its Jacobian in its row of a_out and resumes at
// the same iterate; dump: the first step's first Jacobian into that row).
template <uint32_t kT>
__device__ __forceinline__ void big_tran_lane(const BigArgs &b, uint32_t g, uint32_t lane, ldbl *sm)
{
    const TranArgs &ta = b.ta;
    const OpArgs &a = ta.op;
    const uint32_t tid = threadIdx.x;
    if (a.status[lane] != kTranRunning) return;
    uint32_t s = ta.step[lane];
    if (s >= ta.s1) return;
    if (s < ta.s0) s = ta.s0;
    const DeckProg &dp = a.dp;
    const uint32_t n = dp.n;
    const BigLane L = big_lane<kT>(b, g, sm);
    const double *live = a.live + (size_t)lane * dp.n_live;
    double *lim = a.lim + (size_t)lane * lim_width(dp);
    gdbl *q1 = gptr(ta.q1) + (size_t)lane * n;
    gdbl *ip = gptr(ta.ip) + (size_t)lane * n;
    gdbl *xp = gptr(ta.xp) + (size_t)lane * n;
    gdbl *xg = gptr(a.x) + (size_t)lane * n;
    const LaneResume rs = a.resume[lane];
    const TapeProg T = a.tapes[rs.tape];
    gdbl *aout = gptr(a.a_out) + (size_t)lane * dp.nnz;
    gcu32 *amap = gptr(T.amap);
    for (uint32_t i = tid; i < n; i += kT * kWave) L.x[i] = xg[i];
    __syncthreads();
    if (ta.init) {
        // start at the operating point: limiting state at its own voltages,
        // charges from one evaluation there, no dynamic current
        seed_lim_at<kT * kWave>(dp, live, (const double *)L.x, lim, tid);
        for (uint32_t i = tid; i < n; i += kT * kWave) {
            q1[i] = 0.0;
            ip[i] = 0.0;
            xp[i] = L.x[i];
        }
        __syncthreads();
        big_assemble<kT>(b, T.amap, T.n_tv, live, L.x, lim, L.tv, L, true, 0.0, 0.0, 0.0, q1, ip, tid);
        for (uint32_t i = tid; i < n; i += kT * kWave) q1[i] = L.q[i];
        __syncthreads();
        if (ta.dump) {
            big_assemble<kT>(b, nullptr, dp.nnz, live, L.x, lim, aout, L, true, ta.dt, 1.0 / ta.dt, 0.0, q1, ip, tid);
            return;
        }
    }
    __syncthreads();
    uint32_t iter0 = rs.iter;   // nonzero only when resuming inside a step
    double limit = rs.limit;
    uint32_t status = kTranRunning;
    uint32_t total_it = a.iterations[lane];
    unsigned long long pc[kProfPhases] = {};
    unsigned long long tc = clock64();
    auto lap = [&](int ph) {
        if (a.prof) {
            const unsigned long long now = clock64();
            pc[ph] += now - tc;
            tc = now;
        }
    };
    for (; s < ta.s1 && status == kTranRunning; s++) {
        const double t = (double)(s + 1) * ta.dt;
        const double ag0 = s == 0 ? 1.0 / ta.dt : 2.0 / ta.dt;
        const double ag1 = s == 0 ? 0.0 : 1.0;
        bool converged = false;
        uint32_t iter = iter0;
        for (; iter < a.max_iter; iter++) {
            lap(3);
            big_assemble<kT>(b, T.amap, T.n_tv, live, L.x, lim, L.tv, L, true, t, ag0, ag1, q1, ip, tid);
            if (iter == 0) limit = big_limit_at<kT>(T, n, L, tid);
            __syncthreads();
            lap(0);
            const bool repivot = big_refactor<kT>(T, n, L.tv, L, tid);
            lap(1);
            if (repivot) {
                // the Jacobian again, read out in pattern order for the
                // host's re-pivot; resume at this iterate
                __syncthreads();
                big_assemble<kT>(b, T.amap, T.n_tv, live, L.x, lim, L.tv, L, true, t, ag0, ag1, q1, ip, tid);
                for (uint32_t p = tid; p < dp.nnz; p += kT * kWave) aout[p] = L.tv[amap[p]];
                if (tid == 0) {
                    LaneResume o = rs;
                    o.iter = iter;
                    o.limit = limit;
                    o.fresh = 0;
                    a.resume[lane] = o;
                }
                status = kRepivot;
                break;
            }
            big_solve<kT>(T, n, L.tv, L.rhs, L.sm, tid);
            __syncthreads();
            lap(2);
            const double scaled = big_update<kT>(a, T, L, tid);
            __syncthreads();
            const bool limited = big_limit<kT>(dp, live, L, lim, tid);
            bool ok = !limited && iter != 0 && scaled < 1.0;
            if (ok) {
                bool miss = false;
                for (uint32_t i = tid; i < n; i += kT * kWave) {
                    miss |= !(fabs(L.x[i]) <= limit);
                    miss |= !(fabs(L.rhs[i]) <= __builtin_inf());
                }
                ok = !team_any<kT>(miss, L.scratch);
            }
            __syncthreads();
            if (ok) {
                for (uint32_t i = tid; i < n; i += kT * kWave) L.x[i] = L.xold[i];
                converged = true;
                iter++;
                break;
            }
        }
        total_it += iter - iter0;
        if (status == kRepivot) break;
        iter0 = 0;
        if (!converged) {
            status = kNoConvergence;
            break;
        }
        // accept: q holds the charges of the converged point (the last
        // assembly ran at x_old)
        __syncthreads();
        for (uint32_t i = tid; i < n; i += kT * kWave) {
            const double d = ag0 * (L.q[i] - q1[i]);
            ip[i] = d - ag1 * ip[i];
            q1[i] = L.q[i];
        }
        for (uint32_t k = tid; k < ta.n_probes; k += kT * kWave)
            ta.probes[((size_t)lane * ta.steps + s) * ta.n_probes + k] = L.x[ta.probe_ids[k]];
        __syncthreads();
        seed_lim_at<kT * kWave>(dp, live, (const double *)L.x, lim, tid, true);
        __syncthreads();
        // the next step's first iterate: the last two accepted points
        // extrapolated (tran.zig:1131-1137; lane_device.zig:141-153), then
        // one limit pass against the accepted point (tran.zig:1138)
        if (s + 1 < ta.steps) {
            for (uint32_t i = tid; i < n; i += kT * kWave) {
                const double cu = L.x[i];
                L.x[i] = cu + (cu - xp[i]);
                xp[i] = cu;
            }
            __syncthreads();
            limit_pass<kT * kWave>(dp, live, (gcdbl *)L.x, lim, tid);
            __syncthreads();
        }
    }
    lap(3);
    if (status == kTranRunning && s >= ta.steps) status = kConverged;
    for (uint32_t i = tid; i < n; i += kT * kWave) xg[i] = L.x[i];
    if (tid == 0) {
        if (status != kRepivot) {
            LaneResume o = rs;
            o.iter = 0;
            a.resume[lane] = o;
        }
        ta.step[lane] = s;
        a.status[lane] = status;
        a.iterations[lane] = total_it;
        if (a.prof)
            for (int p = 0; p < kProfPhases; p++) a.prof[(size_t)lane * kProfPhases + p] += pc[p];
    }
}

// One workgroup per lane: the lanes walk the same tape nearly in step, so
// the lanes of an XCD share their words' fetches in its L2.
template <uint32_t kT>
__global__ __launch_bounds__(kT * kWave) void big_lanes(BigArgs b)
{
    const uint32_t g = blockIdx.x;
    const uint32_t lane = uni(b.ta.op.lane_ids[g]);
    extern __shared__ double dyn[];
    ldbl *sm = lptr(dyn);
    if (b.tran) big_tran_lane<kT>(b, g, lane, sm);
    else big_op_lane<kT>(b, g, lane, sm);
}

}  // namespace esl

// Sets the kernel's dynamic LDS limit (before launches, outside graph capture).
extern "C" hipError_t esl_big_attrs(uint32_t team, uint32_t lds_bytes)
{
    const void *f = team == 1 ? (const void *)esl::big_lanes<1> : (const void *)esl::big_lanes<esl::kTeam>;
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(lds_bytes > 65536 ? lds_bytes : 65536));
}

extern "C" hipError_t esl_launch_big(const esl::BigArgs *b, hipStream_t s)
{
    const uint32_t lds = b->lds * (uint32_t)sizeof(double);
    if (b->team == 1) hipLaunchKernelGGL(esl::big_lanes<1>, dim3(b->N), dim3(esl::kWave), lds, s, *b);
    else if (b->team == esl::kTeam)
        hipLaunchKernelGGL(esl::big_lanes<esl::kTeam>, dim3(b->N), dim3(esl::kTeam * esl::kWave), lds, s, *b);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
