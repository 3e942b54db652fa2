// pbb_explorer.h -- the explorer: one IVM branch-and-bound search per
// 64-lane wavefront (navigation, bounding, branching, pruning, interval
// sharing), shared by the one-instance engine kernels (pbb_kernels.hip) and
// the multi-instance pool kernel (pbb_pool.hip).  Device code only; every
// function is force-inlined into the kernels that use it.
#pragma once

#include <utility>

#include "pbb_device.h"
#include "pbb_kernels.h"

namespace pbb {

// ------------------------------------------------------------------ atomics
// Every helper takes the memory scope of the explorers that share the
// words: the agent for a launch over the device, the workgroup for a team
// of explorers in one workgroup (whose release/acquire then need no L2
// writeback or invalidate).
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ int ld_rlx(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, S);
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ unsigned ld_rlx(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, S);
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ unsigned long long ld_rlx(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, S);
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ void st_rel(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, S);
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ void st_rlx(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, S);
}

// lane-0 read-modify-writes, result broadcast to the wavefront
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ int w_add(int *p, int v)
{
    int r = 0;
    if (lane_id() == 0) r = __hip_atomic_fetch_add(p, v, __ATOMIC_ACQ_REL, S);
    return rdlane(r, 0);
}
// Relaxed counters: on this multi-XCD device an agent-scope release writes
// back the wave's L2 and an acquire invalidates it, so the idle mask and the
// work counter, whose values carry no other data, take no fence.
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ void st_rlx64(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, S);
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ unsigned long long w_add64(unsigned long long *p, unsigned long long v)
{
    unsigned long long r = 0;
    if (lane_id() == 0) r = __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, S);
    unsigned lo = (unsigned)rdlane((int)(unsigned)r, 0);
    unsigned hi = (unsigned)rdlane((int)(unsigned)(r >> 32), 0);
    return ((unsigned long long)hi << 32) | lo;
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ bool w_cas(unsigned *p, unsigned expect, unsigned desired)
{
    int ok = 0;
    if (lane_id() == 0) {
        unsigned e = expect;
        ok = __hip_atomic_compare_exchange_strong(p, &e, desired, __ATOMIC_ACQ_REL, __ATOMIC_RELAXED,
                                                  S);
    }
    return rdlane(ok, 0) != 0;
}
template <int S = __HIP_MEMORY_SCOPE_AGENT>
__device__ __forceinline__ void w_min64(unsigned long long *p, unsigned long long v)
{
    if (lane_id() == 0) __hip_atomic_fetch_min(p, v, __ATOMIC_ACQ_REL, S);
}

// ------------------------------------------------------------ LDS layout
struct Lds {
    int *pm;        // [m][PM_STRIDE] machine-major processing times
    int *pmR;       // the same rows, machines reversed: pmR[q] = pm[m-1-q]
    int ps;         // row stride of pm (PM_STRIDE)
    int *minA, *minD, *tot;
    unsigned *jtabL;    // Johnson table staged in LDS (valid when jtl)
    const void *jtabG;  // the table in global memory
    bool jtl, jpacked;
    int nch;        // chunks of 64 pairs (jtwalk)
    bool jtwalk;    // jtabL holds lb2_walk's words (up to 32 jobs)
    int8_t *mat;    // this wave's IVM matrix, row l at mat + lds_mat_row(l, n)
    int *stk;       // this wave's stacks: F entry s at row s, B entry s at row n-s ((n+1) x m)
    int2 *U;        // this wave's LB1 operand block [2][m]
    int *scr;       // this wave's scratch (64 ints; LB2 variant only)
    int2 *sink;     // this wave's 64 int2 where the lanes past a row store: the
                    // row stores of the node loop then need no exec-mask branch
                    // (2066 against 2100-2104 M nodes/s at 50x20)
};

// lb2_walk's table from the one in global memory, by the whole workgroup: a thread
// per column (the columns past the last pair repeat it), a second pass for the
// places.
template <bool WIDE, class Src, class Entry>
__device__ __forceinline__ void stage_walk(const Src *src, Entry *tab, int n, int npairs, int nch)
{
    const int width = 64 * nch;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        const Src *s = src + min(c, npairs - 1);
#pragma unroll 4
        for (int i = 0; i < n; i++) tab[i * width + c] = JWalk<WIDE>::make(s[i * npairs]);
#pragma unroll 4
        for (int i = 0; i < n; i++) {
            unsigned job;
            if constexpr (WIDE) job = (unsigned)s[i * npairs].y & 63u;
            else job = s[i * npairs] & 63u;
            atomicOr((unsigned *)(tab + (int)job * width + c), (unsigned)i << JWalk<WIDE>::PLACE);
        }
    }
}

// jt: bytes set aside for a Johnson table; an instance's is staged if it fits
template <int TAB>
__device__ __forceinline__ Lds lds_setup(const DevInst &I, char *smem, int jt, bool scratch)
{
    Lds L;
    const int n = I.n, mp = I.mp, m = I.m;
    L.ps = PM_STRIDE;
    L.pm = (int *)smem;
    L.pmR = L.pm + m * PM_STRIDE;
    L.minA = L.pmR + m * PM_STRIDE;
    L.minD = L.minA + mp;
    L.tot = L.minD + mp;
    const bool packed = TAB == TAB_PACKED || (TAB == TAB_ANY && I.jpacked);
    const bool walk = n <= 32 && (TAB != TAB_ANY || packed);
    const int bytes = TAB != TAB_ANY || packed ? jtab_lds_bytes(n, I.npairs, packed) : n * I.npairs * 8;
    const bool load_jtab = jt > 0 && bytes <= jt;
    L.jtabL = (unsigned *)(smem + lds_table_bytes(m, 0));
    L.jpacked = packed;
    L.jtabG = I.jtab;
    L.jtl = load_jtab;
    L.nch = jtab_chunks(I.npairs);
    L.jtwalk = load_jtab && walk;
    char *wbase = smem + lds_table_bytes(m, jt) +
                  (size_t)(threadIdx.x >> 6) * lds_wave_bytes(n, m, scratch);
    L.mat = (int8_t *)wbase;
    L.stk = (int *)(wbase + lds_mat_bytes(n));
    L.U = (int2 *)(wbase + lds_mat_bytes(n) + lds_stack_bytes(n, m));
    L.scr = scratch ? (int *)(wbase + lds_mat_bytes(n) + lds_stack_bytes(n, m) + (size_t)m * 16) : nullptr;
    L.sink = (int2 *)(wbase + lds_mat_bytes(n) + lds_stack_bytes(n, m) + (size_t)m * 16 + (scratch ? 64 * 4 : 0));
    for (int i = threadIdx.x; i < n * m; i += blockDim.x) {
        const int q = i / n, j = i - q * n;
        L.pm[q * PM_STRIDE + j] = I.ptm[i];
        L.pmR[(m - 1 - q) * PM_STRIDE + j] = I.ptm[i];
    }
    for (int i = threadIdx.x; i < mp; i += blockDim.x) {
        L.minA[i] = i < m ? I.min_arr[i] : 0;
        L.minD[i] = i < m ? I.min_dep[i] : 0;
        int s = 0;
        if (i < m)
            for (int j = 0; j < n; j++) s += I.ptm[i * n + j];
        L.tot[i] = s;
    }
    if (L.jtwalk) {
        if constexpr (TAB == TAB_WIDE) stage_walk<true>((const int2 *)I.jtab, (int2 *)L.jtabL, n, I.npairs, L.nch);
        else stage_walk<false>((const unsigned *)I.jtab, L.jtabL, n, I.npairs, L.nch);
    } else if (load_jtab) {
        const int words = I.npairs * n * (packed ? 1 : 2);
#pragma unroll 4
        for (int i = threadIdx.x; i < words; i += blockDim.x) L.jtabL[i] = ((const unsigned *)I.jtab)[i];
    }
    __syncthreads();
    return L;
}

// NEH (heuristic/src/fastNEH.cpp:151-243, with the intended partial
// makespan at every insertion position): one wavefront.  Jobs get stable
// ranks by decreasing total time; then job k is inserted into the first k
// at the first position of least partial makespan (lane = position, each
// lane evaluates its candidate sequence on M machines).  The first-minimum
// rule also settles the first two jobs as fastNEH.cpp:233-236 does (the
// original order only when strictly better).  pm: [M][ps] machine-major;
// seq: n ints of the wave's LDS, receives the order.  Returns the makespan.
template <int M>
__device__ __forceinline__ int neh_wave(const int *pm, int ps, int n, int *seq)
{
    const int lane = lane_id();
    int tot = 0;
    if (lane < n)
#pragma unroll
        for (int q = 0; q < M; q++) tot += pm[q * ps + lane];
    int rank = 0;
    for (int i = 0; i < n; i++) {
        const int ti = rdlane(tot, i);
        rank += (ti > tot || (ti == tot && i < lane)) ? 1 : 0;
    }
    if (lane < n) seq[rank] = lane;
    __builtin_amdgcn_wave_barrier();
    int cmin = 0;
    if (n == 1) {
        int c = 0;
#pragma unroll
        for (int q = 0; q < M; q++) c += pm[q * ps + seq[0]];
        return c;
    }
    for (int k = 1; k < n; k++) {
        const int job = seq[k];
        int cost = 0x7fffffff;
        if (lane <= k) {
            int cv[M];
#pragma unroll
            for (int q = 0; q < M; q++) cv[q] = 0;
            for (int i = 0; i <= k; i++) {
                const int j = i < lane ? seq[i] : (i == lane ? job : seq[i - 1]);
                cv[0] += pm[j];
#pragma unroll
                for (int q = 1; q < M; q++) cv[q] = max(cv[q - 1], cv[q]) + pm[q * ps + j];
            }
            cost = cv[M - 1];
        }
        cmin = wave_min(cost);
        const int pb = __ffsll((unsigned long long)ballot(lane <= k && cost == cmin)) - 1;
        const int v = lane < n ? seq[lane] : 0;
        const int vprev = shfl(v, lane > 0 ? lane - 1 : 0);
        __builtin_amdgcn_wave_barrier();
        if (lane == pb) seq[lane] = job;
        else if (lane > pb && lane <= k) seq[lane] = vprev;
        __builtin_amdgcn_wave_barrier();
    }
    return cmin;
}

// instance reference of the one-instance engine: everything from the
// kernel arguments
__device__ __forceinline__ InstRef engine_inst(const KArgs &a)
{
    InstRef r;
    r.ctl = a.ctl;
    r.idle = a.idle;
    r.idle_words = a.idle_words;
    r.member = nullptr;
    r.occ = nullptr;
    r.ub0 = a.initial_ub;
    r.best = a.best;
    r.root_row = a.root_row;
    r.root_dir = a.root_dir;
    r.m = a.I.m;
    r.npairs = a.I.npairs;
    r.pairs_mode = a.pairs_mode;
    r.pair_ab = a.I.pair_ab;
    return r;
}

// ------------------------------------------------------------- explorer
// Stacks: F entry s (row s of stk) = completion times on every machine of
// the first s front jobs, F entry 0 = min_arr (the front of an empty prefix,
// bound_fsp_weak.cpp:67-70); B entry s (row n-s) = reverse completion times
// of the last s back jobs, B entry 0 = min_dep.  nf + nb < n, so the two
// never overlap.  A chain started from min_arr/min_dep equals one started
// from zero, since min_arr[q] never exceeds a single job's head (and min_dep
// its tail).
// REF: 0 LB1 only (boundingMode 0); 1 LB1 + LB1' refinement (boundingMode
// 1/2 as shipped); 2 LB1 + Johnson LB2 refinement.
template <int M, int REF, int SC = __HIP_MEMORY_SCOPE_AGENT, int TAB = TAB_ANY>
struct Explorer {
    static constexpr bool WIDE = TAB == TAB_WIDE;  // form of lb2_walk's table
    const KArgs &a;
    Lds lds;
    InstRef ir;   // the instance this explorer works on
    Ctl *run;     // stop / error words of the launch
    int n, mp, lane, e;
    int rows;     // row count of the HBM explorer state (>= n)
    int L;                            // current line
    int rowv, posv, endv, dirv, remv; // lane vectors (remv: lane q = remaining work on machine q)
    int nf, nb;
    uint64_t free_jobs;               // unscheduled jobs of the current path (REF 2)
    int ftop;                         // lane q < M: top front entry f_q (frow(nf)), else 0
    static constexpr int PCH = (M * (M - 1) / 2 + PBB_WAVE - 1) / PBB_WAVE;  // pair chunks (M >= 2)
    int pinfo[PCH];                   // this lane's Johnson machine pairs (REF 2)
    unsigned places[PCH];             // unscheduled jobs by their places in the pairs' orders (REF 2, lds.jtwalk)
    int local_best;
    unsigned dec, leaves, sb, jb;     // deltas since the last flush
    unsigned mtag;                    // lane i: tag of word i of the last message consumed
    int self;                         // this explorer's member index (bit self / words of word self % words)
    int pollw;                        // next idle word to poll
    int seen;                         // pool: the slot's member word as of the last poll
    unsigned nchk;                    // periodic checks so far (host-word phase)
    bool end_dirty;                   // end moved since pos was last compared with it
    int hist;                         // lane d: nodes decomposed at depth d since the flush
    int jhist;                        // lane d: refinement bounds at depth d (REF != 0)
    unsigned long long t_end;

    __device__ __forceinline__ Explorer(const KArgs &args, const Lds &l, int eid, const InstRef &r, Ctl *runctl,
                                        int n_, int mp_)
        : a(args), lds(l), ir(r), run(runctl), n(n_), mp(mp_), lane(lane_id()), e(eid), rows(args.rows)
    {
        L = 0;
        rowv = posv = endv = dirv = remv = 0;
        nf = nb = 0;
        ftop = 0;
        free_jobs = 0ull;
#pragma unroll
        for (int c = 0; c < PCH; c++) places[c] = 0u;
        if constexpr (REF == 2) pair_lanes<PCH>(r.pair_ab, r.npairs, r.m, r.pairs_mode, pinfo);
        dec = leaves = sb = jb = 0;
        mtag = 0;
        self = eid;
        pollw = seen = 0;
        nchk = (unsigned)eid;  // staggers the host-word reads across explorers
        end_dirty = true;
        hist = jhist = 0;
        local_best = PBB_INF;
        t_end = args.deadline ? wall_clock64() + args.deadline : 0ull;
    }

    __device__ __forceinline__ bool gt_best(int v) const
    {
        return a.find_all ? v > local_best : v >= local_best;
    }

    __device__ __forceinline__ int *frow(int s) const { return lds.stk + s * M; }
    __device__ __forceinline__ int *brow(int s) const { return lds.stk + (n - s) * M; }

    // lane q: p[q][job].  Lanes past the machines read machine M-1 and drop
    // it: an unconditional load, no exec-mask branch around it (as for the
    // other per-machine and per-cell loads of the node loop; 2044-2046
    // against 2068-2070 M nodes/s at 50x20).
    __device__ __forceinline__ int pmach(int job) const
    {
        const int v = lds.pm[(lane < M ? lane : M - 1) * PM_STRIDE + job];
        return lane < M ? v : 0;
    }

    __device__ __forceinline__ int walk_place(int at) const
    {
        return (int)((lds.jtabL[WIDE ? 2 * at : at] >> JWalk<WIDE>::PLACE) & 31u);
    }
    // job j's bit in the place masks: one LDS word per chunk, kept up along the
    // path (rebuilt for every node, it costs what the shorter walk saves)
    __device__ __forceinline__ unsigned place_bit(int c, int j) const
    {
        return 1u << walk_place((j * lds.nch + c) * 64 + lane);
    }
    template <bool ADD>
    __device__ __forceinline__ void mark_places(int j)
    {
        if (!lds.jtwalk) return;
#pragma unroll
        for (int c = 0; c < PCH; c++)
            if (c == 0 || c < lds.nch) {
                const unsigned b = place_bit(c, j);
                places[c] = ADD ? places[c] | b : places[c] & ~b;
            }
    }
    // all jobs unscheduled
    __device__ __forceinline__ void all_free()
    {
        free_jobs = lanes_below(n);
#pragma unroll
        for (int c = 0; c < PCH; c++) places[c] = (unsigned)free_jobs;
    }

    __device__ __forceinline__ void reset_stacks()
    {
        nf = nb = 0;
        ftop = lane < M ? lds.minA[lane] : 0;
        if (lane < M) {
            frow(0)[lane] = ftop;
            brow(0)[lane] = lds.minD[lane];
        }
        remv = lane < M ? lds.tot[lane] : 0;
        if constexpr (REF == 2) all_free();
        __builtin_amdgcn_wave_barrier();
    }

    // schedule job j in direction d: push a new F (d=0) or B (d=1) entry,
    // computed lane-parallel by chain_scan; remain -= p_j.
    __device__ __forceinline__ void push_job(int j, int d)
    {
        const int pk = pmach(j);
        if (d == 0) {
            int c = chain_scan(ftop, pk);
            *(lane < M ? frow(nf + 1) + lane : (int *)(lds.sink + lane)) = c;
            ftop = lane < M ? c : 0;
            nf++;
        } else {
            // back chain runs from machine M-1 down: lane q handles machine M-1-q
            const int qb = lane < M ? lane : M - 1;
            int base = brow(nb)[M - 1 - qb];
            int pr = lds.pmR[qb * PM_STRIDE + j];
            base = lane < M ? base : 0;
            pr = lane < M ? pr : 0;
            int c = chain_scan(base, pr);
            *(lane < M ? brow(nb + 1) + (M - 1 - lane) : (int *)(lds.sink + lane)) = c;
            nb++;
        }
        remv -= pk;
        if constexpr (REF == 2) {
            free_jobs &= ~(1ull << j);
            mark_places<false>(j);
        }
        __builtin_amdgcn_wave_barrier();
    }

    __device__ __forceinline__ void pop_job(int j, int d)
    {
        if (d == 0) {
            nf--;
            ftop = lane < M ? frow(nf)[lane] : 0;
        } else {
            nb--;
        }
        remv += pmach(j);
        if constexpr (REF == 2) {
            free_jobs |= 1ull << j;
            mark_places<true>(j);
        }
    }

    // ivm::beforeEnd (ivm.cpp:152-160): lexicographic pos <= end
    __device__ __forceinline__ bool before_end() const
    {
        const uint64_t in = lanes_below(n);
        uint64_t lt = in & ballot(posv < endv);
        uint64_t gt = in & ballot(posv > endv);
        uint64_t d = lt | gt;
        if (d == 0) return true;
        int f = __ffsll((unsigned long long)d) - 1;
        return (lt >> f) & 1ull;
    }

    // ------------------------------------------------------- LB1 children
    // bound_fsp_weak::addFrontAndBound / addBackAndBound (bound_fsp_weak.cpp:133-191)
    // for all children of the node, both directions in one pass: lane i < 32
    // bounds child base+i in the front direction, lane 32+i the same child in
    // the back direction.  The back recurrence run over machines M-1..0 has
    // the same form as the front one run over 0..M-1, so both halves execute
    // one loop:  t1 = max(x_q, t0); lb = max(lb, t1 + y_q); t0 = t1 + p_q,
    // with (x_q, y_q) = (front_q, remain_q + back_q) in the front half and
    // (back_{M-1-q}, front_{M-1-q} + remain_{M-1-q}) in the back half.
    // The per-wave operand block U holds the front half's pairs in machine
    // order, then the back half's.
    __device__ __forceinline__ void build_operands() const
    {
        const bool in = lane < M;
        const int f = ftop, b = brow(nb)[in ? lane : M - 1], r = remv;
        *(in ? lds.U + lane : lds.sink + lane) = make_int2(f, r + b);
        *(in ? lds.U + M + (M - 1 - lane) : lds.sink + lane) = make_int2(b, f + r);
        __builtin_amdgcn_wave_barrier();
    }

    // lane Q of every 16-lane row, to all lanes of the row (DPP row_newbcast,
    // folded into the instruction that uses it)
    template <int Q>
    __device__ __forceinline__ static int row_bcast_lane(int v)
    {
        return __builtin_amdgcn_update_dpp(0, v, 0x150 + (Q & 15), 0xF, 0xF, false);
    }

    // machine step Q of the fused pass; the step's operand pair is lane Q mod
    // 16 of the row's copy of U (A for Q < 16, A2 above)
    template <int Q>
    __device__ __forceinline__ static void lb1_step(const int2 &A, const int2 &A2, const int (&pj)[M], int &t0,
                                                    int &lb)
    {
        int x, y;
        if constexpr (Q < 16) {
            x = row_bcast_lane<Q>(A.x);
            y = row_bcast_lane<Q>(A.y);
        } else {
            x = row_bcast_lane<Q - 16>(A2.x);
            y = row_bcast_lane<Q - 16>(A2.y);
        }
        if constexpr (Q == 0) {
            t0 = x + pj[0];
            lb = x + y;
        } else {
            const int t1 = max(x, t0);
            lb = max(lb, t1 + y);
            t0 = t1 + pj[Q];
        }
    }

    template <int... Q>
    __device__ __forceinline__ static int lb1_steps(const int2 &A, const int2 &A2, const int (&pj)[M],
                                                    std::integer_sequence<int, Q...>)
    {
        int t0 = 0, lb = 0;
        (lb1_step<Q>(A, A2, pj, t0, lb), ...);
        return lb;
    }

    // one fused pass over children base..base+31; returns this lane's bound.
    // Each 16-lane row reads its half's operand pairs once (two vector LDS
    // reads, no bank conflicts) and every machine step takes its pair from
    // lane q of the row by DPP, instead of M broadcast reads of U.
    __device__ __forceinline__ int lb1_pass(int base, int k) const
    {
        const int half = lane >> 5;
        const int c = base + (lane & 31);
        const int job = base == 0 ? bcast_low_half(rowv) : bcast_high_half(rowv);
        const int jb = c < k ? job : 0;
        // machine-major rows: front lanes walk machines 0..M-1, back lanes M-1..0
        const int *pcol = (half ? lds.pmR : lds.pm) + jb;
        const int ql = lane & 15;
        const int2 *u = lds.U + half * M;
        const int2 A = u[min(ql, M - 1)];
        int2 A2 = make_int2(0, 0);
        if constexpr (M > 16) A2 = u[16 + min(ql, M - 17)];
        int pj[M];
#pragma unroll
        for (int q = 0; q < M; q++) pj[q] = pcol[q * PM_STRIDE];
        return lb1_steps(A, A2, pj, std::make_integer_sequence<int, M>{});
    }

    // row layout (lane = child): cb (front) and ce (back) for k <= 64 children
    __device__ __forceinline__ void lb1_children(int k, int &cb, int &ce) const
    {
        build_operands();
        int lb0 = lb1_pass(0, k);
        if (k <= 32) {
            cb = lb0;
            ce = bcast_high_half(lb0);
        } else {
            int lb1 = lb1_pass(32, k);
            int sh0 = bcast_high_half(lb0), sh1 = bcast_low_half(lb1);
            cb = lane < 32 ? lb0 : sh1;
            ce = lane < 32 ? sh0 : lb1;
        }
    }

    // chooseChildrenSet (ivm_bound.cpp:413-507): lanes beyond the row hold
    // the reference's zero entries and are excluded from every term.
    __device__ __forceinline__ int choose(bool valid, int cb, int ce) const
    {
        switch (a.branching) {
        case -3: return (L % 2) ? 1 : 0;
        case -2: return 1;
        case -1: return 0;
        case 1: {
            int s = wave_sum(valid ? cb - ce : 0);
            return s < 0 ? 1 : 0;
        }
        case 2: {
            int ub = a.single_node ? local_best : ir.ub0;
            const uint64_t vm = ballot(valid);
            int elim = __popcll(vm & ballot(cb >= ub)) - __popcll(vm & ballot(ce >= ub));
            int s = wave_sum(valid ? ((cb < ub ? cb : 0) - (ce < ub ? ce : 0)) : 0);
            if (elim > 0) return 0;
            if (elim < 0) return 1;
            return s < 0 ? 1 : 0;
        }
        default: {
            int ub = a.single_node ? local_best : ir.ub0;
            int mn = wave_min(valid ? min(cb > 0 ? cb : PBB_INF, ce > 0 ? ce : PBB_INF) : PBB_INF);
            const uint64_t vm = ballot(valid);
            int minc = __popcll(vm & ballot(cb == mn)) - __popcll(vm & ballot(ce == mn));
            int elimc = __popcll(vm & ballot(cb >= ub)) - __popcll(vm & ballot(ce >= ub));
            if (minc > 0) return 1;
            if (minc < 0) return 0;
            return elimc > 0 ? 0 : 1;
        }
        }
    }

    // ----------------------------------------------------------- bounding
    // Bound the children of the node at line L (row in rowv, unflagged),
    // choose the direction, refine, prune, reverse (ivm_bound.cpp:141-236,
    // :337-676).  root: boundRoot always uses weakBoundPrune.
    __device__ __forceinline__ void bound_row(bool root)
    {
        const int k = n - L;
        const bool valid = lane < k;
        const int job = valid ? rowv : 0;
        const bool both = a.branching > 0;
        int dir, c1, c2 = 0;
        bool refined = false;
        if constexpr (REF == 0) {
            int cb, ce;
            lb1_children(k, cb, ce);
            if (!both) ce = 0;  // costsEnd[WEAK] stays zero (boundChildren front only)
            sb += (unsigned)(both ? 2 * k : k);
            dir = choose(valid, cb, ce);
            c1 = dir ? ce : cb;
        } else {
            const int mode = root ? 0 : a.bound_mode;
            int cb, ce;
            lb1_children(k, cb, ce);
            if (mode == 1) {
                int csF = 0, csB = 0;
                refine_both(valid, cb, ce, csF, csB);
                dir = choose(valid, csF, csB);
                c1 = c2 = dir ? csB : csF;
                refined = true;
            } else {
                const int back = ce;
                if (!both) ce = 0;
                sb += (unsigned)(both ? 2 * k : k);
                dir = choose(valid, cb, ce);
                c1 = dir ? ce : cb;
                if (mode == 2) {
                    c2 = refine_dir(dir, valid, c1, dir ? back : cb);
                    refined = true;
                }
            }
        }
        bool pr = valid && (gt_best(c1) || (refined && gt_best(c2)));
        int v = pr ? flag_neg(job) : job;
        int prev = L > 0 ? rdlane(dirv, L - 1) : 0;
        if (prev != dir) v = shfl(v, k - 1 - lane);
        rowv = valid ? v : 0;
        dirv = wrlane(dirv, dir, L);
    }

    // ---------------------------------------------------------- refinement
    // LB1' of a child (bound_fsp_weak::bornes_calculer with the child's front or
    // back, bound_fsp_weak.cpp:288-311) is its LB1 bound, so the refinement of REF
    // 1 takes that value and only counts.  With front times f, remaining work r and
    // back times b, LB1' is the maximum over machines i <= q of f_i + r_i + b_q.
    // Back times never grow with the machine: a back chain has b_q >= b_(q+1) +
    // p_q, min_dep sums fewer times, and no time is negative.  So the maximum is at
    // q = i, and f_i + r_i + b_i of the child is the LB1 term of machine i: front,
    // max(f_i, f'_(i-1)) + p_i + (r_i - p_i) + b_i; back, the same from the other
    // end.  A pass of its own with both of the child's chains per lane took half of
    // a node's time (30x17, 6.3 M nodes: 8.1 ms, 6.2 without it).

    // Johnson LB2 of children c0 and c1 (uniform; K = 1: of c0 alone), direction d
    // (bound_fsp_strong::bornes_calculer with the child's partial schedule), to v0
    // and v1.  Half of the wavefront each: the child's front (d = 0) or back
    // (d = 1) completion times come from one lane-parallel chain scan (lane =
    // machine, as a stack push) and go to the wave's LDS, where the pair lanes
    // read them: fs the front times, gs the back times plus the child's
    // remaining work (in the sink, where nothing is read).  Then both children
    // go through the pair lanes together.  Up to 10 machines and 20 jobs the scan,
    // the LDS round trip and the reduction are more of a child's time than its
    // walk, and all are latency.
    template <int K>
    __device__ __forceinline__ void lb2_children(int d, int c0, int c1, int k, int &v0, int &v1)
    {
        const int q = lane & 31, qq = min(q, M - 1);
        const bool up = lane >= 32, in = q < M;
        const int j0 = flag_abs(rdlane(rowv, c0)), j1 = K == 2 ? flag_abs(rdlane(rowv, c1)) : j0;
        const int job = up ? j1 : j0;
        int *fs = lds.scr, *gs = (int *)lds.sink;
        const int ft = bcast_low_half(ftop), rem = bcast_low_half(remv);
        int f;  // the child's front time on machine q
        if (d == 0) {
            const int v = lds.pm[qq * PM_STRIDE + job], pc = in ? v : 0;
            f = chain_scan(ft, pc);
            fs[lane] = f;
            gs[lane] = brow(nb)[qq] + rem - pc;
        } else {
            // back chain over machines M-1..0: lane q handles machine M-1-q
            const int b = brow(nb)[M - 1 - qq], v = lds.pmR[qq * PM_STRIDE + job];
            const int pr = in ? v : 0;
            const int rr = shfl(rem, M - 1 - qq) - pr;
            const int cb = chain_scan(in ? b : 0, pr);
            f = ft;
            fs[lane] = f;
            gs[(up ? 32 : 0) + (in ? M - 1 - q : q)] = cb + rr;
        }
        __builtin_amdgcn_wave_barrier();
        int r[2];
        if (k <= 2) {
            // l2 - l1 <= 2: makespan of the completed permutation (bound_fsp_strong.cpp:543-546);
            // the other job is all the remaining work
            const int o0 = flag_abs(rdlane(rowv, 1 - c0)), o1 = K == 2 ? flag_abs(rdlane(rowv, 1 - c1)) : o0;
            const int v = lds.pm[qq * PM_STRIDE + (up ? o1 : o0)], po = in ? v : 0;
            const int cc = chain_scan(f, po) + gs[lane] - po;
            // both halves' values where the reduction below expects them
            r[0] = up ? 0 : (in ? cc : 0);
            r[1] = up ? (in ? cc : 0) : 0;
        } else if (lds.jtwalk) {
            if (PCH == 1 || lds.nch == 1) walk_children<K, 1>(k - 1, j0, j1, r);
            else if (PCH == 2 || lds.nch == 2) walk_children<K, PCH < 2 ? PCH : 2>(k - 1, j0, j1, r);
            else walk_children<K, PCH>(k - 1, j0, j1, r);
        } else {
#pragma unroll
            for (int i = 0; i < K; i++)
                r[i] = lb2_pairs_any<PCH, TAB>(pinfo, lds.jtl, lds.jtabL, lds.jtabG, lds.jpacked, n, ir.npairs,
                                               fs + 32 * i, gs + 32 * i, free_jobs & ~(1ull << (i ? j1 : j0)));
        }
        if (K == 1) r[1] = r[0];
        const auto h = __builtin_amdgcn_permlane32_swap(r[0], r[1], false, false);
        const int x = scan_max32(max((int)h[0], (int)h[1]));  // lanes 31 and 63: a child's greatest
        v0 = rdlane(x, 31);
        v1 = rdlane(x, 63);
        __builtin_amdgcn_wave_barrier();
    }

    template <int K, int NCH>
    __device__ __forceinline__ void walk_children(int cnt, int j0, int j1, int (&r)[2]) const
    {
        const int *fs = lds.scr, *gs = (const int *)lds.sink;
        unsigned pl[K][NCH];
        int D[K][NCH], best[K][NCH], end[K][NCH];
#pragma unroll
        for (int c = 0; c < NCH; c++) {
            const int info = pinfo[c] < 0 ? 0 : pinfo[c], a = info & 0xff, b = info >> 8;
#pragma unroll
            for (int i = 0; i < K; i++) {
                pl[i][c] = places[c] & ~(1u << walk_place(((i ? j1 : j0) * NCH + c) * 64 + lane));
                D[i][c] = fs[32 * i + a];
                best[i][c] = fs[32 * i + b];
                end[i][c] = D[i][c] + gs[32 * i + a];
            }
        }
        lb2_walk<K, NCH, WIDE>(lds.jtabL, cnt, pl, D, best);
#pragma unroll
        for (int i = 0; i < K; i++) {
            r[i] = 0;
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                const int b = pinfo[c] < 0 ? 0 : pinfo[c] >> 8;
                const int v = max(best[i][c] + gs[32 * i + b], end[i][c]);
                r[i] = max(r[i], pinfo[c] < 0 ? 0 : v);
            }
        }
    }

    // mixed mode (computeStrongBounds, ivm_bound.cpp:141-195): refine the
    // children not pruned by LB1 in the chosen direction (cost cw, zero where only
    // front costs are computed; lb1 is the bound itself); 0 for the others
    __device__ __forceinline__ int refine_dir(int d, bool valid, int cw, int lb1)
    {
        const int k = n - L;
        bool todo = valid && !gt_best(cw);
        uint64_t tmask = ballot(todo);
        jb += (unsigned)__popcll(tmask);
        jhist += lane == L ? __popcll(tmask) : 0;
        if constexpr (REF == 1) return todo ? lb1 : 0;
        int cs = 0;
        uint64_t m = tmask;
        while (m) {
            const int c0 = __ffsll((unsigned long long)m) - 1;
            m &= m - 1;
            int v0, v1;
            if (m) {
                const int c1 = __ffsll((unsigned long long)m) - 1;
                m &= m - 1;
                lb2_children<2>(d, c0, c1, k, v0, v1);
                cs = lane == c1 ? v1 : cs;
            } else {
                lb2_children<1>(d, c0, c0, k, v0, v1);
            }
            cs = lane == c0 ? v0 : cs;
        }
        return cs;
    }

    // strong-only mode (strongBoundPrune, ivm_bound.cpp:668-676)
    __device__ __forceinline__ void refine_both(bool valid, int cb, int ce, int &csF, int &csB)
    {
        const int k = n - L;
        jb += 2u * (unsigned)k;
        jhist += lane == L ? 2 * k : 0;
        if constexpr (REF == 1) {
            csF = valid ? cb : 0;
            csB = valid ? ce : 0;
            return;
        }
        csF = csB = 0;
        for (int c = 0; c < k; c += 2) {
            const int c1 = min(c + 1, k - 1);
#pragma unroll
            for (int d = 0; d < 2; d++) {
                int v0, v1;
                lb2_children<2>(d, c, c1, k, v0, v1);
                int &cs = d ? csB : csF;
                cs = lane == c ? v0 : (lane == c1 ? v1 : cs);
            }
        }
    }

    // -------------------------------------------------------------- leaf
    // ivm_bound::boundLeaf (ivm_bound.cpp:238-271): makespan of front + the
    // last row job + back; the incumbent only moves on strict improvement.
    __device__ __forceinline__ int makespan_with(int r) const
    {
        int c = chain_scan(ftop, pmach(r));
        int b = brow(nb)[lane < M ? lane : M - 1];
        b = lane < M ? b : 0;
        return wave_max(lane < M ? c + b : 0);
    }

    __device__ __forceinline__ void leaf()
    {
        leaves++;
        const int r = rdlane(rowv, 0);
        const int cost = makespan_with(r);
        if (!gt_best(cost)) {
            if (cost < local_best) {
                write_perm(r);
                w_min64<SC>(ir.best, ((unsigned long long)(unsigned)cost << 32) | (unsigned)e);
            }
            local_best = cost;
        }
        rowv = wrlane(rowv, flag_neg(r), 0);
    }

    // decode the leaf schedule (ivm_bound::prepareSchedule) into best_perm[e]
    __device__ __forceinline__ void write_perm(int mid)
    {
        int jl = 0;
        if (lane < L) jl = flag_abs((int)lds.mat[lds_mat_row(lane, n) + posv]);
        uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        uint64_t fr = ballot(lane < L && dirv == 0);
        uint64_t bk = ballot(lane < L && dirv != 0);
        int *dst = a.best_perm + (size_t)e * 64;
        if (lane < L) {
            int p = dirv == 0 ? __popcll(fr & below) : n - 1 - __popcll(bk & below);
            dst[p] = jl;
        }
        if (lane == 0) dst[__popcll(fr)] = mid;
    }

    // ------------------------------------------------------- navigation
    __device__ __forceinline__ void store_row(int line) const
    {
        *(lane < n - line ? lds.mat + lds_mat_row(line, n) + lane : (int8_t *)(lds.sink + lane)) = (int8_t)rowv;
    }

    __device__ __forceinline__ void go_up()
    {
        if (L > 0) {
            posv = wrlane(posv, 0, L);
            L--;
            const int v = (int)lds.mat[lds_mat_row(L, n) + min(lane, n - 1 - L)];
            rowv = lane < n - L ? v : 0;
            const int p = rdlane(posv, L);
            pop_job(flag_abs(rdlane(rowv, p)), rdlane(dirv, L));
            if (lane == p) rowv = flag_neg(rowv);
        } else {
            posv = wrlane(posv, rdlane(posv, 0) + 1, 0);
        }
    }

    // branch on cell c of line L: generate line L+1 (ivm::goDown/generateLine)
    __device__ __forceinline__ void go_down(int c, bool explore)
    {
        store_row(L);
        push_job(flag_abs(rdlane(rowv, c)), rdlane(dirv, L));
        // drop cell c: lanes >= c take their right neighbour (DPP wave_shl:1,
        // lane i reads lane i+1; lane 63 reads 0)
        const int nxt = __builtin_amdgcn_update_dpp(0, rowv, 0x130, 0xF, 0xF, false);
        int v = lane >= c ? nxt : rowv;
        L++;
        rowv = lane < n - L ? flag_abs(v) : 0;
        if (explore) {
            posv = wrlane(posv, 0, L);
            dirv = wrlane(dirv, 0, L);
        }
    }

    // sequentialbb::unfold (sequentialbb.cpp:206-264): bounded, uncounted
    __device__ __forceinline__ void unfold()
    {
        while (L < n - 2) {
            int p = rdlane(posv, L);
            if (rdlane(rowv, p) < 0) {
                if (lane > L) posv = 0;
                break;
            }
            go_down(p, false);
            bound_row(false);
        }
    }

    // One call of sequentialbb::next (sequentialbb.cpp:128-163): returns 1
    // when an interior node was decomposed and bounded, 0 when the interval
    // is exhausted.  The reference tests beforeEnd at every iteration; pos
    // only grows in goRight and at the root line's increment (goUp resets a
    // deeper position to 0, goDown opens a line at 0), and end only shrinks
    // when a donation trims it, so the test runs exactly there and gives the
    // same answers.  goRight then goes down or up in the same iteration.
    __device__ __forceinline__ int step()
    {
        if (end_dirty) {
            end_dirty = false;
            if (!before_end()) return 0;
        }
        while (true) {
            const int p = rdlane(posv, L);
            int c = p;
            if (p < n - L) {
                // first live cell at or after p (ivm::goRight over pruned / visited cells)
                const uint64_t live = lanes_below(n - L) & ballot(rowv >= 0);
                const uint64_t ahead = live & (~0ull << p);
                c = ahead ? __ffsll((unsigned long long)ahead) - 1 : n - L;
                if (c != p) {
                    posv = wrlane(posv, c, L);
                    if (!before_end()) return 0;
                }
            }
            if (c >= n - L) {
                const bool root_line = L == 0;
                go_up();
                if (root_line && !before_end()) return 0;
                continue;
            }
            dec++;
            go_down(c, true);
            hist += (lane == L);
            if (L == n - 1) {
                leaf();
                continue;
            }
            bound_row(false);
            return 1;
        }
    }

    // ------------------------------------------------------ state I/O
    __device__ __forceinline__ void rebuild_stacks()
    {
        reset_stacks();
        for (int l = 0; l < L; l++) {
            int p = rdlane(posv, l);
            int j = uni(flag_abs((int)lds.mat[lds_mat_row(l, n) + p]));
            push_job(j, rdlane(dirv, l));
        }
    }

    __device__ __forceinline__ void load_state()
    {
        L = uni(a.line[e]);
        const int8_t *gm = a.mat + (size_t)e * rows * 64;
        for (int r = 0; r < L; r++)
            if (lane < n - r) lds.mat[lds_mat_row(r, n) + lane] = gm[r * 64 + lane];
        rowv = lane < n - L ? (int)gm[L * 64 + lane] : 0;
        posv = lane < n ? (int)a.pos[(size_t)e * 64 + lane] : 0;
        endv = lane < n ? (int)a.end[(size_t)e * 64 + lane] : 0;
        dirv = lane < n ? (int)a.dir[(size_t)e * 64 + lane] : 0;
        end_dirty = true;
        __builtin_amdgcn_wave_barrier();
        rebuild_stacks();
    }

    __device__ __forceinline__ void save_state(int st)
    {
        int8_t *gm = a.mat + (size_t)e * rows * 64;
        for (int r = 0; r < L; r++)
            if (lane < n - r) gm[r * 64 + lane] = lds.mat[lds_mat_row(r, n) + lane];
        if (lane < n) gm[L * 64 + lane] = (int8_t)rowv;
        if (lane < n) {
            a.pos[(size_t)e * 64 + lane] = (int8_t)posv;
            a.end[(size_t)e * 64 + lane] = (int8_t)endv;
            a.dir[(size_t)e * 64 + lane] = (int8_t)dirv;
        }
        if (lane == 0) {
            a.line[e] = L;
            a.state[e] = st;
            a.mtag[e] = mtag;
        }
    }

    // an idle explorer leaves the launch
    __device__ __forceinline__ void leave_idle()
    {
        if (lane == 0) {
            a.state[e] = ST_IDLE;
            a.mtag[e] = mtag;
        }
    }

    // ------------------------------------------------------------ mailbox
    // An interval is handed over as one message: 64 words of 64 bits, one per
    // lane, written by one store instruction.  The low half of every word
    // carries the message's tag (the previous one's plus 1, mod 64), so a
    // thief that sees the new tag in all 64 words holds the whole message
    // and neither side takes a fence: at agent scope a release writes back
    // the XCD's L2 and an acquire invalidates it.  The high halves carry
    // the front entry (lanes 0-19), the back entry (20-39) of the split
    // line, so the thief replays no push.  Reading the former rows, interval
    // vectors and line back from HBM and replaying the path took 18 us per
    // hand-over (50x20, 98 k hand-overs).
    static_assert(M <= 20, "the high halves of a message hold two vectors of 20 machines");

    __device__ __forceinline__ unsigned long long *my_mail() const { return a.mbox + (size_t)e * 64 + lane; }
    // the last message of this mailbox is consumed (or none was ever sent)
    __device__ __forceinline__ void open_mail() { mtag = mail_tag((unsigned)ld_rlx<SC>(my_mail())); }
    __device__ __forceinline__ unsigned long long peek_mail() const { return ld_rlx<SC>(my_mail()); }
    __device__ __forceinline__ bool mail_here(unsigned long long w) const
    {
        return ballot(mail_tag((unsigned)w) == ((mtag + 1u) & MAIL_TAGS)) == ~0ull;
    }

    __device__ __forceinline__ void take_mail(unsigned long long word)
    {
        const unsigned w = (unsigned)word;
        const int hi = (int)(unsigned)(word >> 32);
        mtag = mail_tag(w);
        const int job = (int)mail_job(w);
        L = __ffsll((unsigned long long)ballot(job == (int)MAIL_NONE)) - 1;
        rowv = mail_cell(w);
        posv = mail_pos(w);
        endv = mail_end(w);
        dirv = mail_dir(w);
        nb = __popcll(lanes_below(L) & ballot(dirv != 0));
        nf = L - nb;
        ftop = lane < M ? hi : 0;
        if (lane < M) frow(nf)[lane] = hi;
        if (lane >= 20 && lane < 20 + M) brow(nb)[lane - 20] = hi;
        remv = lane < M ? lds.tot[lane] : 0;
        if constexpr (REF == 2) all_free();
        for (int r = 0; r < L; r++) {
            const int j = rdlane(job, r);
            if constexpr (REF == 2) {
                free_jobs &= ~(1ull << j);
                mark_places<false>(j);
            }
            *(lane < n - r ? lds.mat + lds_mat_row(r, n) + lane : (int8_t *)(lds.sink + lane)) =
                (int8_t)mail_path_cell(lane, rdlane(posv, r), j);
            remv -= pmach(j);
        }
        end_dirty = true;
        __builtin_amdgcn_wave_barrier();
    }

    // the donor's side: rows 0..l of its path, the split row, the interval
    // [.., cut] .. endE and the stack entries of line l
    __device__ __forceinline__ void send_mail(int thief, unsigned tag, int l, int rowl, int cut, int endE)
    {
        int job = 0;
        if (lane < l) job = flag_abs((int)lds.mat[lds_mat_row(lane, n) + posv]);
        const int nbl = __popcll(lanes_below(l) & ballot(dirv != 0));
        const int qf = lane < M ? lane : M - 1, qb = lane < 20 ? 0 : (lane < 20 + M ? lane - 20 : M - 1);
        const int hi = lane < 20 ? frow(l - nbl)[qf] : brow(nbl)[qb];
        const unsigned lo = mail_word(lane < n - l ? rowl : 0, lane < l ? posv : (lane == l ? cut : 0),
                                      lane < n ? endE : 0, lane < l ? (unsigned)job : MAIL_NONE,
                                      lane <= l ? dirv : 0, tag);
        st_rlx64<SC>(a.mbox + (size_t)thief * 64 + lane, ((unsigned long long)(unsigned)hi << 32) | lo);
    }

    // fresh interval: row 0 = bounded root row, pos/end from HBM
    __device__ __forceinline__ bool start_unfold()
    {
        L = 0;
        rowv = lane < n ? ir.root_row[lane] : 0;
        posv = lane < n ? (int)a.pos[(size_t)e * 64 + lane] : 0;
        endv = lane < n ? (int)a.end[(size_t)e * 64 + lane] : 0;
        dirv = lane == 0 ? ir.root_dir[0] : 0;
        end_dirty = true;
        reset_stacks();
        if (!before_end()) return false;
        unfold();
        return true;
    }

    // the whole search space [0...0, (n-1)...0] from the bounded root row
    // already in rowv / dirv lane 0 (sequentialbb::initFullInterval +
    // initAtInterval, sequentialbb.cpp:66-108)
    __device__ __forceinline__ bool start_root()
    {
        L = 0;
        posv = 0;
        endv = lane < n ? n - 1 - lane : 0;
        dirv = lane == 0 ? dirv : 0;
        end_dirty = true;
        reset_stacks();
        if (!before_end()) return false;
        unfold();
        return true;
    }

    // --------------------------------------------------- work sharing
    // idle-wait pause: 2^k x 512 cycles, k growing to 4 while nothing
    // happens, so thousands of idle wavefronts do not flood the memory
    // system with polls
    __device__ __forceinline__ static void idle_pause(int &nap)
    {
        for (int i = 0; i < nap; i++) __builtin_amdgcn_s_sleep(8);
        if (nap < 16) nap <<= 1;
    }

    // bbthread::shareWork + ivm::cuttingPosition (bbthread.cpp:39-72,
    // ivm.cpp:188-237): split at the first line l whose pos differs from end
    // (l <= L, l < n - margin, the size_d - margin rule of
    // gpu/include/loadbalance.cuh:90); the thief gets the explorable cells after the
    // victim's kept half, rows 0..l and the victim's end; no re-bounding.
    // A line whose cells after pos are all pruned or visited holds no work:
    // its end is trimmed to pos (deeper ends become the maximum, so the
    // victim's interval covers exactly the same live nodes) and the split
    // moves down to the next line.  Node counts are unchanged by either step.
    // An explorer that starts a launch on a fresh interval (the root
    // interval, imported intervals) decomposes `ramp` nodes before it hands
    // work on: a small tree then runs depth-first in one explorer, finding
    // the incumbents the reference's order finds, and a large one fans out
    // after that many nodes (woken and resumed explorers share at once).
    // idle: the mask word loaded before the node's work (peek_idle).  Returns 0
    // when no explorer waits in it, 2 after a hand-over from a large interval
    // (SHARE_DEEP), else 1.
    __device__ __forceinline__ int try_donate(unsigned long long idle)
    {
        idle = uni64(idle);
        const int word = pollw;
        next_word();
        if (!idle) return 0;
        const int lim = min(L, n - 1 - a.steal_margin);  // last line a split may use
        if (lim < 0) return 1;                         // margin >= n: never split
        uint64_t ne = lanes_below(n) & ballot(posv != endv);
        uint64_t limmask = lim >= 64 ? ~0ull : ((1ull << lim) - 1ull);
        uint64_t cand = ne & limmask;
        const int first = cand ? __ffsll((unsigned long long)cand) - 1 : lim;
        int l = first, pl = 0, el = 0, rowl = -1;
        uint64_t expl = 0ull;
        for (;; l++) {
            if (l > lim) return 1;
            pl = rdlane(posv, l);
            el = (l == first) ? rdlane(endv, l) : n - 1 - l;
            if (pl < el) {
                rowl = (l == L) ? rowv : (lane < n - l ? (int)lds.mat[lds_mat_row(l, n) + lane] : -1);
                expl = (lanes_below(el + 1) & ~lanes_below(pl + 1)) & ballot(rowl >= 0);
                if (expl) break;
            }
        }
        // the victim's end once lines first..l-1 are trimmed
        int endE = endv;
        if (l > first) {
            if (lane >= first && lane < l) endE = posv;
            else if (lane >= l && lane < n) endE = n - 1 - lane;
        }
        int nexp = __popcll(expl);
        if (L - l < SHARE_NEAR && nexp < SHARE_CELLS) return 1;
        // Claim one explorer of the word by clearing its bit; each donor starts
        // its choice at another bit.  Relaxed: the claim orders nothing, the
        // donor has published nothing yet.
        const int rot = e & 63;
        const int bit = (__ffsll((idle >> rot) | (idle << (-rot & 63))) - 1 + rot) & 63;
        const int idx = bit * ir.idle_words + word;
        int got = 0, thief = idx;
        if (lane == 0) {
            const unsigned long long old =
                __hip_atomic_fetch_and(ir.idle + (size_t)word * IDLE_STRIDE, ~(1ull << bit), __ATOMIC_RELAXED, SC);
            if (ir.member) thief = ld_rlx<SC>(ir.member + idx);
            got = (int)((old >> bit) & 1ull);
        }
        if (!rdlane(got, 0)) return 1;
        thief = rdlane(thief, 0);
        // The thief is idle and this donor's alone now, so its mailbox holds the
        // last message it consumed: the next one's tag follows from it.  The
        // thief counts as holding an interval before its message is sent (the
        // count's old value has come back: used below), so its own release
        // comes later in the count's order.
        unsigned tag = 0u;
        int held = 0;
        if (lane == 0) {
            held = __hip_atomic_fetch_add(&ir.ctl->work_count, 1, __ATOMIC_RELAXED, SC);
            tag = mail_tag((unsigned)ld_rlx<SC>(a.mbox + (size_t)thief * 64));
        }
        held = rdlane(held, 0);
        tag = ((unsigned)rdlane((int)tag, 0) + 1u) & MAIL_TAGS;
        asm volatile("" : : "s"(held) : "memory");
        int keep = nexp / 2;
        int cut;
        if (keep == 0) {
            cut = pl + 1;
        } else {
            uint64_t mm = expl;
            for (int i = 1; i < keep; i++) mm &= mm - 1;
            cut = __ffsll((unsigned long long)mm);  // index of the keep-th cell + 1
        }
        send_mail(thief, tag, l, rowl, cut, endE);
        // the victim keeps [pos, cut-1] at line l and everything below
        endv = endE;
        if (lane == l) endv = cut - 1;
        if (lane > l && lane < n) endv = n - 1 - lane;
        end_dirty = true;
        return L - l >= SHARE_DEEP ? 2 : 1;
    }

    // member index of this explorer in its instance (the engine's explorers are
    // their own members).  The member word is complete, and the old tag of the
    // mailbox has been read (open_mail, before), when the first registration
    // names this explorer: a donor that claims it at once would otherwise find
    // another explorer's number, or send a message that is taken for the old one.
    // Relaxed accesses to different words have no order, so the wait is explicit (a
    // fence at agent scope would write the L2 back).
    __device__ __forceinline__ void join(int idx)
    {
        self = idx;
        if (ir.member && lane == 0) st_rlx<SC>(const_cast<int *>(ir.member) + idx, e);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(mtag) : : "memory");
        pollw = ir.occ ? 0 : idx % ir.idle_words;
    }

    // the idle word of the next poll (a wavefront passes over all words in turn;
    // a pool slot's over those its members fill so far)
    __device__ __forceinline__ unsigned long long peek_idle()
    {
        if (ir.occ) seen = ld_rlx<SC>(ir.occ);
        return ld_rlx<SC>(ir.idle + (size_t)pollw * IDLE_STRIDE);
    }
    __device__ __forceinline__ void next_word()
    {
        int words = ir.idle_words;
        if (ir.occ) words = min(words, uni(seen) & POOL_MEMBERS);
        pollw = pollw + 1 < words ? pollw + 1 : 0;
    }

    __device__ __forceinline__ void register_idle()
    {
        if (lane == 0)
            __hip_atomic_fetch_or(ir.idle + (size_t)(self % ir.idle_words) * IDLE_STRIDE,
                                  1ull << (self / ir.idle_words), __ATOMIC_RELAXED, SC);
    }

    // give up an exhausted interval; returns true for the explorer whose
    // release emptied the instance (all explorers idle: it is solved).  The
    // registration may take effect before the release: a donor that claims this
    // explorer counts it again before its message arrives, and itself holds an
    // interval meanwhile.
    __device__ __forceinline__ bool go_idle()
    {
        register_idle();
        int left = 0;
        if (lane == 0) left = __hip_atomic_fetch_add(&ir.ctl->work_count, -1, __ATOMIC_RELAXED, SC);
        return rdlane(left, 0) == 1;
    }

    __device__ __forceinline__ void flush_counters()
    {
        if (lane == 0) {
            if (dec) atomicAdd(&ir.ctl->dec, (unsigned long long)dec);
            if (leaves) atomicAdd(&ir.ctl->leaves, (unsigned long long)leaves);
            if (sb) atomicAdd(&ir.ctl->sb, (unsigned long long)sb);
            if (jb) atomicAdd(&ir.ctl->jb, (unsigned long long)jb);
        }
        dec = leaves = sb = jb = 0;
        if (hist && lane <= n) atomicAdd(&ir.ctl->histo[lane], (unsigned long long)hist);
        hist = 0;
        if constexpr (REF != 0) {
            if (jhist && lane <= n) atomicAdd(&ir.ctl->jhisto[lane], (unsigned long long)jhist);
            jhist = 0;
        }
    }

    // incumbent word loaded by the caller (cost << 32 | explorer)
    __device__ __forceinline__ void take_best(unsigned long long b)
    {
        const int bc = uni((int)(unsigned)(b >> 32));
        if (bc < local_best) local_best = bc;
    }

    // periodic: node budget, deadline, host interrupt, incumbent refresh
    __device__ __forceinline__ bool check_stop()
    {
        if (a.node_budget) {
            unsigned long long before = w_add64<SC>(&ir.ctl->dec, (unsigned long long)dec);
            const unsigned long long most = local_best < a.initial_ub ? a.node_budget : a.quiet_budget;
            if (before + dec >= most && lane == 0) st_rlx<SC>(&run->stop, 1);
            dec = 0;
        }
        if (dec >= (1u << 28) || sb >= (1u << 28) || jb >= (1u << 28)) flush_counters();  // 32-bit deltas
        if (t_end && wall_clock64() >= t_end && lane == 0) st_rlx<SC>(&run->stop, 1);
        poll_host_and_best();
        return uni(ld_rlx<SC>(&run->stop)) != 0;
    }

    // The pool's periodic check: the deadline (the launch's or the request's,
    // whichever is first) raises the instance's own stop word.  Returns 0 to
    // go on, 1 when the launch stops (interrupt, error: the explorer leaves),
    // 2 when only this instance stops.
    __device__ __forceinline__ int check_stop_slot(int *slot_stop)
    {
        if (dec >= (1u << 28) || sb >= (1u << 28) || jb >= (1u << 28)) flush_counters();  // 32-bit deltas
        if (t_end && wall_clock64() >= t_end && lane == 0) st_rlx<SC>(slot_stop, 1);
        poll_host_and_best();
        if (uni(ld_rlx<SC>(&run->stop)) != 0) return 1;
        return uni(ld_rlx<SC>(slot_stop)) != 0 ? 2 : 0;
    }

    __device__ __forceinline__ void poll_host_and_best()
    {
        const bool host_turn = (nchk++ & (PBB_HOST_POLL_CHECKS - 1u)) == 0u;
        if (a.host_flag && host_turn && lane == 0) {
            int hf = __hip_atomic_load(a.host_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (hf) st_rlx<SC>(&run->stop, 1);
        }
        unsigned long long b = ld_rlx<SC>(ir.best);
        int bc = uni((int)(unsigned)(b >> 32));
        if (bc < local_best) local_best = bc;
    }
};

}  // namespace pbb
