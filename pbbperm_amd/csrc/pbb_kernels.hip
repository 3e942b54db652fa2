// pbb_kernels.hip -- gfx950 kernels of the IVM branch-and-bound engine.
//
//   k_explore<M,REF,TAB> persistent explorer kernel: one IVM per 64-lane
//                  wavefront, 4 explorers per 256-thread workgroup.  The IVM
//                  matrix (int8 rows) and the front/back completion-time
//                  stacks of each explorer live in LDS; the interval vectors
//                  and the current row live in VGPRs.  Implements
//                  sequentialbb::next / unfold (multicore/src/sequentialbb.cpp:110-264)
//                  with ivm.cpp navigation and ivm_bound.cpp bounding,
//                  branching and pruning.  Work is balanced on the device: an
//                  explorer whose interval is exhausted registers in an idle
//                  mask; busy explorers split their interval as
//                  bbthread::shareWork (multicore/src/bbthread.cpp:39-72) and
//                  hand the upper part to an idle explorer.  No host round
//                  trip until the run ends (all idle, node budget, deadline
//                  or interrupt).  REF selects the bounding variant at
//                  compile time: 0 LB1 only (boundingMode 0), 1 LB1 + LB1'
//                  refinement (modes 1/2 as shipped), 2 LB1 + Johnson LB2,
//                  of the table form TAB.
//   k_bound_root<M> LB1 root bounding, ivm_bound::boundRoot (ivm_bound.cpp:273-330).
//
// Translation units: this file is compiled once per machine count M
// (-DPBB_M=<m>) so the 19 instantiations build in parallel, and once more for the
// kernels of the wide Johnson table (-DPBB_TAB=TAB_WIDE): a process that meets no
// large processing times then never loads them.
#include "pbb_explorer.h"

namespace pbb {

// ------------------------------------------------------------ kernels
// Minimum resident waves per SIMD the compiler must allow (register
// budget): 4 for the LB1 and LB1' explorers (128 VGPRs), 3 with LB2, where the
// 20-machine one spills 21 registers for it (187 VGPRs without the bound, none
// spilled, 2048 explorers).  3 / 2 waves at 18x20: 2.5 M nodes 6.7 / 8.4 ms, 3065
// nodes 1.74 / 1.54; 30x20 3.59 / 3.55.
#ifndef PBB_EXPLORE_MIN_WAVES
#define PBB_EXPLORE_MIN_WAVES 4
#endif

// The explorer loop of one wavefront (explorer e); SC is the memory scope of
// the explorers it shares work with.
template <int M, int REF, int TAB, int SC>
__device__ __forceinline__ void explore_loop(const KArgs &a, const Lds &lds, int e)
{
    Explorer<M, REF, SC, TAB> X(a, lds, e, engine_inst(a), a.ctl, a.I.n, a.I.mp);
    X.local_best = uni((int)(unsigned)(ld_rlx<SC>(a.best) >> 32));
    X.open_mail();
    X.join(e);
    // what the host or the previous launch left is visible at launch start
    int st = uni(ld_rlx<SC>(a.state + e));
    unsigned iter = 0;
    unsigned next = 0;  // node of the next poll
    if (st == ST_UNFOLD) {
        if (X.start_unfold()) {
            st = ST_ACTIVE;
            next = a.ramp;  // none while the ramp holds this explorer's work back
        } else {
            if (X.go_idle() && X.lane == 0) st_rel<SC>(&a.ctl->done, 1);
            st = ST_IDLE;
        }
    } else if (st == ST_ACTIVE) {
        X.load_state();
    } else {
        // An idle explorer enters the idle mask only once it runs (the host
        // leaves the mask empty at every launch), so donors only ever hand
        // work to wavefronts that are resident: one still waiting for a CU
        // (another kernel or process on the device, an occupancy estimate
        // that was too high) holds no work that the others wait for.
        X.register_idle();
    }

    while (true) {
        if (st == ST_IDLE) {
            // wait for a donation, global termination or a stop; the host
            // interrupt word (a PCIe round trip) is read by every 16th
            // explorer, at every 16th pass once its back-off is at the
            // longest, and the first to see it raises the device stop word
            int nap = 1;
            while (true) {
                // one poll: the mailbox and the words a leave depends on, all
                // in flight together
                const unsigned long long mail = X.peek_mail(), bw = ld_rlx<SC>(a.best);
                const int done = ld_rlx<SC>(&a.ctl->done), stop = ld_rlx<SC>(&a.ctl->stop);
                if (X.mail_here(mail)) {
                    st = ST_ACTIVE;
                    X.take_mail(mail);
                    // a donated interval is explored under the current incumbent,
                    // not the one this explorer saw before it went idle
                    X.take_best(bw);
                    if (a.ramp) next = iter;  // a donated interval is shared at once
                    break;
                }
                if (uni(done) || uni(stop) || (X.t_end && wall_clock64() >= X.t_end)) {
                    X.leave_idle();
                    X.flush_counters();
                    return;
                }
                if (a.host_flag && (e & 15) == 0 && nap == 16 && X.lane == 0 &&
                    __hip_atomic_load(a.host_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
                    st_rlx<SC>(&a.ctl->stop, 1);
                if constexpr (SC == __HIP_MEMORY_SCOPE_WORKGROUP) __builtin_amdgcn_s_sleep(2);
                else X.idle_pause(nap);
            }
        }
        // idle-mask poll issued before the node's work so its latency is
        // hidden.  In the workgroup team (at most 16 explorers, workgroup-scope atomics)
        // and with LB2 a donor that saw explorers waiting polls again at the
        // next node, otherwise one that gave from a large interval
        // (PBB_POLL_EVERY, SHARE_DEEP).
        constexpr bool eager = SC == __HIP_MEMORY_SCOPE_WORKGROUP || REF == 2;
        const bool poll = (int)(iter - next) >= 0;
        unsigned long long idle = 0ull;
        if (poll) idle = X.peek_idle();
        const bool refresh = (iter & (PBB_BEST_EVERY - 1)) == 0u;
        unsigned long long bw = ~0ull;
        if (refresh) bw = ld_rlx<SC>(a.best);
        if (!X.step()) {
            if (X.go_idle() && X.lane == 0) st_rel<SC>(&a.ctl->done, 1);
            st = ST_IDLE;
            continue;
        }
        if (refresh) X.take_best(bw);
        if ((++iter & 63u) == 0u && X.check_stop()) {
            X.save_state(ST_ACTIVE);
            X.flush_counters();
            return;
        }
        // one count of nodes for the interval, the eager polls and the ramp: 2106 M
        // nodes/s at 50x20 (2076 with a counter of the ramp's nodes beside it, 2058
        // with that and a flag for the eager polls)
        if (poll) next = iter + (X.try_donate(idle) >= (eager ? 1 : 2) ? 0u : PBB_POLL_EVERY - 1u);
    }
}

template <int M, int REF, int TAB>
__global__ __launch_bounds__(64 * PBB_EXPLORE_WAVES, REF == 2 ? 3 : PBB_EXPLORE_MIN_WAVES) void k_explore(KArgs a)
{
    extern __shared__ __align__(16) char smem[];
    Lds lds = lds_setup<TAB>(a.I, smem, REF == 2 ? a.jt_lds : 0, REF == 2);
    const int e = blockIdx.x * PBB_EXPLORE_WAVES + (threadIdx.x >> 6);
    if (e >= a.E) return;
    explore_loop<M, REF, TAB, __HIP_MEMORY_SCOPE_AGENT>(a, lds, e);
}

// The team launch: explorers 0..a.E-1 as the wavefronts of one workgroup
// (up to team_waves_max(REF)), whose messages, mask word and counters stay in one
// CU's L1 and XCD's L2.  A fresh search starts here: a small tree (a few thousand
// nodes) is solved by the team alone, without a device-wide launch's fan-out; a
// larger one stops at the node budget and the device-wide launch resumes from the
// saved intervals.
template <int M, int REF, int TAB>
__global__ __launch_bounds__(64 * team_waves_max(REF)) void k_team(KArgs a)
{
    extern __shared__ __align__(16) char smem[];
    Lds lds = lds_setup<TAB>(a.I, smem, REF == 2 ? a.jt_lds : 0, REF == 2);
    const int e = threadIdx.x >> 6;
    if (e >= a.E) return;
    explore_loop<M, REF, TAB, __HIP_MEMORY_SCOPE_WORKGROUP>(a, lds, e);
}

template <int M>
__global__ __launch_bounds__(64) void k_bound_root(KArgs a, RootPerm root_perm)
{
    extern __shared__ __align__(16) char smem[];
    Lds lds = lds_setup<TAB_PACKED>(a.I, smem, 0, false);
    Explorer<M, 0> X(a, lds, 0, engine_inst(a), a.ctl, a.I.n, a.I.mp);
    X.local_best = a.initial_ub;
    X.rowv = X.lane < X.n ? root_perm.p[X.lane] : 0;
    X.reset_stacks();
    X.bound_row(true);
    int d0 = rdlane(X.dirv, 0);
    if (X.lane < X.n) a.root_row_out[X.lane] = X.rowv;
    if (X.lane == 0) a.root_dir_out[0] = d0;
}

// ---------------------------------------------------------- host launchers
// the kernel of a bounding variant (the wide form is LB2's)
template <int M, int TAB>
static const void *explore_kernel(const KArgs &a)
{
    if constexpr (TAB == TAB_WIDE) return (const void *)k_explore<M, 2, TAB>;
    else {
        if (a.bound_mode == 0) return (const void *)k_explore<M, 0, TAB>;
        return a.refine == 1 ? (const void *)k_explore<M, 2, TAB> : (const void *)k_explore<M, 1, TAB>;
    }
}
template <int M, int TAB>
static const void *team_kernel(const KArgs &a)
{
    if constexpr (TAB == TAB_WIDE) return (const void *)k_team<M, 2, TAB>;
    else {
        if (a.bound_mode == 0) return (const void *)k_team<M, 0, TAB>;
        return a.refine == 1 ? (const void *)k_team<M, 2, TAB> : (const void *)k_team<M, 1, TAB>;
    }
}

static hipError_t launch_kernel(const void *k, int blocks, int threads, size_t lds, const KArgs &a, hipStream_t s)
{
    if (const hipError_t err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) return err;
    void *args[] = {(void *)&a};
    return hipLaunchKernel(k, dim3(blocks), dim3(threads), args, lds, s);
}

template <int M, int TAB>
hipError_t launch_explore_m(const KArgs &a, int blocks, hipStream_t s)
{
    const bool lb2 = a.bound_mode != 0 && a.refine == 1;
    const size_t lds = explore_lds_bytes(a.I, lb2, lb2 ? a.jt_lds : 0);
    return launch_kernel(explore_kernel<M, TAB>(a), blocks, 64 * PBB_EXPLORE_WAVES, lds, a, s);
}

template <int M, int TAB>
hipError_t launch_team_m(const KArgs &a, hipStream_t s)
{
    const bool lb2 = a.bound_mode != 0 && a.refine == 1;
    const size_t lds = team_lds_bytes(a.I, lb2, lb2 ? a.jt_lds : 0, a.E);
    return launch_kernel(team_kernel<M, TAB>(a), 1, 64 * a.E, lds, a, s);
}

template <int M, int TAB>
hipError_t occupancy_m(const KArgs &a, int *blocks_per_cu)
{
    const bool lb2 = a.bound_mode != 0 && a.refine == 1;
    const size_t lds = explore_lds_bytes(a.I, lb2, lb2 ? a.jt_lds : 0);
    if (lds > 160 * 1024) {
        *blocks_per_cu = 0;
        return hipSuccess;
    }
    const size_t q = residency_lds_bytes(lds);
    const void *k = explore_kernel<M, TAB>(a);
    if (const hipError_t err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)q)) return err;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, k, 64 * PBB_EXPLORE_WAVES, q);
}

template <int M>
hipError_t launch_root_m(const KArgs &a, const RootPerm &root_perm, hipStream_t s)
{
    const size_t lds = root_lds_bytes(a.I);
    if (const hipError_t err =
            hipFuncSetAttribute((const void *)k_bound_root<M>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
        return err;
    hipLaunchKernelGGL(k_bound_root<M>, dim3(1), dim3(64), lds, s, a, root_perm);
    return hipGetLastError();
}

#ifdef PBB_M
#ifndef PBB_TAB
#define PBB_TAB TAB_PACKED
template hipError_t launch_root_m<PBB_M>(const KArgs &, const RootPerm &, hipStream_t);
#endif
template hipError_t launch_explore_m<PBB_M, PBB_TAB>(const KArgs &, int, hipStream_t);
template hipError_t launch_team_m<PBB_M, PBB_TAB>(const KArgs &, hipStream_t);
template hipError_t occupancy_m<PBB_M, PBB_TAB>(const KArgs &, int *);
#endif

}  // namespace pbb
