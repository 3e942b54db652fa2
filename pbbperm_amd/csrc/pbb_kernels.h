// pbb_kernels.h -- kernel argument block and launchers shared by the HIP
// kernels (pbb_kernels.hip) and the host engine (pbb_host.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pbb_device.h"
#include "pbb_slot.h"

namespace pbb {

enum { ST_IDLE = 0, ST_ACTIVE = 1, ST_UNFOLD = 2 };

// Idle explorers register in a bit mask: bit b of mask word w stands for the
// explorer (or pool member) b * words + w.  Each word sits on its own 128-byte
// line (IDLE_STRIDE words of 64 bits apart).  A donor polls one word at a time,
// another at every poll, and claims an explorer by clearing its bit: one atomic
// per attempt, on a line shared with 64 explorers.  One ring for all of them
// (two ticket counters and a count) had every poll and every claim of the
// device on one or two lines: 50 us per attempt at 4096 explorers on a thin
// tree (50x20, 49.7 M nodes, 300 k hand-overs), 77 ms against 29 ms.
#define IDLE_STRIDE 16
__device__ __host__ inline int idle_words_for(int explorers) { return (explorers + 63) / 64; }

// Message word of lane i (low 32 bits; the high 32 carry stack entries):
// bits 0-5 the job of cell i of the split row l, 6 its pruned/visited flag,
// 7-12 pos[i], 13-18 end[i], 19-24 the job chosen at line i (MAIL_NONE from
// line l on), 25 dir[i], 26-31 the message's tag.  63 jobs fit: ids and
// positions are at most 62.
#define MAIL_NONE 63u
#define MAIL_TAGS 63u
__device__ __forceinline__ unsigned mail_word(int cell, int pos, int end, unsigned job, int dir, unsigned tag)
{
    const unsigned c = cell < 0 ? (unsigned)(-cell - 1) | 64u : (unsigned)cell;
    return c | ((unsigned)pos << 7) | ((unsigned)end << 13) | (job << 19) | ((unsigned)dir << 25) | (tag << 26);
}
__device__ __forceinline__ int mail_cell(unsigned w) { return (w & 64u) ? -(int)(w & 63u) - 1 : (int)(w & 63u); }
__device__ __forceinline__ int mail_pos(unsigned w) { return (int)((w >> 7) & 63u); }
__device__ __forceinline__ int mail_end(unsigned w) { return (int)((w >> 13) & 63u); }
__device__ __forceinline__ unsigned mail_job(unsigned w) { return (w >> 19) & 63u; }
__device__ __forceinline__ int mail_dir(unsigned w) { return (int)((w >> 25) & 1u); }
__device__ __forceinline__ unsigned mail_tag(unsigned w) { return w >> 26; }
// Cell i of row r < l of a received interval, pos p, chosen job j.  Lines
// above the split hold no work (their end is their pos): the cells before p
// are dead, and those after it live, so that coming back up to the line ends
// the interval at once by the interval-end test, as on the donor's own row.
__device__ __forceinline__ int mail_path_cell(int i, int p, int j) { return i == p ? j : (i > p ? 0 : -1); }

// A busy explorer of a device-wide launch reads a word of the idle mask every
// PBB_POLL_EVERY decomposed nodes, whether or not explorers wait in it; with
// Johnson LB2, whose node takes several times an LB1 node's time, it reads the
// next word at the next node while it sees explorers waiting.  A poll costs a busy device, a long interval between them a thin
// tree, whose fan-out takes that long per doubling.  Every 16 / 8 / 4 / 1 nodes:
// 50x20 LB1 (49.7 M nodes) 29.3 / 29.0 / 30.5 / 45.8 ms, 20x20 LB1 (0.83 M) 4.3 /
// 3.5 / 3.7 / 4.6 ms; again while explorers wait, 20x20 4.1-4.5 ms.  30x20 LB2
// without the team phase: every 16 / 8 nodes 9.3 / 5.9 ms, again while explorers
// wait 3.0 ms.
#ifndef PBB_POLL_EVERY
#define PBB_POLL_EVERY 8
#endif
// What a donor gives: a split fewer than SHARE_NEAR lines above its own row hands
// over a few nodes, less than the hand-over costs the two of them, unless that
// line has SHARE_CELLS cells left (a wide, shallow tree).  A donor whose split
// was SHARE_DEEP lines up or more holds a large interval and polls again at the
// next node.  20x20 LB1 (0.83 M nodes) 2.9 -> 2.5 ms, 30x17 LB1' 6.2 -> 5.4, 47x17
// LB1 (3.4 M) 5.6 -> 4.7, 19x10 LB2 7.6 -> 6.8; 2 lines and 4 cells 2.5, 5.7, 5.0,
// 7.3; SHARE_DEEP 2, 3, 5 without the lower limit 2.8, 2.65, 2.66 at 20x20.
enum { SHARE_NEAR = 3, SHARE_CELLS = 6, SHARE_DEEP = 4 };
// The pool's explorers poll every PBB_POOL_POLL_EVERY nodes (512-instance batch:
// every 8 / 16 / 32 / 64 nodes 49 / 49 / 51 / 53 ms).
#ifndef PBB_POOL_POLL_EVERY
#define PBB_POOL_POLL_EVERY 16
#endif

// A busy explorer reloads the shared incumbent every PBB_BEST_EVERY decomposed
// nodes (power of two; the load is issued before the node's work and applied
// after it), and an idle one when a donation wakes it, so an improvement found
// by one explorer prunes the others' subtrees within that many nodes.  With a
// frozen incumbent nothing changes.  Measured on the 20x5 NEH-incumbent solve
// (4096 explorers): refreshing only at the periodic check (every 64 nodes,
// which most explorers of a small tree never reach) decomposed 126-136 k nodes
// in 5-6 ms; on wake-up and every 64 / 16 / 8 nodes, 12-13 k / 6-10 k / 6 k
// nodes in 1.1-1.4 ms; the 50x20 explorer is within noise at 16.
#ifndef PBB_BEST_EVERY
#define PBB_BEST_EVERY 16
#endif

// The host's interrupt word lives in host memory, so reading it is a PCIe
// round trip.  A busy explorer reads it at every PBB_HOST_POLL_CHECKS-th
// periodic check (one check per 64 decomposed nodes; explorers start at
// staggered phases), and the first one to see it raises the device-side stop
// word that every explorer reads at each check.  Measured at 50x20 with 4096
// explorers: a host read every 64 nodes held the explorer at 720-1100 M
// nodes/s, varying with the host's load; one every 1024 nodes, 1530-1545 M.
#ifndef PBB_HOST_POLL_CHECKS
#define PBB_HOST_POLL_CHECKS 16
#endif

// Device-resident control block of one engine (or pool slot).  The count of
// working explorers takes atomics at every hand-over and the flags are polled
// by idle explorers, so each sits on its own 128-byte line.
struct Ctl {
    int work_count;            // explorers holding an interval
    int pad1[31];
    int done;                  // set when no explorer holds an interval
    int stop;                  // budget / deadline / interrupt
    int pad2[30];
    unsigned long long dec;    // decomposed nodes
    unsigned long long leaves;
    unsigned long long sb;     // simple (LB1) bounds
    unsigned long long jb;     // refinement bounds
    unsigned long long histo[65];   // decomposed nodes per depth (fixed jobs)
    unsigned long long jhisto[65];  // refinement bounds per depth of the bounded node
};

// The instance one explorer works on: its control block, idle
// mask, incumbent and bounded root row (one per engine, one per pool slot).
struct InstRef {
    Ctl *ctl;
    unsigned long long *idle;   // idle mask words, IDLE_STRIDE apart
    int idle_words;
    const int *member;          // pool: explorer of each member of the slot (nullptr: member = explorer)
    const int *occ;             // pool: members so far (nullptr: all words are in use)
    int ub0;                    // initial UB (branching thresholds when not singleNode)
    unsigned long long *best;   // cost << 32 | explorer
    const int *root_row;
    const int *root_dir;
    int m;                      // machines the pair table refers to
    int npairs;
    int pairs_mode;
    const int *pair_ab;
};

struct KArgs {
    DevInst I;
    int E;              // explorers (wavefronts)
    int rows;           // rows per explorer in mat (the largest n served)
    // explorer state in HBM between launches (row stride 64 bytes; the pool keeps none)
    int8_t *mat;        // [E][n][64]
    int8_t *pos;        // [E][64]
    int8_t *end;        // [E][64]
    int8_t *dir;        // [E][64]
    int *line;          // [E]
    int *state;         // [E]
    unsigned *mtag;     // [E] tag of the last message this explorer consumed
    // mailboxes: a donor hands an interval to an idle explorer as one message
    // of 64 self-tagged words (mail_word)
    unsigned long long *mbox;   // [E][64]
    unsigned long long *idle;   // idle mask words, IDLE_STRIDE apart
    int idle_words;
    Ctl *ctl;
    unsigned long long *best;   // cost << 32 | explorer
    int *best_perm;             // [E][64]
    const int *root_row;        // bounded root row [64]
    const int *root_dir;        // [1]
    int *root_row_out;          // written by k_bound_root
    int *root_dir_out;
    // run control
    unsigned long long node_budget;   // 0 = none
    unsigned long long quiet_budget;  // the same while the incumbent has not moved from initial_ub
    unsigned long long deadline;      // wall_clock64 ticks, 0 = none
    const int *host_flag;             // host-mapped interrupt flag (may be NULL)
    // configuration
    int bound_mode, branching, refine, pairs_mode, find_all, single_node, initial_ub;
    int steal_margin;
    unsigned ramp;      // interior nodes an explorer decomposes in a fresh interval before it donates
    int jt_lds;         // bytes of LDS for the staged Johnson table (0: read from global memory)
};

// The root order of k_bound_root, passed by value (no upload before the launch).
struct RootPerm {
    int p[64];
};

// LDS footprint.  Workgroup tables: the machine-major processing times
// pm[m][PM_STRIDE] and the same rows in reversed machine order pmR, with a
// fixed odd row stride (lanes reading one job on different machines, or
// different jobs on one machine, hit distinct banks, and every per-machine
// offset is a compile-time immediate), min_arr, min_dep, per-machine totals,
// and the packed Johnson table when LB2 is used and it is staged.  Per
// wavefront: the IVM matrix (row l holds its n-l cells, rows packed), the
// front/back stack ((n+1) x m ints), the LB1 operand block (2 x m int2) and,
// for the LB2 variant, 64 ints of scratch, then a 64 x int2 sink for the
// lanes past a row in stores that would otherwise need an exec mask.
#define PM_STRIDE 65
__device__ __host__ inline int lds_pm_stride(int) { return PM_STRIDE; }
// Bytes of the staged Johnson table, packed or wide: up to 32 jobs rows of a
// multiple of 64 pairs (lb2_walk), above that rows of npairs; not less for a
// smaller instance in a pool's larger layout.
__device__ __host__ inline int jtab_chunks(int npairs) { return (npairs + 63) / 64; }
__device__ __host__ inline int jtab_lds_bytes(int n, int npairs, bool packed)
{
    const int walk = (n < 32 ? n : 32) * 64 * jtab_chunks(npairs);
    const int rows = n > 32 ? n * npairs : 0;
    return ((walk > rows ? walk : rows) * (packed ? 4 : 8) + 15) & ~15;
}
// jt: bytes set aside for a Johnson table, a multiple of 16
__device__ __host__ inline size_t lds_table_bytes(int m, int jt)
{
    const int mp = (m + 3) & ~3;
    const size_t off = ((size_t)2 * m * PM_STRIDE + 3 * (size_t)mp) * 4;
    return ((off + 15) & ~(size_t)15) + jt;
}
// offset of IVM row l (rows 0..l-1 hold n, n-1, ..., n-l+1 cells)
__device__ __host__ inline int lds_mat_row(int l, int n) { return l * n - (l * (l - 1)) / 2; }
__device__ __host__ inline size_t lds_mat_bytes(int n)
{
    size_t t = (size_t)n * (n + 1) / 2;
    if (t < (size_t)4 * n) t = (size_t)4 * n;  // also holds n ints (NEH order at admission)
    return (t + 15) & ~(size_t)15;
}
__device__ __host__ inline size_t lds_stack_bytes(int n, int m) { return ((size_t)(n + 1) * m * 4 + 15) & ~(size_t)15; }
__device__ __host__ inline size_t lds_wave_bytes(int n, int m, bool scratch)
{
    return lds_mat_bytes(n) + lds_stack_bytes(n, m) + (size_t)m * 16 + (scratch ? 64 * 4 : 0) + 64 * 8;
}
// Explorers (wavefronts) per workgroup of the one-instance engine; they share
// the workgroup's tables.
#ifndef PBB_EXPLORE_WAVES
#define PBB_EXPLORE_WAVES 4
#endif
// LDS size handed to the occupancy query of the persistent kernels.  Their
// explorers wait on one another (hand-overs, the work count), so every
// workgroup of the grid must be resident at once.  The query's count can be
// one workgroup per CU too high when the workgroups fill the CU's LDS to
// within a granule (12x20 with the Johnson table: 3 x 53904 B of 163840 B
// queried as 3, held 2); rounding each workgroup up to 2 KB keeps the grid
// inside what the hardware actually co-schedules.
inline size_t residency_lds_bytes(size_t lds) { return (lds + 2047) & ~(size_t)2047; }
inline size_t explore_lds_bytes(const DevInst &I, bool lb2, int jt)
{
    return lds_table_bytes(I.m, jt) + PBB_EXPLORE_WAVES * lds_wave_bytes(I.n, I.m, lb2);
}
// The packed Johnson table is staged in LDS when it is at most 24 KB: 20 machines up
// to 32 jobs, 14 at any n.  What is not staged is read from global memory
// (consecutive words per step).
#define JTAB_PACKED_MOST (24 * 1024)
// The bytes an engine's number of explorers is found with: those of the packed
// table where three workgroups still share a CU, as their registers allow (the
// 20-machine pool's two do then as well), else none.  An engine holds as many
// intervals as it has explorers, whatever its times.  The shapes of "none": 59-63
// jobs at 14 machines, 54-58 at 15, 49-51 at 16, 43-45 at 17, 40 at 18 (2048
// explorers with the table, 3072 without), and tables above the limit.
inline int explore_jtab_bytes(const DevInst &I)
{
    const int b = jtab_lds_bytes(I.n, I.npairs, true);
    return b <= JTAB_PACKED_MOST && 3 * residency_lds_bytes(explore_lds_bytes(I, true, b)) <= 160 * 1024 ? b : 0;
}
// The team launch (one workgroup) holds at most 16 explorers with LB1 and LB1' (4 per
// SIMD; their explorers take up to 102 registers of 128) and 8 with LB2 (up to 187).
__device__ __host__ constexpr int team_waves_max(int ref) { return ref == 2 ? 8 : 16; }
inline size_t team_lds_bytes(const DevInst &I, bool lb2, int jt, int waves)
{
    return lds_table_bytes(I.m, jt) + (size_t)waves * lds_wave_bytes(I.n, I.m, lb2);
}
inline size_t root_lds_bytes(const DevInst &I) { return lds_table_bytes(I.m, 0) + lds_wave_bytes(I.n, I.m, false); }

// ------------------------------------------------------------------ pool
// Many instances in one resident launch.  Workgroups of W explorers take one
// instance slot at a time: the first group to pop a slot from the request
// queue admits it (tables, idle mask, root), later groups join running slots
// whose explorers are all busy, up to a per-instance explorer cap; work moves
// between the members of a slot through its idle mask exactly as in the
// one-instance engine.  The last member to leave a solved slot writes its
// result record.  Instances with fewer machines than the pool's M are padded
// with zero-time machines, which changes none of the bounds or makespans.
enum { RES_PENDING = 0, RES_SOLVED = 1, RES_ABORTED = 2, RES_INVALID = 3 };
enum { ROLE_EXIT = 0, ROLE_OWNER = 1, ROLE_HELPER = 2 };

#define PBB_POOL_MAXM 20
#define PBB_POOL_ROW 64

struct PoolReq {                  // one request (host-visible when serving)
    int n, m, ub, tag;
    int ptm[PBB_POOL_MAXM * PBB_POOL_ROW];   // [m][n] machine-major, row stride n
};

struct PoolRes {                  // written once, when the instance retires
    int tag;                      // the request's tag, stored last (completion flag)
    int status;                   // RES_*
    int best;                     // optimum (or the UB when no better schedule exists)
    int improved;                 // 1 when perm holds a schedule of cost best
    unsigned long long dec, leaves, sb, jb;
    unsigned long long t_admit, t_done;      // device wall clock
    int perm[PBB_POOL_ROW];
};

struct PoolQueue {                // request queue: slot ids published by tail
    int tail;
    int closed;
    int started;                  // set by every workgroup of k_pool that starts
    int pad[61];
    int ids[1];                   // [qcap]
};

struct PoolSlot {                 // device header of one instance slot
    Ctl c;
    unsigned long long best;      // cost << 32 | explorer
    unsigned long long t_admit;
    int n, m, ub, tag, npairs, root_dir, best_cost, improved, status, jpacked;
    int root_row[PBB_POOL_ROW];
    int perm[PBB_POOL_ROW];
};

// byte offsets inside one slot's arena (all 256-byte aligned)
struct PoolLayout {
    size_t hdr, ptm, minA, minD, pair, key, jtab, idle, member, stride;
};
__device__ __host__ inline size_t pool_al(size_t x) { return (x + 255) & ~(size_t)255; }
__device__ __host__ inline PoolLayout pool_layout(int nmax, int M, int pmax, int members)
{
    const int mp = (M + 3) & ~3;
    PoolLayout L;
    size_t o = 0;
    L.hdr = o;      o += pool_al(sizeof(PoolSlot));
    L.ptm = o;      o += pool_al((size_t)M * nmax * 4);
    L.minA = o;     o += pool_al((size_t)mp * 4);
    L.minD = o;     o += pool_al((size_t)mp * 4);
    L.pair = o;     o += pool_al((size_t)(pmax > 0 ? pmax : 1) * 4);
    L.key = o;      o += pool_al((size_t)(pmax > 0 ? pmax : 1) * nmax * 4);
    L.jtab = o;     o += pool_al((size_t)(pmax > 0 ? pmax : 1) * nmax * 8);
    L.idle = o;     o += pool_al((size_t)idle_words_for(members) * IDLE_STRIDE * 8);
    L.member = o;   o += pool_al((size_t)members * 4);
    L.stride = o;
    return L;
}

struct PoolArgs {
    char *arena;                  // nslots x layout.stride
    int *occ;                     // [nslots] occupancy words (pbb_slot.h)
    PoolLayout lay;
    int nslots;
    int W;                        // explorers (wavefronts) per workgroup
    int epi;                      // explorer cap per instance
    int nmax;                     // largest n served
    int pmax;                     // pair-table capacity
    int idle_words;               // idle mask words per slot (64 members each)
    int jt_lds;                   // bytes of LDS for a staged Johnson table
    int pairs_mode;               // JohnsonMode: pair list built at admission
    int qcap;                     // queue capacity (power of two)
    int sys;                      // req/res/q live in host-mapped memory
    const PoolReq *req;           // [nslots]
    PoolRes *res;                 // [nslots]
    PoolQueue *q;
    unsigned *q_head;             // consumer ticket (device memory)
    Ctl *run;                     // stop word of the launch
    unsigned long long req_ticks; // per-request budget after admission (wall_clock64 ticks), 0 = none
    int ig_iters;                 // IG helper rounds per instance (0 = no helper wave)
};

__device__ __host__ inline size_t pool_lds_bytes(int nmax, int M, int pmax, int jt_lds, int W)
{
    return lds_table_bytes(M, jt_lds) + (size_t)W * lds_wave_bytes(nmax, M, pmax > 0);
}

// per-M kernels (pbb_kernels.hip, one translation unit per M and table form)
template <int M, int TAB> hipError_t launch_explore_m(const KArgs &a, int blocks, hipStream_t s);
template <int M, int TAB> hipError_t launch_team_m(const KArgs &a, hipStream_t s);
template <int M, int TAB> hipError_t occupancy_m(const KArgs &a, int *blocks_per_cu);
template <int M> hipError_t launch_root_m(const KArgs &a, const RootPerm &root_perm, hipStream_t s);

// batched bounds (pbb_bounds.hip, one translation unit per M and batch size).
// Batches of up to BOUNDS_SMALL schedules go a schedule per wavefront, in tiles of
// four: what bounds them is the time of one chain, and a lane that takes every
// machine of every job is slower for one schedule than a wavefront whose lanes are
// the machines.  A kernel of its own: beside the lane-wise chains it costs LB2 a
// third (50x10, 100 k schedules 102 -> 134 us).  One call, tiles of 16 / this: 256
// schedules at 50x20, children 41.8 / 29.0 us, LB2 53.7 / 36.3; at 20x10 28.7 / 25.0
// and 28.3 / 24.6; 4096 at 50x20, children 42.9 / 32.6, LB2 56.0 / 52.1, 8192 43.3 /
// 40.5 and 61.9 / 75.5.
#define BOUNDS_SMALL 4096
template <int M, bool SMALL>
hipError_t launch_bounds_m(int which, const DevInst &I, int count, const int *perms, const int *l1,
                           const int *l2, int arg, int *o1, int *o2, hipStream_t s);

// pool kernels (pbb_pool.hip, one translation unit per M)
template <int M> hipError_t launch_pool_m(const KArgs &a, const PoolArgs &p, int groups, int init_count,
                                          hipStream_t s);
template <int M> hipError_t pool_occupancy_m(const KArgs &a, const PoolArgs &p, int *groups_per_cu);
template <int M>
hipError_t launch_neh_m(const int *ptms, const long long *off, const int *ns, const int *ms, int count, int nmax,
                        int *perms, int *costs, hipStream_t s);

// iterated greedy (pbb_ig.hip, one translation unit per M): acceptance
// thresholds per instance for cost deltas 0..IG_THR-1
#define IG_THR 256
// LDS of the pool's IG helper wave, after the pool's own LDS: acceptance
// thresholds (IG_THR x u64), job totals (64), heads and tails (2 x M x 64)
// and scratch (64 ints)
__device__ __host__ inline size_t pool_ig_bytes(int M) { return (size_t)IG_THR * 8 + ((size_t)2 * M * 64 + 128) * 4; }
__device__ __host__ inline size_t pool_lds_total(const PoolArgs &p, int M)
{
    return pool_lds_bytes(p.nmax, M, p.pmax, p.jt_lds, p.W) + (p.ig_iters > 0 ? pool_ig_bytes(M) : 0);
}
template <int M>
hipError_t launch_ig_m(const int *ptms, const long long *off, const int *ns, const int *ms, int count, int chains,
                       int iters, unsigned long long seed, const unsigned long long *thr, int *perms, int *costs,
                       hipStream_t s);

// runtime-M dispatch (pbb_dispatch.cpp)
hipError_t launch_explore(const KArgs &a, int blocks, hipStream_t s);
// one workgroup of a.E (<= PBB_TEAM_WAVES) explorers
hipError_t launch_team(const KArgs &a, hipStream_t s);
hipError_t explore_occupancy(const KArgs &a, int *blocks_per_cu);
hipError_t launch_root(const KArgs &a, const RootPerm &root_perm, hipStream_t s);
// engine set-up kernels (pbb_setup.hip, one translation unit): the whole
// search space to explorer 0 and every other explorer idle, with the
// control block cleared; the idle mask emptied and the stop word cleared
// before a launch
hipError_t launch_setup_full(const KArgs &a, hipStream_t s);
hipError_t launch_prelaunch(const KArgs &a, hipStream_t s);
// after a launch that stopped early: messages that arrived at explorers which
// had left already become intervals of the saved state
hipError_t launch_collect(const KArgs &a, hipStream_t s);
// which: 0 lb1 children, 1 lb1 node, 2 lb2 node, 3 makespan
hipError_t launch_bounds(int which, const DevInst &I, int count, const int *perms, const int *l1,
                         const int *l2, int arg, int *o1, int *o2, hipStream_t s);
// init_count > 0: batch launch, the queue holds slots 0..init_count-1
hipError_t launch_pool(int M, const KArgs &a, const PoolArgs &p, int groups, int init_count, hipStream_t s);
hipError_t pool_occupancy(int M, const KArgs &a, const PoolArgs &p, int *groups_per_cu);
hipError_t launch_neh(int M, const int *ptms, const long long *off, const int *ns, const int *ms, int count,
                      int nmax, int *perms, int *costs, hipStream_t s);
hipError_t launch_ig(int M, const int *ptms, const long long *off, const int *ns, const int *ms, int count,
                     int chains, int iters, unsigned long long seed, const unsigned long long *thr, int *perms,
                     int *costs, hipStream_t s);

}  // namespace pbb
