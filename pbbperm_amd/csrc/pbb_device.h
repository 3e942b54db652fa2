// pbb_device.h -- wave64 primitives and the per-wavefront bound routines of
// the gfx950 IVM engine.  One IVM explorer = one 64-lane wavefront:
//   * lane i holds row cell i of the current IVM row (job id, negative when
//     pruned/visited, the flag encoding of common/include/misc.h:19-29);
//   * lane l holds pos[l], end[l], dir[l] of the factoradic interval;
//   * lane s holds entry s of three register stacks (one VGPR per machine):
//       F[s] = completion times of the first s front jobs,
//       B[s] = reverse completion times of the last s back jobs,
//       R[s] = per-machine sum of the jobs still unscheduled at depth s,
//     so the front/back/remain vectors of bound_fsp_weak::computePartial
//     (bounds/src/bound_fsp_weak.cpp:61-130) are read with one v_readlane per
//     machine instead of being recomputed from scratch at every node.
// All arithmetic is int32 max-plus; the recurrences are those of the
// reference, so every value is bit-identical.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define PBB_WAVE 64
#define PBB_INF 0x7fffffff

namespace pbb {

__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ unsigned long long uni64(unsigned long long v)
{
    unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
    unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

__device__ __forceinline__ int rdlane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// write a uniform value into lane l (v_cmp + v_cndmask)
__device__ __forceinline__ int wrlane(int old, int v, int l)
{
    return __lane_id() == l ? v : old;
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// lanes 0..k-1 as a mask, computed in scalar registers (0 <= k <= 64).  A
// ballot of `lane < k && cond` compiles to a VGPR 0/1 select and a second
// compare; lanes_below(k) & ballot(cond) keeps cond's compare mask as is.
__device__ __forceinline__ uint64_t lanes_below(int k) { return k >= 64 ? ~0ull : ((1ull << k) - 1ull); }

__device__ __forceinline__ int shfl(int v, int src) { return __shfl(v, src, PBB_WAVE); }

// Wavefront reductions on DPP lanes moves (row_shr 1,2,4,8 inside each
// 16-lane row, row_bcast:15 and row_bcast:31 across rows): the result is
// complete in lane 63 and read back with v_readlane, without an LDS round
// trip per step.
#define PBB_DPP_REDUCE(NAME, OP, IDENT)                                              \
    __device__ __forceinline__ int NAME(int x)                                       \
    {                                                                                \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x111, 0xF, 0xF, false));   \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x112, 0xF, 0xF, false));   \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x114, 0xF, 0xF, false));   \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x118, 0xF, 0xF, false));   \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x142, 0xA, 0xF, false));   \
        x = OP(x, __builtin_amdgcn_update_dpp(IDENT, x, 0x143, 0xC, 0xF, false));   \
        return __builtin_amdgcn_readlane(x, 63);                                     \
    }

__device__ __forceinline__ int op_add(int a, int b) { return a + b; }
__device__ __forceinline__ int op_min(int a, int b) { return min(a, b); }
__device__ __forceinline__ int op_max(int a, int b) { return max(a, b); }
PBB_DPP_REDUCE(wave_sum, op_add, 0)
PBB_DPP_REDUCE(wave_min, op_min, 0x7fffffff)
PBB_DPP_REDUCE(wave_max, op_max, (int)0x80000000)
#undef PBB_DPP_REDUCE

// ------------------------------------------------------ lane scans (DPP)
// Inclusive prefix scans over lanes 0..31, and over 32..63 by themselves (row_shr
// 1,2,4,8 inside each 16-lane row, then row_bcast:15 into rows 1 and 3).  Lanes
// only combine with lanes to their left, so values in lanes >= the vector length
// are never read.
__device__ __forceinline__ int scan_add32(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);
    return x;
}
__device__ __forceinline__ int scan_max32(int x)
{
    const int lo = (int)0x80000000;
    x = max(x, __builtin_amdgcn_update_dpp(lo, x, 0x111, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(lo, x, 0x112, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(lo, x, 0x114, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(lo, x, 0x118, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(lo, x, 0x142, 0xA, 0xF, false));
    return x;
}

// Max-plus chain of one job over the machines, lane q = machine q:
// c_q = max(base_q, c_{q-1}) + p_q  ==  P_q + max_{i<=q}(base_i - P_{i-1})
// with P the prefix sum of p (the recurrence of bound_fsp_weak.cpp:76-82).
__device__ __forceinline__ int chain_scan(int base, int p)
{
    const int P = scan_add32(p);
    return P + scan_max32(base - (P - p));
}

// lanes i and 32+i both receive x[i] (gfx950 v_permlane32_swap)
__device__ __forceinline__ int bcast_low_half(int x)
{
    return __builtin_amdgcn_permlane32_swap(x, x, false, false)[0];
}
// lanes i and 32+i both receive x[32+i]
__device__ __forceinline__ int bcast_high_half(int x)
{
    return __builtin_amdgcn_permlane32_swap(x, x, false, false)[1];
}

__device__ __forceinline__ int flag_neg(int j) { return j < 0 ? j : -j - 1; }  // misc.h negative()
__device__ __forceinline__ int flag_abs(int j) { return j >= 0 ? j : -j - 1; }  // misc.h absolute()

// Instance tables as seen by the device.
struct DevInst {
    int n, m;
    int mp;               // m, padded to a multiple of 4
    const int *ptm;       // [m][n] machine-major
    const int *min_arr;   // [m] bound_fsp_weak.cpp:270-283
    const int *min_dep;   // [m] bound_fsp_weak.cpp:253-267
    int npairs;
    const int *pair_ab;   // [npairs] a | b << 8, (i<j) lexicographic (bound_fsp_strong.cpp:282-297)
    // [n][npairs]: the i-th job of every pair's Johnson order, packed words
    // (jpacked) or pairs of words
    const void *jtab;
    int jpacked;
};

// Machine pairs of the Johnson bound, one per lane and chunk: chunk c of
// lane l holds pair c*64 + l of the list as a | b << 8, or -1 when there is
// no such pair or the JohnsonMode drops it (pairs_mode 1: pairs ending on the
// last machine; 2: adjacent machines; bound_fsp_strong.cpp:282-297).  Built
// once per explorer, so the pair list is not re-read for every child.
template <int PCH>
__device__ __forceinline__ void pair_lanes(const int *pair_ab, int npairs, int m, int pairs_mode, int (&pinfo)[PCH])
{
    const int lane = lane_id();
#pragma unroll
    for (int c = 0; c < PCH; c++) {
        const int p = c * PBB_WAVE + lane;
        int v = -1;
        if (p < npairs) {
            const int ab = pair_ab[p];
            const int a = ab & 0xff, b = ab >> 8;
            bool use = true;
            if (pairs_mode == 1 && b < m - 1) use = false;
            if (pairs_mode == 2 && b != a + 1) use = false;
            if (use) v = a | (b << 8);
        }
        pinfo[c] = v;
    }
}

// Entry of a Johnson table: job, p_a - p_b and w = p_a + lag, all the bound's
// recurrence needs (lb2_pairs).  Packed in one word when no processing time
// exceeds JPACK_MAX (job in bits 0-5, w in 6-20: at most 19 x 1023; p_a - p_b
// in 21-31), else two words {w, (p_a - p_b) << 6 | job} (times of at most
// 10^6, as the entry points check).
#define JPACK_MAX 1023
__device__ __host__ inline unsigned jpack_word(int job, int pa, int pb, int lag)
{
    return (unsigned)job | ((unsigned)(pa + lag) << 6) | ((unsigned)(pa - pb) << 21);
}
__device__ __host__ inline int2 jpack_pair(int job, int pa, int pb, int lag)
{
    return int2{pa + lag, (int)(((unsigned)(pa - pb) << 6) | (unsigned)job)};
}

// -1 when the job in the low bits of e is unscheduled, else 0
template <bool N32>
__device__ __forceinline__ int job_mask(int e, uint64_t unsched)
{
    if constexpr (N32) return __builtin_amdgcn_sbfe((int)(unsigned)unsched, (unsigned)e, 1u);  // offset: bits 0-4 of e
    else return __builtin_amdgcn_sbfe((int)(unsigned)(unsched >> (e & 63)), 0u, 1u);
}

// The bound from every pair's best (lb2_pairs): the greatest over this lane's
// pairs and the wavefront.
template <int PCH, int ST>
__device__ __forceinline__ int lb2_finish(const int (&pinfo)[PCH], const int (&best)[PCH], const int *fs, const int *gs)
{
    int r = 0;
#pragma unroll
    for (int c = 0; c < PCH; c++) {
        const int info = pinfo[c];
        if (info >= 0) {
            const int a = info & 0xff, b = info >> 8;
            r = max(r, max(best[c] + gs[b * ST], fs[a * ST] + gs[a * ST]));
        }
    }
    return wave_max(r);
}

// Johnson LB2 of one partial schedule over the machine pairs of pinfo
// (bound_fsp_strong.cpp:50-100, :102-162 without early exit, as
// bornes_calculer calls them, :540-560).  fs: its front completion times;
// gs: back completion times plus remaining work (both LDS, by machine, ST words
// apart);
// unsched: the bit set of its unscheduled jobs, not empty.
//
// The reference's recurrence over the unscheduled jobs in Johnson order,
//   t0 += p_a;  t1 = max(t1, t0 + lag) + p_b,
// is t1 = S_b + max(t1_0, max_j (D_j + p_aj + lag_j)) with S_b the sum of all
// p_b and D_j = t0_0 + sum of p_a - p_b over the unscheduled jobs before j, and
// t0 ends at t0_0 + S_a.  So a step is one table word, masked to zero for a
// scheduled job, an add to D and a max, instead of a chain of six dependent
// operations with two selects.  A scheduled job's D + 0 enters the max too:
// never above the true value, since the next unscheduled job's term is at
// least D, and after the last one D + S_b = t0_0 + S_a <= t1.
//
// Lane = pair, all chunks of 64 pairs in one pass (independent chains), the
// table job-major so that the lanes of a step read consecutive words.  The
// former layout (a row of 16-byte entries per pair) had 64 lanes read 64
// cache lines per step from global memory (20 machines), or one LDS bank group
// (n a multiple of 8).  30x20: 42 us per node of 1.4 bounds before.
// Each use of it names one table, in LDS or in global memory: a pointer that
// may be either makes every access a flat load.
template <int PCH, bool N32, bool PACKED, int ST>
__device__ __forceinline__ int lb2_pairs(const int (&pinfo)[PCH], const void *jtab, int n, int npairs,
                                         const int *fs, const int *gs, uint64_t unsched)
{
    const int lane = lane_id();
    int D[PCH], best[PCH], col[PCH];
#pragma unroll
    for (int c = 0; c < PCH; c++) {
        col[c] = min(c * PBB_WAVE + lane, npairs - 1);
        const int ab = pinfo[c] < 0 ? 0 : pinfo[c];
        D[c] = fs[(ab & 0xff) * ST];
        best[c] = fs[(ab >> 8) * ST];
    }
#pragma unroll 4
    for (int i = 0; i < n; i++) {
#pragma unroll
        for (int c = 0; c < PCH; c++) {
            if constexpr (PACKED) {
                int e = (int)((const unsigned *)jtab)[i * npairs + col[c]];
                e &= job_mask<N32>(e, unsched);
                best[c] = max(best[c], D[c] + (int)__builtin_amdgcn_ubfe((unsigned)e, 6u, 15u));
                D[c] += e >> 21;
            } else {
                const int2 e = ((const int2 *)jtab)[i * npairs + col[c]];
                const int m = job_mask<N32>(e.y, unsched);
                best[c] = max(best[c], D[c] + (e.x & m));
                D[c] += (e.y & m) >> 6;
            }
        }
    }
    return lb2_finish<PCH, ST>(pinfo, best, fs, gs);
}

// Entry of the staged table of up to 32 jobs, row i of a pair's column: w of the
// i-th job of the pair's order, the place of job i in that order and p_a - p_b of
// the i-th job.  Packed in one word: w in bits 0-15, the place in 16-20, the
// difference in 21-31; wide in two: w (at most 19 x 10^6) in bits 0-24 and the place
// in 25-29, the difference.
template <bool WIDE>
struct JWalk {
    typedef unsigned Entry;
    static constexpr int PLACE = 16;
    __device__ __forceinline__ static Entry make(unsigned e)
    {
        return ((e >> 6) & 0x7fffu) | (e & 0xffe00000u);
    }
    __device__ __forceinline__ static int w(Entry e) { return (int)(e & 0xffffu); }
    __device__ __forceinline__ static int diff(Entry e) { return (int)e >> 21; }
};
template <>
struct JWalk<true> {
    typedef int2 Entry;
    static constexpr int PLACE = 25;
    __device__ __forceinline__ static Entry make(int2 e) { return make_int2(e.x, e.y >> 6); }
    __device__ __forceinline__ static int w(Entry e) { return e.x & 0x1ffffff; }
    __device__ __forceinline__ static int diff(Entry e) { return e.y; }
};

// The recurrence of lb2_pairs for K children over NCH chunks of 64 pairs, cnt
// steps: places[k][c] has a bit per unscheduled job, at its place in the order
// of this lane's pair, so a step takes the next unscheduled job and the
// scheduled ones cost nothing (7 instructions for each of the n jobs there, 9
// for each unscheduled one here, and those are a third to two thirds of n).
// Rows are a multiple of 64 entries apart, so the lanes of a wavefront read
// distinct banks whatever their places.  512-instance batch 101 -> 86 ms, burst of
// 256 requests 64 -> 46, 30x20 LB2 proof 4.26 -> 4.04.  D and best enter as the children's front
// times on the pair's machines; best leaves without the remaining work.
template <int K, int NCH, bool WIDE>
__device__ __forceinline__ void lb2_walk(const unsigned *tab, int cnt, unsigned (&places)[K][NCH], int (&D)[K][NCH],
                                         int (&best)[K][NCH])
{
    typedef typename JWalk<WIDE>::Entry Entry;
    constexpr unsigned row = 64u * sizeof(Entry);
    const char *col = (const char *)((const Entry *)tab + lane_id());
#pragma unroll 2
    for (int i = 0; i < cnt; i++) {
#pragma unroll
        for (int c = 0; c < NCH; c++) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const unsigned p = (unsigned)__builtin_ctz(places[k][c]);
                places[k][c] &= places[k][c] - 1u;
                const Entry e = *(const Entry *)(col + p * (row * NCH) + c * row);
                best[k][c] = max(best[k][c], D[k][c] + JWalk<WIDE>::w(e));
                D[k][c] += JWalk<WIDE>::diff(e);
            }
        }
    }
}

// lb2_pairs of one schedule with few unscheduled jobs, of a table staged with rows
// of W = 64 PCH words (the columns past the last pair repeat it): place[j * W + c]
// is job j's place in the order of column c.  The lane's mask of places is built
// for the schedule, 3 instructions (4 above 32 jobs) per unscheduled job and
// chunk, and walked as in lb2_walk, 9 (15); lb2_pairs takes 7 (9) for every job.
// 100 k schedules at 50x20, a quarter of the jobs unscheduled on average: 382 -> 276 us.
template <int PCH, bool N32, int ST>
__device__ __forceinline__ int lb2_few(const int (&pinfo)[PCH], const unsigned *tab, const uint8_t *place, const int *fs,
                                       const int *gs, uint64_t unsched)
{
    typedef std::conditional_t<N32, unsigned, uint64_t> Mask;
    constexpr int W = 64 * PCH;
    const int lane = lane_id();
    Mask places[PCH];
    int D[PCH], best[PCH];
#pragma unroll
    for (int c = 0; c < PCH; c++) {
        const int ab = pinfo[c] < 0 ? 0 : pinfo[c];
        D[c] = fs[(ab & 0xff) * ST];
        best[c] = fs[(ab >> 8) * ST];
        places[c] = 0;
    }
    for (uint64_t u = unsched; u; u &= u - 1) {
        const uint8_t *pl = place + (__ffsll((unsigned long long)u) - 1) * W + lane;
#pragma unroll
        for (int c = 0; c < PCH; c++) places[c] |= (Mask)1 << pl[c * 64];
    }
    const int cnt = __popcll(unsched);
#pragma unroll 2
    for (int i = 0; i < cnt; i++) {
#pragma unroll
        for (int c = 0; c < PCH; c++) {
            const int p = N32 ? __builtin_ctz((unsigned)places[c]) : __builtin_ctzll(places[c]);
            places[c] &= places[c] - 1;
            const int e = (int)tab[p * W + c * 64 + lane];
            best[c] = max(best[c], D[c] + (int)__builtin_amdgcn_ubfe((unsigned)e, 6u, 15u));
            D[c] += e >> 21;
        }
    }
    return lb2_finish<PCH, ST>(pinfo, best, fs, gs);
}

// Forms of the Johnson table that an explorer is built for.  The engine has a
// kernel for each (its node loop's registers and code are then one form's); the
// pool's launch meets both, and walks the packed one only.
enum { TAB_ANY = 0, TAB_PACKED = 1, TAB_WIDE = 2 };

// lb2_pairs of an explorer's child where lb2_walk's table does not apply: the
// table of more than 32 jobs in LDS, any in global memory
template <int PCH, int TAB>
__device__ __forceinline__ int lb2_pairs_any(const int (&pinfo)[PCH], bool staged, const unsigned *jtabL,
                                             const void *jtabG, bool packed, int n, int npairs, const int *fs,
                                             const int *gs, uint64_t unsched)
{
    if (TAB == TAB_PACKED || (TAB == TAB_ANY && packed))
        return staged ? lb2_pairs<PCH, false, true, 1>(pinfo, jtabL, n, npairs, fs, gs, unsched)
                      : lb2_pairs<PCH, false, true, 1>(pinfo, jtabG, n, npairs, fs, gs, unsched);
    return staged ? lb2_pairs<PCH, false, false, 1>(pinfo, jtabL, n, npairs, fs, gs, unsched)
                  : lb2_pairs<PCH, false, false, 1>(pinfo, jtabG, n, npairs, fs, gs, unsched);
}

}  // namespace pbb
