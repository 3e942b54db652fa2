// pbb_bounds.hip -- batched bound_abstract calls over device buffers: LB1 of
// all children (bound_fsp_weak::boundChildren, bound_fsp_weak.cpp:193-221), LB1'
// (bornes_calculer, :288-311), Johnson LB2 (bound_fsp_strong.cpp:540-560) and the
// makespan (evalSolution) of explicit partial schedules (perm, l1, l2): front
// perm[0..l1], back perm[l2..n-1], the middle unscheduled.
//
// A workgroup takes tiles of T schedules, its tables staged once:
//   1. chains: one lane per schedule and side, its completion times in
//      registers, so that a job costs 3 instructions per machine for 64 chains
//      (a wavefront per schedule, lane = machine, pays a prefix scan of 25
//      dependent instructions per job for one; small batches take that, BOUNDS_SMALL).
//      Lengths run over 0..n and a wavefront runs as long as its longest chain,
//      so the tile's 2T chains are first sorted by length (a counting sort of 64
//      bins);
//   2. operands: per schedule and machine the front and back times with the
//      remaining work folded in, in LDS;
//   3. the bound: children one lane per child, both directions, over the tile's
//      children laid end to end (a wavefront per schedule leaves the lanes past
//      its k children idle, 12 of 64 in use at 50 jobs over all depths); LB2 one
//      wavefront per schedule, lane = machine pair; the others a lane each.
// What bounds it: the children are LDS reads (two 8-byte operands and a time per
// child and machine) and VALU in about equal parts.
//
// Translation units: compiled once per machine count M (-DPBB_M=<m>), and once more
// for the small batches' kernels (-DPBB_SMALL=true), a code object of their own.
#include "pbb_device.h"
#include "pbb_kernels.h"

namespace pbb {

enum { B_CHILDREN = 0, B_LB1 = 1, B_LB2 = 2, B_MAKESPAN = 3 };

// jobs of a tile's schedules, one byte each; the odd word stride keeps lanes
// that read one position of different schedules on distinct banks
#define BJ_STRIDE 68
#define B_THREADS 256
// schedules of a small batch's tile (BOUNDS_SMALL): one a wavefront
#define B_SMALL (B_THREADS / 64)
// most schedules per tile
__host__ __device__ constexpr int b_tile(int which) { return which == B_LB2 ? 32 : 128; }

// inclusive prefix sum over the 64 lanes
__device__ __forceinline__ int wave_scan(int x)
{
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < PBB_WAVE; o <<= 1) {
        const int y = shfl(x, lane >= o ? lane - o : lane);
        x += lane >= o ? y : 0;
    }
    return x;
}

struct BoundTile {
    int2 *U;                 // [T][2M + 1]: front operands, then back operands (machines reversed)
    uint8_t *jobs;           // [T][BJ_STRIDE]
    uint64_t *mid;           // [T] unscheduled jobs
    int *start;              // [T + 1] first child of every schedule among the tile's
    short *l1, *l2;          // [T]; a malformed schedule has l1 = -2
    unsigned short *order;   // [2T] chains by decreasing length: schedule << 1 | side
    int *hist;               // [64] chains per length, then the next place of each
};

template <int M>
__device__ __host__ inline size_t bound_tile_bytes(int T)
{
    size_t b = (size_t)T * (2 * M + 1) * 8 + (size_t)T * 8 + (size_t)T * BJ_STRIDE;
    b += (size_t)(T + 1) * 4 + 64 * 4 + (size_t)T * 2 * 4;
    return (b + 15) & ~(size_t)15;
}

template <int M>
__device__ __host__ inline size_t bound_table_bytes(const DevInst &I, bool jtab)
{
    size_t b = ((size_t)2 * M * PM_STRIDE + 3 * M) * 4;
    b = (b + 15) & ~(size_t)15;
    if (jtab) b += (size_t)I.n * 64 * jtab_chunks(I.npairs) * 5;  // words, then a byte of place each
    return b;
}

template <int M, int WHICH, bool SMALL>
__global__ __launch_bounds__(B_THREADS) void k_bounds(DevInst I, int count, int tile, const int *perms, const int *l1s,
                                                      const int *l2s, int arg, int *o1, int *o2)
{
    const int T = SMALL ? B_SMALL : tile;
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, lane = lane_id(), wave = uni(tid >> 6);
    const int n = I.n;
    constexpr int US = 2 * M + 1;
    const bool jtab = WHICH == B_LB2 && I.jpacked;

    int *pm = (int *)smem, *pmR = pm + M * PM_STRIDE;
    int *minA = pmR + M * PM_STRIDE, *minD = minA + M, *tot = minD + M;
    unsigned *jtabL = (unsigned *)(smem + bound_table_bytes<M>(I, false));
    BoundTile S;
    S.U = (int2 *)(smem + bound_table_bytes<M>(I, jtab));
    S.mid = (uint64_t *)(S.U + (size_t)T * US);
    S.start = (int *)(S.mid + T);
    S.hist = S.start + T + 1;
    S.l1 = (short *)(S.hist + 64);
    S.l2 = S.l1 + T;
    S.order = (unsigned short *)(S.l2 + T);
    S.jobs = (uint8_t *)(S.order + 2 * T);

    // The next tile's schedules are loaded while this one is worked on, a row
    // per wavefront and register: a load per row and a wait for each took most
    // of the time (50x20: 700 us per million schedules, 473 this way).
    // Ids outside 0..n-1 become 63, which is none of them (n <= 63).
    constexpr int ROWS = (SMALL ? B_SMALL : b_tile(WHICH)) / (B_THREADS / 64);
    int rows[ROWS], pl1 = 0, pl2 = 0;
    const auto prefetch = [&](long long s0) {
        const int ns = (int)max(0ll, min((long long)T, count - s0));
        const int *src = perms + s0 * n;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int t = wave + r * (B_THREADS / 64);
            if (t < ns) rows[r] = src[(size_t)t * n + min(lane, n - 1)];
        }
        if (WHICH != B_MAKESPAN && tid < ns) {
            pl1 = l1s[s0 + tid];
            pl2 = l2s[s0 + tid];
        }
    };
    prefetch((long long)blockIdx.x * T);

#pragma unroll
    for (int r = 0; r < (M + 3) / 4; r++) {
        const int q = wave + 4 * r;
        if (q < M) {
            const int v = I.ptm[q * n + min(lane, n - 1)];
            if (lane < n) pm[q * PM_STRIDE + lane] = pmR[(M - 1 - q) * PM_STRIDE + lane] = v;
            const int sum = wave_sum(lane < n ? v : 0);
            if (lane == 0) tot[q] = sum;
        }
    }
    if (tid < M) {
        minA[tid] = I.min_arr[tid];
        minD[tid] = I.min_dep[tid];
    }
    uint8_t *place = (uint8_t *)(jtabL + (size_t)n * 64 * jtab_chunks(I.npairs));
    if (jtab) {
        const int W = 64 * jtab_chunks(I.npairs);
        for (int i = wave; i < n; i += B_THREADS / 64)
            for (int c = lane; c < W; c += 64) {
                const unsigned e = ((const unsigned *)I.jtab)[i * I.npairs + min(c, I.npairs - 1)];
                jtabL[i * W + c] = e;
                place[(e & 63u) * W + c] = (uint8_t)i;
            }
    }
    constexpr int PCH = (M * (M - 1) / 2 + PBB_WAVE - 1) / PBB_WAVE;
    int pinfo[PCH];
    if constexpr (WHICH == B_LB2) pair_lanes<PCH>(I.pair_ab, I.npairs, I.m, arg, pinfo);
    // the chains of a tile of up to 32 schedules are one wavefront's: no order
    const bool sorted = !SMALL && WHICH != B_MAKESPAN && T > 32;

    for (long long s0 = (long long)blockIdx.x * T; s0 < count; s0 += (long long)gridDim.x * T) {
        const int ns = (int)min((long long)T, count - s0);
        __syncthreads();  // the last tile's readers are done
        if (tid < 64) S.hist[tid] = 0;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int t = wave + r * (B_THREADS / 64);
            if (t < ns) S.jobs[t * BJ_STRIDE + lane] = (uint8_t)(lane < n && (unsigned)rows[r] < (unsigned)n ? rows[r] : 63);
        }
        int l1 = n - 1, l2 = n;  // the makespan is a chain of all jobs
        if constexpr (WHICH != B_MAKESPAN) {
            l1 = pl1;
            l2 = pl2;
        }
        prefetch(s0 + (long long)gridDim.x * T);
        __syncthreads();
        // inputs must be permutations of 0..n-1 with -1 <= l1 < l2 <= n;
        // anything else yields -1 outputs instead of out-of-range table reads
        if (tid < ns) {
            const uint32_t *js = (const uint32_t *)(S.jobs + tid * BJ_STRIDE);
            uint64_t seen = 0ull;
            for (int i = 0; i < n; i += 4) {
                const uint32_t w = js[i >> 2];  // past the jobs: 63
                seen |= (1ull << (w & 63u)) | (1ull << ((w >> 8) & 63u)) | (1ull << ((w >> 16) & 63u)) |
                        (1ull << (w >> 24));
            }
            const bool bad = (seen & ~(1ull << 63)) != lanes_below(n) || l1 < -1 || l2 > n || l1 >= l2;
            if constexpr (WHICH == B_LB1 || WHICH == B_LB2) {
                uint64_t mid = 0ull;
                if (!bad)
                    for (int i = l1 + 1; i < l2; i++) mid |= 1ull << S.jobs[tid * BJ_STRIDE + i];
                S.mid[tid] = mid;
            }
            if (bad) {
                l1 = -2;
                l2 = n;
            }
            S.l1[tid] = (short)l1;
            S.l2[tid] = (short)l2;
            if (sorted) {
                atomicAdd(&S.hist[bad ? 0 : l1 + 1], 1);
                atomicAdd(&S.hist[n - l2], 1);
            } else {
                S.order[tid] = (unsigned short)(2 * tid);
                S.order[ns + tid] = (unsigned short)(2 * tid + 1);
            }
        }
        __syncthreads();
        // places by decreasing length: chains longer than this lane's bin come
        // before it (lane 0 = the longest)
        if (sorted && wave == 0) {
            const int c = S.hist[63 - lane];
            S.hist[63 - lane] = wave_scan(c) - c;
        }
        if (WHICH == B_CHILDREN && wave == 1) {
            int base = 0;
            for (int b = 0; b < ns; b += 64) {
                const int t = b + lane;
                const int k = t < ns && S.l1[t] >= -1 ? S.l2[t] - S.l1[t] - 1 : 0;
                const int x = wave_scan(k);
                if (t < ns) S.start[t] = base + x - k;
                base += rdlane(x, 63);
            }
            if (lane == 0) S.start[ns] = base;
        }
        if (sorted) {
            __syncthreads();
            if (tid < ns) {
                S.order[atomicAdd(&S.hist[l1 < -1 ? 0 : l1 + 1], 1)] = (unsigned short)(2 * tid);
                S.order[atomicAdd(&S.hist[n - l2], 1)] = (unsigned short)(2 * tid + 1);
            }
        }
        __syncthreads();
        // chains: front over machines 0..M-1 from min_arr, back over machines
        // M-1..0 from min_dep (as starting from zero, bound_fsp_weak.cpp:61-110)
        if constexpr (SMALL) {
            // a wavefront per schedule, half of it per side, lane = machine: a job
            // costs the wavefront a scan, but the chain is short
            if (wave < ns) {
                const int side = lane >> 5, q = lane & 31, qq = min(q, M - 1);
                const int lf = uni(S.l1[wave] < -1 ? 0 : S.l1[wave] + 1), lb = uni(n - S.l2[wave]);
                const int len = side ? lb : lf, step = side ? -1 : 1;
                const uint8_t *js = S.jobs + wave * BJ_STRIDE + (side ? n - 1 : 0);
                const int *tab = (side ? pmR : pm) + qq * PM_STRIDE;
                int f = side ? minD[M - 1 - qq] : minA[qq], w = 0;
                int v = tab[js[0]];
                const int steps = max(lf, lb);
                for (int i = 0; i < steps; i++) {
                    js += step;
                    const int next = tab[js[0] & 63];  // past the chain: unused
                    const int p = i < len && q < M ? v : 0;
                    const int c = chain_scan(q < M ? f : 0, p);
                    f = i < len ? c : f;
                    w += p;
                    v = next;
                }
                if (q < M) S.U[(size_t)wave * US + side * M + q] = make_int2(f, w);
            }
        } else {
            for (int c = tid; c < 2 * ns; c += B_THREADS) {
                const int s = S.order[c] >> 1, side = S.order[c] & 1;
                const int len = side ? n - S.l2[s] : (S.l1[s] < -1 ? 0 : S.l1[s] + 1);
                const uint8_t *js = S.jobs + s * BJ_STRIDE + (side ? n - 1 : 0);
                const int *tab = side ? pmR : pm;
                const int step = side ? -1 : 1;
                int f[M], w[M], v[M];
#pragma unroll
                for (int q = 0; q < M; q++) {
                    f[q] = side ? minD[M - 1 - q] : minA[q];
                    w[q] = 0;
                }
                // the next job's times are read before this one's are used (one
                // past the chain: any byte, kept inside the table and unused)
                int next = js[step] & 63;
                {
                    const int *p = tab + js[0];
#pragma unroll
                    for (int q = 0; q < M; q++) v[q] = p[q * PM_STRIDE];
                }
                for (int i = 0; i < len; i++) {
                    const int *p = tab + next;
                    js += step;
                    next = js[step] & 63;
                    int t = 0;
#pragma unroll
                    for (int q = 0; q < M; q++) {
                        t = max(t, f[q]) + v[q];  // times are not negative: t = 0 before the first machine
                        f[q] = t;
                        w[q] += v[q];
                        v[q] = p[q * PM_STRIDE];
                    }
                }
                int2 *u = S.U + (size_t)s * US + side * M;
#pragma unroll
                for (int q = 0; q < M; q++) u[q] = make_int2(f[q], w[q]);
            }
        }
        __syncthreads();
        // (f, work in front), (b, work behind) -> (f, r + b), (b, f + r)
        for (int i = tid; i < ns * M; i += B_THREADS) {
            const int s = i / M, q = i - s * M;
            int2 *u = S.U + (size_t)s * US;
            const int2 x = u[q], y = u[M + M - 1 - q];
            const int r = tot[q] - x.y - y.y;
            u[q].y = r + y.x;
            u[M + M - 1 - q].y = x.x + r;
        }
        if constexpr (WHICH == B_CHILDREN) {
            // jobs that are no children get 0, malformed schedules -1
            int *r1 = o1 + s0 * n, *r2 = arg ? o2 + s0 * n : nullptr;
            for (int s = wave; s < ns; s += B_THREADS / 64) {
                const int v = S.l1[s] < -1 ? -1 : 0;
                if (lane < n) {
                    r1[(size_t)s * n + lane] = v;
                    if (arg) r2[(size_t)s * n + lane] = v;
                }
            }
            __syncthreads();
            const int kids = S.start[ns];
            for (int c = tid; c < kids; c += B_THREADS) {
                // the schedule of child c: the last one that starts at or before it
                int s = 0, hi = ns;
                while (hi - s > 1) {
                    const int h = (s + hi) >> 1;
                    if (S.start[h] <= c) s = h;
                    else hi = h;
                }
                const int job = S.jobs[s * BJ_STRIDE + S.l1[s] + 1 + (c - S.start[s])];
                const int2 *u = S.U + (size_t)s * US;
                int p[M];
#pragma unroll
                for (int q = 0; q < M; q++) p[q] = pm[q * PM_STRIDE + job];
                int t = 0, lb = 0;
#pragma unroll
                for (int q = 0; q < M; q++) {
                    const int2 x = u[q];
                    t = max(t, x.x);
                    lb = max(lb, t + x.y);
                    t += p[q];
                }
                r1[(size_t)s * n + job] = lb;
                if (arg) {
                    t = lb = 0;
#pragma unroll
                    for (int q = 0; q < M; q++) {
                        const int2 x = u[M + q];
                        t = max(t, x.x);
                        lb = max(lb, t + x.y);
                        t += p[M - 1 - q];
                    }
                    r2[(size_t)s * n + job] = lb;
                }
            }
        } else {
            __syncthreads();
            // a lane per schedule: LB1' and, where at most one job (LB2) or
            // none is left, the makespan of the completed permutation
            // (bound_fsp_strong.cpp:543-546)
            for (int s = tid; s < ns; s += B_THREADS) {
                const int2 *u = S.U + (size_t)s * US;
                const int k = WHICH == B_MAKESPAN ? 0 : __popcll(S.mid[s]);
                int v = 0, t = 0;
                if (S.l1[s] < -1) {
                    v = -1;
                } else if (WHICH == B_LB1 && k > 0) {
                    // t = max over machines up to q of f + r
#pragma unroll
                    for (int q = 0; q < M; q++) {
                        const int2 y = u[M + M - 1 - q];
                        t = max(t, y.y);
                        v = max(v, t + y.x);
                    }
                } else {
                    const int *p = pm + (k ? __ffsll((unsigned long long)S.mid[s]) - 1 : 0);
#pragma unroll
                    for (int q = 0; q < M; q++) {
                        const int pq = k ? p[q * PM_STRIDE] : 0;
                        const int x = u[q].x;
                        t = k ? max(t, x) + pq : x;
                        v = max(v, t + u[M + M - 1 - q].x);
                    }
                }
                if (WHICH != B_LB2 || k <= 1) o1[s0 + s] = v;
            }
            if constexpr (WHICH == B_LB2) {
                for (int s = wave; s < ns; s += B_THREADS / 64) {
                    const uint64_t mid = uni64(S.mid[s]);
                    if (__popcll(mid) <= 1) continue;
                    const int *fs = (const int *)(S.U + (size_t)s * US);
                    const int k = __popcll(mid);
                    int v;
                    if (!jtab) v = lb2_pairs<PCH, false, false, 2>(pinfo, I.jtab, n, I.npairs, fs, fs + 1, mid);
                    else if (n <= 32)
                        v = 12 * k < 7 * n ? lb2_few<PCH, true, 2>(pinfo, jtabL, place, fs, fs + 1, mid)
                                           : lb2_pairs<PCH, true, true, 2>(pinfo, jtabL, n, 64 * PCH, fs, fs + 1, mid);
                    else
                        v = 19 * k < 9 * n ? lb2_few<PCH, false, 2>(pinfo, jtabL, place, fs, fs + 1, mid)
                                           : lb2_pairs<PCH, false, true, 2>(pinfo, jtabL, n, 64 * PCH, fs, fs + 1, mid);
                    if (lane == 0) o1[s0 + s] = v;
                }
            }
        }
    }
}

// Tile size: up to 128 schedules, as many as leave room for three workgroups
// per CU beside the tables (two with a Johnson table); a smaller batch is spread
// over the CUs in smaller tiles, 16 schedules at least.
template <int M, int WHICH, bool SMALL>
static hipError_t launch(const DevInst &I, int count, const int *perms, const int *l1, const int *l2, int arg, int *o1,
                         int *o2, hipStream_t s)
{
    const size_t tab = bound_table_bytes<M>(I, WHICH == B_LB2 && I.jpacked);
    const size_t room = 160 * 1024 / (WHICH == B_LB2 ? 2 : 3) - 2048;
    const auto tiles = [&](int T) { return (int)(((long long)count + T - 1) / T); };
    int T = SMALL ? B_SMALL : b_tile(WHICH);
    while (T > 16 && tab + bound_tile_bytes<M>(T) > room) T -= 16;
    while (T > 16 && tiles(T) < 512) T -= 16;
    const size_t lds = tab + bound_tile_bytes<M>(T);
    if (lds > 64 * 1024)
        if (const hipError_t err = hipFuncSetAttribute((const void *)k_bounds<M, WHICH, SMALL>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
            return err;
    const int resident = 256 * (int)(160 * 1024 / lds < 8 ? 160 * 1024 / lds : 8);
    const int grid = tiles(T) < resident ? tiles(T) : resident;
    hipLaunchKernelGGL((k_bounds<M, WHICH, SMALL>), dim3(grid), dim3(B_THREADS), lds, s, I, count, T, perms, l1, l2,
                       arg, o1, o2);
    return hipGetLastError();
}

template <int M, bool SMALL>
hipError_t launch_bounds_m(int which, const DevInst &I, int count, const int *perms, const int *l1, const int *l2,
                           int arg, int *o1, int *o2, hipStream_t s)
{
    switch (which) {
    case B_CHILDREN: return launch<M, B_CHILDREN, SMALL>(I, count, perms, l1, l2, arg, o1, o2, s);
    case B_LB1: return launch<M, B_LB1, SMALL>(I, count, perms, l1, l2, arg, o1, o2, s);
    case B_LB2: return launch<M, B_LB2, SMALL>(I, count, perms, l1, l2, arg, o1, o2, s);
    default: return launch<M, B_MAKESPAN, SMALL>(I, count, perms, l1, l2, arg, o1, o2, s);
    }
}

#ifdef PBB_M
#ifndef PBB_SMALL
#define PBB_SMALL false
#endif
template hipError_t launch_bounds_m<PBB_M, PBB_SMALL>(int, const DevInst &, int, const int *, const int *, const int *,
                                                      int, int *, int *, hipStream_t);
#endif

}  // namespace pbb
