// pbb_setup.hip -- set-up kernels of the one-instance engine (compiled once,
// independent of the machine count).  They replace host-to-device copies of
// explorer-sized arrays, so pbb_init_full and pbb_run issue launches on the
// engine's stream and the host waits once, after the explorer kernel.
#include <stddef.h>

#include "pbb_kernels.h"

namespace pbb {

// sequentialbb::initFullInterval (multicore/src/sequentialbb.cpp:66-81): the
// interval [0...0, (n-1)...0] goes to explorer 0, every other explorer is
// idle; the control block is cleared with one explorer holding work.  One
// thread per explorer (pos/end rows of 64 bytes) and per control-block word.
__global__ __launch_bounds__(256) void k_setup_full(KArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < a.E) {
        a.state[t] = t == 0 ? ST_UNFOLD : ST_IDLE;
        int *pw = (int *)(a.pos + (size_t)t * 64);
        int *ew = (int *)(a.end + (size_t)t * 64);
        for (int w = 0; w < 16; w++) {
            pw[w] = 0;
            int packed = 0;
            if (t == 0)
                for (int b = 0; b < 4; b++) {
                    const int i = 4 * w + b;
                    const int d = i < a.I.n ? a.I.n - 1 - i : 0;
                    packed |= (d & 0xff) << (8 * b);
                }
            ew[w] = packed;
        }
    }
    constexpr int words = (int)(sizeof(Ctl) / sizeof(int));
    if (t < words) {
        constexpr int wc = (int)(offsetof(Ctl, work_count) / sizeof(int));
        ((int *)a.ctl)[t] = t == wc ? 1 : 0;
    }
}

// before every explorer launch: the idle mask empty and the stop word clear
__global__ __launch_bounds__(256) void k_prelaunch(KArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < a.idle_words) a.idle[(size_t)t * IDLE_STRIDE] = 0ull;
    if (t == 0) a.ctl->stop = 0;
}

// One wavefront per explorer: a message newer than the one its explorer last
// consumed was handed over while the launch stopped (the donor had claimed the
// explorer, which then left on the stop word).  It becomes the explorer's saved
// interval, as the explorer would have saved it.
__global__ __launch_bounds__(64) void k_collect(KArgs a)
{
    const int e = blockIdx.x, lane = threadIdx.x, n = a.I.n;
    const unsigned w = (unsigned)a.mbox[(size_t)e * 64 + lane];
    if (a.state[e] != ST_IDLE || mail_tag(w) == a.mtag[e]) return;  // uniform: one tag per message
    const int l = __ffsll((unsigned long long)__ballot(mail_job(w) == MAIL_NONE)) - 1;
    int8_t *gm = a.mat + (size_t)e * a.rows * 64;
    for (int r = 0; r < l; r++) {
        const unsigned wr = (unsigned)__shfl((int)w, r, 64);
        gm[r * 64 + lane] = (int8_t)mail_path_cell(lane, mail_pos(wr), (int)mail_job(wr));
    }
    gm[l * 64 + lane] = (int8_t)mail_cell(w);
    a.pos[(size_t)e * 64 + lane] = (int8_t)mail_pos(w);
    a.end[(size_t)e * 64 + lane] = (int8_t)mail_end(w);
    a.dir[(size_t)e * 64 + lane] = (int8_t)mail_dir(w);
    if (lane == 0) {
        a.line[e] = l;
        a.state[e] = ST_ACTIVE;
        a.mtag[e] = mail_tag(w);
    }
}

hipError_t launch_setup_full(const KArgs &a, hipStream_t s)
{
    constexpr int words = (int)(sizeof(Ctl) / sizeof(int));
    const int threads = a.E > words ? a.E : words;
    hipLaunchKernelGGL(k_setup_full, dim3((threads + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_prelaunch(const KArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_prelaunch, dim3((a.idle_words + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_collect(const KArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_collect, dim3(a.E), dim3(64), 0, s, a);
    return hipGetLastError();
}

}  // namespace pbb
