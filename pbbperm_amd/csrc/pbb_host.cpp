// pbb_host.cpp -- host side of the MI355X IVM engine: the C ABI of
// include/pbb_engine.h.  Instance tables are built here and uploaded once;
// everything on the node path runs in the HIP kernels of pbb_kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cctype>
#include <chrono>
#include <cstddef>
#include <climits>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <sstream>
#include <string>
#include <thread>
#include <vector>

#include "../../include/pbb_engine.h"
#include "pbb_internal.h"
#include "pbb_kernels.h"

using namespace pbb;

// ------------------------------------------------------------ device tables
void pbb::build_tables(const int32_t *ptm, int n, int m, HostTables &T)
{
    T.n = n;
    T.m = m;
    T.mp = (m + 3) & ~3;
    T.ptm.assign(ptm, ptm + (size_t)n * m);
    // bound_fsp_weak::fillMinTimeArrDep (bound_fsp_weak.cpp:248-286)
    T.min_arr.assign(m, INT_MAX);
    T.min_dep.assign(m, INT_MAX);
    T.min_arr[0] = 0;
    T.min_dep[m - 1] = 0;
    for (int j = 0; j < n; j++) {
        int tail = 0;
        for (int k = m - 2; k >= 0; k--) {
            tail += ptm[(k + 1) * n + j];
            T.min_dep[k] = std::min(T.min_dep[k], tail);
        }
        int head = 0;
        for (int k = 1; k < m; k++) {
            head += ptm[(k - 1) * n + j];
            T.min_arr[k] = std::min(T.min_arr[k], head);
        }
    }
    // machine pairs and Johnson/Mitten orders (bound_fsp_strong.cpp:264-436).
    // Ties inside a key leave the two-machine optimum unchanged; a stable
    // order by (set, key) is used.
    T.npairs = m * (m - 1) / 2;
    T.pair_ab.clear();
    T.jtab.assign((size_t)T.npairs * n, int4{0, 0, 0, 0});
    int p = 0;
    for (int a = 0; a < m - 1; a++)
        for (int b = a + 1; b < m; b++, p++) {
            T.pair_ab.push_back(a | (b << 8));
            std::vector<int> lag(n), set(n), key(n), ord(n);
            for (int j = 0; j < n; j++) {
                int l = 0;
                for (int k = a + 1; k < b; k++) l += ptm[k * n + j];
                lag[j] = l;
                bool first = ptm[a * n + j] < ptm[b * n + j];
                set[j] = first ? 1 : 2;
                key[j] = (first ? ptm[a * n + j] : ptm[b * n + j]) + l;
                ord[j] = j;
            }
            std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) {
                if (set[x] != set[y]) return set[x] < set[y];
                return set[x] == 1 ? key[x] < key[y] : key[x] > key[y];
            });
            for (int i = 0; i < n; i++) {
                int j = ord[i];
                T.jtab[(size_t)p * n + i] = int4{j, ptm[a * n + j], ptm[b * n + j], lag[j]};
            }
        }
    T.jpacked = *std::max_element(T.ptm.begin(), T.ptm.end()) <= JPACK_MAX;
    T.jdev.resize(T.jtab.size() * (T.jpacked ? 1 : 2));
    for (int q = 0; q < T.npairs; q++)
        for (int i = 0; i < n; i++) {
            const int4 e = T.jtab[(size_t)q * n + i];
            const size_t at = (size_t)i * T.npairs + q;
            if (T.jpacked) {
                T.jdev[at] = jpack_word(e.x, e.y, e.z, e.w);
            } else {
                const int2 v = jpack_pair(e.x, e.y, e.z, e.w);
                T.jdev[2 * at] = (unsigned)v.x;
                T.jdev[2 * at + 1] = (unsigned)v.y;
            }
        }
}

// The tables in one device allocation, filled by one copy: a table of its own
// each, and an engine's state in 11 more, were 17 allocations and 6 copies of an
// engine's creation (20x5 solve with its creation 1.03 -> 0.86 ms).
struct DevTables {
    char *mem = nullptr;
    DevInst I{};
};

static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

// Offsets of ptm, min_arr, min_dep, pair_ab and jtab (in either form).
struct TableLayout {
    size_t min_arr, min_dep, pair_ab, jtab, bytes;
    explicit TableLayout(const HostTables &T)
    {
        min_arr = al256(T.ptm.size() * 4);
        min_dep = min_arr + al256((size_t)T.m * 4);
        pair_ab = min_dep + al256((size_t)T.m * 4);
        jtab = pair_ab + al256((size_t)T.npairs * 4);
        bytes = jtab + T.jtab.size() * 8;
    }
};

// the tables as they lie in DevTables::mem, up to the end of the Johnson table's present form
static std::vector<char> pack_tables(const HostTables &T)
{
    const TableLayout L(T);
    std::vector<char> v(L.jtab + T.jdev.size() * 4);
    memcpy(v.data(), T.ptm.data(), T.ptm.size() * 4);
    memcpy(v.data() + L.min_arr, T.min_arr.data(), (size_t)T.m * 4);
    memcpy(v.data() + L.min_dep, T.min_dep.data(), (size_t)T.m * 4);
    if (T.npairs) {
        memcpy(v.data() + L.pair_ab, T.pair_ab.data(), (size_t)T.npairs * 4);
        memcpy(v.data() + L.jtab, T.jdev.data(), T.jdev.size() * 4);
    }
    return v;
}

static int upload_tables(const HostTables &T, DevTables &D)
{
    const TableLayout L(T);
    const std::vector<char> v = pack_tables(T);
    HIPCHK(hipMalloc(&D.mem, L.bytes));
    HIPCHK(hipMemcpy(D.mem, v.data(), v.size(), hipMemcpyHostToDevice));
    D.I.n = T.n;
    D.I.m = T.m;
    D.I.mp = T.mp;
    D.I.ptm = (const int *)D.mem;
    D.I.min_arr = (const int *)(D.mem + L.min_arr);
    D.I.min_dep = (const int *)(D.mem + L.min_dep);
    D.I.npairs = T.npairs;
    D.I.pair_ab = (const int *)(D.mem + L.pair_ab);
    D.I.jtab = D.mem + L.jtab;
    D.I.jpacked = T.jpacked ? 1 : 0;
    return PBB_OK;
}

static void free_tables(DevTables &D)
{
    hipFree(D.mem);
    D = DevTables{};
}

int pbb::check_device()
{
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count < 1) return fail(PBB_E_NODEVICE, "no HIP device available");
    return PBB_OK;
}

// ------------------------------------------------------------ bound library
struct pbb_bounds {
    HostTables T;
    DevTables D;
};

extern "C" int pbb_bounds_create(const int32_t *ptm, int n, int m, pbb_bounds **out)
{
    if (!out) return fail(PBB_E_ARG, "null out");
    int rc = check_shape(ptm, n, m);
    if (rc) return rc;
    if ((rc = check_device())) return rc;
    pbb_bounds *b = new pbb_bounds();
    build_tables(ptm, n, m, b->T);
    rc = upload_tables(b->T, b->D);
    if (rc) {
        free_tables(b->D);
        delete b;
        return rc;
    }
    *out = b;
    return PBB_OK;
}

extern "C" int pbb_bounds_destroy(pbb_bounds *b)
{
    if (!b) return PBB_OK;
    free_tables(b->D);
    delete b;
    return PBB_OK;
}

static int bounds_call(pbb_bounds *b, int which, int count, const int *perms, const int *l1,
                       const int *l2, int arg, int *o1, int *o2, void *stream)
{
    if (!b || count < 0 || !perms || !o1) return fail(PBB_E_ARG, "bad bound batch arguments");
    if (which != 3 && (!l1 || !l2)) return fail(PBB_E_ARG, "null l1/l2");
    if (which == 0 && arg && !o2) return fail(PBB_E_ARG, "null ce with both=1");
    if (count == 0) return PBB_OK;
    HIPCHK(launch_bounds(which, b->D.I, count, perms, l1, l2, arg, o1, o2, (hipStream_t)stream));
    return PBB_OK;
}

extern "C" int pbb_lb1_children_batch(pbb_bounds *b, int count, const int *perms, const int *l1,
                                      const int *l2, int both, int *cb, int *ce, void *stream)
{
    return bounds_call(b, 0, count, perms, l1, l2, both ? 1 : 0, cb, ce, stream);
}

extern "C" int pbb_lb1_node_batch(pbb_bounds *b, int count, const int *perms, const int *l1,
                                  const int *l2, int *lb, void *stream)
{
    return bounds_call(b, 1, count, perms, l1, l2, 0, lb, nullptr, stream);
}

extern "C" int pbb_lb2_node_batch(pbb_bounds *b, int count, const int *perms, const int *l1,
                                  const int *l2, int pairs, int *lb, void *stream)
{
    if (pairs < 0 || pairs > 2) return fail(PBB_E_ARG, "pairs mode %d", pairs);
    return bounds_call(b, 2, count, perms, l1, l2, pairs, lb, nullptr, stream);
}

extern "C" int pbb_makespan_batch(pbb_bounds *b, int count, const int *perms, int *cmax, void *stream)
{
    return bounds_call(b, 3, count, perms, nullptr, nullptr, 0, cmax, nullptr, stream);
}

// ------------------------------------------------------------------ engine
// Launches with one form of the Johnson table: the bytes of LDS it is staged in (0:
// read from global memory), the explorers that are resident with them and the
// explorers of the team launch (0: none fits).  The resident ones can be fewer than
// the engine's (a wide table of 30 jobs and 20 machines, 46 KB, leaves one or two
// workgroups per CU); a launch then uses the table with so many as long as they
// hold all intervals, else all explorers without it.  A wide table is staged whatever
// it costs: read from global memory beside thousands of polling explorers, a step
// of the recurrence takes a memory round trip (times of 11 to 1089, global / staged:
// 18x20, 3065 nodes 11.5 / 1.7 ms; 30x20, 268 k nodes 35 / 3.7 ms; 45x17, 28 k nodes
// 23 / 3.8 ms).
struct JForm {
    int bytes, explorers, team;
};

struct pbb_engine {
    pbb_config cfg;
    HostTables T;
    DevTables D;
    int n, m, E;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // device buffers, in one allocation
    char *mem = nullptr;
    int8_t *mat = nullptr, *pos = nullptr, *end = nullptr, *dir = nullptr;
    int *line = nullptr, *state = nullptr;
    unsigned *mtag = nullptr;
    unsigned long long *mbox = nullptr;
    unsigned long long *idle = nullptr;
    Ctl *ctl = nullptr;
    unsigned long long *best = nullptr;
    int *best_perm = nullptr, *root_row = nullptr, *root_dir = nullptr;
    int *host_flag = nullptr, *host_flag_d = nullptr;
    // pinned, in one allocation with host_flag: read-back of the control block and
    // the incumbent word after a launch
    Ctl *ctl_h = nullptr;
    unsigned long long *best_h = nullptr;
    JForm form[2]{};  // wide, packed (DevInst::jpacked)
    int top = 0;      // all intervals are held by explorers below this
    // host state
    std::vector<int> root_perm;
    int inc_cost;
    std::vector<int> inc_perm;
    int initial_ub;
    bool root_bounded = false;
    bool initialized = false;
    unsigned long long exported_dec = 0, exported_leaves = 0;
    // counters carried in from a checkpoint file (works::init_infile restores
    // simpleBounds, distributed/src/works.cpp:81-83; the unit's exploredNodes)
    unsigned long long dec_base = 0, sb_base = 0;
    // the device control block's done flag and node count as of the last
    // set-up or launch (nothing else writes them between launches)
    bool done_host = false;
    unsigned long long dec_dev = 0;
    // whether the next pbb_run starts with the team launch (set by pbb_init_full)
    bool team_pending = false;
    double last_ms = 0.0;
    int wall_khz = 100000;
};

static KArgs make_args(pbb_engine *e)
{
    KArgs a{};
    a.I = e->D.I;
    a.E = e->E;
    a.rows = e->n;
    a.mat = e->mat;
    a.pos = e->pos;
    a.end = e->end;
    a.dir = e->dir;
    a.line = e->line;
    a.state = e->state;
    a.mtag = e->mtag;
    a.mbox = e->mbox;
    a.idle = e->idle;
    a.idle_words = idle_words_for(e->E);
    a.ctl = e->ctl;
    a.best = e->best;
    a.best_perm = e->best_perm;
    a.root_row = e->root_row;
    a.root_dir = e->root_dir;
    a.root_row_out = e->root_row;
    a.root_dir_out = e->root_dir;
    a.host_flag = e->host_flag_d;
    a.bound_mode = e->cfg.bound_mode;
    a.branching = e->cfg.branching;
    a.refine = e->cfg.refine;
    a.pairs_mode = e->cfg.johnson_pairs;
    a.find_all = e->cfg.find_all;
    a.single_node = e->cfg.single_node;
    a.initial_ub = e->initial_ub;
    a.steal_margin = e->cfg.steal_margin;
    a.ramp = (unsigned)e->cfg.ramp_nodes;
    return a;
}

// Every copy of engine state is ordered on the engine's stream (launches are
// not followed by a wait of their own; the host waits where it reads).
static hipError_t copy_sync(pbb_engine *e, void *dst, const void *src, size_t bytes, hipMemcpyKind kind)
{
    hipError_t r = hipMemcpyAsync(dst, src, bytes, kind, e->stream);
    if (r == hipSuccess) r = hipStreamSynchronize(e->stream);
    return r;
}

// resident explorers of a device-wide launch of the given form with jt bytes of LDS for its table
static int capacity(pbb_engine *e, int packed, int jt, int *explorers)
{
    KArgs a = make_args(e);
    a.I.jpacked = packed;
    a.jt_lds = jt;
    int bpc = 0;
    HIPCHK(explore_occupancy(a, &bpc));
    if (bpc < 1) return fail(PBB_E_CAPACITY, "explorer kernel does not fit one workgroup per CU (LDS)");
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    int cus = 0;
    HIPCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    *explorers = bpc * cus * PBB_EXPLORE_WAVES;
    return PBB_OK;
}

static bool with_lb2(const pbb_engine *e) { return e->cfg.bound_mode != 0 && e->cfg.refine == 1; }

// The engine's explorers: what is resident with the packed table's bytes, and
// without a table where the instance is of the wide form (no fewer).  The query loads
// the form's kernels, a tenth of a millisecond the first time, so the packed form asks
// for its own only; a retargeted engine, which starts from explorer 0 alone, launches
// as many of the other form as plan_form finds.
static int engine_explorers(pbb_engine *e)
{
    int cap = 0, wide = 0;
    const bool lb2 = with_lb2(e);
    if (const int rc = capacity(e, 1, lb2 ? explore_jtab_bytes(e->D.I) : 0, &cap)) return rc;
    if (lb2 && !e->D.I.jpacked) {
        if (const int rc = capacity(e, 0, 0, &wide)) return rc;
        cap = std::min(cap, wide);
    }
    e->E = std::max(1, std::min(e->cfg.nb_ivms, cap));
    return PBB_OK;
}

// The present form's launches (JForm), found once per form.
static int plan_form(pbb_engine *e)
{
    const int packed = e->D.I.jpacked;
    JForm &f = e->form[packed];
    if (f.explorers) return PBB_OK;
    const bool lb2 = with_lb2(e);
    JForm g{0, e->E, 0};
    if (lb2) g.bytes = jtab_lds_bytes(e->n, e->D.I.npairs, packed);
    if (packed ? g.bytes > JTAB_PACKED_MOST : explore_lds_bytes(e->D.I, lb2, g.bytes) > 160 * 1024) g.bytes = 0;
    if (g.bytes && !(packed && g.bytes == explore_jtab_bytes(e->D.I))) {
        int cap = 0;
        if (const int rc = capacity(e, packed, g.bytes, &cap)) return rc;
        g.explorers = std::min(e->E, cap);
    }
    // the team: up to team_waves_max explorers whose LDS fits one workgroup
    g.team = std::min(e->E, team_waves_max(e->cfg.bound_mode == 0 ? 0 : (lb2 ? 2 : 1)));
    if (e->cfg.team_waves > 0) g.team = std::min(g.team, e->cfg.team_waves);
    while (g.team > 0 && team_lds_bytes(e->D.I, lb2, g.bytes, g.team) > 160 * 1024) g.team--;
    f = g;
    return PBB_OK;
}
static const JForm &form_of(const pbb_engine *e) { return e->form[e->D.I.jpacked]; }

extern "C" int pbb_destroy(pbb_engine *e)
{
    if (!e) return PBB_OK;
    hipFree(e->mem);
    if (e->host_flag) hipHostFree(e->host_flag);
    if (e->ev0) hipEventDestroy(e->ev0);
    if (e->ev1) hipEventDestroy(e->ev1);
    if (e->stream) hipStreamDestroy(e->stream);
    free_tables(e->D);
    delete e;
    return PBB_OK;
}

extern "C" int pbb_create(const int32_t *ptm, int n, int m, const pbb_config *cfg, int ub,
                          const int *ub_perm, pbb_engine **out)
{
    if (!out || !cfg) return fail(PBB_E_ARG, "null argument");
    *out = nullptr;
    int rc = check_shape(ptm, n, m);
    if (rc) return rc;
    if ((rc = validate(cfg))) return rc;
    // an incumbent cost is a makespan: a negative one (PBB_UB_NEH of the pool
    // entry points, say) would prune every root child and report it as optimal
    if (ub < 0) return fail(PBB_E_ARG, "incumbent cost %d is negative (INT_MAX = none)", ub);
    if (ub_perm && !is_perm(ub_perm, n)) return fail(PBB_E_ARG, "incumbent order is not a permutation of 0..%d", n - 1);
    if ((rc = check_device())) return rc;
    pbb_engine *e = new pbb_engine();
    e->cfg = *cfg;
    e->n = n;
    e->m = m;
    e->inc_cost = ub;
    e->initial_ub = ub;
    e->inc_perm.resize(n);
    for (int i = 0; i < n; i++) e->inc_perm[i] = ub_perm ? ub_perm[i] : i;
    e->root_perm.resize(n);
    for (int i = 0; i < n; i++) e->root_perm[i] = i;
    build_tables(ptm, n, m, e->T);
#define TRY(x)                \
    do {                      \
        int r_ = (x);         \
        if (r_) {             \
            pbb_destroy(e);   \
            return r_;        \
        }                     \
    } while (0)
#define HTRY(x) TRY(([&]() -> int { HIPCHK(x); return PBB_OK; })())
    TRY(upload_tables(e->T, e->D));
    HTRY(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
    HTRY(hipEventCreate(&e->ev0));
    HTRY(hipEventCreate(&e->ev1));
    TRY(engine_explorers(e));
    TRY(plan_form(e));
    size_t E = (size_t)e->E;
    // cleared once: mailboxes, idle mask, state words, tags
    const size_t idle_bytes = (size_t)idle_words_for(e->E) * IDLE_STRIDE * 8;
    const size_t share_bytes = E * 64 * 8 + idle_bytes + E * 8;
    size_t bytes = 0;
    const auto part = [&](size_t b) {
        const size_t at = bytes;
        bytes += al256(b);
        return at;
    };
    const size_t mat = part(E * n * 64), pos = part(E * 64), end = part(E * 64), dir = part(E * 64), line = part(E * 4);
    const size_t mbox = part(share_bytes), ctl = part(sizeof(Ctl)), best = part(8), best_perm = part(E * 64 * 4);
    const size_t root_row = part(64 * 4), root_dir = part(4);
    HTRY(hipMalloc(&e->mem, bytes));
    e->mat = (int8_t *)(e->mem + mat);
    e->pos = (int8_t *)(e->mem + pos);
    e->end = (int8_t *)(e->mem + end);
    e->dir = (int8_t *)(e->mem + dir);
    e->line = (int *)(e->mem + line);
    e->mbox = (unsigned long long *)(e->mem + mbox);
    e->idle = e->mbox + E * 64;
    e->state = (int *)((char *)e->idle + idle_bytes);
    e->mtag = (unsigned *)(e->state + E);
    e->ctl = (Ctl *)(e->mem + ctl);
    e->best = (unsigned long long *)(e->mem + best);
    e->best_perm = (int *)(e->mem + best_perm);
    e->root_row = (int *)(e->mem + root_row);
    e->root_dir = (int *)(e->mem + root_dir);
    // the interrupt word on a line of its own
    HTRY(hipHostMalloc((void **)&e->host_flag, 256 + al256(sizeof(Ctl)) + 8, hipHostMallocMapped));
    e->ctl_h = (Ctl *)((char *)e->host_flag + 256);
    e->best_h = (unsigned long long *)((char *)e->ctl_h + al256(sizeof(Ctl)));
    *e->host_flag = 0;
    HTRY(hipHostGetDevicePointer((void **)&e->host_flag_d, e->host_flag, 0));
    int dev = 0;
    HTRY(hipGetDevice(&dev));
    HTRY(hipDeviceGetAttribute(&e->wall_khz, hipDeviceAttributeWallClockRate, dev));
    HTRY(hipMemsetAsync(e->mbox, 0, share_bytes, e->stream));
    unsigned long long packed = ((unsigned long long)(unsigned)ub << 32) | 0xffffffffull;
    HTRY(copy_sync(e, e->best, &packed, 8, hipMemcpyHostToDevice));
#undef HTRY
#undef TRY
    *out = e;
    return PBB_OK;
}

extern "C" int pbb_set_root(pbb_engine *e, const int *root_perm)
{
    if (!e || !root_perm) return fail(PBB_E_ARG, "null argument");
    std::vector<int> seen(e->n, 0);
    for (int i = 0; i < e->n; i++) {
        if (root_perm[i] < 0 || root_perm[i] >= e->n || seen[root_perm[i]]++)
            return fail(PBB_E_ARG, "root order is not a permutation");
    }
    e->root_perm.assign(root_perm, root_perm + e->n);
    e->root_bounded = false;
    return PBB_OK;
}

// take the device incumbent word (read back already) into the host's copy
static int take_incumbent(pbb_engine *e, unsigned long long packed)
{
    int cost = (int)(packed >> 32);
    unsigned who = (unsigned)(packed & 0xffffffffull);
    if (cost < e->inc_cost && who != 0xffffffffu && (int)who < e->E) {
        std::vector<int> p(64);
        HIPCHK(copy_sync(e, p.data(), e->best_perm + (size_t)who * 64, 64 * 4, hipMemcpyDeviceToHost));
        e->inc_cost = cost;
        e->inc_perm.assign(p.begin(), p.begin() + e->n);
    }
    return PBB_OK;
}

static int sync_incumbent(pbb_engine *e)
{
    HIPCHK(copy_sync(e, e->best_h, e->best, 8, hipMemcpyDeviceToHost));
    return take_incumbent(e, *e->best_h);
}

// ivm_bound::boundRoot (ivm_bound.cpp:273-330) under the current incumbent:
// the host's copy is current here (every launch ends by reading the device
// word back, and pbb_set_incumbent writes both).  The launch is only
// enqueued; the set-up and explorer launches after it on the same stream
// read its output.
static int bound_root(pbb_engine *e)
{
    if (e->root_bounded) return PBB_OK;
    e->initial_ub = e->inc_cost;
    RootPerm rp{};
    std::copy(e->root_perm.begin(), e->root_perm.end(), rp.p);
    KArgs a = make_args(e);
    HIPCHK(launch_root(a, rp, e->stream));
    e->root_bounded = true;
    return PBB_OK;
}

// reset the explorer pool: explorers in `active` get (pos, end) and unfold,
// the others are registered idle.
static int setup_pool(pbb_engine *e, const std::vector<int> &ids, const int *pos, const int *end)
{
    const int n = e->n, E = e->E;
    std::vector<int> state(E, ST_IDLE);
    std::vector<int8_t> hp((size_t)E * 64, 0), he((size_t)E * 64, 0);
    for (size_t k = 0; k < ids.size(); k++) {
        int id = ids[k];
        state[id] = ST_UNFOLD;
        for (int i = 0; i < n; i++) {
            hp[(size_t)id * 64 + i] = (int8_t)pos[k * n + i];
            he[(size_t)id * 64 + i] = (int8_t)end[k * n + i];
        }
    }
    // The idle mask starts empty: idle explorers register themselves when
    // their wavefront runs (pbb_run empties it again before every launch).
    Ctl c;
    memset(&c, 0, sizeof c);
    c.work_count = (int)ids.size();
    c.done = ids.empty() ? 1 : 0;
    HIPCHK(copy_sync(e, e->state, state.data(), (size_t)E * 4, hipMemcpyHostToDevice));
    HIPCHK(copy_sync(e, e->pos, hp.data(), hp.size(), hipMemcpyHostToDevice));
    HIPCHK(copy_sync(e, e->end, he.data(), he.size(), hipMemcpyHostToDevice));
    HIPCHK(copy_sync(e, e->ctl, &c, sizeof c, hipMemcpyHostToDevice));
    e->exported_dec = e->exported_leaves = 0;
    e->dec_base = e->sb_base = 0;
    e->done_host = c.done != 0;
    e->dec_dev = 0;
    e->team_pending = false;
    e->top = ids.empty() ? 0 : *std::max_element(ids.begin(), ids.end()) + 1;
    e->initialized = true;
    return PBB_OK;
}

// The whole search space to explorer 0, the others idle: two launches
// enqueued on the engine's stream (root bounding, set-up), no copy and no
// wait; pbb_run's launches follow them on the stream.
extern "C" int pbb_init_full(pbb_engine *e)
{
    if (!e) return fail(PBB_E_ARG, "null engine");
    int rc = bound_root(e);
    if (rc) return rc;
    KArgs a = make_args(e);
    HIPCHK(launch_setup_full(a, e->stream));
    e->exported_dec = e->exported_leaves = 0;
    e->dec_base = e->sb_base = 0;
    e->done_host = false;
    e->dec_dev = 0;
    e->top = 1;
    e->initialized = true;
    e->team_pending = form_of(e).team > 0 && e->cfg.team_nodes > 0;
    return PBB_OK;
}

extern "C" int pbb_init_intervals(pbb_engine *e, int nb, const int *ids, const int *pos, const int *end)
{
    if (!e || nb < 0 || (nb > 0 && (!ids || !pos || !end))) return fail(PBB_E_ARG, "bad arguments");
    if (nb > e->E) return fail(PBB_E_CAPACITY, "cannot handle more than %d intervals", e->E);
    std::vector<int> seen(e->E, 0), idv(nb);
    for (int k = 0; k < nb; k++) {
        if (ids[k] < 0 || ids[k] >= e->E || seen[ids[k]]++)
            return fail(PBB_E_ARG, "interval id %d invalid or repeated", ids[k]);
        for (int i = 0; i < e->n; i++) {
            int lim = e->n - i;
            if (pos[k * e->n + i] < 0 || pos[k * e->n + i] >= lim || end[k * e->n + i] < 0 ||
                end[k * e->n + i] >= lim)
                return fail(PBB_E_ARG, "interval %d: factoradic digit %d out of range", k, i);
        }
        idv[k] = ids[k];
    }
    int rc = bound_root(e);
    if (rc) return rc;
    return setup_pool(e, idv, pos, end);
}

// One launch: empty the idle mask and clear the stop word (explorers idle at
// the end of the previous launch register again when they run, so the mask
// never names a wavefront that is not resident), then the explorers, either
// the device-wide grid or the one-workgroup team; the control block and the
// incumbent word come back into pinned memory behind them, and the host
// waits once.  Returns the launch's device time in *ms.
static int launch_once(pbb_engine *e, bool team, uint64_t node_budget, uint64_t quiet_budget, double time_budget_s,
                       float *ms)
{
    *e->host_flag = 0;
    KArgs a = make_args(e);
    const JForm &f = form_of(e);
    if (team) {
        a.E = f.team;
        a.jt_lds = f.bytes;
    } else if (f.bytes && e->top <= f.explorers) {
        a.E = f.explorers;
        a.jt_lds = f.bytes;
    }
    a.idle_words = idle_words_for(a.E);
    e->top = std::max(e->top, a.E);
    a.node_budget = node_budget ? e->dec_dev + node_budget : 0;
    a.quiet_budget = e->dec_dev + quiet_budget;
    a.deadline = time_budget_s > 0 ? (unsigned long long)(time_budget_s * e->wall_khz * 1000.0) : 0;
    HIPCHK(launch_prelaunch(a, e->stream));
    HIPCHK(hipEventRecord(e->ev0, e->stream));
    if (team) HIPCHK(launch_team(a, e->stream));
    else HIPCHK(launch_explore(a, (a.E + PBB_EXPLORE_WAVES - 1) / PBB_EXPLORE_WAVES, e->stream));
    HIPCHK(hipEventRecord(e->ev1, e->stream));
    HIPCHK(hipMemcpyAsync(e->ctl_h, e->ctl, sizeof(Ctl), hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipMemcpyAsync(e->best_h, e->best, 8, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    HIPCHK(hipEventElapsedTime(ms, e->ev0, e->ev1));
    const Ctl &c = *e->ctl_h;
    e->done_host = c.done != 0;
    e->dec_dev = c.dec;
    if (!c.done) HIPCHK(launch_collect(a, e->stream));
    return take_incumbent(e, *e->best_h);
}

// Nodes of the team phase while the incumbent has not moved, and once it has.
// team_nodes as the caller set it, unless it is the default: then the engine
// chooses.  The team pays on trees that end within it; on a larger one it holds
// the device back, so it gets about the time that a device-wide launch needs to
// fan out: a quarter of team_nodes with LB1 (0.15-0.18 us a node), an eighth with a
// refinement bound (0.42 and 0.78 us with LB2 at 10 and 20 machines).  A quarter / a
// half / all of it with LB1: 2457 nodes 0.46 / 0.46 / 0.46 ms, 5394 nodes 1.0 / 1.07 /
// 0.8, 31 k nodes 1.58 / 1.8 / 2.35; an eighth 1735 nodes 0.67 against 0.47.  An
// eighth / all of it with LB2: 20x10 (3636 nodes) 1.13 / 1.34, 30x20 (14 k nodes) 2.5 /
// 7.6; LB1' 20x10 (8 k nodes) 1.1 / 1.2, 30x17 (45 k) 1.47 / 2.4.  Once the team has
// found a better schedule it keeps all of team_nodes, a quarter with LB2: more
// explorers would search more of what the next one prunes (20x5 from NEH, the share /
// this: LB1 1.08 / 0.8, LB1' 1.3 / 0.87, LB2 1.9 / 1.1; with LB2 half of it brings no
// more, and 256 instances of the batch one after the other take 0.376 s at the share,
// 0.386 at a quarter, 0.408 at half, 0.458 at all).  An engine of no more explorers
// than the team has nothing to gain from the second launch, and a run for fewer
// nodes than team_nodes stays with the team, which stops within a few hundred nodes of
// its budget; thousands of explorers, each of which looks every 64 nodes, overrun it by
// as many.
struct TeamBudget {
    uint64_t quiet, moved;
};
static TeamBudget team_budget(const pbb_engine *e, uint64_t node_budget)
{
    const uint64_t most = (uint64_t)e->cfg.team_nodes;
    if (node_budget && node_budget <= most) return {node_budget, node_budget};
    if (e->cfg.team_nodes != PBB_TEAM_NODES_DEFAULT || e->E <= form_of(e).team) return {most, most};
    if (with_lb2(e)) return {most / 8, most / 4};
    return {most / (e->cfg.bound_mode == 0 ? 4 : 8), most};
}

// A search started by pbb_init_full runs first on the team (one workgroup)
// for team_budget() decomposed nodes; what is left then continues on the
// device-wide grid from the team's saved intervals.
extern "C" int pbb_run(pbb_engine *e, uint64_t node_budget, double time_budget_s, int *all_done)
{
    if (!e) return fail(PBB_E_ARG, "null engine");
    if (!e->initialized) return fail(PBB_E_STATE, "pbb_run before pbb_init_full/pbb_init_intervals");
    if (all_done) *all_done = 0;
    if (e->done_host) {
        if (all_done) *all_done = 1;
        return PBB_OK;
    }
    e->last_ms = 0.0;
    float ms = 0.f;
    if (e->team_pending) {
        e->team_pending = false;
        const TeamBudget tb = team_budget(e, node_budget);
        const uint64_t before = e->dec_dev;
        const auto t0 = std::chrono::steady_clock::now();
        int rc = launch_once(e, true, tb.moved, tb.quiet, time_budget_s, &ms);
        if (rc) return rc;
        e->last_ms += ms;
        if (e->done_host) {
            if (all_done) *all_done = 1;
            return PBB_OK;
        }
        const uint64_t used = e->dec_dev - before;
        if (node_budget) {
            if (used >= node_budget) return PBB_OK;
            node_budget -= used;
        }
        if (time_budget_s > 0) {
            time_budget_s -= std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (time_budget_s <= 0) return PBB_OK;
        }
    }
    int rc = launch_once(e, false, node_budget, node_budget, time_budget_s, &ms);
    if (rc) return rc;
    e->last_ms += ms;
    if (all_done) *all_done = e->done_host ? 1 : 0;
    return PBB_OK;
}

// every active explorer's interval (state != idle)
static int export_intervals(pbb_engine *e, int *pos, int *end, int *ids, int *nb, int max)
{
    const int n = e->n, E = e->E;
    std::vector<int> st(E);
    std::vector<int8_t> hp((size_t)E * 64), he((size_t)E * 64);
    HIPCHK(copy_sync(e, st.data(), e->state, (size_t)E * 4, hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, hp.data(), e->pos, hp.size(), hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, he.data(), e->end, he.size(), hipMemcpyDeviceToHost));
    memset(pos, 0, sizeof(int) * (size_t)max * n);
    memset(end, 0, sizeof(int) * (size_t)max * n);
    int k = 0;
    for (int i = 0; i < E; i++)
        if (st[i] != ST_IDLE) {
            ids[k] = i;
            for (int d = 0; d < n; d++) {
                pos[(size_t)k * n + d] = hp[(size_t)i * 64 + d];
                end[(size_t)k * n + d] = he[(size_t)i * 64 + d];
            }
            k++;
        }
    *nb = k;
    return PBB_OK;
}

extern "C" int pbb_get_intervals(pbb_engine *e, int *pos, int *end, int *ids, int *nb, int max,
                                 uint64_t *decomposed, uint64_t *leaves)
{
    if (!e || !pos || !end || !ids || !nb) return fail(PBB_E_ARG, "null argument");
    if (max < e->E) return fail(PBB_E_CAPACITY, "buffer too small (%d < %d)", max, e->E);
    int rc = export_intervals(e, pos, end, ids, nb, max);
    if (rc) return rc;
    Ctl c;
    HIPCHK(copy_sync(e, &c, e->ctl, sizeof c, hipMemcpyDeviceToHost));
    if (decomposed) *decomposed = c.dec - e->exported_dec;
    if (leaves) *leaves = c.leaves - e->exported_leaves;
    e->exported_dec = c.dec;
    e->exported_leaves = c.leaves;
    return PBB_OK;
}

extern "C" int pbb_get_incumbent(pbb_engine *e, int *cost, int *perm)
{
    if (!e || !cost) return fail(PBB_E_ARG, "null argument");
    int rc = sync_incumbent(e);
    if (rc) return rc;
    *cost = e->inc_cost;
    if (perm) std::copy(e->inc_perm.begin(), e->inc_perm.end(), perm);
    return PBB_OK;
}

extern "C" int pbb_set_incumbent(pbb_engine *e, int cost, const int *perm)
{
    if (!e) return fail(PBB_E_ARG, "null engine");
    if (cost < 0) return fail(PBB_E_ARG, "incumbent cost %d is negative", cost);
    if (perm && !is_perm(perm, e->n)) return fail(PBB_E_ARG, "incumbent order is not a permutation of 0..%d", e->n - 1);
    int rc = sync_incumbent(e);
    if (rc) return rc;
    if (cost >= e->inc_cost) return PBB_OK;  // solution::update keeps strict improvements
    e->inc_cost = cost;
    if (perm) e->inc_perm.assign(perm, perm + e->n);
    unsigned long long packed = ((unsigned long long)(unsigned)cost << 32) | 0xffffffffull;
    HIPCHK(copy_sync(e, e->best, &packed, 8, hipMemcpyHostToDevice));
    return PBB_OK;
}

extern "C" int pbb_get_stats(pbb_engine *e, pbb_stats *st)
{
    if (!e || !st) return fail(PBB_E_ARG, "null argument");
    Ctl c;
    HIPCHK(copy_sync(e, &c, e->ctl, sizeof c, hipMemcpyDeviceToHost));
    memset(st, 0, sizeof *st);
    st->decomposed = e->dec_base + c.dec;
    st->leaves = c.leaves;
    st->simple_bounds = e->sb_base + c.sb;
    st->johnson_bounds = c.jb;
    st->explorers = e->E;
    // a finished search leaves every explorer idle
    int act = 0;
    if (!c.done) {
        std::vector<int> s(e->E);
        HIPCHK(copy_sync(e, s.data(), e->state, (size_t)e->E * 4, hipMemcpyDeviceToHost));
        for (int v : s) act += v != ST_IDLE;
    }
    st->active = act;
    st->kernel_ms = e->last_ms;
    for (int i = 0; i <= PBB_MAX_JOBS + 1; i++) {
        st->depth_histo[i] = c.histo[i];
        st->refine_histo[i] = c.jhisto[i];
    }
    return PBB_OK;
}

extern "C" int pbb_get_deep_subproblems(pbb_engine *e, int *perms, int max, int *count)
{
    if (!e || !count || max < 0 || (max > 0 && !perms)) return fail(PBB_E_ARG, "bad arguments");
    *count = 0;
    if (!e->initialized || max == 0) return PBB_OK;
    const int n = e->n, m = e->m, E = e->E;
    std::vector<int> st(E), line(E);
    std::vector<int8_t> pos((size_t)E * 64), dir((size_t)E * 64), mat((size_t)E * n * 64);
    HIPCHK(copy_sync(e, st.data(), e->state, (size_t)E * 4, hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, line.data(), e->line, (size_t)E * 4, hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, pos.data(), e->pos, pos.size(), hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, dir.data(), e->dir, dir.size(), hipMemcpyDeviceToHost));
    HIPCHK(copy_sync(e, mat.data(), e->mat, mat.size(), hipMemcpyDeviceToHost));
    std::vector<std::pair<int, int>> order;  // (cost, explorer)
    std::vector<int> sched((size_t)E * n);
    for (int i = 0; i < E; i++) {
        if (st[i] != ST_ACTIVE) continue;
        const int L = line[i];
        if (L < 0 || L >= n) continue;
        const int8_t *rows = mat.data() + (size_t)i * n * 64;
        int *sc = sched.data() + (size_t)i * n;
        int l1 = 0, l2 = n - 1;
        for (int l = 0; l < L; l++) {
            const int p = pos[(size_t)i * 64 + l];
            const int v = rows[l * 64 + p];
            const int job = v < 0 ? -v - 1 : v;
            if (dir[(size_t)i * 64 + l] == 0) sc[l1++] = job;
            else sc[l2--] = job;
        }
        for (int c = 0; c < n - L; c++) {
            const int v = rows[L * 64 + c];
            sc[l1 + c] = v < 0 ? -v - 1 : v;
        }
        order.emplace_back(host_partial_makespan(e->T.ptm.data(), n, m, sc, n), i);
    }
    std::sort(order.begin(), order.end());
    const int k = std::min((int)order.size(), max);
    for (int j = 0; j < k; j++)
        std::copy(sched.begin() + (size_t)order[j].second * n, sched.begin() + (size_t)(order[j].second + 1) * n,
                  perms + (size_t)j * n);
    *count = k;
    return PBB_OK;
}

extern "C" int pbb_interrupt(pbb_engine *e)
{
    if (!e) return fail(PBB_E_ARG, "null engine");
    __atomic_store_n(e->host_flag, 1, __ATOMIC_SEQ_CST);
    return PBB_OK;
}

extern "C" int pbb_query_explorers(int n, int m, const pbb_config *cfg, int *explorers)
{
    if (!cfg || !explorers) return fail(PBB_E_ARG, "null argument");
    std::vector<int32_t> ptm((size_t)n * m, 1);
    pbb_engine *e = nullptr;
    int rc = pbb_create(ptm.data(), n, m, cfg, INT_MAX, nullptr, &e);
    if (rc) return rc;
    *explorers = e->E;
    return pbb_destroy(e);
}

// ------------------------------------------------- plain stream replay
// The one-instance engine re-pointed at a new instance of the same shape:
// tables re-uploaded into the existing buffers, incumbent and root reset.
static int engine_retarget(pbb_engine *e, const int32_t *ptm, int ub, const int *ub_perm)
{
    build_tables(ptm, e->n, e->m, e->T);
    const HostTables &T = e->T;
    const std::vector<char> v = pack_tables(T);
    HIPCHK(copy_sync(e, e->D.mem, v.data(), v.size(), hipMemcpyHostToDevice));
    e->D.I.jpacked = T.jpacked ? 1 : 0;
    if (const int rc = plan_form(e)) return rc;
    e->inc_cost = ub;
    e->initial_ub = ub;
    for (int i = 0; i < e->n; i++) {
        e->root_perm[i] = i;
        e->inc_perm[i] = ub_perm ? ub_perm[i] : i;
    }
    e->root_bounded = false;
    e->initialized = false;
    *e->host_flag = 0;
    unsigned long long packed = ((unsigned long long)(unsigned)ub << 32) | 0xffffffffull;
    HIPCHK(copy_sync(e, e->best, &packed, 8, hipMemcpyHostToDevice));
    return PBB_OK;
}

extern "C" int pbb_plain_replay(const pbb_config *cfg, int count, const int32_t *ptms, const int *n,
                                const int *m, const int *ub, const double *arrival_s, double time_budget_s,
                                double request_budget_s, pbb_result *out, double *latency_ms, double *wall_s)
{
    if (!cfg || count < 0 || (count > 0 && (!ptms || !n || !m || !ub || !arrival_s || !out || !latency_ms)))
        return fail(PBB_E_ARG, "bad replay arguments");
    if (request_budget_s < 0) return fail(PBB_E_ARG, "negative request budget");
    std::vector<size_t> off(count + 1, 0);
    for (int i = 0; i < count; i++) {
        int rc = check_shape(ptms + off[i], n[i], m[i]);
        if (rc) return rc;
        off[i + 1] = off[i] + (size_t)n[i] * m[i];
    }
    // one engine per shape, created before the clock starts
    std::map<std::pair<int, int>, pbb_engine *> eng;
    auto cleanup = [&]() {
        for (auto &kv : eng) pbb_destroy(kv.second);
    };
    for (int i = 0; i < count; i++) {
        auto key = std::make_pair(n[i], m[i]);
        if (eng.count(key)) continue;
        pbb_engine *e = nullptr;
        int rc = pbb_create(ptms + off[i], n[i], m[i], cfg, INT_MAX, nullptr, &e);
        if (rc) {
            cleanup();
            return rc;
        }
        eng[key] = e;
    }
    const double budget = time_budget_s > 0 ? time_budget_s : 600.0;
    const auto t0 = std::chrono::steady_clock::now();
    auto now_s = [&]() { return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(); };
    double t_last = 0.0;
    int rc = PBB_OK;
    for (int i = 0; i < count; i++) {
        memset(&out[i], 0, sizeof out[i]);
        out[i].tag = i;
        out[i].status = PBB_RES_ABORTED;
        out[i].best = ub[i];
        latency_ms[i] = -1.0;
    }
    for (int i = 0; i < count && rc == PBB_OK; i++) {
        while (now_s() < arrival_s[i]) std::this_thread::yield();
        double left = budget - now_s();
        if (left <= 0) break;
        if (request_budget_s > 0 && request_budget_s < left) left = request_budget_s;
        pbb_engine *e = eng[std::make_pair(n[i], m[i])];
        // PBB_UB_NEH (any negative ub): the incumbent is the host NEH's, as the
        // pool computes it on the device at admission; its time counts in the
        // request's latency there too
        int u = ub[i];
        std::vector<int> neh_perm;
        if (u < 0) {
            neh_perm.resize(n[i]);
            for (int j = 0; j < n[i]; j++) neh_perm[j] = j;
            if ((rc = pbb_neh(ptms + off[i], n[i], m[i], neh_perm.data(), &u))) break;
        }
        if ((rc = engine_retarget(e, ptms + off[i], u, u == ub[i] ? nullptr : neh_perm.data()))) break;
        const double t_admit = now_s();
        int all_done = 0;
        if ((rc = pbb_init_full(e))) break;
        if ((rc = pbb_run(e, 0, left, &all_done))) break;
        int cost = 0;
        std::vector<int> perm(e->n);
        if ((rc = pbb_get_incumbent(e, &cost, perm.data()))) break;
        pbb_stats st;
        if ((rc = pbb_get_stats(e, &st))) break;
        const double tc = now_s();
        pbb_result &o = out[i];
        o.status = all_done ? PBB_RES_SOLVED : PBB_RES_ABORTED;
        o.best = cost;
        // improved: perm holds a schedule of cost best (the NEH order counts)
        o.improved = (cost < u || u != ub[i]) ? 1 : 0;
        o.decomposed = st.decomposed;
        o.leaves = st.leaves;
        o.simple_bounds = st.simple_bounds;
        o.johnson_bounds = st.johnson_bounds;
        o.admit_ms = t_admit * 1e3;
        o.done_ms = tc * 1e3;
        for (int j = 0; j < PBB_MAX_JOBS; j++) o.perm[j] = (o.improved && j < e->n) ? perm[j] : -1;
        latency_ms[i] = (tc - arrival_s[i]) * 1e3;
        t_last = tc;
        replay_progress("plain replay", i, i + 1, count);
    }
    cleanup();
    if (wall_s) *wall_s = count ? t_last - arrival_s[0] : 0.0;
    return rc;
}

// ----------------------------------------------------------- checkpoint
extern "C" int pbb_checkpoint_save(pbb_engine *e, const char *path)
{
    if (!e || !path) return fail(PBB_E_ARG, "null argument");
    if (!e->initialized) return fail(PBB_E_STATE, "checkpoint before pbb_init_full/pbb_init_intervals");
    const int n = e->n, E = e->E;
    std::vector<int> pos((size_t)E * n), end((size_t)E * n), ids(E);
    int nb = 0;
    int rc = export_intervals(e, pos.data(), end.data(), ids.data(), &nb, E);
    if (rc) return rc;
    if ((rc = sync_incumbent(e))) return rc;
    pbb_stats st;
    if ((rc = pbb_get_stats(e, &st))) return rc;
    pbb_checkpoint c;
    memset(&c, 0, sizeof c);
    c.n = n;
    c.root_cost = e->initial_ub;
    for (int i = 0; i < n; i++) {
        c.root_perm[i] = e->root_perm[i];
        c.best_perm[i] = e->inc_perm[i];
    }
    c.simple_bounds = st.simple_bounds;
    c.best_cost = e->inc_cost;
    c.work_id = 0;
    c.max_intervals = E;
    c.explored = st.decomposed;
    c.nb = nb;
    int len = 0;
    if ((rc = pbb_checkpoint_format(&c, ids.data(), pos.data(), end.data(), nullptr, 0, &len))) return rc;
    std::vector<char> buf(len + 1);
    if ((rc = pbb_checkpoint_format(&c, ids.data(), pos.data(), end.data(), buf.data(), len + 1, &len))) return rc;
    FILE *f = fopen(path, "w");
    if (!f) return fail(PBB_E_ARG, "cannot write %s", path);
    size_t w = fwrite(buf.data(), 1, len, f);
    fclose(f);
    if (w != (size_t)len) return fail(PBB_E_ARG, "short write to %s", path);
    return PBB_OK;
}

extern "C" int pbb_checkpoint_load(pbb_engine *e, const char *path, pbb_checkpoint *info)
{
    if (!e || !path) return fail(PBB_E_ARG, "null argument");
    std::ifstream f(path);
    if (!f) return fail(PBB_E_ARG, "cannot read %s", path);
    std::stringstream ss;
    ss << f.rdbuf();
    const std::string text = ss.str();
    const int n = e->n, E = e->E;
    std::vector<int> pos((size_t)E * n), end((size_t)E * n), ids(E);
    pbb_checkpoint c;
    int rc = pbb_checkpoint_parse(text.c_str(), n, &c, ids.data(), pos.data(), end.data(), E);
    if (rc) return rc;
    if (!is_perm(c.best_perm, n)) return fail(PBB_E_ARG, "%s: incumbent is not a permutation of 0..%d", path, n - 1);
    if ((rc = pbb_set_root(e, c.root_perm))) return rc;
    if ((rc = pbb_set_incumbent(e, c.best_cost, c.best_perm))) return rc;
    for (int k = 0; k < c.nb; k++) ids[k] = k;  // interval k -> explorer k
    if ((rc = pbb_init_intervals(e, c.nb, ids.data(), pos.data(), end.data()))) return rc;
    // the file's counters carry on (works::init_infile restores simpleBounds,
    // distributed/src/works.cpp:81-83): pbb_get_stats and the next save
    // report the whole run, not the segment since this load
    e->dec_base = c.explored;
    e->sb_base = c.simple_bounds;
    if (info) *info = c;
    return PBB_OK;
}
