// Pieces shared by the FP32 walk (walk.hip) and the FP64 walk (walk64.hip): the walk control block,
// the wave-level stack and scan helpers of the breadth-ordered traversal, and the field layout.
#pragma once

#include <algorithm>

#include "ptg_common.hpp"

#define WALK_FN static __device__ __forceinline__
#include "walk_tasks.hpp"

#define WALK_WAVES 4
#define SCAP 768       // LDS traversal stack entries per wave (>= 512, the most children one step pushes)
#define SPILL 256      // entries refilled from global memory at a time (<= SCAP - 512)
#define GCAP 16384     // global spill entries per wave

template <typename T> struct alignas(4 * sizeof(T)) V4 {
    T x, y, z, w;
};

template <int FIELDS> struct NW {
    static constexpr int POT = (FIELDS & PTG_POT) ? 1 : 0;
    static constexpr int ACC = (FIELDS & PTG_ACC) ? 1 : 0;
    static constexpr int TID = (FIELDS & PTG_TIDAL) ? 1 : 0;
    static constexpr int W = POT + 3 * ACC + 9 * TID;
};

// per-target accumulators: phi, g(3), T(6 independent)
template <typename T> struct Acc {
    T phi, gx, gy, gz, txx, tyy, tzz, txy, txz, tyz;
};

// gap between x and the interval [lo, hi] (0 inside): bmin - x and x - bmax are exact differences,
// so this equals the two-sided branch form bit for bit
__device__ __forceinline__ float box_gap(float x, float lo, float hi) { return fmaxf(fmaxf(lo - x, x - hi), 0.f); }
__device__ __forceinline__ double box_gap(double x, double lo, double hi) { return fmax(fmax(lo - x, x - hi), 0.0); }

// Stack spill: when sp entries plus the tot children about to be pushed exceed SCAP, the bottom
// ks entries (the excess rounded up to 64, at most sp; tot <= 512 <= SCAP so ks >= the excess)
// go to the wave's global spill stack and the rest move down.  Any order of visits gives the same
// accepted sets, so the global stack is refilled from its top when the LDS stack runs empty.
static_assert(SCAP >= 512 && SPILL >= 64 && SPILL <= SCAP - 512, "stack geometry");
__device__ __forceinline__ int spill_count(int sp, int tot)
{
    const int ex = sp + tot - SCAP;
    return std::min(sp, (ex + 63) & ~63);
}
__device__ __forceinline__ void spill_bottom(int *stack, int *dst, int sp, int ks, int lane)
{
    for (int q = lane; q < ks; q += 64) dst[q] = stack[q];
    __builtin_amdgcn_wave_barrier();
    // read [ks + q, ks + q + 64) before writing [q, q + 64); later reads lie above earlier writes
    for (int q = 0; q < sp - ks; q += 64) {
        const int v = (q + lane < sp - ks) ? stack[ks + q + lane] : 0;
        __builtin_amdgcn_wave_barrier();
        if (q + lane < sp - ks) stack[q + lane] = v;
        __builtin_amdgcn_wave_barrier();
    }
}

// lanes below this one whose bit is set in m
__device__ __forceinline__ int lanes_below(uint64_t m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// exclusive prefix sum across the wave of v in [0, 15] (children counts), one ballot per bit;
// tot receives the wave total
__device__ __forceinline__ int small_excl_scan(int v, int &tot)
{
    int below = 0, t = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const uint64_t m = ptg_ballot((v >> b) & 1);
        below += lanes_below(m) << b;
        t += (int)__popcll(m) << b;
    }
    tot = t;
    return below;
}

// FIELDS of the angle-binned column density's six sums (walk64.hip)
#define BINS 8

template <int FIELDS> struct Sums {
    static constexpr int WI = FIELDS == BINS ? 6 : NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC + 6 * NW<FIELDS>::TID;
    static constexpr int WO = FIELDS == BINS ? 6 : NW<FIELDS>::W;  // output row
};

// the entries of output row o[] that sum c of a target fills: the tidal tensor is kept as xx xy xz yy yz zz,
// and an off-diagonal component fills two
template <int FIELDS> __device__ __forceinline__ void store_sum(double *o, int c, double v)
{
    constexpr int PA = FIELDS == BINS ? 6 : NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC;
    if (!NW<FIELDS>::TID || c < PA) {
        o[c] = v;
        return;
    }
    const int k = c - PA;
    const int i = k < 3 ? 0 : k < 5 ? 1 : 2, j = k < 3 ? k : k < 5 ? k - 2 : 2;
    o[PA + 3 * i + j] = v;
    o[PA + 3 * j + i] = v;
}

// ---- deferred traversals ----
// A group whose box is wide against its surroundings (a run of the Morton order across a high-level cell
// boundary, or few targets in a large domain) opens a large part of the tree, and one wave walking it
// alone sets the kernel's time.  A traversal past a budget of visits is therefore cut: the wave stores
// the sums it has (a row) and saves its stack as interleaved shares, tasks of a second launch.  There the
// waves draw tickets for the tasks; a task past the budget is cut again, its shares published for the
// waves that wait, and whoever finishes the last share of a task or group adds the shares' rows to it in
// their order.  Where a traversal is cut depends on the group alone, also where the tables fill up
// (walk_tasks.hpp), so results do not depend on scheduling or on what else is walked.
//
// The second launch costs 3 us where nothing was deferred; a launch per generation of tasks and one per
// level of sums cost 30.  Its waves end when no task is open; which wave walks which task is in
// walk_tasks.hpp.  What one wave writes and another reads within it (records, stacks, rows) goes
// through agent-scope accesses, ordered by the writer's wait before it publishes or counts down.
#define WALK_LOOKS (1 << 26)  // a wave gives up after some minutes without a task and reports it

// The workspace: the control block, the flags of the task slots and the bits of the groups put back (these
// cleared before each walk), the spill stacks of the waves, and WALK_POOL bytes for what deferral needs.  The
// tables are sized by the row alone, so that what fits does not depend on the call.
#define WALK_AGAIN (4u << 20)  // bytes of the bits: 3.4e7 groups
#define WALK_POOL (48u << 20)  // the listed and drawn cases use at most a third
#define WALK_ENTRIES (WALK_POOL / 4)
#define WALK_COUNTS (WALK_MAX_TASKS / 8 * 4 * sizeof(int64_t))

// words of the bits of `groups` groups
static __host__ __device__ __forceinline__ int64_t walk_words(int64_t groups) { return (groups + 255) / 256 * 8; }

static constexpr size_t walk_align(size_t x) { return (x + 255) & ~(size_t)255; }
#define WALK_READY_AT walk_align(sizeof(WalkCtl))
#define WALK_AGAIN_AT (WALK_READY_AT + walk_align(WALK_MAX_TASKS * sizeof(int64_t)))

static inline size_t walk_control_bytes(size_t again = WALK_AGAIN) { return WALK_AGAIN_AT + walk_align(again); }

// A walk's workspace as its kernels take it: few words, since they are held in scalar registers through the
// traversal.  The tables behind it are found where they are needed (walk_pool).
struct WalkHot {
    int *spill;  // per-wave global stacks, gcap entries each
    int gcap;
    int budget;       // of visits, before a traversal is cut
    int most0, most;  // shares of a deferred group: stack >> WALK_DIV0, at most most0; of a task: >> WALK_DIV, most
    int tcount;       // slots of the task table, 8 per entry for groups (0: nothing is deferred)
    uint32_t pool_at;  // of the tables, from the control block, in units of 256 bytes
};
#define WALK_DIV0 4
#define WALK_DIV 2

static __host__ __device__ __forceinline__ WalkPool walk_pool(WalkCtl *ctl, const WalkHot &h)
{
    char *ws = (char *)ctl, *p = ws + (size_t)h.pool_at * 256;
    WalkPool b;
    b.ready = (int64_t *)(ws + WALK_READY_AT);
    b.again = (int32_t *)(ws + WALK_AGAIN_AT);
    b.entries = (int *)p;
    b.ecap = (int)(WALK_ENTRIES / sizeof(int));
    b.counts = (int64_t *)(p + WALK_ENTRIES);
    b.tasks = (WalkTask *)(p + WALK_ENTRIES + WALK_COUNTS);
    b.tcount = h.tcount;
    b.gcount = h.tcount / 8;
    b.partial = p + WALK_ENTRIES + WALK_COUNTS + walk_align((size_t)(b.gcount + b.tcount) * sizeof(WalkTask));
    return b;
}
// The pool within a walk: the barrier keeps the addresses where they are used, moved out of the traversal they are
// scalar registers again.  The task pass, which uses them between any two traversals, takes them as an argument.
template <bool TASKS>
__device__ __forceinline__ WalkPool walk_pool(WalkCtl *ctl, const WalkHot &h, const WalkPool &arg)
{
    if (TASKS) return arg;
    asm volatile("" : "+s"(ctl));
    return walk_pool(ctl, h);
}

// groups: at most, again: bytes of their bits (too few: nothing is deferred), gcap: spill entries per wave,
// row: bytes of one partial row
static ptg_status walk_carve(WalkHot &h, char *ws, size_t ws_bytes, int64_t groups, size_t again, int64_t waves, int gcap,
                             size_t row)
{
    const size_t spill_at = walk_control_bytes(again), at = spill_at + walk_align((size_t)waves * gcap * sizeof(int));
    if (at + WALK_POOL > ws_bytes) {
        ptg_set_error("ptg_walk: workspace too small (%zu < %zu)", ws_bytes, at + WALK_POOL);
        return PTG_ERR_WORKSPACE;
    }
    h.spill = (int *)(ws + spill_at);
    h.gcap = gcap;
    h.pool_at = (uint32_t)(at / 256);
    const int64_t left = WALK_POOL - WALK_ENTRIES - WALK_COUNTS - 256, nine = 9 * (int64_t)(row + sizeof(WalkTask));
    h.tcount = 8 * (int)std::min<int64_t>(WALK_MAX_TASKS / 8, left / nine);
    if (walk_words(groups) * (int64_t)sizeof(int32_t) > (int64_t)again) h.tcount = 0;
    return PTG_OK;
}

// clears the control block, the task flags and the bits of the groups: n int4
__global__ static void k_walk_init(int4 *ws, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        ws[i] = int4{0, 0, 0, 0};
}
static inline ptg_status walk_clear(void *ws, int64_t groups, size_t again, hipStream_t s)
{
    const size_t bits = std::min<size_t>(again, walk_words(groups) * sizeof(int32_t));
    const int64_t n = (int64_t)((WALK_AGAIN_AT + bits) / sizeof(int4));
    k_walk_init<<<(unsigned)std::min<int64_t>(2048, (n + 1023) / 1024), 256, 0, s>>>((int4 *)ws, n);
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

template <typename V> __device__ __forceinline__ V agent_load(const V *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V> __device__ __forceinline__ void agent_store(V *p, V v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the wave's stores so far have completed
__device__ __forceinline__ void wave_stores_done()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

struct WalkSpan {
    int64_t a0;  // first target
    int mt;      // targets
    bool over;   // a supplied group holds targets past gs (not evaluated)
};

__device__ __forceinline__ WalkSpan walk_span(const int32_t *goff, int gs, int64_t nt, int64_t g)
{
    const int64_t a0 = goff ? (int64_t)goff[g] : g * gs;
    const int64_t e0 = goff ? (int64_t)goff[g + 1] : nt;
    const int64_t b0 = e0 < a0 + gs ? e0 : a0 + gs;
    return WalkSpan{a0, (int)(b0 - a0), goff && e0 > b0};
}

// the memory of the task pass (walk_tasks.hpp)
struct AgentMem {
    static constexpr int LANES = 64;
    static __device__ __forceinline__ int32_t load(const int32_t *p) { return agent_load(p); }
    static __device__ __forceinline__ void store(int32_t *p, int32_t v) { agent_store(p, v); }
    static __device__ __forceinline__ int32_t add(int32_t *p, int32_t v) { return atomicAdd(p, v); }
    static __device__ __forceinline__ int32_t sub(int32_t *p, int32_t v) { return atomicSub(p, v); }
    static __device__ __forceinline__ bool cas(int32_t *p, int32_t is, int32_t v) { return atomicCAS(p, is, v) == is; }
    static __device__ __forceinline__ void max(int32_t *p, int32_t v) { atomicMax(p, v); }
    static __device__ __forceinline__ void set(int32_t *p, int32_t bits) { atomicOr(p, bits); }
    static __device__ __forceinline__ int64_t load(const int64_t *p) { return agent_load(p); }
    static __device__ __forceinline__ void store(int64_t *p, int64_t v) { agent_store(p, v); }
    // one store of the wave
    static __device__ __forceinline__ void record(WalkTask *p, const WalkTask &T, int lane)
    {
        const int32_t v[WALK_TASK_WORDS] = {T.group, T.parent, T.root, T.level, T.off, T.count, T.child0, T.nchild, T.wait};
        int32_t w = v[0];
#pragma unroll
        for (int i = 1; i < WALK_TASK_WORDS; i++) w = lane == i ? v[i] : w;
        if (lane < WALK_TASK_WORDS) agent_store((int32_t *)p + lane, w);
    }
    static __device__ __forceinline__ void settle() { wave_stores_done(); }
};

// Cuts a traversal: takes room for its shares (gsp spilled entries below sp in LDS) and saves the stack.
// share: as a share of a group is cut, not as a group.  `self` is the task's entry of tasks (a group's is taken
// here where it is negative).  Returns the number of shares, 0 if the traversal is one that is not cut, -1 if
// there is no room; the row is stored next, then walk_publish makes the shares tasks.
template <bool TASKS>
__device__ __forceinline__ int walk_cut(WalkCtl *ctl, const WalkHot &h, const WalkPool &arg, bool share, const int *stack, int sp,
                                        const int *spill, int gsp, int lane, int &self, int &off, int &child0)
{
    const WalkPool B = walk_pool<TASKS>(ctl, h, arg);
    const int cnt = gsp + sp;
    const int most = share ? h.most : h.most0, part = cnt >> (share ? WALK_DIV : WALK_DIV0);
    const int nchild = part > most ? most : part < 1 ? 1 : part;
    if (cnt > nchild * SCAP) return 0;
    int room = 0;
    if (lane == 0) room = walk_room<AgentMem>(ctl, B, cnt, nchild, self, off, child0);
    if (!__builtin_amdgcn_readfirstlane(room)) return -1;
    self = __builtin_amdgcn_readfirstlane(self);
    off = __builtin_amdgcn_readfirstlane(off);
    child0 = __builtin_amdgcn_readfirstlane(child0);
#pragma unroll 1
    for (int q = lane; q < gsp; q += 64) agent_store(&B.entries[off + q], spill[q]);
#pragma unroll 1
    for (int q = lane; q < sp; q += 64) agent_store(&B.entries[off + gsp + q], stack[q]);
    return nchild;
}

// a budget of visits at a level
__device__ __forceinline__ int walk_budget(int budget, int level)
{
    return level == 0 ? budget : level < 8 && budget < 0x7fffffff >> 3 * level ? budget << 3 * level : 0x7fffffff;
}

// The next task of the task pass (its entry of tasks), or -1 when none is open any more.  Block b is of
// class b mod 8, as it runs on XCD b mod 8.  ticket, closed: the wave's (task_look), uniform.
__device__ __forceinline__ int walk_ticket(WalkCtl *ctl, const WalkPool &B, int lane, int &ticket, int &closed, int &parent)
{
    for (int looks = 0; looks < WALK_LOOKS; looks++) {
        int t = TASK_NONE;
        if (lane == 0)
            t = task_look<AgentMem>(ctl, B, blockIdx.x % NXCD, blockIdx.x % WALK_DONE, looks, ticket, closed, parent);
        t = __builtin_amdgcn_readfirstlane(t);
        parent = __builtin_amdgcn_readfirstlane(parent);
        ticket = __builtin_amdgcn_readfirstlane(ticket);
        closed = __builtin_amdgcn_readfirstlane(closed);
        if (t != TASK_NONE) return t == TASK_END ? -1 : B.gcount + t;
        __builtin_amdgcn_s_sleep(32);  // 0.9 us
    }
    if (lane == 0) atomicOr(&ctl->err, 8);
    return -1;
}

// a record of the task table in the wave's lanes: one load, where a load per field waited for each in turn
struct TaskWords {
    int32_t word = 0;
    TaskWords() = default;
    __device__ __forceinline__ TaskWords(const WalkTask *T, int lane)
    {
        word = agent_load((const int32_t *)T + (lane < WALK_TASK_WORDS ? lane : 0));
    }
    template <int32_t WalkTask::*F> __device__ __forceinline__ int get() const
    {
        constexpr WalkTask T{};
        return __builtin_amdgcn_readlane(word, (int)(&(T.*F) - &T.group));
    }
};

// the row of a share of entry p is stored: counts p's shares down; the last share's wave adds them up,
// and so on up to the group, whose total is the result.  Returns the group's entry then, or -1.
template <int FIELDS, typename R>
__device__ __forceinline__ int walk_add_up(WalkCtl *ctl, const WalkPool &B, int p, const WalkSpan &grp, int gs,
                                           const int64_t *perm, double G, double *out, int lane)
{
    constexpr int WI = Sums<FIELDS>::WI;
    const int nv = grp.mt * WI;
    const int64_t rs = (int64_t)gs * WI;
    R *rows = (R *)B.partial;
    for (;;) {
        wave_stores_done();
        int last = 0;
        if (lane == 0) last = task_close<AgentMem>(B, p);
        if (!__builtin_amdgcn_readfirstlane(last)) return -1;
        asm volatile("" ::: "memory");
        const TaskWords T(&B.tasks[p], lane);
        const int nchild = T.get<&WalkTask::nchild>(), kid0 = T.get<&WalkTask::child0>();
        const bool own = T.get<&WalkTask::off>() >= 0;  // p has a row
        if (p < B.gcount && T.get<&WalkTask::root>()) {  // a share found no room
            if (lane == 0) walk_put_back<AgentMem>(ctl, B, true, T.word);  // lane 0: the group
            return -1;
        }
        const R *slots = rows + B.gcount * rs;
#pragma unroll 1
        for (int v = lane; v < nv; v += 64) {
            R s = agent_load(own ? &rows[p * rs + v] : &slots[kid0 * rs + v]);
#pragma unroll 1
            for (int k0 = own ? 0 : 1; k0 < nchild; k0 += 16) {
                R t[16];  // the loads go out together
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const int e = kid0 + (k0 + u < nchild ? k0 + u : nchild - 1);
                    t[u] = agent_load(&slots[(e < B.tcount ? e : e - B.tcount) * rs + v]);  // the slots go round
                }
#pragma unroll
                for (int u = 0; u < 16; u++)
                    if (k0 + u < nchild) s += t[u];
            }
            if (p >= B.gcount) {
                agent_store(&rows[p * rs + v], s);
            } else {
                const int64_t i = grp.a0 + v / WI, o = perm ? perm[i] : i;
                store_sum<FIELDS>(out + o * Sums<FIELDS>::WO, v % WI, G * (double)s);
            }
        }
        if (p < B.gcount) return p;
        p = T.get<&WalkTask::parent>();
    }
}

// ---- FP64 walk (walk64.hip) ----
struct Walk64Args {
    const V4<double> *xyzm;
    const V4<double> *aux;
    const int2 *kids;
    const double *quad;  // 8 per slot
    const double *pos;
    const double *soft;   // NULL: none
    const int64_t *perm;  // NULL: the targets in the order given
    int sorted;  // pos/soft are indexed by the sorted target position (perm maps the outputs only)
    int64_t nslots;
    int64_t nt;
    int64_t ngroups;
    const int32_t *goff;    // optional group offsets (ngroups + 1), else fixed groups of gs
    const int32_t *gcount;  // device group count when goff is given
    int gs;
    double theta, inv_theta;
    double G;
    double ox, oy, oz;
    int64_t nsys;         // 0: one tree; else group g walks the tree of the system holding its first target
    const int64_t *soff;  // (nsys + 1) system target ranges
    double *out;
    int64_t *counters;
    WalkCtl *ctl;
    const int32_t *start;  // subtree walks: device slot of the element every walk starts at (nullable)
};

// launches the walk on a workspace whose control block ws starts with (cleared by the caller); gcap =
// spill entries per wave; cus = the device's compute units
// angle-binned column density (colden.hip): groups of gs <= 64 sorted targets, six sums each (soft and
// perm NULL: no softening, rows in target order), scaled by G
ptg_status ptg_walk64_bins(const Walk64Args &a, int cus, int gcap, size_t again, char *ws, size_t ws_bytes, hipStream_t s);
ptg_status ptg_walk64_launch(const Walk64Args &a, int fields, bool quad, int cus, int gcap, size_t again, char *ws, size_t ws_bytes,
                             hipStream_t s);
