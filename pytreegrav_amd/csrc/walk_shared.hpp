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
// their order.  Where a traversal is cut depends on the group alone, so results do not depend on
// scheduling or on what else is walked (unless the tables fill up: then the rest is walked in place, the
// same terms summed in another order).
//
// The second launch costs 3 us where nothing was deferred; a launch per generation of tasks and one per
// level of sums cost 30.  Its waves end when no task is open; which wave walks which task is in
// walk_tasks.hpp.  What one wave writes and another reads within it (records, stacks, rows) goes
// through agent-scope accesses, ordered by the writer's wait before it publishes or counts down.
#define WALK_LOOKS (1 << 26)  // a wave gives up after a minute without a task and reports it

// the workspace behind the control block: the spill stacks of `waves` waves, then what deferral needs.
// row: bytes of one partial row
static ptg_status walk_carve(WalkPool &b, char *ws, size_t ws_bytes, int64_t waves, int gcap, size_t row)
{
    size_t at = ptg_align256(sizeof(WalkCtl));
    auto take = [&](size_t bytes) {
        char *p = ws + at;
        at += ptg_align256(bytes);
        return p;
    };
    b.ready = (int32_t *)take(WALK_MAX_TASKS * sizeof(int32_t));  // where the control block's clearing expects it
    b.gcap = gcap;
    b.spill = (int *)take((size_t)waves * gcap * sizeof(int));
    if (at > ws_bytes) {
        ptg_set_error("ptg_walk: workspace too small (%zu < %zu)", ws_bytes, at);
        return PTG_ERR_WORKSPACE;
    }
    const size_t left = ws_bytes - at;
    const size_t ebytes = std::min<size_t>(left / 8 * 3, 48u << 20);
    const size_t nrows = left > ebytes + 1024 ? (left - ebytes - 1024) / (row + sizeof(WalkTask)) : 0;
    b.gcount = b.tcount = 0;
    if (nrows >= 1024) {
        b.ecap = (int)(ebytes / sizeof(int));
        b.entries = (int *)take(ebytes);
        b.tcount = (int)std::min<size_t>(WALK_MAX_TASKS, nrows / 8 * 7);
        b.gcount = b.tcount / 8;
        b.tasks = (WalkTask *)take((size_t)(b.gcount + b.tcount) * sizeof(WalkTask));
        b.partial = take((size_t)(b.gcount + b.tcount) * row);
    }
    return PTG_OK;
}

static inline size_t walk_control_bytes()
{
    return ptg_align256(sizeof(WalkCtl)) + ptg_align256(WALK_MAX_TASKS * sizeof(int32_t));
}

// clears the control block and the task flags behind it
__global__ static void k_walk_init(int4 *ws, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) ws[i] = int4{0, 0, 0, 0};
}
static inline ptg_status walk_clear(void *ws, hipStream_t s)
{
    const int n = (int)(walk_control_bytes() / sizeof(int4));
    k_walk_init<<<(n + 1023) / 1024, 256, 0, s>>>((int4 *)ws, n);
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
    static __device__ __forceinline__ void settle() { wave_stores_done(); }
};

// Cuts a traversal: takes room for its shares (gsp spilled entries below sp in LDS) and saves the stack.
// `self` is the task's entry of tasks (a group's is taken here).  Returns the number of shares, 0 if
// there is no room (the wave goes on); the row is stored next, then walk_publish makes the shares tasks.
template <bool TASKS>
__device__ __forceinline__ int walk_cut(WalkCtl *ctl, const WalkPool &B, const int *stack, int sp, const int *spill,
                                        int gsp, int lane, int &self, int &off, int &child0)
{
    const int cnt = gsp + sp;
    const int most = TASKS ? B.most : B.most0, part = cnt >> (TASKS ? B.div : B.div0);
    const int nchild = part > most ? most : part < 1 ? 1 : part;
    off = -1;
    if (lane == 0 && cnt <= nchild * SCAP) {
        // tasks last: one that was taken is published (a ticket would wait for it)
        if (!TASKS) self = walk_take<AgentMem>(&ctl->ngroup, 1, B.gcount);
        off = self >= 0 ? walk_take<AgentMem>(&ctl->npool, cnt, B.ecap) : -1;
        child0 = off >= 0 ? walk_take<AgentMem>(&ctl->ntask, nchild, B.tcount) : -1;
        if (child0 < 0) off = -1;
        child0 += B.gcount;
    }
    self = __builtin_amdgcn_readfirstlane(self);
    off = __builtin_amdgcn_readfirstlane(off);
    child0 = __builtin_amdgcn_readfirstlane(child0);
    if (off < 0) return 0;
#pragma unroll 1
    for (int q = lane; q < gsp; q += 64) agent_store(&B.entries[off + q], spill[q]);
#pragma unroll 1
    for (int q = lane; q < sp; q += 64) agent_store(&B.entries[off + gsp + q], stack[q]);
    return nchild;
}

// The next task of the task pass (its entry of tasks), or -1 when none is open any more.  Block b is of
// class b mod 8, as it runs on XCD b mod 8.  ticket, closed: the wave's (task_look), uniform.
__device__ __forceinline__ int walk_ticket(WalkCtl *ctl, const WalkPool &B, int lane, int &ticket, int &closed)
{
    for (int looks = 0; looks < WALK_LOOKS; looks++) {
        int t = TASK_NONE;
        if (lane == 0)
            t = task_look<AgentMem>(ctl, B, blockIdx.x % NXCD, blockIdx.x % WALK_DONE, looks, ticket, closed);
        t = __builtin_amdgcn_readfirstlane(t);
        ticket = __builtin_amdgcn_readfirstlane(ticket);
        closed = __builtin_amdgcn_readfirstlane(closed);
        if (t != TASK_NONE) return t == TASK_END ? -1 : B.gcount + t;
        __builtin_amdgcn_s_sleep(32);  // 0.9 us
    }
    if (lane == 0) atomicOr(&ctl->err, 8);
    return -1;
}

// the row of task `self` is stored: counts its parent's shares down; the last share's wave adds them up,
// and so on up to the group, whose total is the result
template <int FIELDS, typename R>
__device__ __forceinline__ void walk_add_up(const WalkPool &B, int self, const WalkSpan &grp, int gs, const int64_t *perm,
                                            double G, double *out, int lane)
{
    constexpr int WI = Sums<FIELDS>::WI;
    const int nv = grp.mt * WI;
    const int64_t rs = (int64_t)gs * WI;
    R *rows = (R *)B.partial;
    for (;;) {
        wave_stores_done();
        const int p = __builtin_amdgcn_readfirstlane(agent_load(&B.tasks[self].parent));
        WalkTask *T = &B.tasks[p];
        int w = 0;
        if (lane == 0) w = atomicSub(&T->wait, 1);
        if (__builtin_amdgcn_readfirstlane(w) != 1) return;
        asm volatile("" ::: "memory");
        const int nchild = __builtin_amdgcn_readfirstlane(agent_load(&T->nchild));
        const int64_t kids = __builtin_amdgcn_readfirstlane(agent_load(&T->child0)) * rs;
#pragma unroll 1
        for (int v = lane; v < nv; v += 64) {
            R s = agent_load(&rows[p * rs + v]);
#pragma unroll 4
            for (int k = 0; k < nchild; k++) s += agent_load(&rows[kids + k * rs + v]);
            if (p >= B.gcount) {
                agent_store(&rows[p * rs + v], s);
            } else {
                const int64_t i = grp.a0 + v / WI, o = perm ? perm[i] : i;
                store_sum<FIELDS>(out + o * Sums<FIELDS>::WO, v % WI, G * (double)s);
            }
        }
        if (p < B.gcount) return;
        self = p;
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
ptg_status ptg_walk64_bins(const Walk64Args &a, int cus, int gcap, char *ws, size_t ws_bytes, hipStream_t s);
ptg_status ptg_walk64_launch(const Walk64Args &a, int fields, bool quad, int cus, int gcap, char *ws, size_t ws_bytes,
                             hipStream_t s);
