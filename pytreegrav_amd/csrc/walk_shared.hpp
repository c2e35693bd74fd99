// Pieces shared by the FP32 walk (walk.hip) and the FP64 walk (walk64.hip): the walk control block,
// the wave-level stack and scan helpers of the breadth-ordered traversal, and the field layout.
#pragma once

#include <algorithm>

#include "ptg_common.hpp"

#define WALK_WAVES 4
#define SCAP 768       // LDS traversal stack entries per wave (>= 512, the most children one step pushes)
#define SPILL 256      // entries refilled from global memory at a time (<= SCAP - 512)
#define GCAP 16384     // global spill entries per wave
#define NXCD 8
#define CTR_STRIDE 32  // int32 words between per-XCD counters (128 B)

template <typename T> struct alignas(4 * sizeof(T)) V4 {
    T x, y, z, w;
};

#define WALK_DONE 16  // copies of the word that ends the task pass, each on its own line

struct WalkCtl {
    int32_t ctr[NXCD * CTR_STRIDE];   // per-XCD group counters
    int32_t err;
    int32_t hwm;  // deepest global spill stack (entries) any wave reached in the last walk
    int32_t pad[30];
    // deferral: entries taken of the deferred groups, of the tasks and of the saved stacks; tasks not yet
    // finished; tickets drawn by the task pass, per XCD
    int32_t ngroup, ntask, npool, pad2[29];
    int32_t open, pad3[31];
    int32_t ticket[NXCD * CTR_STRIDE];
    int32_t done[WALK_DONE * 32];
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
// level of sums cost 30.  Its waves end when no task is open: running waves wait for nothing, so the open
// count falls to zero.  What one wave writes and another reads within it (records, stacks, rows) goes
// through agent-scope accesses, ordered by the writer's wait before it publishes or counts down.
struct WalkTask {
    int32_t group;
    int32_t parent;              // entry of tasks (-1: a deferred group)
    int32_t off, stride, count;  // saved stack entries entries[off + i * stride], i < count
    int32_t child0, nchild;      // its shares (a group or a task that was cut)
    int32_t wait;                // shares not yet added
};

#define WALK_MAX_TASKS 196608
#define WALK_POLLS (1 << 26)  // a wave gives up after a minute without a task and reports it

struct WalkPool {
    int *spill;  // per-wave global stacks, gcap entries each
    int gcap;
    int *entries;  // saved stacks
    int ecap;
    WalkTask *tasks;  // gcount deferred groups, then tcount tasks
    int32_t *ready;   // [WALK_MAX_TASKS] task published (cleared before the walk)
    int gcount, tcount;  // 0: nothing is deferred
    void *partial;    // one row of gs * (sums per target) per entry of tasks, in the walk's type
    int budget, most0, div0, most, div;  // shares of a deferred group (task): stack >> div0 (div), at most most0 (most)

    // the workspace behind the control block: the spill stacks of `waves` waves, then what deferral needs.
    // row: bytes of one partial row
    ptg_status carve(char *ws, size_t ws_bytes, int64_t waves, int gcap_, size_t row)
    {
        size_t at = ptg_align256(sizeof(WalkCtl));
        auto take = [&](size_t bytes) {
            char *p = ws + at;
            at += ptg_align256(bytes);
            return p;
        };
        ready = (int32_t *)take(WALK_MAX_TASKS * sizeof(int32_t));  // where the control block's clearing expects it
        gcap = gcap_;
        spill = (int *)take((size_t)waves * gcap * sizeof(int));
        if (at > ws_bytes) {
            ptg_set_error("ptg_walk: workspace too small (%zu < %zu)", ws_bytes, at);
            return PTG_ERR_WORKSPACE;
        }
        const size_t left = ws_bytes - at;
        const size_t ebytes = std::min<size_t>(left / 8 * 3, 48u << 20);
        const size_t nrows = left > ebytes + 1024 ? (left - ebytes - 1024) / (row + sizeof(WalkTask)) : 0;
        gcount = tcount = 0;
        if (nrows >= 1024) {
            ecap = (int)(ebytes / sizeof(int));
            entries = (int *)take(ebytes);
            tcount = (int)std::min<size_t>(WALK_MAX_TASKS, nrows / 8 * 7);
            gcount = tcount / 8;
            tasks = (WalkTask *)take((size_t)(gcount + tcount) * sizeof(WalkTask));
            partial = take((size_t)(gcount + tcount) * row);
        }
        return PTG_OK;
    }
};

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

// n entries of a table of cap counted by *counter: the first one's index, or -1 (one lane calls).  The
// counter is added to once and never taken back: when thousands of waves reach their budgets together,
// compare-and-swap loops on it took 27 ms.
__device__ __forceinline__ int walk_take(int32_t *counter, int n, int cap)
{
    if (agent_load(counter) > cap - n) return -1;
    const int at = atomicAdd(counter, n);
    return at > cap - n ? -1 : at;
}

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
        if (!TASKS) self = walk_take(&ctl->ngroup, 1, B.gcount);
        off = self >= 0 ? walk_take(&ctl->npool, cnt, B.ecap) : -1;
        child0 = off >= 0 ? walk_take(&ctl->ntask, nchild, B.tcount) : -1;
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

// after the row of `self` is stored: its record, then its shares' records, then their flags
template <bool TASKS>
__device__ __forceinline__ void walk_publish(WalkCtl *ctl, const WalkPool &B, int64_t g, int cnt, int nchild, int off,
                                             int child0, int self, int lane)
{
    if (lane == 0) {
        WalkTask *T = &B.tasks[self];
        if (!TASKS) {
            agent_store(&T->group, (int32_t)g);
            agent_store(&T->parent, -1);
        }
        agent_store(&T->child0, child0);
        agent_store(&T->nchild, nchild);
        agent_store(&T->wait, nchild);
        atomicAdd(&ctl->open, nchild);
    }
#pragma unroll 1
    for (int q = lane; q < nchild; q += 64) {
        WalkTask *T = &B.tasks[child0 + q];
        agent_store(&T->group, (int32_t)g);
        agent_store(&T->parent, self);
        agent_store(&T->off, off + q);
        agent_store(&T->stride, nchild);
        agent_store(&T->count, (cnt - q + nchild - 1) / nchild);
    }
    wave_stores_done();
#pragma unroll 1
    for (int q = lane; q < nchild; q += 64) agent_store(&B.ready[child0 - B.gcount + q], 1);
}

// The next task of the task pass (its entry of tasks), or -1 when none is open any more.  Task t is drawn
// by XCD t mod 8 (block b runs on XCD b mod 8; the grid holds blocks of each).  closed: tasks this wave has
// finished since it last counted them off, which it does before it waits: a count per task on one word
// would take milliseconds.
__device__ __forceinline__ int walk_ticket(WalkCtl *ctl, const WalkPool &B, int lane, int &closed)
{
    const int x = blockIdx.x % NXCD;
    int t = 0;
    if (lane == 0) t = x + NXCD * atomicAdd(&ctl->ticket[x * CTR_STRIDE], 1);
    t = __builtin_amdgcn_readfirstlane(t);
    for (int polls = 0; polls < WALK_POLLS; polls++) {
        int r = 0, d = 0;
        if (lane == 0) {
            if (t < B.tcount) r = agent_load(&B.ready[t]);
            if (polls) d = agent_load(&ctl->done[(blockIdx.x % WALK_DONE) * 32]);
        }
        if (__builtin_amdgcn_readfirstlane(r)) return B.gcount + t;
        if (__builtin_amdgcn_readfirstlane(d)) return -1;
        if (closed) {
            int o = 0;
            if (lane == 0) o = atomicSub(&ctl->open, closed);
            if (__builtin_amdgcn_readfirstlane(o) == closed && lane < WALK_DONE) agent_store(&ctl->done[lane * 32], 1);
            closed = 0;
        }
        if (t >= B.tcount) return -1;  // all that there can be have been drawn
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
