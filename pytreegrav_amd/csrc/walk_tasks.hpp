// Scheduling of cut traversals (walk_shared.hpp): who walks which task, and when the task pass ends.
// Plain C++ over a memory policy M (loads, stores and read-modify-writes that every wave of the device
// sees), so that the CPU test runs the same source with a thread for each wave.  Functions whose comment
// says so are called by one lane.
//
// Task t belongs to class t mod NXCD, and a wave draws tickets from the counter of its block's class: one
// counter for all took milliseconds.  A wave whose task is not published yet waits with its ticket; every
// STEAL_POLLS looks it also takes a published task of another class that nobody has drawn.  So a task waits
// only for a wave that runs, of whichever class: no wave waits for a block to be placed, and a pass that
// shares the device with another one (a walk on another stream) ends however the two are placed.
#pragma once

#include <stdint.h>

#define NXCD 8
#define CTR_STRIDE 32  // int32 words between per-XCD counters (128 B)
#define WALK_DONE 16   // copies of the word that ends the task pass, each on its own line
#define WALK_MAX_TASKS 196608
#define STEAL_POLLS 16

struct WalkCtl {
    int32_t ctr[NXCD * CTR_STRIDE];  // per-XCD group counters
    int32_t err;
    int32_t hwm;  // deepest global spill stack (entries) any wave reached in the last walk
    int32_t pad[30];
    // deferral: entries taken of the deferred groups, of the tasks and of the saved stacks; tasks not yet
    // finished; tickets drawn by the task pass, per class
    int32_t ngroup, ntask, npool, pad2[29];
    int32_t open, pad3[31];
    int32_t ticket[NXCD * CTR_STRIDE];
    int32_t done[WALK_DONE * 32];
};

struct WalkTask {
    int32_t group;
    int32_t parent;              // entry of tasks (-1: a deferred group)
    int32_t off, stride, count;  // saved stack entries entries[off + i * stride], i < count
    int32_t child0, nchild;      // its shares (a group or a task that was cut)
    int32_t wait;                // shares not yet added
};

struct WalkPool {
    int *spill;  // per-wave global stacks, gcap entries each
    int gcap;
    int *entries;  // saved stacks
    int ecap;
    WalkTask *tasks;     // gcount deferred groups, then tcount tasks
    int32_t *ready;      // [WALK_MAX_TASKS] task published (cleared before the walk)
    int gcount, tcount;  // 0: nothing is deferred
    void *partial;       // one row of gs * (sums per target) per entry of tasks, in the walk's type
    int budget, most0, div0, most, div;  // shares of a deferred group (task): stack >> div0 (div), at most most0 (most)
};

// n entries of a table of cap counted by *counter: the first one's index, or -1 (one lane).  The counter
// is added to once and never taken back: when thousands of waves reach their budgets together,
// compare-and-swap loops on it took 27 ms.
template <typename M> WALK_FN int walk_take(int32_t *counter, int n, int cap)
{
    if (M::load(counter) > cap - n) return -1;
    const int at = M::add(counter, n);
    return at > cap - n ? -1 : at;
}

// after the row of `self` is stored: its record, then its shares' records, then their flags
// (lane: this one of M::LANES that all call)
template <typename M>
WALK_FN void walk_publish(WalkCtl *ctl, const WalkPool &B, bool task, int group, int cnt, int nchild, int off, int child0,
                          int self, int lane)
{
    if (lane == 0) {
        WalkTask *T = &B.tasks[self];
        if (!task) {
            M::store(&T->group, group);
            M::store(&T->parent, -1);
        }
        M::store(&T->child0, child0);
        M::store(&T->nchild, nchild);
        M::store(&T->wait, nchild);
        M::add(&ctl->open, nchild);
    }
#pragma unroll 1
    for (int q = lane; q < nchild; q += M::LANES) {
        WalkTask *T = &B.tasks[child0 + q];
        M::store(&T->group, group);
        M::store(&T->parent, self);
        M::store(&T->off, off + q);
        M::store(&T->stride, nchild);
        M::store(&T->count, (cnt - q + nchild - 1) / nchild);
    }
    M::settle();
#pragma unroll 1
    for (int q = lane; q < nchild; q += M::LANES) M::store(&B.ready[child0 - B.gcount + q], 1);
}

enum { TASK_END = -1, TASK_NONE = -2 };

// One look for a task by a wave of class x (one lane): its index, TASK_NONE (look again), or TASK_END when
// no task is open any more.  ticket: the task drawn and not yet walked (-1: none).  closed: tasks this wave
// has finished since it last counted them off, which it does before it waits: a count per task on one
// word would take milliseconds.
template <typename M>
WALK_FN int task_look(WalkCtl *ctl, const WalkPool &B, int x, int line, int looks, int &ticket, int &closed)
{
    if (ticket < 0) ticket = x + NXCD * M::add(&ctl->ticket[x * CTR_STRIDE], 1);
    if (ticket < B.tcount && M::load(&B.ready[ticket])) {
        const int t = ticket;
        ticket = -1;
        return t;
    }
    if (looks && M::load(&ctl->done[line * 32])) return TASK_END;
    if (closed) {
        if (M::sub(&ctl->open, closed) == closed)
            for (int i = 0; i < WALK_DONE; i++) M::store(&ctl->done[i * 32], 1);
        closed = 0;
    }
    if (looks % STEAL_POLLS == STEAL_POLLS - 1) {
        int v[NXCD], r[NXCD];  // the loads of a kind go out together
#pragma unroll
        for (int y = 0; y < NXCD; y++) v[y] = M::load(&ctl->ticket[y * CTR_STRIDE]);
#pragma unroll
        for (int y = 0; y < NXCD; y++) {
            const int t = y + NXCD * v[y];
            r[y] = t < B.tcount ? M::load(&B.ready[t]) : 0;
        }
#pragma unroll
        for (int y = 0; y < NXCD; y++)
            if (r[y] && M::cas(&ctl->ticket[y * CTR_STRIDE], v[y], v[y] + 1)) return y + NXCD * v[y];
    }
    return TASK_NONE;
}
