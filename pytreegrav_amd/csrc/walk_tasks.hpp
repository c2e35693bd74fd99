// Scheduling of cut traversals (walk_shared.hpp): who walks which task, what happens when the tables are
// full, and when the task pass ends.  Plain C++ over a memory policy M (loads, stores and
// read-modify-writes that every wave of the device sees), so that the CPU test runs the same source with a
// thread for each wave.  Functions whose comment says so are called by one lane.
//
// Task t belongs to class t mod NXCD, and a wave draws tickets from the counter of its block's class: one
// counter for all took milliseconds.  A wave whose task is not published yet waits with its ticket; every
// STEAL_LOOKS looks it also takes a published task of another class that nobody has drawn.  So a task waits
// only for a wave that runs, of whichever class: no wave waits for a block to be placed, and a pass that
// shares the device with another one (a walk on another stream) ends however the two are placed.
//
// A group that finds the tables full is put back, with whatever was walked of it, and walked again from its
// root once all open tasks are done and the tables are empty: first with others (a batch), and alone in
// the end.  One that does not fit alone is walked with eight times the budget, and so on.  What it is cut
// into is therefore its own affair, whatever else is walked and however waves are scheduled.
#pragma once

#include <stdint.h>

#define NXCD 8
#define CTR_STRIDE 32  // int32 words between per-XCD counters (128 B)
#define WALK_DONE 16   // copies of the word that ends the task pass, each on its own line
#define WALK_MAX_TASKS 196608
#define STEAL_LOOKS 64

struct WalkCtl {
    int32_t ctr[NXCD * CTR_STRIDE];  // per-XCD group counters
    int32_t err;
    int32_t hwm;  // deepest global spill stack (entries) any wave reached in the last walk
    int32_t pad[30];
    // deferral: entries taken of the deferred groups, of the tasks (numbered on from batch to batch) and of
    // the saved stacks; INT32_MAX - the first task number that was refused (0: none)
    int32_t ngroup, ntask, npool, refused, pad2[28];
    int32_t open, pad3[31];  // tasks not yet finished
    int32_t ticket[NXCD * CTR_STRIDE];  // tickets drawn, per class
    int32_t done[WALK_DONE * 32];
    // groups put back; 1: some were before the task pass, which starts with a task in `open` for them
    int32_t back, resume;
    // the batch: tasks below base + tcount - 1 fit; its groups (0: the group pass) and those put back of it,
    // its last group and that one's level, the word of `again` to look on from
    int32_t base, batch, failed, last, level, word;
    int32_t words;  // of `again`, a multiple of 8: written by the group pass
    int32_t pad4[23];
};

// a group or a task that was cut; its shares need no more than their number and its entry, which their flags hold
struct WalkTask {
    int32_t group;
    int32_t parent;         // entry of tasks (-1: a deferred group)
    int32_t root;           // its group's entry; of a group: 1 if a share of it found no room
    int32_t level;          // budgets are 8^level times the ordinary
    int32_t off, count;     // saved stack: share q's are entries[off + q + i * nchild]; off -1: a group from its root
    int32_t child0, nchild;  // its shares' slots
    int32_t wait;           // shares not yet added
    int32_t pad[3];
};
#define WALK_TASK_WORDS 9

struct WalkPool {
    int *entries;  // saved stacks
    int ecap;
    WalkTask *tasks;     // gcount deferred groups, then tcount slots: task t is in slot t mod tcount
    int64_t *counts;     // 4 per deferred group: its tasks' interactions, visits, particle interactions, folds
    int64_t *ready;      // [WALK_MAX_TASKS] task t of the slot is published: t + 1 and its parent's entry << 32
    int32_t *again;      // a bit per group, set while it is put back (cleared before the walk)
    int gcount, tcount;  // 0: nothing is deferred
    void *partial;       // one row of gs * (sums per target) per entry of tasks, in the walk's type
};

// room for a group's (self < 0: takes its entry) or a task's cut into nchild shares of cnt stack entries:
// the entries' offset and the shares' first task number; false if there is none (one lane).  A counter is
// added to once and never taken back: when thousands of waves reach their budgets together,
// compare-and-swap loops on it took 27 ms.
template <typename M>
WALK_FN bool walk_room(WalkCtl *ctl, const WalkPool &B, int cnt, int nchild, int &self, int &off, int &child0)
{
    const int group = self < 0 ? M::load(&ctl->ngroup) : -1, pool = M::load(&ctl->npool), task = M::load(&ctl->ntask);
    const int cap = M::load(&ctl->base) + B.tcount - 1;
    if (group >= B.gcount || pool > B.ecap - cnt || task > cap - nchild) return false;
    if (self < 0 && (self = M::add(&ctl->ngroup, 1)) >= B.gcount) return false;
    off = M::add(&ctl->npool, cnt);
    if (off > B.ecap - cnt) return false;
    // tasks last: numbers that were taken are published (a ticket would wait for them)
    child0 = M::add(&ctl->ntask, nchild);
    if (child0 <= cap - nchild) return true;
    M::max(&ctl->refused, INT32_MAX - child0);
    return false;
}

// a task's parent in its flag
#define WALK_FLAG(t, parent) ((int64_t)(parent) << 32 | ((t) + 1))

// after the row and the stack of `self` are stored: its record, then its shares' flags (lane: this one of
// M::LANES that all call)
template <typename M>
WALK_FN void walk_publish(WalkCtl *ctl, const WalkPool &B, const WalkTask &T, int child0, int self, int lane)
{
    M::record(&B.tasks[self], T, lane);
    if (lane == 0) M::add(&ctl->open, T.nchild);
    M::settle();
#pragma unroll 1
    for (int q = lane; q < T.nchild; q += M::LANES)
        M::store(&B.ready[(child0 + q) % B.tcount], WALK_FLAG(child0 + q, self));
}

// puts group g back, in the group pass or the task pass (one lane)
template <typename M> WALK_FN void walk_put_back(WalkCtl *ctl, const WalkPool &B, bool task, int g)
{
    M::set(&B.again[g >> 5], (int32_t)(1u << (g & 31)));
    if (task) M::add(&ctl->failed, 1);
    if (M::add(&ctl->back, 1) == 0 && !task) {
        M::add(&ctl->open, 1);
        M::store(&ctl->resume, 1);
    }
}

// No task is open and every other wave waits (one lane of the wave that counted the last one off): the next
// batch of groups that were put back, or the end.  A batch is a quarter of the groups the group pass cut,
// then twice the last one, or half of what got through of it.
template <typename M> WALK_FN void task_refill(WalkCtl *ctl, const WalkPool &B)
{
    const int back = M::load(&ctl->back);
    if (back == 0) {
        for (int i = 0; i < WALK_DONE; i++) M::store(&ctl->done[i * 32], 1);
        return;
    }
    const int was = M::load(&ctl->batch), failed = M::load(&ctl->failed);
    const int refused = M::load(&ctl->refused), top = refused ? INT32_MAX - refused : M::load(&ctl->ntask);
    const bool alone = was == 1 && failed;
    const int cut = M::load(&ctl->ngroup) < B.gcount ? M::load(&ctl->ngroup) : B.gcount;
    int n = was == 0 ? cut / 4 : failed ? (was - failed) / 2 : 2 * was;
    if (n > back) n = back;
    if (n > B.gcount) n = B.gcount;
    if (n > B.tcount / 2) n = B.tcount / 2;
    if (n > 4096) n = 4096;  // one lane writes them all
    if (n < 1) n = 1;
    const int level = alone ? M::load(&ctl->level) + 1 : 0, words = M::load(&ctl->words);
    int got = 0, w = M::load(&ctl->word), last = M::load(&ctl->last);
    auto put = [&](int g) {
        const WalkTask T{g, -1, 0, level, -1, 0, (top + got) % B.tcount, 1, 1, {}};
        for (int i = 0; i < M::LANES; i++) M::record(&B.tasks[got], T, i);
        for (int i = 0; i < 4; i++) M::store(&B.counts[4 * got + i], (int64_t)0);
        last = g;
        got++;
    };
    if (alone) {
        M::store(&B.again[last >> 5], (int32_t)((uint32_t)M::load(&B.again[last >> 5]) & ~(1u << (last & 31))));
        put(last);
    }
    for (int seen = 0; got < n && seen <= words; seen += 8) {
        int32_t bits[8];
#pragma unroll
        for (int i = 0; i < 8; i++) bits[i] = M::load(&B.again[w + i]);
        for (int i = 0; i < 8 && got < n; i++) {
            uint32_t b = (uint32_t)bits[i];
            if (!b) continue;
            for (; b && got < n; b &= b - 1) put(32 * (w + i) + __builtin_ctz(b));
            M::store(&B.again[w + i], (int32_t)b);
        }
        if (got < n) w = w + 8 < words ? w + 8 : 0;
    }
    M::store(&ctl->back, back - got);
    M::store(&ctl->ngroup, got);
    M::store(&ctl->npool, 0);
    M::store(&ctl->ntask, top + got);
    M::store(&ctl->refused, 0);
    M::store(&ctl->base, top + 1);
    M::store(&ctl->batch, got);
    M::store(&ctl->failed, 0);
    M::store(&ctl->last, last);
    M::store(&ctl->level, level);
    M::store(&ctl->word, w);
    M::store(&ctl->open, got);
    M::settle();
    for (int i = 0; i < got; i++) M::store(&B.ready[(top + i) % B.tcount], WALK_FLAG(top + i, i));
}

// share q of a task of `count` saved entries
WALK_FN int share_count(int count, int nchild, int q) { return (count - q + nchild - 1) / nchild; }

enum { TASK_END = -1, TASK_NONE = -2 };

// One look for a task by a wave of class x (one lane): its slot, TASK_NONE (look again), or TASK_END when
// no task is open any more and no group put back.  parent: the task's parent's entry.  ticket: the task drawn
// and not yet walked (-1: none).  closed: tasks this wave has finished since it last counted them off, which
// it does before it waits: a count per task on one word would take milliseconds.
template <typename M>
WALK_FN int task_look(WalkCtl *ctl, const WalkPool &B, int x, int line, int looks, int &ticket, int &closed,
                      int &parent)
{
    if (ticket < 0) ticket = x + NXCD * M::add(&ctl->ticket[x * CTR_STRIDE], 1);
    const int slot = ticket % B.tcount;
    const int64_t flag = M::load(&B.ready[slot]);
    if ((int32_t)flag == ticket + 1) {
        ticket = -1;
        parent = (int)(flag >> 32);
        return slot;
    }
    if (looks && M::load(&ctl->done[line * 32])) return TASK_END;
    if (closed) {
        M::settle();  // what it put back is counted before its tasks are
        if (M::sub(&ctl->open, closed) == closed) task_refill<M>(ctl, B);
        closed = 0;
    }
    if (looks % STEAL_LOOKS == STEAL_LOOKS - 1) {
        int v[NXCD];
        int64_t r[NXCD];  // the loads of a kind go out together
        const int resume = M::load(&ctl->resume);
#pragma unroll
        for (int y = 0; y < NXCD; y++) v[y] = M::load(&ctl->ticket[y * CTR_STRIDE]);
#pragma unroll
        for (int y = 0; y < NXCD; y++) r[y] = M::load(&B.ready[(y + NXCD * v[y]) % B.tcount]);
#pragma unroll
        for (int y = 0; y < NXCD; y++) {
            const int t = y + NXCD * v[y];
            if ((int32_t)r[y] == t + 1 && M::cas(&ctl->ticket[y * CTR_STRIDE], v[y], v[y] + 1)) {
                parent = (int)(r[y] >> 32);
                return t % B.tcount;
            }
        }
        if (resume && M::cas(&ctl->resume, 1, 0)) closed++;
    }
    return TASK_NONE;
}

// the row of a share of entry p is stored, or one of its group found no room: true if p has all its shares' rows
// now (one lane)
template <typename M> WALK_FN bool task_close(const WalkPool &B, int p) { return M::sub(&B.tasks[p].wait, 1) == 1; }
