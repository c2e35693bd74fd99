// Runs the scheduling of cut traversals (pytreegrav_amd/csrc/walk_tasks.hpp) with a thread for each wave.
// argv: the classes that have a running wave (bit mask), threads per class, deferred groups.
// Exit status 0: every published task was walked exactly once and every wave saw the end.
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#define WALK_FN static inline
#include "walk_tasks.hpp"

struct HostMem {
    static constexpr int LANES = 1;
    static int32_t load(const int32_t *p) { return __atomic_load_n(p, __ATOMIC_SEQ_CST); }
    static void store(int32_t *p, int32_t v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
    static int32_t add(int32_t *p, int32_t v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
    static int32_t sub(int32_t *p, int32_t v) { return __atomic_fetch_sub(p, v, __ATOMIC_SEQ_CST); }
    static bool cas(int32_t *p, int32_t is, int32_t v)
    {
        return __atomic_compare_exchange_n(p, &is, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
    }
    static void settle() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }
};

static WalkCtl ctl;
static WalkPool pool;
static std::vector<int32_t> walked;

// a task or group of `size` steps of work that is past its budget: published as nchild shares
static bool cut(bool task, int group, int self, int size)
{
    const int nchild = 1 + size / 4 % 7;
    const int child0 = walk_take<HostMem>(&ctl.ntask, nchild, pool.tcount);
    if (child0 < 0) return false;
    walk_publish<HostMem>(&ctl, pool, task, group, size, nchild, 0, pool.gcount + child0, self, 0);
    return true;
}

static bool wave(int x, int id)
{
    int ticket = -1, closed = 0;
    for (int looks = 0; looks < 20000000; looks++) {
        const int t = task_look<HostMem>(&ctl, pool, x, id % WALK_DONE, looks, ticket, closed);
        if (t == TASK_END) return true;
        if (t == TASK_NONE) {
            std::this_thread::yield();
            continue;
        }
        const WalkTask *T = &pool.tasks[pool.gcount + t];
        HostMem::add(&walked[t], 1);
        const int size = HostMem::load(&T->count);
        if (size > 8) cut(true, HostMem::load(&T->group), pool.gcount + t, size);
        closed++;
        looks = -1;
    }
    return false;
}

int main(int argc, char **argv)
{
    const int classes = argc > 1 ? atoi(argv[1]) : 255, per = argc > 2 ? atoi(argv[2]) : 2, groups = argc > 3 ? atoi(argv[3]) : 100;
    pool.gcount = groups;
    pool.tcount = 4096;
    std::vector<WalkTask> tasks(pool.gcount + pool.tcount);
    std::vector<int32_t> ready(WALK_MAX_TASKS);
    walked.assign(pool.tcount, 0);
    pool.tasks = tasks.data();
    pool.ready = ready.data();
    for (int g = 0; g < groups; g++) cut(false, g, g, 20 + g * 7 % 200);
    std::vector<std::thread> th;
    std::vector<int> ok(NXCD * per, 1);
    for (int x = 0; x < NXCD; x++)
        for (int i = 0; i < per; i++)
            if (classes >> x & 1) th.emplace_back([&, x, i] { ok[x * per + i] = wave(x, x + NXCD * i); });
    for (auto &t : th) t.join();
    const int n = ctl.ntask < pool.tcount ? ctl.ntask : pool.tcount;
    for (int t = 0; t < n; t++)
        if (walked[t] != ready[t]) {
            printf("task %d: published %d, walked %d\n", t, ready[t], walked[t]);
            return 1;
        }
    for (int v : ok)
        if (!v) {
            printf("a wave waited in vain\n");
            return 2;
        }
    printf("%d tasks\n", n);
    return 0;
}
