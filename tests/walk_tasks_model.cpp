// Runs the scheduling of cut traversals (pytreegrav_amd/csrc/walk_tasks.hpp) with a thread for each wave.
// A traversal is a stack of numbers: v is summed and pushes v / 2 and (v - 1) / 2.  Sums are hashes that
// depend on the order of every term, so a group's result shows what it was cut into.
//
// argv: the classes that have a running wave (bit mask), threads per class, groups, the largest group's
// number, slots of the task table, saved stack entries, entries for groups.
// Exit status 0: each group's result and counts are those it has alone, and every wave saw the end.
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#define WALK_FN static inline
#include "walk_tasks.hpp"

struct HostMem {
    static constexpr int LANES = 1;
    template <typename T> static T load(const T *p) { return __atomic_load_n(p, __ATOMIC_SEQ_CST); }
    template <typename T> static void store(T *p, T v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
    static void record(WalkTask *p, const WalkTask &T, int)
    {
        for (int i = 0; i < WALK_TASK_WORDS; i++) store((int32_t *)p + i, ((const int32_t *)&T)[i]);
    }
    static int32_t add(int32_t *p, int32_t v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
    static int32_t sub(int32_t *p, int32_t v) { return __atomic_fetch_sub(p, v, __ATOMIC_SEQ_CST); }
    static void set(int32_t *p, int32_t b) { __atomic_fetch_or(p, b, __ATOMIC_SEQ_CST); }
    static void max(int32_t *p, int32_t v)
    {
        int32_t is = load(p);
        while (is < v && !cas(p, is, v)) is = load(p);
    }
    static bool cas(int32_t *p, int32_t is, int32_t v)
    {
        return __atomic_compare_exchange_n(p, &is, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
    }
    static void settle() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }
};
typedef HostMem M;

static WalkCtl ctl;
static WalkPool pool;
static int groups, largest;
static std::vector<uint64_t> rows, out;
static std::vector<int64_t> visits;

static int number(int g) { return g == groups / 2 ? largest : 1 + (int)((uint32_t)g * 2654435761u % 97); }
static int budget(bool share, int level) { return (share ? 6 : 10) << (level < 8 ? 3 * level : 24); }
static int shares(bool share, int cnt)
{
    const int most = share ? 11 : 5, n = cnt >> 1;
    return n > most ? most : n < 1 ? 1 : n;
}

// walks the stack until it is empty or the budget is reached
static void traverse(std::vector<int> &stack, int budget, uint64_t &sum, int64_t &n)
{
    sum = 0;
    n = 0;
    while (!stack.empty() && n < budget) {
        const int v = stack.back();
        stack.pop_back();
        sum = sum * 6364136223846793005ull + v;
        n++;
        if (v > 1) stack.push_back(v / 2);
        if (v > 2) stack.push_back((v - 1) / 2);
    }
}
static uint64_t join(uint64_t a, uint64_t b) { return a * 1000003u ^ b; }

// the result of a traversal alone, the tasks and stack entries its cuts take, and its visits
static uint64_t alone(std::vector<int> stack, bool share, int level, int64_t &ntask, int64_t &nentry, int64_t &n)
{
    uint64_t s;
    int64_t k;
    traverse(stack, budget(share, level), s, k);
    n += k;
    if (stack.empty()) return s;
    const int cnt = (int)stack.size(), nchild = shares(share, cnt);
    ntask += nchild;
    nentry += cnt;
    for (int q = 0; q < nchild; q++) {
        std::vector<int> part;
        for (int i = q; i < cnt; i += nchild) part.push_back(stack[i]);
        s = join(s, alone(part, true, level, ntask, nentry, n));
    }
    return s;
}

// the row of a share of entry p is there (or its group found no room)
static void add_up(int p)
{
    for (;;) {
        M::settle();
        if (!task_close<M>(pool, p)) return;
        const WalkTask *T = &pool.tasks[p];
        if (p < pool.gcount && M::load(&T->root)) return walk_put_back<M>(&ctl, pool, true, M::load(&T->group));
        const bool own = M::load(&T->off) >= 0;
        const int kid0 = M::load(&T->child0), nchild = M::load(&T->nchild);
        uint64_t s = M::load(&rows[own ? p : pool.gcount + kid0]);
        for (int k = own ? 0 : 1; k < nchild; k++) s = join(s, M::load(&rows[pool.gcount + (kid0 + k) % pool.tcount]));
        if (p < pool.gcount) {
            const int g = M::load(&T->group);
            out[g] = s;
            visits[g] += M::load(&pool.counts[4 * p]);
            return;
        }
        M::store(&rows[p], s);
        p = M::load(&T->parent);
    }
}

// a group (self < 0) or a task
static void walk(int g, int self, int parent)
{
    const bool task = self >= 0;
    const WalkTask *T = task ? &pool.tasks[parent] : nullptr;
    const int level = task ? M::load(&T->level) : 0, off0 = task ? M::load(&T->off) : -1;
    const bool share = off0 >= 0;
    const int root = !task ? -1 : parent < pool.gcount ? parent : M::load(&T->root);
    if (task) g = M::load(&T->group);
    std::vector<int> stack;
    if (share) {
        const int n = M::load(&T->nchild), q = (self - pool.gcount - M::load(&T->child0) + pool.tcount) % pool.tcount;
        for (int i = 0; i < share_count(M::load(&T->count), n, q); i++) stack.push_back(M::load(&pool.entries[off0 + q + i * n]));
    } else {
        stack.push_back(number(g));
    }
    uint64_t s;
    int64_t n;
    traverse(stack, budget(share, level), s, n);
    int off = 0, child0 = 0;
    const int cnt = (int)stack.size(), nchild = shares(share, cnt);
    const bool cut = cnt > 0;
    if (cut && !walk_room<M>(&ctl, pool, cnt, nchild, self, off, child0)) {
        if (!task) return walk_put_back<M>(&ctl, pool, false, g);
        M::store(&pool.tasks[root].root, 1);
        return add_up(parent);
    }
    if (!task && !cut) {
        out[g] = s;
        visits[g] += n;
        return;
    }
    if (!task) M::store(&pool.counts[4 * self], n);
    else __atomic_fetch_add(&pool.counts[4 * root], n, __ATOMIC_SEQ_CST);
    M::store(&rows[self], s);
    if (!cut) return add_up(parent);
    for (int i = 0; i < cnt; i++) M::store(&pool.entries[off + i], stack[i]);
    walk_publish<M>(&ctl, pool, WalkTask{g, parent, task ? root : 0, level, off, cnt, child0 % pool.tcount, nchild, nchild, {}},
                    child0, self, 0);
}

static bool wave(int x, int id)
{
    int ticket = -1, closed = 0, parent = -1;
    if (M::load(&ctl.open) == 0) return true;
    for (int looks = 0; looks < 20000000; looks++) {
        const int t = task_look<M>(&ctl, pool, x, id % WALK_DONE, looks, ticket, closed, parent);
        if (t == TASK_END) return true;
        if (t == TASK_NONE) {
            std::this_thread::yield();
            continue;
        }
        walk(-1, pool.gcount + t, parent);
        closed++;
        looks = -1;
    }
    return false;
}

int main(int argc, char **argv)
{
    auto arg = [&](int i, int def) { return argc > i ? atoi(argv[i]) : def; };
    const int classes = arg(1, 255), per = arg(2, 2);
    groups = arg(3, 100);
    largest = arg(4, 1000);
    pool.tcount = arg(5, 4096);
    pool.ecap = arg(6, 65536);
    pool.gcount = arg(7, 512);
    std::vector<WalkTask> tasks(pool.gcount + pool.tcount);
    std::vector<int64_t> ready(WALK_MAX_TASKS);
    std::vector<int32_t> again(ctl.words = (groups + 255) / 256 * 8);
    std::vector<int64_t> counts(4 * pool.gcount);
    std::vector<int> entries(pool.ecap);
    pool.tasks = tasks.data();
    pool.ready = ready.data();
    pool.again = again.data();
    pool.counts = counts.data();
    pool.entries = entries.data();
    rows.resize(tasks.size());
    out.resize(groups);
    visits.resize(groups);
    std::vector<std::thread> th;
    for (int i = 0; i < 4; i++)
        th.emplace_back([] {
            for (int g; (g = M::add(&ctl.ctr[0], 1)) < groups;) walk(g, -1, -1);
        });
    for (auto &t : th) t.join();
    const int was_back = ctl.back;
    th.clear();
    std::vector<int> ok(NXCD * per, 1);
    for (int x = 0; x < NXCD; x++)
        for (int i = 0; i < per; i++)
            if (classes >> x & 1) th.emplace_back([&, x, i] { ok[x * per + i] = wave(x, x + NXCD * i); });
    for (auto &t : th) t.join();
    for (int v : ok)
        if (!v) {
            printf("a wave waited in vain\n");
            return 2;
        }
    int deepest = 0;
    for (int g = 0; g < groups; g++) {
        uint64_t want = 0;
        int64_t n = 0;
        for (int level = 0; level <= 8; level++) {
            int64_t ntask = 0, nentry = 0;
            n = 0;
            want = alone({number(g)}, false, level, ntask, nentry, n);
            if (level > deepest) deepest = level;
            if (ntask <= pool.tcount - 1 && nentry <= pool.ecap) break;
        }
        if (out[g] != want || visits[g] != n) {
            printf("group %d: another result than alone (visits %lld, %lld alone)\n", g, (long long)visits[g], (long long)n);
            return 1;
        }
    }
    printf("%d groups put back by the group pass, level %d\n", was_back, deepest);
    return 0;
}
