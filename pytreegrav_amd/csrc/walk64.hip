// Grouped Barnes-Hut walk in FP64 with the reference's branch set (grouped_treewalk.py:45-241): the
// decisions of its opening test bit for bit, and per pair r2 > 0, softened iff r < max(h_s, h_t).
//
// The reference's groups hold 8 targets by default, an eighth of a wavefront, so the wave splits into
// slices: lane l holds target l mod P (P = group size rounded up to a power of two) and evaluates the
// list entries l / P, l / P + 64 / P, ...; the slices' sums are added by shuffles at the end.  Accepted
// nodes need neither the self test nor the softening (the opening test keeps every target farther than
// max(h_s, h_t) from them) and take one reciprocal square root; particles outside every softening
// radius of the group join them (monopole walks).
//
// The reference's groups are runs of the Morton order.  A run that crosses a high-level cell boundary
// in a sparse region has a box as wide as the domain, opens nearly every node, and one wave walking it
// alone sets the kernel's time (1.48e6 of the 2.9e8 visits of a 1e6-particle Plummer sphere are one
// group's).  A task past its budget of visits is therefore deferred: it saves its stack, cut into
// interleaved shares, as tasks of the next round, and k_walk64_sum adds the shares' partial sums in
// their order.  The cut depends only on the group's own traversal, so results do not depend on
// scheduling (unless the task tables fill up: then the rest is walked in place, the same terms summed
// in another order).
//
// Bound: instruction issue, about 60 % of it the traversal (250 instructions per 64-element step).
// Whole calls, against one wave per group evaluating every entry for 8 of its 64 lanes with IEEE
// square roots and divisions: 1e6-particle Plummer sphere 333 -> 6.1 ms (the walk 3.2 ms of it where
// it took 332), uniform cube of 1e5 6.0 -> 0.87 ms, tidal tensors with quadrupoles of 6e4 23.3 -> 1.6 ms.

#include "walk_shared.hpp"

#define LIST 32           // a list is evaluated in multiples of LIST entries once it holds LIST
#define ICAP (LIST + 64)  // LIST - 1 entries + one step's 64
#define BUDGET 4096       // visits after which a task is deferred (not in the last round), at least
#define SHARES0 64        // tasks a deferred group is cut into, at most (of DIV0 stack entries or more)
#define DIV0 16
#define SHARES 128        // tasks a deferred task is cut into, at most (of DIV stack entries or more)
#define DIV 4
#define SHARE_BYTES 262144  // of partial sums, past 16 tasks: large groups are cut into fewer
#define MAX_BLOCKS_PER_CU 4
#define MAX_TASKS 196608  // of round 1; a quarter of it in each later round, an eighth deferred groups

struct Walk64Task {
    int32_t group;
    int32_t child0, nchild;      // its shares in the task tables (deferred tasks; else nchild 0)
    int32_t off, stride, count;  // saved stack entries pool[off + i * stride], i < count
};

struct Walk64Pool {
    int *spill;  // per-wave global stacks, gcap entries each
    int gcap;
    int *entries;  // saved stacks
    int ecap;
    // task tables: the deferred groups, then the tasks of rounds 1, 2, ..; table k starts at base[k]
    // and holds cap[k] (cap[0] = 0: nothing is deferred)
    Walk64Task *tasks;
    int base[WALK_ROUNDS], cap[WALK_ROUNDS];
    int budget, shares0, shares;
    double *partial;    // one row of gs * WI sums per task and deferred group, in the order of tasks
};

template <bool QUAD> struct Lds64 {
    int stack[SCAP];
    V4<double> nodes[ICAP];  // elements no target can be inside the softening of: x y z m
    double nq[QUAD ? 6 * ICAP : 1];
    V4<double> parts[ICAP];  // particles: x y z m
    double ph[ICAP];
};

// 1/sqrt(x) and 1/x: the hardware estimate (2^-24) with one cubic step, 1-2 ulp
__device__ __forceinline__ double rsqrt64(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double rcp64(double x)
{
    const double y = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// squared distances are capped so that the refinement of 1/sqrt stays finite (r2 = inf gives nan)
#define R2_MAX 1e300

template <int FIELDS>
__device__ __forceinline__ void add_pair(Acc<double> &a, double phi, double K, double Q, double dx, double dy, double dz)
{
    if (NW<FIELDS>::POT) a.phi += phi;
    if (NW<FIELDS>::ACC) {
        a.gx += K * dx;
        a.gy += K * dy;
        a.gz += K * dz;
    }
    if (NW<FIELDS>::TID) {
        const double qx = Q * dx, qy = Q * dy;
        a.txx += qx * dx - K;
        a.tyy += qy * dy - K;
        a.tzz += Q * dz * dz - K;
        a.txy += qx * dy;
        a.txz += qx * dz;
        a.tyz += qy * dz;
    }
}

template <int FIELDS, bool QUAD>
__device__ __forceinline__ void pair_node(Acc<double> &a, const V4<double> &s, const double *q, double tx, double ty,
                                          double tz)
{
    const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    const double r2 = fmin(dx * dx + dy * dy + dz * dz, R2_MAX);
    const double rinv = rsqrt64(r2), rinv2 = rinv * rinv;
    const double mr = s.w * rinv, K = mr * rinv2;
    add_pair<FIELDS>(a, -mr, K, 3.0 * K * rinv2, dx, dy, dz);
    if (QUAD) {
        const double qxx = q[0], qxy = q[1], qxz = q[2], qyy = q[3], qyz = q[4], qzz = q[5];
        const double r5inv = rinv2 * rinv2 * rinv, r7inv = r5inv * rinv2;
        const double qdx = qxx * dx + qxy * dy + qxz * dz;
        const double qdy = qxy * dx + qyy * dy + qyz * dz;
        const double qdz = qxz * dx + qyz * dy + qzz * dz;
        const double A = dx * qdx + dy * qdy + dz * qdz;
        if (NW<FIELDS>::POT) a.phi += -0.5 * A * r5inv;
        if (NW<FIELDS>::ACC) {
            const double f = 2.5 * A * r7inv;
            a.gx += f * dx - qdx * r5inv;
            a.gy += f * dy - qdy * r5inv;
            a.gz += f * dz - qdz * r5inv;
        }
        if (NW<FIELDS>::TID) {
            const double diag = -2.5 * A * r7inv, fac = 17.5 * A * r7inv * rinv2;
            const double fx = fac * dx, fy = fac * dy;
            const double px = qdx * r7inv, py = qdy * r7inv, pz = qdz * r7inv;
            a.txx += qxx * r5inv - 10.0 * dx * px + diag + fx * dx;
            a.tyy += qyy * r5inv - 10.0 * dy * py + diag + fy * dy;
            a.tzz += qzz * r5inv - 10.0 * dz * pz + diag + fac * dz * dz;
            a.txy += qxy * r5inv - 5.0 * (dx * py + dy * px) + fx * dy;
            a.txz += qxz * r5inv - 5.0 * (dx * pz + dz * px) + fx * dz;
            a.tyz += qyz * r5inv - 5.0 * (dy * pz + dz * py) + fy * dz;
        }
    }
}

// the M4 spline softening of kernel.py:4-75 at 0 < r < h
template <int FIELDS>
__device__ __forceinline__ void spline64(double r, double rinv, double h, double &phi, double &K, double &Q)
{
    const double hinv = rcp64(h), q = r * hinv;
    const double hinv2 = hinv * hinv, hinv3 = hinv2 * hinv;
    if (q <= 0.5) {
        const double q2 = q * q;
        if (NW<FIELDS>::POT)
            phi = (-2.8 + q2 * (5.33333333333333333 + q2 * (6.4 * q - 9.6))) * hinv;
        K = (10.666666666666666666 + q2 * (-38.4 + 32.0 * q)) * hinv3;
        if (NW<FIELDS>::TID) Q = (76.8 - 96.0 * q) * hinv3 * hinv2;
    } else {
        const double qinv = h * rinv, qinv3 = qinv * qinv * qinv;
        if (NW<FIELDS>::POT)
            phi = (-3.2 + 0.066666666666666666666 * qinv +
                   q * q * (10.666666666666666666666 + q * (-16.0 + q * (9.6 - 2.1333333333333333333333 * q)))) *
                  hinv;
        K = (21.333333333333 - 48.0 * q + 38.4 * q * q - 10.666666666667 * q * q * q - 0.066666666667 * qinv3) * hinv3;
        if (NW<FIELDS>::TID) Q = (48.0 * qinv - 76.8 + 32.0 * q - 0.2 * qinv3 * qinv * qinv) * hinv3 * hinv2;
    }
}

template <int FIELDS>
__device__ __forceinline__ void pair_part(Acc<double> &a, const V4<double> &s, double hs, double tx, double ty, double tz,
                                          double th)
{
    const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    const double r2 = fmin(dx * dx + dy * dy + dz * dz, R2_MAX);
    const double h = fmax(hs, th);
    const bool apart = r2 > 0.0;
    const double rinv = apart ? rsqrt64(r2) : 0.0, rinv2 = rinv * rinv;
    const double mr = s.w * rinv;
    double phi = -mr, K = mr * rinv2, Q = 3.0 * K * rinv2;
    const bool soft = apart && r2 < h * h;
    if (ptg_ballot(soft)) {
        if (soft) {
            spline64<FIELDS>(r2 * rinv, rinv, h, phi, K, Q);
            phi *= s.w;
            K *= s.w;
            Q *= s.w;
        }
    }
    add_pair<FIELDS>(a, phi, K, Q, dx, dy, dz);
}

// components of one target's sums, in the order they are stored in a partial row
template <int FIELDS, typename F> __device__ __forceinline__ void each_sum(Acc<double> &a, F f)
{
    if (NW<FIELDS>::POT) f(a.phi);
    if (NW<FIELDS>::ACC) {
        f(a.gx);
        f(a.gy);
        f(a.gz);
    }
    if (NW<FIELDS>::TID) {
        f(a.txx);
        f(a.txy);
        f(a.txz);
        f(a.tyy);
        f(a.tyz);
        f(a.tzz);
    }
}
template <int FIELDS> struct Sums {
    static constexpr int WI = NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC + 6 * NW<FIELDS>::TID;
};

// the output row o[] entries that sum c of a target fills (two for an off-diagonal tidal component)
template <int FIELDS> __device__ __forceinline__ void store_sum(double *o, int c, double v)
{
    constexpr int PA = NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC;
    if (!NW<FIELDS>::TID || c < PA) {
        o[c] = v;
        return;
    }
    const int k = c - PA;
    const int i = k < 3 ? 0 : k < 5 ? 1 : 2, j = k < 3 ? k : k < 5 ? k - 2 : 2;
    o[PA + 3 * i + j] = v;
    o[PA + 3 * j + i] = v;
}

struct Group64 {
    int64_t a0;  // first target
    int mt;      // targets
    int over;    // targets of a supplied group past gs (not evaluated)
};

__device__ __forceinline__ Group64 group_of(const Walk64Args &A, int64_t g)
{
    const int64_t a0 = A.goff ? (int64_t)A.goff[g] : g * A.gs;
    const int64_t e0 = A.goff ? (int64_t)A.goff[g + 1] : A.nt;
    const int64_t b0 = e0 < a0 + A.gs ? e0 : a0 + A.gs;
    return Group64{a0, (int)(b0 - a0), A.goff && e0 > b0};
}

// n consecutive entries of a table of cap counted by *counter: the first one's index (one lane calls).
// Past cap - n they do not fit: cap if nothing was taken, else the entries below cap are the caller's
// all the same.  The counter is added to once and never taken back: when thousands of waves reach
// their budgets together, compare-and-swap loops on it took 27 ms.
__device__ __forceinline__ int take(int32_t *counter, int n, int cap)
{
    const int seen = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return seen > cap - n ? cap : atomicAdd(counter, n);
}

// waves per SIMD the registers are capped for: four where the LDS lets four blocks onto a CU
template <int TPL, int FIELDS, bool QUAD> struct Occ64 {
    static constexpr int waves = TPL == 1 && !QUAD && !NW<FIELDS>::TID ? 4 : 1;
};

template <int TPL, int FIELDS, bool QUAD>
__global__ __launch_bounds__(64 * WALK_WAVES) __attribute__((amdgpu_waves_per_eu(Occ64<TPL, FIELDS, QUAD>::waves)))
void k_walk64(const Walk64Args A, const Walk64Pool B, int round)
{
    constexpr int WI = Sums<FIELDS>::WI;
    __shared__ Lds64<QUAD> lds[WALK_WAVES];
    const int wave = threadIdx.x >> 6, lane = ptg_lane();
    Lds64<QUAD> &L = lds[wave];
    int *spill = B.spill + ((int64_t)blockIdx.x * WALK_WAVES + wave) * (int64_t)B.gcap;
    const int xcd = blockIdx.x % NXCD;
    int64_t n_int = 0, n_vis = 0, n_part = 0;
    int ghw = 0;
    const int64_t ngroups = A.goff ? (int64_t)__builtin_amdgcn_readfirstlane(*A.gcount) : A.ngroups;
    const int ntask = round ? std::min(__builtin_amdgcn_readfirstlane(A.ctl->ntask[round]), B.cap[round]) : 0;
    if (round && ntask == 0) return;
    // targets per slice, a power of two
    int P = 64;
    if (TPL == 1)
        while (P > 1 && P / 2 >= A.gs) P /= 2;
    const int tl = lane & (P - 1), sl = lane / P, slices = 64 / P;

    // groups (round 0) or tasks from per-XCD counters, as the FP32 walk takes its groups
    const int64_t nwork = round ? ntask : ngroups;
    int32_t *ctr = round ? A.ctl->tctr + (round - 1) * NXCD * CTR_STRIDE : A.ctl->ctr;
    for (int attempt = 0; attempt < NXCD; attempt++) {
        const int x = (xcd + attempt) % NXCD;
        const int64_t w_lo = nwork * x / NXCD, w_hi = nwork * (x + 1) / NXCD;
        for (;;) {
            int wi = 0;
            if (lane == 0) wi = atomicAdd(&ctr[x * CTR_STRIDE], 1);
            const int64_t work = w_lo + __builtin_amdgcn_readfirstlane(wi);
            if (work >= w_hi) break;
            int64_t g = work;
            int t_off = 0, t_stride = 0, t_count = 0;
            if (round) {
                const Walk64Task *T = &B.tasks[B.base[round] + work];
                g = __builtin_amdgcn_readfirstlane(T->group);
                t_off = __builtin_amdgcn_readfirstlane(T->off);
                t_stride = __builtin_amdgcn_readfirstlane(T->stride);
                t_count = __builtin_amdgcn_readfirstlane(T->count);
            }
            const Group64 grp = group_of(A, g);
            const int64_t a0 = grp.a0;
            const int mt = grp.mt;
            if (grp.over && lane == 0) atomicOr(&A.ctl->err, 2);  // a supplied group larger than group_size
            int root = 0;
            if (A.nsys > 0) {
                int64_t lo = 0, hi = A.nsys;  // last system with soff[s] <= a0
                while (hi - lo > 1) {
                    const int64_t mid = (lo + hi) >> 1;
                    if (A.soff[mid] <= a0) lo = mid;
                    else hi = mid;
                }
                root = (int)lo;
            }

            // ---- targets: lane holds a0 + tl + 64 j; the slices hold the same targets ----
            double tx[TPL], ty[TPL], tz[TPL], th[TPL];
            int64_t tidx[TPL];
            bool tval[TPL];
            double bmin0 = INFINITY, bmin1 = INFINITY, bmin2 = INFINITY;
            double bmax0 = -INFINITY, bmax1 = -INFINITY, bmax2 = -INFINITY, hmax = -INFINITY;
            const double ox = A.nsys > 0 ? 0.0 : A.ox, oy = A.nsys > 0 ? 0.0 : A.oy, oz = A.nsys > 0 ? 0.0 : A.oz;
#pragma unroll
            for (int j = 0; j < TPL; j++) {
                const int o = tl + 64 * j;
                tval[j] = o < mt;
                tidx[j] = tval[j] ? A.perm[a0 + o] : 0;
                if (tval[j]) {
                    const int64_t src = A.sorted ? a0 + o : tidx[j];
                    tx[j] = A.pos[3 * src] - ox;
                    ty[j] = A.pos[3 * src + 1] - oy;
                    tz[j] = A.pos[3 * src + 2] - oz;
                    th[j] = A.soft[src];
                    bmin0 = std::min(bmin0, tx[j]);
                    bmin1 = std::min(bmin1, ty[j]);
                    bmin2 = std::min(bmin2, tz[j]);
                    bmax0 = std::max(bmax0, tx[j]);
                    bmax1 = std::max(bmax1, ty[j]);
                    bmax2 = std::max(bmax2, tz[j]);
                    hmax = std::max(hmax, th[j]);
                } else {
                    tx[j] = ty[j] = tz[j] = th[j] = 0.0;
                }
            }
            bmin0 = ptg_wave_min(bmin0);
            bmin1 = ptg_wave_min(bmin1);
            bmin2 = ptg_wave_min(bmin2);
            bmax0 = ptg_wave_max(bmax0);
            bmax1 = ptg_wave_max(bmax1);
            bmax2 = ptg_wave_max(bmax2);
            hmax = ptg_wave_max(hmax);
            Acc<double> acc[TPL];
#pragma unroll
            for (int j = 0; j < TPL; j++) acc[j] = Acc<double>{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

            int sp = 1, gsp = 0, nn = 0, np = 0, visits = 0;
            bool overflow = false;
            if (round) {
                sp = t_count;  // <= SCAP: deeper stacks are not deferred
                for (int q = lane; q < sp; q += 64) L.stack[q] = B.entries[t_off + (int64_t)q * t_stride];
            } else {
                // the root of system s occupies walk slot s; a subtree walk starts at its element's slot
                // instead (wave-uniform; an out-of-range slot is reported, and dropped when popped like
                // any corrupt link, so it walks nothing)
                int first = root;
                if (A.start) {
                    first = __builtin_amdgcn_readfirstlane(*A.start);
                    if ((first < 0 || first >= A.nslots) && lane == 0) atomicOr(&A.ctl->err, 4);
                }
                if (lane == 0) L.stack[0] = first;
            }
            __builtin_amdgcn_wave_barrier();
            // The more groups share the device, the longer one may run alone, and the fewer should pay for
            // being cut: 4096 visits against 8192 take 0.83 / 0.95 ms (walk and build, 1e5 particles), 8192
            // against 16384 2.88 / 3.30 (3e5), 12288 against 8192 6.8 / 8.0 (6e5, clumpy).  Counted per
            // system, so that a system's cuts are those it has alone.
            const int64_t sg = (A.nsys > 0 ? A.soff[root + 1] - A.soff[root] : A.nt) / A.gs;
            int budget = B.budget * (round || sg <= 16384 ? 1 : sg <= 65536 ? 2 : sg <= 262144 ? 3 : 16);
            if (round == WALK_ROUNDS - 1 || B.cap[0] == 0) budget = 0x7fffffff;
            int child0 = -1, nchild = 0, slot = round ? B.base[round] + (int)work : -1;

            for (;;) {
                if (sp == 0) {
                    if (gsp == 0) break;
                    const int k = std::min(gsp, SPILL);
                    for (int q = lane; q < k; q += 64) L.stack[q] = spill[gsp - k + q];
                    __builtin_amdgcn_wave_barrier();
                    gsp -= k;
                    sp = k;
                }
                if (visits >= budget) {
                    // save the stack as interleaved shares of the next round; out of room: go on here
                    const int cnt = gsp + sp;
                    nchild = std::max(1, round ? std::min(B.shares, cnt / DIV) : std::min(B.shares0, cnt / DIV0));
                    const int cap = B.cap[round + 1];
                    int off = -1, at = cap;
                    if (lane == 0 && cnt <= nchild * SCAP) {
                        if (round == 0) slot = take(&A.ctl->ntask[0], 1, B.cap[0]);
                        if (round || slot < B.cap[0]) {
                            at = take(&A.ctl->ntask[round + 1], nchild, cap);
                            if (at <= cap - nchild) off = take(&A.ctl->npool, cnt, B.ecap);
                            if (off > B.ecap - cnt) off = -1;
                            if (off >= 0) child0 = B.base[round + 1] + at;
                            // a record without shares, should there be no room
                            B.tasks[slot].group = (int32_t)g;
                            B.tasks[slot].child0 = child0;
                            B.tasks[slot].nchild = off >= 0 ? nchild : 0;
                        }
                    }
                    slot = __builtin_amdgcn_readfirstlane(slot);
                    at = __builtin_amdgcn_readfirstlane(at);
                    off = __builtin_amdgcn_readfirstlane(off);
                    child0 = __builtin_amdgcn_readfirstlane(child0);
                    // the entries taken below cap are filled in any case: the next round reads all of them
                    for (int q = lane; q < nchild && at + q < cap; q += 64) {
                        Walk64Task &T = B.tasks[B.base[round + 1] + at + q];
                        T.group = (int32_t)g;
                        T.nchild = 0;
                        T.off = off + q;
                        T.stride = nchild;
                        T.count = off >= 0 ? (cnt - q + nchild - 1) / nchild : 0;
                    }
                    if (child0 >= 0) {
                        for (int q = lane; q < gsp; q += 64) B.entries[off + q] = spill[q];
                        for (int q = lane; q < sp; q += 64) B.entries[off + gsp + q] = L.stack[q];
                        break;
                    }
                    budget = 0x7fffffff;
                }
                const int k = std::min(sp, 64);
                const int base = sp - k;
                int e = lane < k ? L.stack[base + lane] : 0;
                const bool ve = lane < k && e >= 0 && e < A.nslots;  // a corrupt link is dropped, not followed
                if (!ve) e = 0;
                __builtin_amdgcn_wave_barrier();
                sp = base;
                visits += k;
                const V4<double> X = A.xyzm[e];
                const V4<double> X2 = A.aux[e];
                const int2 K = A.kids[e];
                const bool ispart = K.y == 0;
                const double dxm = box_gap(X.x, bmin0, bmax0), dym = box_gap(X.y, bmin1, bmax1);
                const double dzm = box_gap(X.z, bmin2, bmax2);
                const double r2m = dxm * dxm + dym * dym + dzm * dzm;
                const double hh = X2.x > hmax ? X2.x : hmax;
                // the reference's test r_min > max(size/theta + delta, h + 0.6 size + delta): decided on
                // the squares unless they agree to 1e-14 (or could underflow), then as written
                const double c2 = hh + X2.y * 0.6 + X2.z;
                const double cq = std::max(X2.y * A.inv_theta + X2.z, c2), cc = cq * cq;
                bool acc_node = ve & !ispart & (r2m > cc);
                const bool close = ve & !ispart & !(fabs(r2m - cc) > fma(1e-14, cc, 1e-290));
                if (ptg_ballot(close)) {
                    const double r_min = sqrt(r2m), c1 = X2.y / A.theta + X2.z;
                    if (close) acc_node = r_min > (c1 > c2 ? c1 : c2);
                }
                // a particle farther from the box than every softening radius needs neither the softening
                // nor the self test; with quadrupoles it stays a particle (no quadrupole terms)
                const bool far_part = !QUAD & ve & ispart & (r2m > hh * hh);
                const bool acc_part = ve & ispart & !far_part;
                const bool open = ve & !ispart & !acc_node;
                acc_node |= far_part;
                const uint64_t bp = ptg_ballot(acc_part), bn = ptg_ballot(acc_node);
                if (acc_part) {
                    const int at = np + lanes_below(bp);
                    L.parts[at] = X;
                    L.ph[at] = X2.x;
                }
                if (acc_node) {
                    const int at = nn + lanes_below(bn);
                    L.nodes[at] = X;
                    if (QUAD) {
                        const double *q = A.quad + 8 * (int64_t)e;
#pragma unroll
                        for (int c = 0; c < 6; c++) L.nq[6 * at + c] = q[c];
                    }
                }
                np += (int)__popcll(bp);
                nn += (int)__popcll(bn);
                if (A.counters) {
                    n_int += (int64_t)(__popcll(bp) + __popcll(bn)) * mt;
                    n_part += (int64_t)(__popcll(bp) + __popcll(ptg_ballot(far_part))) * mt;
                }

                const int cnt = open ? std::min(std::max(K.y, 0), 8) : 0;
                int tot;
                const int below = small_excl_scan(cnt, tot);
                if (sp + tot > SCAP) {
                    const int ks = spill_count(sp, tot);
                    if (gsp + ks > B.gcap) {
                        overflow = true;
                        break;
                    }
                    spill_bottom(L.stack, spill + gsp, sp, ks, lane);
                    gsp += ks;
                    sp -= ks;
                    ghw = std::max(ghw, gsp);
                }
                {
                    int *dst = &L.stack[sp + below];
#pragma unroll
                    for (int c = 0; c < 8; c++)
                        if (c < cnt) dst[c] = K.x + c;
                }
                sp += tot;
                __builtin_amdgcn_wave_barrier();

                if (nn >= LIST) {
                    const int c = nn & ~(LIST - 1);  // c >= LIST > nn - c
                    for (int q = sl; q < c; q += slices) {
                        const V4<double> s = L.nodes[q];
#pragma unroll
                        for (int j = 0; j < TPL; j++)
                            pair_node<FIELDS, QUAD>(acc[j], s, &L.nq[QUAD ? 6 * q : 0], tx[j], ty[j], tz[j]);
                    }
                    __builtin_amdgcn_wave_barrier();
                    if (lane < nn - c) {  // reads [c, nn) and writes [0, nn - c): disjoint
                        L.nodes[lane] = L.nodes[c + lane];
                        if (QUAD)
                            for (int q = 0; q < 6; q++) L.nq[6 * lane + q] = L.nq[6 * (c + lane) + q];
                    }
                    __builtin_amdgcn_wave_barrier();
                    nn -= c;
                }
                if (np >= LIST) {
                    const int c = np & ~(LIST - 1);
                    for (int q = sl; q < c; q += slices) {
                        const V4<double> s = L.parts[q];
#pragma unroll
                        for (int j = 0; j < TPL; j++) pair_part<FIELDS>(acc[j], s, L.ph[q], tx[j], ty[j], tz[j], th[j]);
                    }
                    __builtin_amdgcn_wave_barrier();
                    if (lane < np - c) {  // disjoint ranges, as above
                        L.parts[lane] = L.parts[c + lane];
                        L.ph[lane] = L.ph[c + lane];
                    }
                    __builtin_amdgcn_wave_barrier();
                    np -= c;
                }
            }
            n_vis += visits;
            if (overflow) {
                if (lane == 0) atomicOr(&A.ctl->err, 1);
                nn = np = 0;  // a task's row is still written: the sums read every task's
            }
            for (int q = sl; q < nn; q += slices) {
                const V4<double> s = L.nodes[q];
#pragma unroll
                for (int j = 0; j < TPL; j++)
                    pair_node<FIELDS, QUAD>(acc[j], s, &L.nq[QUAD ? 6 * q : 0], tx[j], ty[j], tz[j]);
            }
            for (int q = sl; q < np; q += slices) {
                const V4<double> s = L.parts[q];
#pragma unroll
                for (int j = 0; j < TPL; j++) pair_part<FIELDS>(acc[j], s, L.ph[q], tx[j], ty[j], tz[j], th[j]);
            }
            __builtin_amdgcn_wave_barrier();
            for (int d = P; d < 64; d <<= 1) {
#pragma unroll
                for (int j = 0; j < TPL; j++) each_sum<FIELDS>(acc[j], [&](double &v) { v += __shfl_xor(v, d, 64); });
            }

            // ---- G * fields in the caller's order, or the task's row of partial sums ----
            const bool whole = round == 0 && child0 < 0;
#pragma unroll
            for (int j = 0; j < TPL; j++) {
                if (!tval[j] || sl != 0) continue;
                int c = 0;
                if (whole) {
                    double *o = A.out + tidx[j] * NW<FIELDS>::W;
                    each_sum<FIELDS>(acc[j], [&](double &v) { store_sum<FIELDS>(o, c++, A.G * v); });
                } else {
                    double *o = B.partial + ((int64_t)slot * A.gs + tl + 64 * j) * WI;
                    each_sum<FIELDS>(acc[j], [&](double &v) { o[c++] = v; });
                }
            }
        }
    }
    if (lane == 0 && ghw > 0) atomicMax(&A.ctl->hwm, ghw);
    if (lane == 0 && A.counters) {
        atomicAdd((unsigned long long *)&A.counters[0], (unsigned long long)n_int);
        atomicAdd((unsigned long long *)&A.counters[1], (unsigned long long)n_vis);
        atomicAdd((unsigned long long *)&A.counters[2], (unsigned long long)n_part);
    }
}

// Adds to the row of each deferred task of round `level` the rows of its shares, in order; level 0:
// the deferred groups, whose totals are the results.  One wave per deferred task, deepest level first.
template <int FIELDS>
__global__ __launch_bounds__(256) void k_walk64_sum(const Walk64Args A, const Walk64Pool B, int level)
{
    constexpr int WI = Sums<FIELDS>::WI;
    const int nt = std::min(__builtin_amdgcn_readfirstlane(A.ctl->ntask[level]), B.cap[level]);
    const int64_t rs = (int64_t)A.gs * WI;
    for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < nt; t += gridDim.x * 4) {
        const Walk64Task T = B.tasks[B.base[level] + t];
        if (T.nchild == 0) continue;
        const Group64 grp = group_of(A, T.group);
        const int nv = grp.mt * WI;
        double *row = B.partial + (B.base[level] + t) * rs;
        const double *kids = B.partial + T.child0 * rs;
        for (int v = ptg_lane(); v < nv; v += 64) {
            double s = row[v];
#pragma unroll 8
            for (int k = 0; k < T.nchild; k++) s += kids[k * rs + v];
            if (level) {
                row[v] = s;
            } else {
                const int64_t o = A.perm[grp.a0 + v / WI];
                store_sum<FIELDS>(A.out + o * NW<FIELDS>::W, v % WI, A.G * s);
            }
        }
    }
}

// ============================================================================================
// host side
// ============================================================================================
template <int TPL, int FIELDS, bool QUAD>
static ptg_status launch(const Walk64Args &a, int cus, int gcap, char *ws, size_t ws_bytes, hipStream_t s)
{
    static int per_cu = 0;
    if (per_cu == 0) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_walk64<TPL, FIELDS, QUAD>, 64 * WALK_WAVES, 0) !=
                hipSuccess ||
            nb < 1)
            nb = 1;
        per_cu = std::min(nb, MAX_BLOCKS_PER_CU);
    }
    // the workspace after the control block: the spill stacks of the resident waves, then what deferral
    // needs; none is left over only on a device with more waves than the workspace was sized for
    Walk64Pool b{};
    size_t at = ptg_align256(sizeof(WalkCtl));
    auto carve = [&](size_t bytes) {
        char *p = ws + at;
        at += ptg_align256(bytes);
        return p;
    };
    b.gcap = gcap;
    b.spill = (int *)carve((size_t)cus * per_cu * WALK_WAVES * gcap * sizeof(int));
    const size_t left = ws_bytes > at ? ws_bytes - at : 0;
    const size_t pool = std::min<size_t>(left / 8 * 3, 48u << 20);
    const size_t row = (size_t)a.gs * Sums<FIELDS>::WI * sizeof(double);
    // an ordinary group's traversal stays well inside the budget: it grows as 1 / theta^2 and with the group
    const double open = a.theta < 0.7 ? 0.49 / (a.theta * a.theta) : 1.0;
    b.budget = (int)std::min(1e8, BUDGET * open * (a.gs <= 16 ? 1 : a.gs <= 64 ? 2 : 4));
    b.shares0 = (int)std::min<size_t>(SHARES0, std::max<size_t>(16, SHARE_BYTES / row));
    b.shares = (int)std::min<size_t>(SHARES, std::max<size_t>(16, SHARE_BYTES / row));
    const size_t nrows = left > pool + 1024 ? (left - pool - 1024) / (row + sizeof(Walk64Task)) : 0;
    const int most = (int)std::min<size_t>(MAX_TASKS, nrows * 3 / 5);
    if (most >= SHARES) {
        b.ecap = (int)(pool / sizeof(int));
        b.entries = (int *)carve(pool);
        int n = 0;
        for (int k = 0; k < WALK_ROUNDS; k++) {  // nrows * 0.6 * (1/8 + 1 + 1/4 + 1/4) rows at most
            b.base[k] = n;
            n += b.cap[k] = k == 0 ? most / 8 : k == 1 ? most : most / 4;
        }
        b.tasks = (Walk64Task *)carve(n * sizeof(Walk64Task));
        b.partial = (double *)carve(n * row);
    }
    const int64_t blocks = (int64_t)cus * per_cu;
    // a task of round r is what r budgets left of one traversal, which visits a slot once
    const int rounds = b.cap[0] ? (int)std::min<int64_t>(WALK_ROUNDS, 1 + a.nslots / b.budget) : 1;
    for (int round = 0; round < rounds; round++) {
        const int64_t nb = round || a.goff ? blocks : std::min(blocks, ptg_cdiv(a.ngroups, WALK_WAVES));
        k_walk64<TPL, FIELDS, QUAD><<<(unsigned)nb, 64 * WALK_WAVES, 0, s>>>(a, b, round);
        PTG_LAUNCH_CHECK();
    }
    for (int level = rounds - 2; level >= 0; level--) {
        k_walk64_sum<FIELDS><<<256, 256, 0, s>>>(a, b, level);
        PTG_LAUNCH_CHECK();
    }
    return PTG_OK;
}

template <int TPL>
static ptg_status launch_fields(const Walk64Args &a, int fields, bool quad, int cus, int gcap, char *ws, size_t ws_bytes,
                                hipStream_t s)
{
#define PTG_F(F)                                                             \
    case F:                                                                  \
        return quad ? launch<TPL, F, true>(a, cus, gcap, ws, ws_bytes, s)    \
                    : launch<TPL, F, false>(a, cus, gcap, ws, ws_bytes, s);
    switch (fields) {
        PTG_F(1) PTG_F(2) PTG_F(3) PTG_F(4) PTG_F(5) PTG_F(6) PTG_F(7)
    }
#undef PTG_F
    ptg_set_error("ptg_walk: fields must be a nonzero combination of PTG_POT|PTG_ACC|PTG_TIDAL");
    return PTG_ERR_ARG;
}

ptg_status ptg_walk64_launch(const Walk64Args &a, int fields, bool quad, int cus, int gcap, char *ws, size_t ws_bytes,
                             hipStream_t s)
{
    if (a.gs <= 64) return launch_fields<1>(a, fields, quad, cus, gcap, ws, ws_bytes, s);
    if (a.gs <= 128) return launch_fields<2>(a, fields, quad, cus, gcap, ws, ws_bytes, s);
    return launch_fields<4>(a, fields, quad, cus, gcap, ws, ws_bytes, s);
}
