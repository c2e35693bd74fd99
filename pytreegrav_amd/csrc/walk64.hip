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
// The reference's groups are runs of the Morton order; those that cross a high-level cell boundary in a
// sparse region open nearly every node (1.48e6 of the 2.9e8 visits of a 1e6-particle Plummer sphere are
// one group's) and are deferred (walk_shared.hpp).
//
// Bound: instruction issue, about 60 % of it the traversal (250 instructions per 64-element step).
// Whole calls, against one wave per group evaluating every entry for 8 of its 64 lanes with IEEE
// square roots and divisions: 1e6-particle Plummer sphere 333 -> 4.3 ms, uniform cube of 1e5 6.0 -> 0.73
// ms, tidal tensors with quadrupoles of 6e4 23.3 -> 1.24 ms.  Angle-binned columns of 2e5 particles
// against their own walk (two waves per SIMD, six selected adds and a division a pair): 4.9 -> 2.05 ms.

#include "walk_shared.hpp"

#define LIST 32           // a list is evaluated in multiples of LIST entries once it holds LIST
#define ICAP (LIST + 64)  // LIST - 1 entries + one step's 64
#define BUDGET 3072  // visits after which a traversal is cut, at least
#define MAX_BLOCKS_PER_CU 4

// FIELDS of the angle-binned column density (treewalk.py:976-1028, :1197-1276): six sums per target, kept
// in LDS, since which of them a pair adds to differs from lane to lane (one LDS add instead of six
// selected ones)
#define SKY_BIN (4.0 * 3.14159265358979323846 / 6.0)  // solid angle of a bin

template <int FIELDS, bool QUAD> struct Lds64 {
    int stack[SCAP];
    V4<double> nodes[ICAP];  // elements no target can be inside the softening of: x y z m
    double nq[QUAD ? 6 * ICAP : 1];
    V4<double> parts[ICAP];  // particles: x y z m
    double ph[ICAP];
    double bins[FIELDS == BINS ? 6 * 64 : 1];  // [bin][lane]
};

// A group is walked WIDE where a coordinate of it or of its tree is not at most this large, or a target's softening: no
// other squared distance can overflow.  Caps in every pair cost 6 to 18 % of the walk (groups of 64 to 256).
#define ORDINARY 1e153

__device__ __forceinline__ bool is_nan3(double x, double y, double z) { return !(x == x) | !(y == y) | !(z == z); }

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

template <int FIELDS, bool QUAD, bool WIDE>
__device__ __forceinline__ void pair_node(Acc<double> &a, const V4<double> &s, const double *q, double tx, double ty,
                                          double tz)
{
    const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double rinv = ptg_rsqrt64<WIDE>(r2), rinv2 = rinv * rinv;
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
template <int FIELDS, bool WIDE>
__device__ __forceinline__ void spline64(double r, double rinv, double h, double &phi, double &K, double &Q)
{
    const double hinv = ptg_rcp64<WIDE>(h), q = r * hinv;
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

// A particle's pair: the spline where it is softened, nothing where it coincides (SOFT: with that branch).
struct Pair64 {
    double dx, dy, dz, r2, h;
    bool apart, soft;
};
template <bool WIDE>
__device__ __forceinline__ Pair64 part_pair(const V4<double> &s, double hs, double tx, double ty, double tz, double th)
{
    Pair64 p;
    p.dx = s.x - tx;
    p.dy = s.y - ty;
    p.dz = s.z - tz;
    p.r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
    p.h = fmax(hs, th);
    p.apart = p.r2 > 0.0;
    p.soft = p.apart & (!WIDE | (th == th)) & (p.r2 < p.h * p.h);  // a target whose softening is a nan is never softened
    return p;
}
template <int FIELDS, bool SOFT, bool WIDE>
__device__ __forceinline__ void part_add(Acc<double> &a, const Pair64 &p, double m)
{
    const double rinv = p.apart ? ptg_rsqrt64<WIDE>(p.r2) : 0.0, rinv2 = rinv * rinv;
    const double mr = m * rinv;
    double phi = -mr, K = mr * rinv2, Q = 3.0 * K * rinv2;
    if (SOFT && p.soft) {
        spline64<FIELDS, WIDE>(p.r2 * rinv, rinv, p.h, phi, K, Q);
        phi *= m;
        K *= m;
        Q *= m;
    }
    add_pair<FIELDS>(a, phi, K, Q, p.dx, p.dy, p.dz);
}

// U entries of a lane's slice of a list together: their LDS reads are issued at once and their chains
// overlap, and the spline is evaluated only where a pair of the batch is softened.  The terms are added in
// the order of the list.
template <int U, int TPL, int FIELDS, bool QUAD, bool WIDE, typename L>
__device__ __forceinline__ void add_nodes(const L &l, int at, int step, Acc<double> (&acc)[TPL], const double (&tx)[TPL],
                                          const double (&ty)[TPL], const double (&tz)[TPL])
{
    V4<double> s[U];
#pragma unroll
    for (int u = 0; u < U; u++) s[u] = l.nodes[at + u * step];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < TPL; j++)
            pair_node<FIELDS, QUAD, WIDE>(acc[j], s[u], &l.nq[QUAD ? 6 * (at + u * step) : 0], tx[j], ty[j], tz[j]);
}
template <int U, int TPL, int FIELDS, bool WIDE, typename L>
__device__ __forceinline__ void add_parts(const L &l, int at, int step, Acc<double> (&acc)[TPL], const double (&tx)[TPL],
                                          const double (&ty)[TPL], const double (&tz)[TPL], const double (&th)[TPL])
{
    V4<double> s[U];
    double hs[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        s[u] = l.parts[at + u * step];
        hs[u] = l.ph[at + u * step];
    }
#pragma unroll
    for (int j = 0; j < TPL; j++) {
        Pair64 p[U];
        bool soft = false;
#pragma unroll
        for (int u = 0; u < U; u++) {
            p[u] = part_pair<WIDE>(s[u], hs[u], tx[j], ty[j], tz[j], th[j]);
            soft |= p[u].soft;
        }
        if (ptg_ballot(soft)) {
            // the barrier keeps this a branch: as selects, every pair went through the spline's 27 instructions
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < U; u++) part_add<FIELDS, true, WIDE>(acc[j], p[u], s[u].w);
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) part_add<FIELDS, false, WIDE>(acc[j], p[u], s[u].w);
        }
    }
}
// entries [0, c) of the lists, this lane's slice of them
template <int U, int TPL, int FIELDS, bool QUAD, bool WIDE, typename L>
__device__ __forceinline__ void sum_nodes(const L &l, int sl, int slices, int c, Acc<double> (&acc)[TPL],
                                          const double (&tx)[TPL], const double (&ty)[TPL], const double (&tz)[TPL])
{
    int q = sl;
#pragma unroll 1
    for (; q + (U - 1) * slices < c; q += U * slices) add_nodes<U, TPL, FIELDS, QUAD, WIDE>(l, q, slices, acc, tx, ty, tz);
#pragma unroll 1
    for (; U > 1 && q < c; q += slices) add_nodes<1, TPL, FIELDS, QUAD, WIDE>(l, q, slices, acc, tx, ty, tz);
}
template <int U, int TPL, int FIELDS, bool WIDE, typename L>
__device__ __forceinline__ void sum_parts(const L &l, int sl, int slices, int c, Acc<double> (&acc)[TPL],
                                          const double (&tx)[TPL], const double (&ty)[TPL], const double (&tz)[TPL],
                                          const double (&th)[TPL])
{
    int q = sl;
#pragma unroll 1
    for (; q + (U - 1) * slices < c; q += U * slices) add_parts<U, TPL, FIELDS, WIDE>(l, q, slices, acc, tx, ty, tz, th);
#pragma unroll 1
    for (; U > 1 && q < c; q += slices) add_parts<1, TPL, FIELDS, WIDE>(l, q, slices, acc, tx, ty, tz, th);
}

// angle-binned columns of one lane: LDS sums bins[64 * bin] (units of mass / distance^2) and the part
// that goes to every bin alike
struct Sky {
    double *bins;
    double iso;

    __device__ __forceinline__ void add(double dx, double dy, double dz, double v)
    {
        // angular_bin_scalar (treewalk.py:38-45)
        const double ax = fabs(dx), ay = fabs(dy), az = fabs(dz);
        const bool x = ax > ay && ax > az, y = ay > az;
        const double d = x ? dx : y ? dy : dz;
        const int bin = (x ? 0 : y ? 2 : 4) + (d > 0 ? 0 : 1);
        __hip_atomic_fetch_add(bins + 64 * bin, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    // an element farther than its radius: a point mass
    template <bool WIDE> __device__ __forceinline__ void node(const V4<double> &s, double tx, double ty, double tz)
    {
        const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
        add(dx, dy, dz, s.w * ptg_rcp64<WIDE>(dx * dx + dy * dy + dz * dz));
    }
    // a particle: a point mass outside its radius h, a blend of the isotropic and directed limits inside
    template <bool WIDE> __device__ __forceinline__ void part(const V4<double> &s, double h, double tx, double ty, double tz)
    {
        const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
        const double r2 = dx * dx + dy * dy + dz * dz, hh = h * h;
        const bool out = r2 > hh;
        double v = s.w * ptg_rcp64<WIDE>(out ? r2 : 1.0);
        if (ptg_ballot(!out)) {
            if (!out) {
                v = 0.0;
                if (h > 0) {
                    const double hinv = ptg_rcp64<WIDE>(h), col0 = s.w * (3.0 / (4.0 * 3.14159265358979323846) * SKY_BIN) * hinv * hinv;
                    const double fac = r2 == 0 ? 0.0 : r2 * ptg_rsqrt64<WIDE>(r2) * hinv;
                    iso += (1.0 - fac) * col0;
                    v = 2.0 * col0 * fac;
                }
            }
        }
        add(dx, dy, dz, v);
    }
};

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
// waves per SIMD the registers are capped for: as many as the sums leave room for and the LDS lets onto a CU
template <int TPL, int FIELDS, bool QUAD> struct Occ64 {
    static constexpr int sums = TPL * Sums<FIELDS>::WI;
    static constexpr int waves = FIELDS == BINS ? 3 : !QUAD && TPL == 1 ? (sums <= 4 ? 4 : sums <= 9 ? 3 : 1)
                                                 : sums >= 12 && sums <= 24 ? 2 : 1;
};

template <int TPL, int FIELDS, bool QUAD, bool TASKS>
__global__ __launch_bounds__(64 * WALK_WAVES) __attribute__((amdgpu_waves_per_eu(Occ64<TPL, FIELDS, QUAD>::waves)))
void k_walk64(const Walk64Args A, const WalkHot H, const WalkPool pool)
{
    constexpr int WI = Sums<FIELDS>::WI;
    // entries evaluated together (nodes, particles).  Quadrupoles, three waves per SIMD, have the registers for 4
    // and 2: acceleration of 2e5 particles 2.31 -> 2.11 ms, of 1e5 in groups of 256 2.29 -> 2.06 (2 and 2: 2.19,
    // 2.40).  Monopole sums at four waves have not: 4 and 2 spill 10 registers, 2 and 2 took the time of 1 and 1,
    // which gain from the spline's branch alone (1e6 particles 4.45 -> 4.34 ms).
    constexpr int UN = QUAD ? 4 : 1, UP = QUAD || NW<FIELDS>::TID ? 2 : 1;
    __shared__ Lds64<FIELDS, QUAD> lds[WALK_WAVES];
    const int wave = threadIdx.x >> 6, lane = ptg_lane();
    Lds64<FIELDS, QUAD> &L = lds[wave];
    int *spill = H.spill + ((int64_t)blockIdx.x * WALK_WAVES + wave) * (int64_t)H.gcap;
    const int xcd = blockIdx.x % NXCD;
    int64_t total[3] = {0, 0, 0};  // interactions, visits, particle interactions of the groups this wave finished
    int ghw = 0;
    const int64_t ngroups = A.goff ? (int64_t)__builtin_amdgcn_readfirstlane(*A.gcount) : A.ngroups;
    int ticket = -1, closed = 0;
    if (!TASKS && blockIdx.x == 0 && threadIdx.x == 0) A.ctl->words = (int32_t)walk_words(ngroups);
    if (TASKS && agent_load(&A.ctl->open) == 0) return;  // nothing was deferred, or all of it is done
    // targets per slice, a power of two
    int P = 64;
    if (TPL == 1)
        while (P > 1 && P / 2 >= A.gs) P /= 2;
    const int tl = lane & (P - 1), sl = lane / P, slices = 64 / P;

    // groups from per-XCD counters, as the FP32 walk takes them; or tasks by ticket
    for (int attempt = 0; attempt < (TASKS ? 1 : NXCD); attempt++) {
        const int x = (xcd + attempt) % NXCD;
        const int64_t w_lo = ngroups * x / NXCD, w_hi = ngroups * (x + 1) / NXCD;
        for (;;) {
            int self = -1, parent = -1;
            int64_t g;
            TaskWords rec;  // the parent's
            if (TASKS) {
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                self = walk_ticket(A.ctl, B, lane, ticket, closed, parent);
                if (self < 0) break;
                rec = TaskWords(&B.tasks[parent], lane);
                g = rec.get<&WalkTask::group>();
            } else {
                int wi = 0;
                if (lane == 0) wi = atomicAdd(&A.ctl->ctr[x * CTR_STRIDE], 1);
                g = w_lo + __builtin_amdgcn_readfirstlane(wi);
                if (g >= w_hi) break;
            }
            const WalkSpan grp = walk_span(A.goff, A.gs, A.nt, g);
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
                tidx[j] = !tval[j] ? 0 : A.perm ? A.perm[a0 + o] : a0 + o;
                if (tval[j]) {
                    const int64_t src = A.sorted ? a0 + o : tidx[j];
                    tx[j] = A.pos[3 * src] - ox;
                    ty[j] = A.pos[3 * src + 1] - oy;
                    tz[j] = A.pos[3 * src + 2] - oz;
                    th[j] = A.soft ? A.soft[src] : -INFINITY;
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
            // a target with a nan coordinate bounds nothing; of binned columns it gets what the particles' own radii
            // give it, so none of its group's particles is taken for a far one
            const bool near_all = FIELDS == BINS && ptg_ballot(is_nan3(tx[0], ty[0], tz[0])) != 0;
            const V4<double> top = A.xyzm[root];
            const double far = fmax(fmax(fabs(top.x), fabs(top.y)), fabs(top.z)) + A.aux[root].y;
            bool odd = !(far <= ORDINARY);
#pragma unroll
            for (int j = 0; j < TPL; j++)
                odd |= !(fabs(tx[j]) <= ORDINARY) | !(fabs(ty[j]) <= ORDINARY) | !(fabs(tz[j]) <= ORDINARY) | !(th[j] <= ORDINARY);
            const bool wide = ptg_ballot(odd) != 0;
            Acc<double> acc[TPL];
#pragma unroll
            for (int j = 0; j < TPL; j++) acc[j] = Acc<double>{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            Sky sky{&L.bins[FIELDS == BINS ? lane : 0], 0.0};
            if (FIELDS == BINS)
                for (int q = 0; q < 6; q++) L.bins[64 * q + lane] = 0.0;

            // entries [0, c) of a list, this lane's slice of them
            auto nodes_now = [&](int c) {
                if constexpr (FIELDS == BINS) {
                    if (wide) {
#pragma unroll 1
                        for (int q = sl; q < c; q += slices) sky.template node<true>(L.nodes[q], tx[0], ty[0], tz[0]);
                    } else {
                        for (int q = sl; q < c; q += slices) sky.template node<false>(L.nodes[q], tx[0], ty[0], tz[0]);
                    }
                } else if (wide) {
                    sum_nodes<1, TPL, FIELDS, QUAD, true>(L, sl, slices, c, acc, tx, ty, tz);
                } else {
                    sum_nodes<UN, TPL, FIELDS, QUAD, false>(L, sl, slices, c, acc, tx, ty, tz);
                }
            };
            auto parts_now = [&](int c) {
                if constexpr (FIELDS == BINS) {
                    if (wide) {
#pragma unroll 1
                        for (int q = sl; q < c; q += slices)
                            sky.template part<true>(L.parts[q], L.ph[q], tx[0], ty[0], tz[0]);
                    } else {
                        for (int q = sl; q < c; q += slices)
                            sky.template part<false>(L.parts[q], L.ph[q], tx[0], ty[0], tz[0]);
                    }
                } else if (wide) {
                    sum_parts<1, TPL, FIELDS, true>(L, sl, slices, c, acc, tx, ty, tz, th);
                } else {
                    sum_parts<UP, TPL, FIELDS, false>(L, sl, slices, c, acc, tx, ty, tz, th);
                }
            };

            int sp = 1, gsp = 0, nn = 0, np = 0, visits = 0, n_list = 0, n_part = 0;
            bool overflow = false;
            const bool share = TASKS && rec.get<&WalkTask::off>() >= 0;  // else a group from its root
            if (share) {
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                const int stride = rec.get<&WalkTask::nchild>(), q0 = self - B.gcount - rec.get<&WalkTask::child0>();
                const int share_no = q0 < 0 ? q0 + B.tcount : q0;
                const int *entries = B.entries + rec.get<&WalkTask::off>() + share_no;
                sp = share_count(rec.get<&WalkTask::count>(), stride, share_no);  // <= SCAP: deeper stacks are not cut
                for (int q = lane; q < sp; q += 64) L.stack[q] = agent_load(&entries[(int64_t)q * stride]);
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
            // being cut: budgets of 3072 against 8192 take 0.79 / 0.95 ms (walk and build, uniform 1e5), 4
            // against 3 times 3072 6.8 / 8.3 ms (clumpy 6e5).  Counted per system, so that a system's cuts
            // are those it has alone.
            const int64_t sg = (A.nsys > 0 ? A.soff[root + 1] - A.soff[root] : A.nt) / A.gs;
            int budget = H.budget * (share || sg <= 16384 ? 1 : sg <= 65536 ? 2 : sg <= 262144 ? 4 : 16);
            if (TASKS) budget = walk_budget(budget, rec.get<&WalkTask::level>());
            if (H.tcount == 0) budget = 0x7fffffff;
            bool cut = false;
            int nchild = 0, off = 0, child0 = 0, troot = -1;

            for (;;) {  // once more only for a traversal that is not cut
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
                        cut = true;
                        break;
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
                    const bool far_part = !QUAD & ve & ispart & (r2m > hh * hh) & !near_all;
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
                        n_list += (int)(__popcll(bp) + __popcll(bn));
                        n_part += (int)(__popcll(bp) + __popcll(ptg_ballot(far_part)));
                    }

                    const int cnt = open ? std::min(std::max(K.y, 0), 8) : 0;
                    int tot;
                    const int below = small_excl_scan(cnt, tot);
                    if (sp + tot > SCAP) {
                        const int ks = spill_count(sp, tot);
                        if (gsp + ks > H.gcap) {
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
                        nodes_now(c);
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
                        parts_now(c);
                        __builtin_amdgcn_wave_barrier();
                        if (lane < np - c) {  // disjoint ranges, as above
                            L.parts[lane] = L.parts[c + lane];
                            L.ph[lane] = L.ph[c + lane];
                        }
                        __builtin_amdgcn_wave_barrier();
                        np -= c;
                    }
                }
                if (!cut) break;
                nchild = walk_cut<TASKS>(A.ctl, H, pool, share, L.stack, sp, spill, gsp, lane, self, off, child0);
                cut = nchild > 0;
                if (nchild) break;
                budget = 0x7fffffff;
            }
            if (TASKS) troot = parent < walk_pool<TASKS>(A.ctl, H, pool).gcount ? parent : rec.get<&WalkTask::root>();
            if (nchild < 0) {  // no room: the group is walked again
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                if (!TASKS) {
                    if (lane == 0) walk_put_back<AgentMem>(A.ctl, B, false, (int)g);
                    continue;
                }
                if (lane == 0) agent_store(&B.tasks[troot].root, 1);
                nn = np = 0;  // its row and counts are not used any more
            }
            if (A.counters) {
                const int64_t n[3] = {(int64_t)n_list * mt, visits, (int64_t)n_part * mt};
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    if (!TASKS && !cut) total[q] += n[q];
                    else if (lane != 0) continue;
                    else if (TASKS) atomicAdd((unsigned long long *)&walk_pool<TASKS>(A.ctl, H, pool).counts[4 * troot + q], (unsigned long long)n[q]);
                    else agent_store(&walk_pool<TASKS>(A.ctl, H, pool).counts[4 * self + q], n[q]);
                }
            }
            if (overflow) {
                if (lane == 0) atomicOr(&A.ctl->err, 1);
                nn = np = 0;  // a task's row is still written: the sums read every task's
            }
            nodes_now(nn);
            parts_now(np);
            __builtin_amdgcn_wave_barrier();
            [[maybe_unused]] double bin[FIELDS == BINS ? 6 : 1];
            if constexpr (FIELDS == BINS) {
#pragma unroll
                for (int q = 0; q < 6; q++) bin[q] = L.bins[64 * q + lane] + sky.iso;
                for (int d = P; d < 64; d <<= 1) {
#pragma unroll
                    for (int q = 0; q < 6; q++) bin[q] += __shfl_xor(bin[q], d, 64);
                }
            }
            if (FIELDS != BINS && wide) {  // a target with a nan coordinate meets nothing
#pragma unroll
                for (int j = 0; j < TPL; j++)
                    if (is_nan3(tx[j], ty[j], tz[j])) acc[j] = Acc<double>{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            }
            for (int d = P; FIELDS != BINS && d < 64; d <<= 1) {
#pragma unroll
                for (int j = 0; j < TPL; j++) each_sum<FIELDS>(acc[j], [&](double &v) { v += __shfl_xor(v, d, 64); });
            }

            // ---- G * fields in the caller's order, or the task's row of partial sums ----
            const bool whole = !TASKS && !cut;
#pragma unroll
            for (int j = 0; j < TPL; j++) {
                if (!tval[j] || sl != 0) continue;
                int c = 0;
                if (whole) {
                    double *o = A.out + tidx[j] * Sums<FIELDS>::WO;
                    each_sum<FIELDS>(acc[j], [&](double &v) { store_sum<FIELDS>(o, c++, A.G * v); });
                    if constexpr (FIELDS == BINS) {
#pragma unroll
                        for (int q = 0; q < 6; q++) o[q] = A.G * bin[q];
                    }
                } else {
                    double *o = (double *)walk_pool<TASKS>(A.ctl, H, pool).partial + ((int64_t)self * A.gs + tl + 64 * j) * WI;
                    each_sum<FIELDS>(acc[j], [&](double &v) { agent_store(&o[c++], v); });
                    if constexpr (FIELDS == BINS) {
#pragma unroll
                        for (int q = 0; q < 6; q++) agent_store(&o[q], bin[q]);
                    }
                }
            }
            if (cut) {
                const WalkPool P = walk_pool<TASKS>(A.ctl, H, pool);
                walk_publish<AgentMem>(A.ctl, P, WalkTask{(int)g, parent, TASKS ? troot : 0, TASKS ? rec.get<&WalkTask::level>() : 0, off,
                                                     gsp + sp, child0 % P.tcount, nchild, nchild, {}}, child0, self, lane);
            } else if (TASKS) {
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                const int p = walk_add_up<FIELDS, double>(A.ctl, B, parent, grp, A.gs, A.perm, A.G, A.out, lane);
                if (p >= 0 && A.counters)
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        const int64_t n = agent_load(&walk_pool<TASKS>(A.ctl, H, pool).counts[4 * p + q]);
                        total[q] += (int64_t)__builtin_amdgcn_readfirstlane((int)(n >> 32)) << 32 |
                                    (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
                    }
            }
            if (TASKS) closed++;
        }
    }
    if (lane == 0 && ghw > 0) atomicMax(&A.ctl->hwm, ghw);
    if (lane == 0 && A.counters) {
        for (int q = 0; q < (FIELDS == BINS ? 2 : 3); q++)
            atomicAdd((unsigned long long *)&A.counters[q], (unsigned long long)total[q]);
    }
}

// ============================================================================================
// host side
// ============================================================================================
template <int TPL, int FIELDS, bool QUAD>
static ptg_status launch(const Walk64Args &a, int cus, int gcap, size_t again, char *ws, size_t ws_bytes, hipStream_t s)
{
    static int per_cu = 0;
    if (per_cu == 0) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_walk64<TPL, FIELDS, QUAD, false>, 64 * WALK_WAVES, 0) !=
                hipSuccess ||
            nb < 1)
            nb = 1;
        per_cu = std::min(nb, MAX_BLOCKS_PER_CU);
    }
    // an ordinary group's traversal stays well inside the budget: it grows as 1 / theta^2 and with the
    // group; large groups (large rows of sums) are cut into fewer shares
    const size_t row = (size_t)a.gs * Sums<FIELDS>::WI * sizeof(double);
    const double open = a.theta < 0.7 ? 0.49 / (a.theta * a.theta) : 1.0;
    const int share = (int)std::max<size_t>(16, 262144 / row);
    WalkHot b{};
    b.budget = (int)std::min(1e8, BUDGET * open * (a.gs <= 16 ? 1 : a.gs <= 64 ? 2 : 4));
    b.most0 = std::min(64, share);
    b.most = std::min(128, share);
    const int64_t blocks = (int64_t)cus * per_cu;
    const ptg_status st = walk_carve(b, ws, ws_bytes, a.goff ? a.nt : a.ngroups, again, blocks * WALK_WAVES, gcap, row);
    if (st) return st;
    const int64_t nb = a.goff ? blocks : std::min(blocks, ptg_cdiv(a.ngroups, WALK_WAVES));
    k_walk64<TPL, FIELDS, QUAD, false><<<(unsigned)nb, 64 * WALK_WAVES, 0, s>>>(a, b, walk_pool(a.ctl, b));
    PTG_LAUNCH_CHECK();
    if (b.tcount && a.nslots > b.budget) {  // a traversal visits a slot once
        k_walk64<TPL, FIELDS, QUAD, true><<<(unsigned)blocks, 64 * WALK_WAVES, 0, s>>>(a, b, walk_pool(a.ctl, b));
        PTG_LAUNCH_CHECK();
    }
    return PTG_OK;
}

template <int TPL>
static ptg_status launch_fields(const Walk64Args &a, int fields, bool quad, int cus, int gcap, size_t again, char *ws, size_t ws_bytes,
                                hipStream_t s)
{
#define PTG_F(F)                                                             \
    case F:                                                                  \
        return quad ? launch<TPL, F, true>(a, cus, gcap, again, ws, ws_bytes, s)    \
                    : launch<TPL, F, false>(a, cus, gcap, again, ws, ws_bytes, s);
    switch (fields) {
        PTG_F(1) PTG_F(2) PTG_F(3) PTG_F(4) PTG_F(5) PTG_F(6) PTG_F(7)
    }
#undef PTG_F
    ptg_set_error("ptg_walk: fields must be a nonzero combination of PTG_POT|PTG_ACC|PTG_TIDAL");
    return PTG_ERR_ARG;
}

ptg_status ptg_walk64_launch(const Walk64Args &a, int fields, bool quad, int cus, int gcap, size_t again, char *ws, size_t ws_bytes,
                             hipStream_t s)
{
    if (a.gs <= 64) return launch_fields<1>(a, fields, quad, cus, gcap, again, ws, ws_bytes, s);
    if (a.gs <= 128) return launch_fields<2>(a, fields, quad, cus, gcap, again, ws, ws_bytes, s);
    return launch_fields<4>(a, fields, quad, cus, gcap, again, ws, ws_bytes, s);
}

ptg_status ptg_walk64_bins(const Walk64Args &a, int cus, int gcap, size_t again, char *ws, size_t ws_bytes, hipStream_t s)
{
    return launch<1, BINS, false>(a, cus, gcap, again, ws, ws_bytes, s);
}
