// Grouped Barnes-Hut walk for gfx950: one wavefront walks the tree for one group of Morton-
// consecutive targets (grouped_treewalk.py:163-241).  Traversal is breadth-ordered over a stack in
// LDS: each step pops up to 64 elements (one per lane), evaluates the opening test against the
// group's bounding box in parallel, appends accepted elements to LDS interaction lists with
// ballot/popcount compaction and pushes the children of opened nodes with a wave prefix sum.
// When a list holds 64 entries the wave evaluates them against its targets, every lane reading the
// same LDS entry (broadcast).  Persistent waves take groups from per-XCD counters.
//
// Group expansion (FP32 monopole walks, no reference counterpart): an accepted element far enough
// from the group's centre that a third-order Taylor expansion of its field about that centre is
// within the tolerance is not listed; the lane that accepted it adds its derivative tensors to the
// lane's local-expansion coefficients, the wave sums them once per group and every target
// evaluates the expansion at its offset from the centre.

#include <algorithm>
#include <mutex>

#include "walk_shared.hpp"

#define BUDGET 4096  // visits after which a traversal is cut (walk_shared.hpp), at least

// groups a system has at least where its traversals are cut
__host__ __device__ constexpr int cut_groups(int fields) { return fields & PTG_TIDAL ? 2048 : 1024; }

// a list is evaluated in multiples of LF entries once it holds LF (a power of 2: 64, or 32 for the
// six-wave variant); a list holds LF - 1 + one step's 64 entries (ICAP)

template <typename T, bool QUAD, int LF> struct WaveLds {
    static constexpr int ICAP = LF + 64;
    int stack[SCAP];
    V4<T> nodes[ICAP];  // accepted nodes: x y z m
    T nq[QUAD ? 6 * ICAP : 1];
    V4<T> parts[ICAP];  // particles: x y z m
    T ph[ICAP];
};

template <typename T> struct WalkArgs {
    const V4<T> *xyzm;
    const V4<T> *aux;
    const int2 *kids;
    const T *quad;  // 8 per slot
    const double *pos;
    const double *soft;
    const int64_t *perm;
    int sorted;  // pos/soft are indexed by the sorted target position (perm maps the outputs only)
    int64_t nslots;
    int64_t nt;
    int64_t ngroups;
    const int32_t *goff;    // optional group offsets (ngroups + 1), else fixed groups of gs
    const int32_t *gcount;  // device group count when goff is given
    int gs;
    T theta;
    T inv_theta;  // FP32 path: 1 / theta
    int crit;  // 0: geometric (treewalk.py:22-25); 1: quadrupole error bound; 2: learned
    T eps;     // criterion 1/2: per-node acceleration error tolerance (already divided by 3.5)
    T eps_exp;                 // group expansion: per-element tolerance of the expansion test
    T exp_rel;                 // group expansion: cap of the truncation bound relative to M / D^2 (0: none)
    const double *eps_scale;   // nullable: eps_exp * eps_scale[system] (one scale per system)
    double G;
    double ox, oy, oz;
    // forest: group g walks the tree of the system s holding its first target (root at slot s),
    // with coordinates relative to that system's cube centre (FP32) or absolute (FP64)
    int64_t nsys;          // 0: one tree
    const int64_t *soff;   // (nsys + 1) system target ranges
    const double *cubes;   // (nsys, 4)
    double *out;
    int64_t *counters;
    WalkCtl *ctl;
};

__device__ __forceinline__ float fast_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }

// Accepted node on one target, fast path: the acceptance test guarantees r > h_t, h_s and r > 0.
template <typename T, int FIELDS, bool QUAD>
__device__ __forceinline__ void interact_node_fast(Acc<T> &a, V4<T> s, const T *q, T tx, T ty, T tz)
{
    constexpr bool P = NW<FIELDS>::POT, G = NW<FIELDS>::ACC, D = NW<FIELDS>::TID;
    T dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    T r2 = dx * dx + dy * dy + dz * dz;
    T rinv = fast_rsqrt(r2);
    T rinv2 = rinv * rinv;
    T mr = s.w * rinv;
    if (P) a.phi -= mr;
    T K = mr * rinv2;
    if (G) {
        a.gx += K * dx;
        a.gy += K * dy;
        a.gz += K * dz;
    }
    if (D) {
        T Q = T(3) * K * rinv2;
        a.txx += Q * dx * dx - K;
        a.tyy += Q * dy * dy - K;
        a.tzz += Q * dz * dz - K;
        a.txy += Q * dx * dy;
        a.txz += Q * dx * dz;
        a.tyz += Q * dy * dz;
    }
    if (QUAD) {
        T qxx = q[0], qxy = q[1], qxz = q[2], qyy = q[3], qyz = q[4], qzz = q[5];
        T r5inv = rinv2 * rinv2 * rinv;
        T r7inv = r5inv * rinv2;
        T qdx = qxx * dx + qxy * dy + qxz * dz;
        T qdy = qxy * dx + qyy * dy + qyz * dz;
        T qdz = qxz * dx + qyz * dy + qzz * dz;
        T A = dx * qdx + dy * qdy + dz * qdz;
        if (P) a.phi += T(-0.5) * A * r5inv;
        if (G) {
            T f = T(2.5) * A * r7inv;
            a.gx += f * dx - qdx * r5inv;
            a.gy += f * dy - qdy * r5inv;
            a.gz += f * dz - qdz * r5inv;
        }
        if (D) {
            T diag = T(-2.5) * A * r7inv;
            T fac = T(17.5) * A * r7inv * rinv2;
            a.txx += qxx * r5inv - T(10.0) * dx * qdx * r7inv + diag + fac * dx * dx;
            a.tyy += qyy * r5inv - T(10.0) * dy * qdy * r7inv + diag + fac * dy * dy;
            a.tzz += qzz * r5inv - T(10.0) * dz * qdz * r7inv + diag + fac * dz * dz;
            a.txy += qxy * r5inv - T(5.0) * (dx * qdy + dy * qdx) * r7inv + fac * dx * dy;
            a.txz += qxz * r5inv - T(5.0) * (dx * qdz + dz * qdx) * r7inv + fac * dx * dz;
            a.tyz += qyz * r5inv - T(5.0) * (dy * qdz + dz * qdy) * r7inv + fac * dy * dz;
        }
    }
}

// The M4 spline terms for r < h (kernel.py:4-75) with reciprocals instead of IEEE divisions, for
// the FP32 fast path: hinv = 1/h, qinv = h/r = h * rinv.
template <typename T> struct SplineFast {
    T K, phi, Q;
};
template <typename T, bool P, bool D>
__device__ __forceinline__ SplineFast<T> spline_fast(T r, T rinv, T h)
{
    T hinv = __builtin_amdgcn_rcpf(h);
    T q = r * hinv;
    T hinv2 = hinv * hinv;
    T hinv3 = hinv2 * hinv;
    SplineFast<T> o;
    o.phi = 0;
    o.Q = 0;
    if (q <= T(0.5)) {
        T q2 = q * q;
        o.K = (T(10.666666666666666666) + q2 * (T(-38.4) + T(32.0) * q)) * hinv3;
        if (P) o.phi = (T(-2.8) + q2 * (T(5.33333333333333333) + q2 * (T(6.4) * q - T(9.6)))) * hinv;
        if (D) o.Q = (T(76.8) - T(96.0) * q) * hinv3 * hinv2;
    } else {
        T qinv = h * rinv;
        T qinv3 = qinv * qinv * qinv;
        o.K = (T(21.333333333333) - T(48.0) * q + T(38.4) * q * q - T(10.666666666667) * q * q * q -
               T(0.066666666667) * qinv3) * hinv3;
        if (P)
            o.phi = (T(-3.2) + T(0.066666666666666666666) * qinv +
                     q * q * (T(10.666666666666666666666) + q * (T(-16.0) + q * (T(9.6) - T(2.1333333333333333333333) * q)))) *
                    hinv;
        if (D) o.Q = (T(48.0) * qinv - T(76.8) + T(32.0) * q - T(0.2) * qinv3 * qinv * qinv) * hinv3 * hinv2;
    }
    return o;
}

// Particle on one target, fast path: point mass unless any lane is inside the softening radius, in which
// case those lanes evaluate the spline; r2 == 0 contributes zero.  part_pair says whether this lane's pair is
// softened, part_add adds it (SOFT: with the spline branch).
template <typename T> struct PartPair {
    T dx, dy, dz, r2, ht;
    bool nonzero, soft;
};
template <typename T>
__device__ __forceinline__ PartPair<T> part_pair(const V4<T> &s, T hs, T tx, T ty, T tz, T th)
{
    PartPair<T> p;
    p.dx = s.x - tx;
    p.dy = s.y - ty;
    p.dz = s.z - tz;
    p.r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
    p.ht = fmaxf(hs, th);
    p.nonzero = p.r2 > T(0);
    p.soft = p.nonzero && p.r2 < p.ht * p.ht;
    return p;
}
template <typename T, int FIELDS, bool SOFT>
__device__ __forceinline__ void part_add(Acc<T> &a, const PartPair<T> &p, T m)
{
    constexpr bool P = NW<FIELDS>::POT, G = NW<FIELDS>::ACC, D = NW<FIELDS>::TID;
    const T dx = p.dx, dy = p.dy, dz = p.dz;
    T rinv = p.nonzero ? fast_rsqrt(p.r2) : T(0);
    T rinv2 = rinv * rinv;
    T mr = m * rinv;
    T phi = -mr;
    T K = mr * rinv2;
    T Q = T(3) * K * rinv2;
    if (SOFT && p.soft) {
        SplineFast<T> sp = spline_fast<T, P, D>(p.r2 * rinv, rinv, p.ht);
        if (P) phi = m * sp.phi;
        K = m * sp.K;
        if (D) Q = m * sp.Q;
    }
    if (P) {
#pragma clang fp contract(off)  // rounded as in the soft branch, whichever other lanes and entries share the batch
        a.phi += phi;
    }
    if (G) {
        a.gx += K * dx;
        a.gy += K * dy;
        a.gz += K * dz;
    }
    if (D) {
        a.txx += fma(Q * dx, dx, -K);
        a.tyy += fma(Q * dy, dy, -K);
        a.tzz += fma(Q * dz, dz, -K);
        a.txy += Q * dx * dy;
        a.txz += Q * dx * dz;
        a.tyz += Q * dy * dz;
    }
}

// ---- group expansion ----
// A point mass M at D = y - c from the group centre c acts on a target at c + u through
// f(D - u) = 1/|D - u| = f - u.f1 + (1/2) u f2 u - (1/6) f3 uuu + O(|u|^4 / |D|^5) with the
// derivative tensors of 1/r at D: f1 = -D/D^3, f2 = 3 D D / D^5 - I / D^3,
// f3 = -15 D D D / D^7 + 3 (D I + I D + (I D)^T) / D^5.  Summed over the folded elements:
// a0 = sum M f, g = -sum M f1, a2 = sum M f2, a3 = sum M f3; then at u
//   phi = -a0 - u.g - (1/2) u a2 u + (1/6) a3 uuu,    acc = g + a2 u - (1/2) a3 uu.
// a2 and a3 are trace-free (1/r is harmonic), so five and seven components are kept:
// a2zz = -(xx + yy), a3xzz = -(xxx + xyy), a3yzz = -(xxy + yyy), a3zzz = -(xxz + yyz).
// Error bound: the dropped terms of 1/|D - u| are |u|^l P_l(cos g) / D^(l+1), l >= 4, and the
// gradient of the solid harmonic r^l P_l(cos) is at most l r^(l-1) long, so for |u| <= R < D the
// acceleration misses by at most (M / D^2) sum_{l>=4} l x^(l-1) = (M / D^2) x^3 (4 - 3x) / (1 - x)^2
// with x = R / D (the potential by (M / D) x^4 / (1 - x)); an element is folded when that is below
// the tolerance.
template <typename T> struct GroupExp {
    T a0, gx, gy, gz;
    T xx, yy, xy, xz, yz;
    T xxx, xxy, xxz, xyy, xyz, yyy, yyz;
};

template <typename T>
__device__ __forceinline__ void exp_add(GroupExp<T> &E, T M, T Dx, T Dy, T Dz, T rinv)
{
    const T rinv2 = rinv * rinv;
    const T mr = M * rinv;
    const T m3 = mr * rinv2;
    E.a0 += mr;
    E.gx += m3 * Dx;
    E.gy += m3 * Dy;
    E.gz += m3 * Dz;
    const T p = T(3) * m3 * rinv2;
    const T pDx = p * Dx, pDy = p * Dy;
    E.xx += pDx * Dx - m3;
    E.yy += pDy * Dy - m3;
    E.xy += pDx * Dy;
    E.xz += pDx * Dz;
    E.yz += pDy * Dz;
    const T q = T(-5) * p * rinv2;
    const T qxx = q * Dx * Dx, qyy = q * Dy * Dy;
    E.xxx += (qxx + T(3) * p) * Dx;
    E.xxy += (qxx + p) * Dy;
    E.xxz += (qxx + p) * Dz;
    E.xyy += (qyy + p) * Dx;
    E.xyz += q * Dx * Dy * Dz;
    E.yyy += (qyy + T(3) * p) * Dy;
    E.yyz += (qyy + p) * Dz;
}

// the fold test: truncation bound of the expansion about a centre at offset -D, radius rg, below
// the absolute tolerance eps and, when rel > 0, below rel times the element's own field M / D^2
// (bound / (M / D^2) = x^3 (4 - 3x) / (1 - x)^2 depends on x alone, so rel caps x)
template <typename T>
__device__ __forceinline__ bool fold_test(T M, T Dx, T Dy, T Dz, T rg, T eps, T rel, T &rinv)
{
    const T D2 = Dx * Dx + Dy * Dy + Dz * Dz;
    rinv = fast_rsqrt(D2);  // D2 == 0 gives x = inf or nan: no fold
    const T x = rg * rinv, omx = T(1) - x;
    const T lhs = x * x * x * (T(4) - T(3) * x);
    const T rhs = omx * omx;
    return x < T(1) && M * lhs < eps * D2 * rhs && (rel <= T(0) || lhs < rel * rhs);
}

__device__ __forceinline__ float wave_fsum(float v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ void exp_wave_sum(GroupExp<float> &E)
{
    E.a0 = wave_fsum(E.a0);
    E.gx = wave_fsum(E.gx);
    E.gy = wave_fsum(E.gy);
    E.gz = wave_fsum(E.gz);
    E.xx = wave_fsum(E.xx);
    E.yy = wave_fsum(E.yy);
    E.xy = wave_fsum(E.xy);
    E.xz = wave_fsum(E.xz);
    E.yz = wave_fsum(E.yz);
    E.xxx = wave_fsum(E.xxx);
    E.xxy = wave_fsum(E.xxy);
    E.xxz = wave_fsum(E.xxz);
    E.xyy = wave_fsum(E.xyy);
    E.xyz = wave_fsum(E.xyz);
    E.yyy = wave_fsum(E.yyy);
    E.yyz = wave_fsum(E.yyz);
}

template <typename T, int FIELDS>
__device__ __forceinline__ void exp_eval(Acc<T> &a, const GroupExp<T> &E, T ux, T uy, T uz)
{
    const T zz = -(E.xx + E.yy);
    const T xzz = -(E.xxx + E.xyy), yzz = -(E.xxy + E.yyy), zzz = -(E.xxz + E.yyz);
    const T a2x = E.xx * ux + E.xy * uy + E.xz * uz;
    const T a2y = E.xy * ux + E.yy * uy + E.yz * uz;
    const T a2z = E.xz * ux + E.yz * uy + zz * uz;
    const T uxx = ux * ux, uyy = uy * uy, uzz = uz * uz;
    const T uxy = T(2) * ux * uy, uxz = T(2) * ux * uz, uyz = T(2) * uy * uz;
    const T a3x = E.xxx * uxx + E.xyy * uyy + xzz * uzz + E.xxy * uxy + E.xxz * uxz + E.xyz * uyz;
    const T a3y = E.xxy * uxx + E.yyy * uyy + yzz * uzz + E.xyy * uxy + E.xyz * uxz + E.yyz * uyz;
    const T a3z = E.xxz * uxx + E.yyz * uyy + zzz * uzz + E.xyz * uxy + xzz * uxz + yzz * uyz;
    if (NW<FIELDS>::POT)
        a.phi += -E.a0 - (ux * E.gx + uy * E.gy + uz * E.gz) - T(0.5) * (ux * a2x + uy * a2y + uz * a2z) +
                 T(1.0 / 6.0) * (ux * a3x + uy * a3y + uz * a3z);
    if (NW<FIELDS>::ACC) {
        a.gx += E.gx + a2x - T(0.5) * a3x;
        a.gy += E.gy + a2y - T(0.5) * a3y;
        a.gz += E.gz + a2z - T(0.5) * a3z;
    }
}

// U entries of a list are evaluated together: their LDS reads are issued at once and their chains overlap.  One
// at a time, every entry waited for its read and 4 of a node's 19 instructions were the loop's; for particles the
// spline was evaluated whether a lane was softened or not.  The terms are added in the order of the list.
// Whole calls, one entry -> U: 1000 targets on 1e5 particles 2.43 -> 1.54 ms, FP32 acceleration of
// 5e4 particles 0.93 -> 0.84, of 1e6 2.10 -> 1.95, a learned step of 1e7 9.57 -> 9.25.
template <typename T, int TPL, int FIELDS, bool QUAD, int LF, int U>
__device__ __forceinline__ void add_nodes(const WaveLds<T, QUAD, LF> &L, int k, Acc<T> (&acc)[TPL],
                                          const T (&tx)[TPL], const T (&ty)[TPL], const T (&tz)[TPL])
{
    V4<T> s[U];
    T q[U][6];
#pragma unroll
    for (int u = 0; u < U; u++) {
        s[u] = L.nodes[k + u];
        if (QUAD) {
#pragma unroll
            for (int c = 0; c < 6; c++) q[u][c] = L.nq[6 * (k + u) + c];
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < TPL; j++) interact_node_fast<T, FIELDS, QUAD>(acc[j], s[u], q[u], tx[j], ty[j], tz[j]);
}

template <int U, typename T, int TPL, int FIELDS, bool QUAD, int LF>
__device__ __forceinline__ void flush_nodes(const WaveLds<T, QUAD, LF> &L, int cnt, Acc<T> (&acc)[TPL],
                                            const T (&tx)[TPL], const T (&ty)[TPL], const T (&tz)[TPL])
{
    int k = 0;
#pragma unroll 1
    for (; k + U <= cnt; k += U) add_nodes<T, TPL, FIELDS, QUAD, LF, U>(L, k, acc, tx, ty, tz);
#pragma unroll 1
    for (; U > 1 && k < cnt; k++) add_nodes<T, TPL, FIELDS, QUAD, LF, 1>(L, k, acc, tx, ty, tz);
}

template <typename T, int TPL, int FIELDS, bool QUAD, int LF, int U>
__device__ __forceinline__ void add_parts(const WaveLds<T, QUAD, LF> &L, int k, Acc<T> (&acc)[TPL],
                                          const T (&tx)[TPL], const T (&ty)[TPL], const T (&tz)[TPL],
                                          const T (&th)[TPL])
{
    V4<T> s[U];
    T hs[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        s[u] = L.parts[k + u];
        hs[u] = L.ph[k + u];
    }
#pragma unroll
    for (int j = 0; j < TPL; j++) {
        PartPair<T> p[U];
        bool soft = false;
#pragma unroll
        for (int u = 0; u < U; u++) {
            p[u] = part_pair(s[u], hs[u], tx[j], ty[j], tz[j], th[j]);
            soft |= p[u].soft;
        }
        if (U == 1 || ptg_ballot(soft)) {
            // the barrier keeps this a branch: as selects, every pair went through the spline's 40 instructions
            if (U > 1) __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < U; u++) part_add<T, FIELDS, true>(acc[j], p[u], s[u].w);
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) part_add<T, FIELDS, false>(acc[j], p[u], s[u].w);
        }
    }
}

template <int U, typename T, int TPL, int FIELDS, bool QUAD, int LF>
__device__ __forceinline__ void flush_parts(const WaveLds<T, QUAD, LF> &L, int cnt, Acc<T> (&acc)[TPL],
                                            const T (&tx)[TPL], const T (&ty)[TPL], const T (&tz)[TPL],
                                            const T (&th)[TPL])
{
    int k = 0;
#pragma unroll 1
    for (; k + U <= cnt; k += U) add_parts<T, TPL, FIELDS, QUAD, LF, U>(L, k, acc, tx, ty, tz, th);
#pragma unroll 1
    for (; U > 1 && k < cnt; k++) add_parts<T, TPL, FIELDS, QUAD, LF, 1>(L, k, acc, tx, ty, tz, th);
}

// Kernel variants of the FP32 one-target-per-lane walk (ptg_criterion.variant; the autotuner picks
// one per problem).  The traversal is latency-bound (3 -> 4 waves per SIMD: 4.5 -> 3.7 ms on the
// 1e7-particle walk), so registers are capped to fit more waves:
//   0: 5 waves per SIMD, lists evaluated at 64 entries (7.7 KB of LDS per wave, five 4-wave blocks per CU)
//   1: 4 waves per SIMD, lists at 64 (more registers per lane)
//   2: 6 waves per SIMD, lists at 32 (6.4 KB of LDS per wave, six blocks per CU)
// Every variant evaluates the same terms; variants 0 and 1 in the same order (bit-identical results),
// variant 2's shorter lists interleave the node and particle list evaluations differently, so its
// FP32 sums differ at the rounding level.
#define WALK_NVARIANTS 3
template <typename T, int TPL, int VAR> struct WalkOcc {
    static constexpr bool fast = TPL == 1;
    static constexpr int waves = !fast ? 1 : VAR == 1 ? 4 : VAR == 2 ? 6 : 5;
    static constexpr int lf = fast && VAR == 2 ? 32 : 64;
    static constexpr int blocks_per_cu = fast && VAR == 2 ? 6 : 5;
};

// PASS: the groups' walks that are never cut, those that may be, the tasks of those that were
enum { WHOLE, CUT, TASK };

template <typename T, int TPL, int FIELDS, bool QUAD, bool EXP, int VAR, int PASS>
__global__ __launch_bounds__(64 * WALK_WAVES) __attribute__((amdgpu_waves_per_eu(WalkOcc<T, TPL, VAR>::waves)))
void k_walk(const WalkArgs<T> A, const WalkHot H, const WalkPool pool)
{
    constexpr int LF = WalkOcc<T, TPL, VAR>::lf;
    constexpr bool TASKS = PASS == TASK;
    // entries evaluated together (nodes, particles): 4 where the registers of five waves per SIMD hold them.
    // The expansion's 16 sums leave room for 2 (with 4: 13 spilled registers), and in the six-wave variant for
    // none; tidal or quadrupole particles take 2.  4 and 2 against 1 and 1 with quadrupoles: 2.20 against 2.33 ms
    // for 1e6 particles, 2.89 against 3.60 with tidal tensors of 1e5 targets; 8 nodes were no faster than 4.  Two
    // and four targets per lane fill the chain alone: 2 nodes 0.81 against 0.83 ms (groups of 128, 3e5
    // particles), with quadrupoles 1 (2.75 ms for groups of 256; 2.89 with 2).
    constexpr int UN = VAR == 2 ? (EXP ? 1 : 2) : TPL > 1 ? (QUAD ? 1 : 2) : EXP ? 2 : 4;
    constexpr int UP = VAR == 2 ? UN : TPL > 1 ? 1 : EXP || QUAD || NW<FIELDS>::TID ? 2 : 4;
    static_assert(!EXP || (!QUAD && !NW<FIELDS>::TID), "the group expansion is a monopole potential/acceleration path");
    __shared__ WaveLds<T, QUAD, LF> lds[WALK_WAVES];
    const int wave = threadIdx.x >> 6, lane = ptg_lane();
    WaveLds<T, QUAD, LF> &L = lds[wave];
    // each wave's counts, added to the caller's when it ends: added per group they serialised on one line
    // (the learned walk of 1e7 particles took 10.3 ms with counters, 4.1 without)
    __shared__ unsigned long long counts[WALK_WAVES][4];
    if (lane < 4) counts[wave][lane] = 0;
    __builtin_amdgcn_wave_barrier();
    int *spill = H.spill + ((int64_t)blockIdx.x * WALK_WAVES + wave) * (int64_t)H.gcap;
    const int xcd = blockIdx.x % NXCD;
    int ghw = 0;  // this wave's deepest spill
    const int64_t ngroups = A.goff ? (int64_t)__builtin_amdgcn_readfirstlane(*A.gcount) : A.ngroups;

    int ticket = -1, closed = 0;
    if (!TASKS && blockIdx.x == 0 && threadIdx.x == 0) A.ctl->words = (int32_t)walk_words(ngroups);
    if (TASKS && agent_load(&A.ctl->open) == 0) return;  // nothing was deferred, or all of it is done

    for (int attempt = 0; attempt < (TASKS ? 1 : NXCD); attempt++) {
        const int x = (xcd + attempt) % NXCD;
        const int64_t g_lo = ngroups * x / NXCD, g_hi = ngroups * (x + 1) / NXCD;
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
                int gi = 0;
                if (lane == 0) gi = atomicAdd(&A.ctl->ctr[x * CTR_STRIDE], 1);
                g = g_lo + __builtin_amdgcn_readfirstlane(gi);
                if (g >= g_hi) break;
            }
            const WalkSpan grp = walk_span(A.goff, A.gs, A.nt, g);
            const int64_t a0 = grp.a0;
            const int mt = grp.mt;
            if (grp.over && lane == 0) atomicOr(&A.ctl->err, 2);  // a supplied group larger than group_size
            int root = 0;
            double ox = A.ox, oy = A.oy, oz = A.oz;
            if (A.nsys > 0) {
                int64_t lo = 0, hi = A.nsys;  // last system with soff[s] <= a0
                while (hi - lo > 1) {
                    const int64_t mid = (lo + hi) >> 1;
                    if (A.soff[mid] <= a0) lo = mid;
                    else hi = mid;
                }
                root = (int)lo;
                ox = A.cubes[4 * lo];
                oy = A.cubes[4 * lo + 1];
                oz = A.cubes[4 * lo + 2];
            }

            // ---- targets: lane holds a0 + lane + 64 j ----
            T tx[TPL], ty[TPL], tz[TPL], th[TPL];
            bool tval[TPL];
            int64_t tidx[TPL];  // rows of out, where the registers for them are there
            T bmin0 = INFINITY, bmin1 = INFINITY, bmin2 = INFINITY;
            T bmax0 = -INFINITY, bmax1 = -INFINITY, bmax2 = -INFINITY, hmax = -INFINITY;
#pragma unroll
            for (int j = 0; j < TPL; j++) {
                const int o = lane + 64 * j;
                tval[j] = o < mt;
                if (PASS == WHOLE) tidx[j] = tval[j] ? A.perm[a0 + o] : 0;
                if (tval[j]) {
                    const int64_t src = A.sorted ? a0 + o : PASS == WHOLE ? tidx[j] : A.perm[a0 + o];
                    tx[j] = (T)(A.pos[3 * src] - ox);
                    ty[j] = (T)(A.pos[3 * src + 1] - oy);
                    tz[j] = (T)(A.pos[3 * src + 2] - oz);
                    th[j] = (T)A.soft[src];
                    bmin0 = std::min(bmin0, tx[j]);
                    bmin1 = std::min(bmin1, ty[j]);
                    bmin2 = std::min(bmin2, tz[j]);
                    bmax0 = std::max(bmax0, tx[j]);
                    bmax1 = std::max(bmax1, ty[j]);
                    bmax2 = std::max(bmax2, tz[j]);
                    hmax = std::max(hmax, th[j]);
                } else {
                    tx[j] = ty[j] = tz[j] = th[j] = T(0);
                }
            }
            bmin0 = ptg_wave_min(bmin0);
            bmin1 = ptg_wave_min(bmin1);
            bmin2 = ptg_wave_min(bmin2);
            bmax0 = ptg_wave_max(bmax0);
            bmax1 = ptg_wave_max(bmax1);
            bmax2 = ptg_wave_max(bmax2);
            hmax = ptg_wave_max(hmax);
            // invalid lanes sit at the box corner so they never divide by zero
#pragma unroll
            for (int j = 0; j < TPL; j++)
                if (!tval[j]) {
                    tx[j] = bmin0 - T(1);
                    ty[j] = bmin1 - T(1);
                    tz[j] = bmin2 - T(1);
                }

            Acc<T> acc[TPL];
#pragma unroll
            for (int j = 0; j < TPL; j++) acc[j] = Acc<T>{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

            // group expansion: centre and radius of the group's box, this system's tolerance
            T cx = 0, cy = 0, cz = 0, rg = 0, eps_x = 0;
            GroupExp<T> E{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            if constexpr (EXP) {
                cx = T(0.5) * (bmin0 + bmax0);
                cy = T(0.5) * (bmin1 + bmax1);
                cz = T(0.5) * (bmin2 + bmax2);
                const T hx = T(0.5) * (bmax0 - bmin0), hy = T(0.5) * (bmax1 - bmin1), hz = T(0.5) * (bmax2 - bmin2);
                // rounded up by a relative 1e-6 so every target's offset from the centre is within rg
                rg = sqrt(hx * hx + hy * hy + hz * hz) * T(1.000001);
                eps_x = A.eps_exp * (A.eps_scale ? (T)A.eps_scale[root] : T(1));
            }

            int sp = 1, gsp = 0, nn = 0, np = 0;
            bool overflow = false, cut = false;
            const bool share = TASKS && rec.get<&WalkTask::off>() >= 0;  // else a group from its root
            if (share) {
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                const int stride = rec.get<&WalkTask::nchild>(), q0 = self - B.gcount - rec.get<&WalkTask::child0>();
                const int share_no = q0 < 0 ? q0 + B.tcount : q0;
                const int *entries = B.entries + rec.get<&WalkTask::off>() + share_no;
                sp = share_count(rec.get<&WalkTask::count>(), stride, share_no);  // <= SCAP: deeper stacks are not cut
                for (int q = lane; q < sp; q += 64) L.stack[q] = agent_load(&entries[(int64_t)q * stride]);
            } else if (lane == 0) {
                L.stack[0] = root;  // the root of system s occupies walk slot s
            }
            __builtin_amdgcn_wave_barrier();
            // Visits after which the traversal is cut.  Few groups: none, each opens much of the tree and its
            // sums run over up to all particles in FP32, so that another order of the terms moves the
            // fields (1e-4 of their RMS for 200 targets among 3e6 clumpy particles, tidal tensors 1e-3;
            // with the groups asked for 8e-6, 8e-6).  Middling: the longest traversal sets the time (66000
            // targets among 3e6 clumpy particles 22.4 -> 1.8 ms).  Many: the device is full without, and
            // the tables would fill (1e6 clumpy targets of 1e6 particles: 14.5 ms, 9.8 as here, 14.6 with
            // BUDGET; 2.2e6: 36 ms, 42 with BUDGET).  By the targets of the group's own system, so that a
            // system's cuts are those it has alone.
            int budget = 0x7fffffff;
            if (share) {
                budget = H.budget;
            } else if (PASS != WHOLE) {
                const int64_t sg = (A.nsys > 0 ? A.soff[root + 1] - A.soff[root] : A.nt) / A.gs;
                const float many = fmaxf(1.0f, (float)sg * (1.0f / 5120));
                if (sg >= cut_groups(FIELDS)) budget = (int)fminf((float)H.budget * many * sqrtf(many), 2e9f);
            }
            if (TASKS) budget = walk_budget(budget, rec.get<&WalkTask::level>());
            int nchild = 0, off = 0, child0 = 0, troot = -1;
            // counts of this traversal: elements visited, listed, listed as particles; folded (per lane)
            int n_vis = 0, n_list = 0, n_part = 0, n_exp = 0;

            for (;;) {  // once more only for a traversal that is not cut
                for (;;) {
                    // pop up to 64 stack entries, one per lane, refilling the LDS stack from the spill
                    // region when it is empty
                    if (sp == 0) {
                        if (gsp > 0) {
                            const int k = std::min(gsp, SPILL);
                            for (int q = lane; q < k; q += 64) L.stack[q] = spill[gsp - k + q];
                            __builtin_amdgcn_wave_barrier();
                            gsp -= k;
                            sp = k;
                        } else {
                            break;
                        }
                    }
                    if (PASS != WHOLE && n_vis >= budget) {
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
                    n_vis += k;
                    const V4<T> X = A.xyzm[e];
                    const V4<T> X2 = A.aux[e];
                    const int2 K = A.kids[e];
                    const bool ispart = K.y == 0;
                    // distance to the box per axis: max(bmin - x, x - bmax, 0), the same value as the
                    // two-sided test (one max3 per axis)
                    const T dxm = box_gap(X.x, bmin0, bmax0), dym = box_gap(X.y, bmin1, bmax1), dzm = box_gap(X.z, bmin2, bmax2);
                    const T r2m = dxm * dxm + dym * dym + dzm * dzm;
                    const T hh = X2.x > hmax ? X2.x : hmax;
                    // the reference's test (treewalk.py:22-25) on squared distances (every threshold is >= 0),
                    // with 1/theta; evaluated without branches (bitwise &) so the slot's aux record is one
                    // load issued with the others, not a second round trip inside a branch
                    const T c1 = X2.y * A.inv_theta + X2.z;
                    const T c2 = hh + X2.y * T(0.6) + X2.z;
                    const T c = c1 > c2 ? c1 : c2;
                    bool acc_node = ve & !ispart & (r2m > c * c);
                    // a particle farther from the group's box than every softening radius (and not
                    // inside it) needs neither the softening nor the self test -> node list
                    const bool far_part = ve & ispart & (r2m > hh * hh);
                    if (A.crit == 1) {
                        // error-bounded: also require the quadrupole term the monopole drops,
                        // 3.5 |Q| / r^4, to stay below eps (theta is then only a loose cap)
                        acc_node = acc_node & (X2.w < A.eps * r2m * r2m);
                    } else if (A.crit == 2) {
                        // learned: r_min beyond the node's predicted opening radius
                        acc_node = acc_node & (r2m > X2.w * X2.w);
                    }
                    bool acc_part = ve && ispart && !far_part;
                    acc_node = acc_node || far_part;
                    bool open = ve && !ispart && !acc_node;
                    if constexpr (EXP) {
                        if (acc_node) {
                            // accepted elements are outside every softening radius and r_min > 0,
                            // so D >= r_min > 0; fold if the truncation bound is within the tolerance
                            const T Dx = X.x - cx, Dy = X.y - cy, Dz = X.z - cz;
                            T rinv;
                            if (fold_test(X.w, Dx, Dy, Dz, rg, eps_x, A.exp_rel, rinv)) {
                                exp_add(E, X.w, Dx, Dy, Dz, rinv);
                                acc_node = false;
                                n_exp++;
                            }
                        }
                    }

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
                            const T *q = A.quad + 8 * (int64_t)e;
#pragma unroll
                            for (int c = 0; c < 6; c++) L.nq[6 * at + c] = q[c];
                        }
                    }
                    const int addp = (int)__popcll(bp), addn = (int)__popcll(bn);
                    np += addp;
                    nn += addn;
                    n_list += addp + addn;
                    n_part += addp;

                    // push the children of opened nodes
                    const int cnt = open ? std::min(std::max(K.y, 0), 8) : 0;
                    int tot;
                    const int below = small_excl_scan(cnt, tot);
                    if (sp + tot > SCAP) {
                        // move the bottom ks entries of the LDS stack to this wave's global region
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
                        // unrolled: eight masked LDS stores with immediate offsets, no per-lane loop
                        int *dst = &L.stack[sp + below];
#pragma unroll
                        for (int c = 0; c < 8; c++)
                            if (c < cnt) dst[c] = K.x + c;
                    }
                    sp += tot;
                    __builtin_amdgcn_wave_barrier();

                    if (nn >= LF) {
                        const int c = nn & ~(LF - 1);  // c >= LF > nn - c
                        flush_nodes<UN, T, TPL, FIELDS, QUAD, LF>(L, c, acc, tx, ty, tz);
                        __builtin_amdgcn_wave_barrier();
                        if (lane < nn - c) {  // reads [c, nn) and writes [0, nn - c): disjoint
                            L.nodes[lane] = L.nodes[c + lane];
                            if (QUAD)
                                for (int q = 0; q < 6; q++) L.nq[6 * lane + q] = L.nq[6 * (c + lane) + q];
                        }
                        __builtin_amdgcn_wave_barrier();
                        nn -= c;
                    }
                    if (np >= LF) {
                        const int c = np & ~(LF - 1);
                        flush_parts<UP, T, TPL, FIELDS, QUAD, LF>(L, c, acc, tx, ty, tz, th);
                        __builtin_amdgcn_wave_barrier();
                        if (lane < np - c) {  // disjoint ranges, as above
                            L.parts[lane] = L.parts[c + lane];
                            L.ph[lane] = L.ph[c + lane];
                        }
                        __builtin_amdgcn_wave_barrier();
                        np -= c;
                    }
                }
                if (PASS == WHOLE || !cut) break;
                nchild = walk_cut<TASKS>(A.ctl, H, pool, share, L.stack, sp, spill, gsp, lane, self, off, child0);
                cut = nchild > 0;
                if (nchild) break;
                budget = 0x7fffffff;
            }
            if (TASKS) troot = parent < walk_pool<TASKS>(A.ctl, H, pool).gcount ? parent : rec.get<&WalkTask::root>();
            if (PASS != WHOLE && nchild < 0) {  // no room: the group is walked again
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
                if (!TASKS) {
                    if (lane == 0) walk_put_back<AgentMem>(A.ctl, B, false, (int)g);
                    continue;
                }
                if (lane == 0) agent_store(&B.tasks[troot].root, 1);
                nn = np = 0;  // its row and counts are not used any more
            }
            if (A.counters) {
                if (EXP) {
#pragma unroll
                    for (int d = 32; d >= 1; d >>= 1) n_exp += __shfl_xor(n_exp, d, 64);  // lanes fold separately
                }
                if (lane == 0) {
                    const int64_t n[4] = {(int64_t)n_list * mt, n_vis, (int64_t)n_part * mt, n_exp};
                    for (int q = 0; q < (EXP ? 4 : 3); q++) {
                        if (PASS == CUT && cut) agent_store(&walk_pool<TASKS>(A.ctl, H, pool).counts[4 * self + q], n[q]);
                        else if (TASKS) atomicAdd((unsigned long long *)&walk_pool<TASKS>(A.ctl, H, pool).counts[4 * troot + q], (unsigned long long)n[q]);
                        else counts[wave][q] += (unsigned long long)n[q];
                    }
                }
            }
            if (overflow) {
                if (lane == 0) atomicOr(&A.ctl->err, 1);
                if (!TASKS) continue;
                nn = np = 0;  // a task's row is written all the same: the sums read every task's
            }
            flush_nodes<UN, T, TPL, FIELDS, QUAD, LF>(L, nn, acc, tx, ty, tz);
            flush_parts<UP, T, TPL, FIELDS, QUAD, LF>(L, np, acc, tx, ty, tz, th);
            __builtin_amdgcn_wave_barrier();
            if constexpr (EXP) {
                exp_wave_sum(E);
#pragma unroll
                for (int j = 0; j < TPL; j++) exp_eval<T, FIELDS>(acc[j], E, tx[j] - cx, ty[j] - cy, tz[j] - cz);
            }

            // ---- G * fields in the caller's order, or the row of a deferred group or a task ----
            constexpr int W = NW<FIELDS>::W, WI = NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC + 6 * NW<FIELDS>::TID;
            if (TASKS || cut) {
                const WalkPool B = walk_pool<TASKS>(A.ctl, H, pool);
#pragma unroll
                for (int j = 0; j < TPL; j++) {
                    if (!tval[j]) continue;
                    T *o = (T *)B.partial + ((int64_t)self * A.gs + lane + 64 * j) * WI;
                    int c = 0;
                    if (NW<FIELDS>::POT) agent_store(&o[c++], acc[j].phi);
                    if (NW<FIELDS>::ACC) {
                        agent_store(&o[c++], acc[j].gx);
                        agent_store(&o[c++], acc[j].gy);
                        agent_store(&o[c++], acc[j].gz);
                    }
                    if (NW<FIELDS>::TID) {
                        agent_store(&o[c++], acc[j].txx);
                        agent_store(&o[c++], acc[j].txy);
                        agent_store(&o[c++], acc[j].txz);
                        agent_store(&o[c++], acc[j].tyy);
                        agent_store(&o[c++], acc[j].tyz);
                        agent_store(&o[c++], acc[j].tzz);
                    }
                }
                if (cut) {
                    const WalkPool P = walk_pool<TASKS>(A.ctl, H, pool);
                    walk_publish<AgentMem>(A.ctl, P, WalkTask{(int)g, parent, TASKS ? troot : 0, TASKS ? rec.get<&WalkTask::level>() : 0, off,
                                                         gsp + sp, child0 % P.tcount, nchild, nchild, {}}, child0, self, lane);
                } else {
                    const int p = walk_add_up<FIELDS, T>(A.ctl, B, parent, grp, A.gs, A.perm, A.G, A.out, lane);
                    if (p >= 0 && A.counters && lane < (EXP ? 4 : 3))
                        counts[wave][lane] += (unsigned long long)agent_load(&B.counts[4 * p + lane]);
                }
                if (TASKS) closed++;
                continue;
            }
#pragma unroll
            for (int j = 0; j < TPL; j++) {
                if (!tval[j]) continue;
                double *o = A.out + (PASS == WHOLE ? tidx[j] : A.perm[a0 + lane + 64 * j]) * W;
                int c = 0;
                if (NW<FIELDS>::POT) o[c++] = A.G * (double)acc[j].phi;
                if (NW<FIELDS>::ACC) {
                    o[c++] = A.G * (double)acc[j].gx;
                    o[c++] = A.G * (double)acc[j].gy;
                    o[c++] = A.G * (double)acc[j].gz;
                }
                if (NW<FIELDS>::TID) {
                    double xx = A.G * (double)acc[j].txx, yy = A.G * (double)acc[j].tyy, zz = A.G * (double)acc[j].tzz;
                    double xy = A.G * (double)acc[j].txy, xz = A.G * (double)acc[j].txz, yz = A.G * (double)acc[j].tyz;
                    o[c++] = xx; o[c++] = xy; o[c++] = xz;
                    o[c++] = xy; o[c++] = yy; o[c++] = yz;
                    o[c++] = xz; o[c++] = yz; o[c++] = zz;
                }
            }
        }
    }
    if (lane == 0 && ghw > 0) atomicMax(&A.ctl->hwm, ghw);
    __builtin_amdgcn_wave_barrier();
    if (A.counters && lane < (EXP ? 4 : 3) && counts[wave][lane])
        atomicAdd((unsigned long long *)&A.counters[lane], counts[wave][lane]);
}


// ============================================================================================
// host side
// ============================================================================================
static int g_num_cus = 0;

static int num_cus()
{
    if (g_num_cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) dev = 0;
        hipDeviceProp_t p;
        if (hipGetDeviceProperties(&p, dev) == hipSuccess) g_num_cus = p.multiProcessorCount;
        if (g_num_cus <= 0) g_num_cus = 256;
    }
    return g_num_cus;
}

#define WALK_MAX_BLOCKS_PER_CU 6  // the most any variant runs (variant 2)

// persistent grid: resident blocks per CU from the occupancy API, capped by the variant's plan and
// by the spill allocation
static int64_t walk_grid_blocks(int variant = -1)
{
    const int per = variant == 2 ? 6 : variant < 0 ? WALK_MAX_BLOCKS_PER_CU : 5;
    return (int64_t)num_cus() * per;
}

// bytes of the bits of a walk's groups, at most one per target
static size_t walk_again_bytes(int64_t nt)
{
    return std::max<size_t>(WALK_AGAIN, walk_words(nt) * sizeof(int32_t));
}

extern "C" size_t ptg_walk_workspace_bytes(int64_t nt, int group_size)
{
    (void)group_size;
    size_t waves = (size_t)walk_grid_blocks() * WALK_WAVES;
    return walk_control_bytes(walk_again_bytes(nt)) + ptg_align256(waves * GCAP * sizeof(int)) + WALK_POOL;
}

// ---- static scratch of ptg_walk_noalloc ----
// Callers that cannot allocate (code under HIP graph capture, serving loops, harnesses that forbid
// hipMalloc) walk with this file-scope array as the workspace: the walk control block (per-XCD group
// counters, overflow flag), the per-wave global spill stacks and the cut traversals.  Every GPU that runs the library
// holds its own copy until the process ends; every call on a device shares it, so calls that
// overlap on one device (different streams) race.  Host code never passes the array's name to a
// kernel (that is a host-side stand-in): it uses the address hipGetSymbolAddress returns, looked up
// once per device with that device current and kept per device.
// 4096 spill entries per wave for 5120 resident waves
#define NOALLOC_BYTES ((80u << 20) + (1u << 20) + WALK_AGAIN + WALK_POOL)
#define NOALLOC_MIN_GCAP 2048  // spill entries per wave the static scratch must leave
#define NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) char scratch[NOALLOC_BYTES];
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[NOALLOC_MAX_DEVICES];

static ptg_status noalloc_scratch(void **p)
{
    int dev = 0;
    PTG_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
        ptg_set_error("ptg_walk_noalloc: device %d beyond the %d the library tracks", dev, NOALLOC_MAX_DEVICES);
        return PTG_ERR_ARG;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            ptg_set_error("ptg_walk_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                          hipGetErrorString(e));
            return PTG_ERR_HIP;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *p = g_scratch_ptr[dev];
    return PTG_OK;
}

// spill entries per wave the static scratch leaves for `blocks` resident blocks (a multiple of 64,
// at most GCAP)
static int noalloc_gcap(int64_t blocks)
{
    const int64_t waves = blocks * WALK_WAVES;
    int64_t per = (int64_t)(NOALLOC_BYTES - WALK_POOL - walk_control_bytes()) / (waves * (int64_t)sizeof(int));
    per = std::min<int64_t>(per, GCAP) & ~(int64_t)63;
    return (int)per;
}

__global__ void k_walk_err_out(const WalkCtl *ctl, int32_t *err)
{
    if (threadIdx.x == 0) *err = ctl->err;
}

struct WalkWs {  // a walk's workspace
    char *p;
    size_t bytes;
    size_t again;  // bytes of the bits of the groups put back
    int gcap;  // global spill entries per wave (GCAP, or what the static scratch of ptg_walk_noalloc gives)
};


template <typename T, int TPL, int FIELDS, bool QUAD, bool EXP, int VAR = 0>
static ptg_status launch_t(const WalkArgs<T> &a, int64_t max_blocks, const WalkWs &ws, hipStream_t s)
{
    static int per_cu = 0;
    if (per_cu == 0) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_walk<T, TPL, FIELDS, QUAD, EXP, VAR, CUT>,
                                                         64 * WALK_WAVES, 0) != hipSuccess ||
            nb < 1)
            nb = 1;
        per_cu = std::min(nb, WalkOcc<T, TPL, VAR>::blocks_per_cu);
    }
    const int64_t blocks = std::min<int64_t>(max_blocks, (int64_t)num_cus() * per_cu);
    constexpr int WI = NW<FIELDS>::POT + 3 * NW<FIELDS>::ACC + 6 * NW<FIELDS>::TID;
    WalkHot b{};
    const double open = a.theta < T(0.7) ? 0.49 / ((double)a.theta * a.theta) : 1.0;
    b.budget = (int)std::min(1e8, BUDGET * open * TPL);
    b.most0 = 16;
    b.most = 128;
    ptg_status st = walk_carve(b, ws.p, ws.bytes, a.goff ? a.nt : a.ngroups, ws.again, blocks * WALK_WAVES, ws.gcap,
                               (size_t)a.gs * WI * sizeof(T));
    if (st) return st;
    // a traversal visits a slot once, and no system has more targets than there are: where none can be
    // cut, the kernel without (its scalar registers do not spill; 2 to 7 % of the longest traversals)
    if (b.tcount == 0 || a.nslots <= b.budget || a.nt / a.gs < cut_groups(FIELDS)) {
        k_walk<T, TPL, FIELDS, QUAD, EXP, VAR, WHOLE><<<(unsigned)blocks, 64 * WALK_WAVES, 0, s>>>(a, b, walk_pool(a.ctl, b));
    } else {
        k_walk<T, TPL, FIELDS, QUAD, EXP, VAR, CUT><<<(unsigned)blocks, 64 * WALK_WAVES, 0, s>>>(a, b, walk_pool(a.ctl, b));
        PTG_LAUNCH_CHECK();
        k_walk<T, TPL, FIELDS, QUAD, EXP, VAR, TASK><<<(unsigned)blocks, 64 * WALK_WAVES, 0, s>>>(a, b, walk_pool(a.ctl, b));
    }
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

// the monopole potential/acceleration kernels of the one-target-per-lane FP32 walk come in
// WALK_NVARIANTS variants; every other kernel in variant 0
template <typename T, int TPL, int FIELDS, bool EXP>
static ptg_status launch_var(const WalkArgs<T> &a, int variant, int64_t blocks, const WalkWs &ws, hipStream_t s)
{
    if constexpr (TPL == 1) {
        if (variant == 1) return launch_t<T, TPL, FIELDS, false, EXP, 1>(a, blocks, ws, s);
        if (variant == 2) return launch_t<T, TPL, FIELDS, false, EXP, 2>(a, blocks, ws, s);
    }
    return launch_t<T, TPL, FIELDS, false, EXP, 0>(a, blocks, ws, s);
}

template <typename T, int TPL>
static ptg_status launch_fq(const WalkArgs<T> &a, int fields, bool quad, bool expand, int variant, int64_t blocks,
                            const WalkWs &ws, hipStream_t s)
{
    if (expand) {  // checked by the caller: monopole, potential and/or acceleration
        if (fields == PTG_POT) return launch_var<T, TPL, PTG_POT, true>(a, variant, blocks, ws, s);
        if (fields == PTG_ACC) return launch_var<T, TPL, PTG_ACC, true>(a, variant, blocks, ws, s);
        return launch_var<T, TPL, PTG_POT | PTG_ACC, true>(a, variant, blocks, ws, s);
    }
    if (!quad) {
        if (fields == PTG_POT) return launch_var<T, TPL, PTG_POT, false>(a, variant, blocks, ws, s);
        if (fields == PTG_ACC) return launch_var<T, TPL, PTG_ACC, false>(a, variant, blocks, ws, s);
        if (fields == (PTG_POT | PTG_ACC)) return launch_var<T, TPL, PTG_POT | PTG_ACC, false>(a, variant, blocks, ws, s);
    }
#define PTG_F(F)                                                              \
    case F:                                                                   \
        return quad ? launch_t<T, TPL, F, true, false>(a, blocks, ws, s)          \
                    : launch_t<T, TPL, F, false, false>(a, blocks, ws, s);
    switch (fields) {
        PTG_F(1) PTG_F(2) PTG_F(3) PTG_F(4) PTG_F(5) PTG_F(6) PTG_F(7)
    }
#undef PTG_F
    ptg_set_error("ptg_walk: fields must be a nonzero combination of PTG_POT|PTG_ACC|PTG_TIDAL");
    return PTG_ERR_ARG;
}

template <typename T>
static ptg_status launch_walk(const WalkArgs<T> &a, int fields, bool quad, bool expand, int variant, int64_t blocks,
                              const WalkWs &ws, hipStream_t s)
{
    if (a.gs <= 64) return launch_fq<T, 1>(a, fields, quad, expand, variant, blocks, ws, s);
    if (a.gs <= 128) return launch_fq<T, 2>(a, fields, quad, expand, variant, blocks, ws, s);
    return launch_fq<T, 4>(a, fields, quad, expand, variant, blocks, ws, s);
}

// ptg_walk and ptg_walk_noalloc: ws/ws_bytes is the caller's workspace, or nullptr with noalloc set
// (the static scratch below; err_out then receives the overflow flag)
static ptg_status walk_impl(const ptg_walk_tree *wt, const ptg_forest *forest, const double *pos, const double *soft,
                            const int64_t *perm, int targets_sorted, int64_t nt, int fields, int quadrupole,
                            int group_size, const int32_t *group_offsets, const int32_t *group_count, double theta,
                            const ptg_criterion *criterion, double G, int exact, double *out, int64_t *counters,
                            void *ws, size_t ws_bytes, bool noalloc, int32_t *err_out, void *stream,
                            const int32_t *start_slot = nullptr)
{
    hipStream_t s = (hipStream_t)stream;
    if (!wt || nt < 0 || (nt > 0 && (!pos || !soft || !perm || !out))) {
        ptg_set_error("ptg_walk: bad arguments");
        return PTG_ERR_ARG;
    }
    if (forest && (forest->nsys < 1 || !forest->offsets || !forest->cubes)) {
        ptg_set_error("ptg_walk: a forest needs nsys >= 1, offsets and cubes");
        return PTG_ERR_ARG;
    }
    if (forest && forest->nsys > 1 && !group_offsets) {
        ptg_set_error("ptg_walk: a forest walk needs group offsets that respect system boundaries "
                      "(ptg_target_groups with the forest)");
        return PTG_ERR_ARG;
    }
    if (group_size < 1 || group_size > 256) {
        ptg_set_error("ptg_walk: group_size must be in [1, 256], got %d", group_size);
        return PTG_ERR_ARG;
    }
    if (!(theta > 0)) {
        ptg_set_error("ptg_walk: theta must be positive");
        return PTG_ERR_ARG;
    }
    if (quadrupole && (!wt->has_quad || !wt->quad)) {
        ptg_set_error("ptg_walk: quadrupole=True requires a walk tree packed with quadrupoles");
        return PTG_ERR_ARG;
    }
    if (fields < 1 || fields > 7) {
        ptg_set_error("ptg_walk: fields must be a nonzero combination of PTG_POT|PTG_ACC|PTG_TIDAL");
        return PTG_ERR_ARG;
    }
    if ((group_offsets == nullptr) != (group_count == nullptr)) {
        ptg_set_error("ptg_walk: group_offsets and group_count must be given together");
        return PTG_ERR_ARG;
    }
    const int crit = criterion ? criterion->criterion : PTG_CRIT_THETA;
    if (crit != PTG_CRIT_THETA && crit != PTG_CRIT_QERR && crit != PTG_CRIT_RADIUS) {
        ptg_set_error("ptg_walk: unknown criterion %d", crit);
        return PTG_ERR_ARG;
    }
    if (crit == PTG_CRIT_QERR && (exact || !(criterion->eps > 0))) {
        ptg_set_error("ptg_walk: the error-bounded criterion needs eps > 0 and the FP32 walk");
        return PTG_ERR_ARG;
    }
    if (crit == PTG_CRIT_RADIUS && (exact || wt->prec != PTG_F32)) {
        ptg_set_error("ptg_walk: the radius criterion runs on the FP32 walk with radii from ptg_open_radii");
        return PTG_ERR_ARG;
    }
    const double eps = crit == PTG_CRIT_QERR ? criterion->eps / 3.5 : 0.0;
    const bool expand = criterion && criterion->group_expansion != 0;
    if (expand) {
        if (exact || wt->prec != PTG_F32 || quadrupole || (fields & PTG_TIDAL)) {
            ptg_set_error("ptg_walk: the group expansion runs on the FP32 walk with monopole interactions, "
                          "for the potential and/or the acceleration");
            return PTG_ERR_ARG;
        }
        if (!(criterion->expansion_eps > 0)) {
            ptg_set_error("ptg_walk: the group expansion needs expansion_eps > 0");
            return PTG_ERR_ARG;
        }
        if (!(criterion->expansion_rel >= 0.0f)) {
            ptg_set_error("ptg_walk: expansion_rel must be >= 0 (0 = no relative cap)");
            return PTG_ERR_ARG;
        }
    }
    const double eps_exp = expand ? criterion->expansion_eps : 0.0;
    const double *eps_scale = expand ? criterion->eps_scale : nullptr;
    if (expand && criterion->group_expansion != 1) {
        ptg_set_error("ptg_walk: group_expansion must be 0 (off) or 1");
        return PTG_ERR_ARG;
    }
    const int variant = criterion ? criterion->variant : 0;
    if (variant < 0 || variant >= WALK_NVARIANTS) {
        ptg_set_error("ptg_walk: variant must be in [0, %d), got %d", WALK_NVARIANTS, variant);
        return PTG_ERR_ARG;
    }
    int64_t blocks = walk_grid_blocks(variant);
    int gcap = GCAP;
    if (noalloc) {
        if (!err_out) {
            ptg_set_error("ptg_walk_noalloc: err (a device int32 that receives the overflow flag) is required");
            return PTG_ERR_ARG;
        }
        ptg_status st = noalloc_scratch(&ws);
        if (st) return st;
        ws_bytes = NOALLOC_BYTES;
        gcap = noalloc_gcap(blocks);
        if (gcap < NOALLOC_MIN_GCAP) {
            ptg_set_error("ptg_walk_noalloc: %lld resident waves leave %d spill entries each in the %u-byte static "
                          "scratch (at least %d needed); use ptg_walk with a workspace",
                          (long long)(blocks * WALK_WAVES), gcap, NOALLOC_BYTES, NOALLOC_MIN_GCAP);
            return PTG_ERR_ARG;
        }
    }
    if (nt == 0) return PTG_OK;
    const size_t base_bytes = noalloc ? ws_bytes : ptg_walk_workspace_bytes(nt, group_size);
    const size_t need = base_bytes;
    if (ws_bytes < need || !ws) {
        ptg_set_error("ptg_walk: workspace too small (%zu < %zu)", ws_bytes, need);
        return PTG_ERR_WORKSPACE;
    }
    WalkCtl *ctl = (WalkCtl *)ws;
    const int64_t fn = forest ? forest->nsys : 0;
    const int64_t *fo = forest ? forest->offsets : nullptr;
    const double *fc = forest ? forest->cubes : nullptr;
    const size_t again = noalloc ? WALK_AGAIN : walk_again_bytes(nt);
    ptg_status st = walk_clear(ctl, group_offsets ? nt : ptg_cdiv(nt, group_size), again, s);
    if (st) return st;
    if (wt->prec == PTG_F32) {
        WalkArgs<float> a{(const V4<float> *)wt->xyzm, (const V4<float> *)wt->aux, (const int2 *)wt->kids,
                          (const float *)wt->quad, pos, soft, perm, targets_sorted != 0, wt->nslots, nt, ptg_cdiv(nt, group_size), group_offsets, group_count,
                          group_size, (float)theta, (float)(1.0 / theta), crit, (float)eps, (float)eps_exp,
                          expand ? criterion->expansion_rel : 0.0f, eps_scale, G, wt->origin[0], wt->origin[1],
                          wt->origin[2],
                          fn, fo, fc, out, counters, ctl};
        if (exact) {
            ptg_set_error("ptg_walk: the exact branch set is evaluated in FP64; use prec=PTG_F64");
            return PTG_ERR_ARG;
        }
        st = launch_walk<float>(a, fields, quadrupole != 0, expand, variant, blocks, WalkWs{(char *)ws, ws_bytes, again, gcap}, s);
    } else if (wt->prec == PTG_F64) {
        Walk64Args a{(const V4<double> *)wt->xyzm, (const V4<double> *)wt->aux, (const int2 *)wt->kids,
                     (const double *)wt->quad, pos, soft, perm, targets_sorted != 0, wt->nslots, nt,
                     ptg_cdiv(nt, group_size), group_offsets, group_count, group_size, theta, 1.0 / theta, G,
                     wt->origin[0], wt->origin[1], wt->origin[2], fn, fo, out, counters, ctl, start_slot};
        st = ptg_walk64_launch(a, fields, quadrupole != 0, num_cus(), gcap, again, (char *)ws, ws_bytes, s);
    } else {
        ptg_set_error("ptg_walk: prec must be PTG_F32 or PTG_F64");
        return PTG_ERR_ARG;
    }
    if (st == PTG_OK && noalloc) {
        k_walk_err_out<<<1, 64, 0, s>>>(ctl, err_out);
        PTG_LAUNCH_CHECK();
    }
    return st;
}

extern "C" ptg_status ptg_walk(const ptg_walk_tree *wt, const ptg_forest *forest, const double *pos,
                               const double *soft, const int64_t *perm, int targets_sorted, int64_t nt, int fields,
                               int quadrupole, int group_size, const int32_t *group_offsets,
                               const int32_t *group_count, double theta, const ptg_criterion *criterion, double G,
                               int exact, double *out, int64_t *counters, void *ws, size_t ws_bytes, void *stream)
{
    return walk_impl(wt, forest, pos, soft, perm, targets_sorted, nt, fields, quadrupole, group_size, group_offsets,
                     group_count, theta, criterion, G, exact, out, counters, ws, ws_bytes, false, nullptr, stream);
}

extern "C" ptg_status ptg_walk_noalloc(const ptg_walk_tree *wt, const ptg_forest *forest, const double *pos,
                                       const double *soft, const int64_t *perm, int targets_sorted, int64_t nt,
                                       int fields, int quadrupole, int group_size, const int32_t *group_offsets,
                                       const int32_t *group_count, double theta, const ptg_criterion *criterion,
                                       double G, int exact, double *out, int64_t *counters, int32_t *err,
                                       void *stream)
{
    return walk_impl(wt, forest, pos, soft, perm, targets_sorted, nt, fields, quadrupole, group_size, group_offsets,
                     group_count, theta, criterion, G, exact, out, counters, nullptr, 0, true, err, stream);
}

// every target walks the subtree of one element (treewalk.py:78-277 with no >= 0, stopping at
// subtree_end :28-34): the FP64 walk with the reference's branches, one target per group
extern "C" ptg_status ptg_walk_subtree(const ptg_walk_tree *wt, const int32_t *start_slot, const double *pos,
                                       const double *soft, const int64_t *perm, int64_t nt, int fields,
                                       int quadrupole, double theta, double G, double *out, int64_t *counters,
                                       void *ws, size_t ws_bytes, void *stream)
{
    if (!wt || !start_slot) {
        ptg_set_error("ptg_walk_subtree: bad arguments (walk tree and start slot are required)");
        return PTG_ERR_ARG;
    }
    if (wt->prec != PTG_F64) {
        ptg_set_error("ptg_walk_subtree: the per-target walks run on the FP64 walk tree (prec=PTG_F64)");
        return PTG_ERR_ARG;
    }
    return walk_impl(wt, nullptr, pos, soft, perm, 0, nt, fields, quadrupole, 1, nullptr, nullptr, theta, nullptr, G,
                     1, out, counters, ws, ws_bytes, false, nullptr, stream, start_slot);
}

// overflow flag of the last walk on this workspace (0 = fine); synchronises the stream
extern "C" ptg_status ptg_walk_check(void *ws, void *stream)
{
    int32_t err = 0;
    hipStream_t s = (hipStream_t)stream;
    PTG_HIP_CHECK(hipMemcpyAsync(&err, &((WalkCtl *)ws)->err, 4, hipMemcpyDeviceToHost, s));
    PTG_HIP_CHECK(hipStreamSynchronize(s));
    if (err & 2) {
        ptg_set_error("ptg_walk: a supplied target group holds more than group_size targets (its rows past "
                      "group_size were not evaluated)");
        return PTG_ERR_ARG;
    }
    if (err & 4) {
        ptg_set_error("ptg_walk_subtree: the start element's slot is outside the walk tree (nothing was walked)");
        return PTG_ERR_ARG;
    }
    if (err & 8) {
        ptg_set_error("ptg_walk: waves of the task pass gave up waiting for deferred traversals");
        return PTG_ERR_OVERFLOW;
    }
    if (err) {
        ptg_set_error("ptg_walk: a traversal stack exceeded its spill capacity");
        return PTG_ERR_OVERFLOW;
    }
    return PTG_OK;
}
