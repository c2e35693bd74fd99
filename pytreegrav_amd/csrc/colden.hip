// Column density through the octree (treewalk.py:821-1276): particles are uniform spheres of radius
// equal to their softening.
//
// Ray-traced: exact, a node is opened whenever its bounding sphere, inflated by the largest particle radius in
// it, could meet the ray; only particles contribute, by the closed-form chord integral.  Three walks:
//   k_column_bundles (ptg_column_bundles): shared unit rays, one wavefront for 64 targets that neighbour each
//     other across the ray, 64 elements a step over a stack in LDS; sums in the bundle's order.
//   k_column_rays_wave (ptg_column_rays with the FP64 pack): rays of each target's own, or of any length, one
//     wavefront for 64 targets along one ray index, one element a step; sums in the reference's order.
//   k_column_rays (ptg_column_rays without): one thread per (target, ray) along the tree's depth-first links,
//     with no stack, for trees deeper than the stacks of the others; sums in the reference's order.
//
// Angular-binned (ptg_column_binned), the reference's grouped estimator: a node whose distance to
// the box of group_size consecutive targets passes the opening test puts its mass in one of six
// equal-area sky bins per target; particles are summed per target.  For group_size <= 64 it is the FP64
// grouped walk (walk64.hip) with the bins as its sums.  Larger groups take one thread per group along the
// depth-first links.
#include <algorithm>

#include "walk_shared.hpp"

#define CD_THREADS 256

// one 32-byte record of the FP64 walk pack
struct alignas(32) D4 {
    double x, y, z, w;
};

// a corrupt link (index out of range, or a chain longer than the element count) stops the walk and
// sets err[0]; the depth-first chain visits each element at most once
__device__ __forceinline__ bool cd_bad(int64_t no, int64_t ne, int64_t &visits)
{
    return no >= ne || ++visits > ne;
}

// adds one wave's counts to ctr[k] with one atomic (every lane of the wave takes part)
__device__ __forceinline__ void cd_count(unsigned long long *ctr, int k, int64_t v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    if (ptg_lane() == 0 && v) atomicAdd(ctr + k, (unsigned long long)v);
}

// An element at d from a target, against a ray u: its squared distance, its distance along the ray and its squared
// distance across it, each product and sum rounded as in the reference's arithmetic.  An element exactly along the
// ray (as on a lattice) is at b2 = 0; with fused multiply-adds its sign was a product's rounding error, and half of
// such elements, particles and whole nodes, were skipped.
struct Across {
    double r2, z, b2;
    __device__ __forceinline__ Across(double dx, double dy, double dz, double ux, double uy, double uz)
    {
#pragma clang fp contract(off)
        r2 = dx * dx + dy * dy + dz * dz;
        z = ux * dx + uy * dy + uz * dz;
        b2 = r2 - z * z;
    }
};

// column along ray i from target j; visits counts the elements the walk touched
__device__ __forceinline__ double ray_column(const ptg_tree_arrays &t, int64_t n, int64_t ne, const double *tp,
                                             const double *rays, int64_t nr, int per_target, int64_t i, int64_t j,
                                             int32_t *err, int64_t &visits)
{
    const double *ray = per_target ? rays + 3 * (j * nr + i) : rays + 3 * i;
    const double rx = ray[0], ry = ray[1], rz = ray[2];
    const double px = tp[3 * j], py = tp[3 * j + 1], pz = tp[3 * j + 2];
    const double fac_density = 3.0 / (4.0 * 3.14159265358979323846);
    double column = 0.0;
    int64_t no = n;
    const int64_t stop = t.next_branch[n];
    while (no > -1 && no != stop) {
        if (cd_bad(no, ne, visits)) {
            atomicOr(err, 1);
            break;
        }
        const double dx = t.coordinates[3 * no] - px, dy = t.coordinates[3 * no + 1] - py;
        const double dz = t.coordinates[3 * no + 2] - pz;
        const Across e(dx, dy, dz, rx, ry, rz);
        const double r = sqrt(e.r2), z = e.z, b2 = e.b2;
        if (b2 < 0) {  // rounding below zero: skipped, as ColumnDensityWalk_singleray does
            no = t.next_branch[no];
            continue;
        }
        const double h_no = t.softenings[no];
        if (no < n) {
            if (h_no > 0) {  // a zero radius has no cross-section
                const double hinv = 1.0 / h_no;
                const double fac = fac_density * t.masses[no] * hinv * hinv;
                const double r_proj = sqrt(b2);
                const double q = r_proj * hinv;
                if (r_proj < h_no) {
                    if (r > h_no) {  // target outside the sphere: the whole chord if it lies ahead
                        if (z > 0) column += fac * 2 * sqrt(1 - q * q);
                    } else {  // target inside: the forward half-chord
                        column += fac * (z * hinv + sqrt(1 - q * q));
                    }
                }
            }
            no = t.next_branch[no];
        } else {
            const double reach = h_no + t.sizes[no] * 0.8660254037844386 + t.deltas[no];
            bool open = r < reach;  // the node holds the ray's origin
            if (!open && z > 0) open = b2 < reach * reach;
            no = open ? t.first_subnode[no] : t.next_branch[no];
        }
    }
    return column;
}

__global__ __launch_bounds__(CD_THREADS) void k_column_rays(const ptg_tree_arrays t, int64_t n, int64_t ne,
                                                            const double *tp, int64_t nt, const double *rays,
                                                            int64_t nr, int per_target, double *out, int32_t *err,
                                                            unsigned long long *ctr)
{
    const int64_t id = (int64_t)blockIdx.x * CD_THREADS + threadIdx.x;
    int64_t visits = 0;
    if (id < nt * nr) {
        const int64_t i = id / nt, j = id - (id / nt) * nt;  // ray i, target j
        out[j * nr + i] = ray_column(t, n, ne, tp, rays, nr, per_target, i, j, err, visits);
    }
    if (ctr) cd_count(ctr, 0, visits);
}

// ---- ray-traced walk, one wavefront per 64 targets along one ray index ----
// The wavefront walks the union of its lanes' walks in depth-first preorder over the FP64 walk pack:
// a stack of (first slot, count, lane mask) sibling ranges, one element per iteration, its record
// read once for all lanes.  Each lane applies exactly the tests of the per-thread walk to the
// elements its own walk would reach (those whose ancestors it opened), in the same order, so every
// column gets the same terms summed in the same sequence.
#define CR_WAVES 4
#define CR_DEPTH 256  // sibling ranges on the stack (one per tree level on the current path)

struct CrLds {
    int s[CR_DEPTH], c[CR_DEPTH];
    uint64_t m[CR_DEPTH];
};

__global__ __launch_bounds__(64 * CR_WAVES) void k_column_rays_wave(const D4 *xyzm, const D4 *aux, const int2 *kids,
                                                                    int64_t nslots, const double *tp, int64_t nt,
                                                                    const double *rays, int64_t nr, int per_target,
                                                                    const int64_t *order, double *out, int32_t *err,
                                                                    unsigned long long *ctr)
{
    __shared__ CrLds lds[CR_WAVES];
    const int wave = threadIdx.x >> 6, lane = ptg_lane();
    CrLds &S = lds[wave];
    const int64_t ntb = (nt + 63) / 64;
    const int64_t task = (int64_t)blockIdx.x * CR_WAVES + wave;
    if (task >= ntb * nr) return;  // whole wavefronts only: task is uniform
    const int64_t i = task / ntb, jr = (task % ntb) * 64 + lane;  // ray i, rank jr of the target
    const bool live = jr < nt;
    // the target order of ray i (if given) puts targets whose rays run side by side in one wavefront
    const int64_t j = live && order ? order[i * nt + jr] : jr;
    double rx = 0, ry = 0, rz = 0, px = 0, py = 0, pz = 0;
    if (live) {
        const double *ray = per_target ? rays + 3 * (j * nr + i) : rays + 3 * i;
        rx = ray[0];
        ry = ray[1];
        rz = ray[2];
        px = tp[3 * j];
        py = tp[3 * j + 1];
        pz = tp[3 * j + 2];
    }
    const double fac_density = 3.0 / (4.0 * 3.14159265358979323846);
    const uint64_t me = 1ull << lane;
    double column = 0.0;
    int64_t visits = 0;
    int top = 0;
    const uint64_t all = ptg_ballot(live);  // outside the lane-0 branch: a ballot sees the active lanes only
    if (lane == 0) {
        S.s[0] = 0;  // the root's walk slot
        S.c[0] = 1;
        S.m[0] = all;
    }
    __builtin_amdgcn_wave_barrier();
    while (top >= 0) {
        const int sl = S.s[top], cnt = S.c[top];
        const uint64_t m = S.m[top];
        __builtin_amdgcn_wave_barrier();
        if (cnt > 1) {
            if (lane == 0) {
                S.s[top] = sl + 1;
                S.c[top] = cnt - 1;
            }
        } else {
            top--;
        }
        if (sl < 0 || sl >= nslots) {  // a corrupt range is reported, never followed
            if (lane == 0) atomicOr(err, 1);
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        const D4 X = xyzm[sl], X2 = aux[sl];
        const int2 K = kids[sl];
        bool open = false;
        if (m & me) {
            visits++;
            const double dx = X.x - px, dy = X.y - py, dz = X.z - pz;
            const Across a(dx, dy, dz, rx, ry, rz);
            const double r = sqrt(a.r2), z = a.z, b2 = a.b2;
            if (!(b2 < 0)) {  // rounding below zero: skipped, as ColumnDensityWalk_singleray does
                const double h_no = X2.x;
                if (K.y == 0) {
                    if (h_no > 0) {  // a zero radius has no cross-section
                        const double hinv = 1.0 / h_no;
                        const double fac = fac_density * X.w * hinv * hinv;
                        const double r_proj = sqrt(b2);
                        const double q = r_proj * hinv;
                        if (r_proj < h_no) {
                            if (r > h_no) {
                                if (z > 0) column += fac * 2 * sqrt(1 - q * q);
                            } else {
                                column += fac * (z * hinv + sqrt(1 - q * q));
                            }
                        }
                    }
                } else {
                    const double reach = h_no + X2.y * 0.8660254037844386 + X2.z;
                    open = r < reach;
                    if (!open && z > 0) open = b2 < reach * reach;
                }
            }
        }
        const uint64_t mo = ptg_ballot(open);
        if (mo && K.y > 0) {
            if (top + 1 >= CR_DEPTH) {  // deeper than the stack: the caller reruns the stackless walk
                if (lane == 0) atomicOr(err, 2);
                break;
            }
            top++;
            if (lane == 0) {
                S.s[top] = K.x;
                S.c[top] = std::min(K.y, 8);
                S.m[top] = mo;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (live) out[j * nr + i] = column;
    if (ctr) cd_count(ctr, 0, visits);
}

// ---- ray-traced walk of bundles: 64 targets that neighbour each other across one shared ray ----
// One wavefront walks the tree once for its bundle, 64 elements per step (one per lane): an element is
// opened or listed when it could meet any of the bundle's rays, tested in coordinates across the ray
// against the bundle's rectangle, and, where the rectangle is wide against the element's reach, against
// four quarter bundles' rectangles and then their targets one by one.  Listed particles are evaluated for
// all 64 targets by the chord formulae of the per-target walk.  A superset of each target's own path is
// walked, so every particle its ray crosses is met; the others add nothing.
//
// Bound: instruction issue (about 14 FP64 instructions per listed particle, 200 per step) and, in
// launches of few bundles, the chain of loads per step.  Six axis rays of 1e5 targets in a Gaussian
// cloud: 8.3 -> 0.85 ms against one element per step for all lanes (k_column_rays_wave, still the walk
// of per-target rays, whose bundles are not parallel).
#define CN_WAVES 4
#define CN_SCAP 1024  // LDS stack; near its top a step takes fewer elements, so it needs no spill
#define CN_LIST 32    // the list is evaluated in multiples of CN_LIST
#define CN_ICAP (CN_LIST + 64)
#define CN_WIDE 4.0   // a rectangle wider than CN_WIDE reaches is refined: 1.60 ms against 1.70 at 1, 11.8 if never

struct CnLds {
    int stack[CN_SCAP];
    D4 part[CN_ICAP];     // x, y, z and the weight 3 m / (4 pi h^2)
    double h[CN_ICAP], hinv[CN_ICAP];
    double a[64], b[64];  // the targets across the ray
};

__device__ __forceinline__ double cn_sqrt(double x) { return x > 0.0 ? x * ptg_rsqrt64(x) : 0.0; }

__device__ __forceinline__ void cn_flush(const CnLds &S, int c, double px, double py, double pz, double rx, double ry,
                                         double rz, double &column)
{
    for (int k = 0; k < c; k++) {
        const D4 P = S.part[k];
        const double h = S.h[k];
        const double dx = P.x - px, dy = P.y - py, dz = P.z - pz;
        const Across e(dx, dy, dz, rx, ry, rz);
        const double b2 = e.b2, z = e.z, hh = h * h;
        // b2 < 0 by rounding: skipped, as ColumnDensityWalk_singleray does
        const bool inside = !(e.r2 > hh);
        if (b2 >= 0 && b2 < hh && (inside || z > 0)) {
            const double hinv = S.hinv[k];
            const double half = cn_sqrt(1.0 - b2 * (hinv * hinv));
            column += P.w * (inside ? z * hinv + half : 2.0 * half);
        }
    }
}

__global__ __launch_bounds__(64 * CN_WAVES) __attribute__((amdgpu_waves_per_eu(4))) void k_column_bundles(const D4 *xyzm, const D4 *aux, const int2 *kids,
                                                                  int64_t nslots, const double *tp, int64_t nt,
                                                                  const double *rays, int64_t nr, const int64_t *order,
                                                                  double *out, int32_t *err)
{
    __shared__ CnLds lds[CN_WAVES];
    const int wave = threadIdx.x >> 6, lane = ptg_lane();
    CnLds &S = lds[wave];
    const int64_t ntb = (nt + 63) / 64;
    // contiguous runs of bundles per XCD (block b runs on XCD b mod 8; the grid is a multiple of 8): neighbours share their paths in its L2
    const int64_t per = gridDim.x / 8, blk = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int64_t task = blk * CN_WAVES + wave;
    if (task >= ntb * nr) return;  // whole wavefronts only: task is uniform
    const int64_t i = task / ntb, jr = (task % ntb) * 64 + lane;
    const bool live = jr < nt;
    const int64_t jl = live ? jr : nt - 1;  // idle lanes repeat the last target
    const int64_t j = order ? order[i * nt + jl] : jl;
    const double rx = rays[3 * i], ry = rays[3 * i + 1], rz = rays[3 * i + 2];
    const double px = tp[3 * j], py = tp[3 * j + 1], pz = tp[3 * j + 2];
    // A ray that is not of unit length has no geometry to bundle by: its columns are what the formulae give along
    // each target's own walk, which the caller makes.
    if (!(fabs(rx * rx + ry * ry + rz * rz - 1.0) < 1e-13)) {
        if (lane == 0) atomicOr(err, 4);
        return;
    }
    // frame of the bundle: origin at its first finite target, e1 and e2 across the ray, e3 along it
    const bool fin = isfinite(px) && isfinite(py) && isfinite(pz);  // others see no column and bound nothing
    const uint64_t mf = ptg_ballot(fin);
    const int ol = mf ? (int)__ffsll((unsigned long long)mf) - 1 : 0;
    const double ox = __shfl(px, ol, 64), oy = __shfl(py, ol, 64), oz = __shfl(pz, ol, 64);
    const double ax = fabs(rx) < 0.9 ? 1.0 : 0.0, ay = 1.0 - ax;
    double e1x = -rz * ay, e1y = rz * ax, e1z = rx * ay - ry * ax;
    const double en = 1.0 / sqrt(e1x * e1x + e1y * e1y + e1z * e1z);
    e1x *= en;
    e1y *= en;
    e1z *= en;
    const double e2x = ry * e1z - rz * e1y, e2y = rz * e1x - rx * e1z, e2z = rx * e1y - ry * e1x;
    const double qx = fin ? px - ox : 0.0, qy = fin ? py - oy : 0.0, qz = fin ? pz - oz : 0.0;
    const double ta = e1x * qx + e1y * qy + e1z * qz, tb = e2x * qx + e2y * qy + e2z * qz;
    const double tc = rx * qx + ry * qy + rz * qz;
    S.a[lane] = ta;
    S.b[lane] = tb;
    // rectangles of the quarters (lanes 16 s .. 16 s + 15) and of the bundle, and its nearest start
    double alo = ta, ahi = ta, blo = tb, bhi = tb;
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        alo = fmin(alo, __shfl_xor(alo, d, 64));
        ahi = fmax(ahi, __shfl_xor(ahi, d, 64));
        blo = fmin(blo, __shfl_xor(blo, d, 64));
        bhi = fmax(bhi, __shfl_xor(bhi, d, 64));
    }
    const double qalo = alo, qahi = ahi, qblo = blo, qbhi = bhi;
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) {
        alo = fmin(alo, __shfl_xor(alo, d, 64));
        ahi = fmax(ahi, __shfl_xor(ahi, d, 64));
        blo = fmin(blo, __shfl_xor(blo, d, 64));
        bhi = fmax(bhi, __shfl_xor(bhi, d, 64));
    }
    const double clo = ptg_wave_min(tc);
    const double side = fmax(ahi - alo, bhi - blo);
    const double tmax = fmax(fmax(fabs(alo), fabs(ahi)), fmax(fabs(blo), fabs(bhi)));
    const double fac_density = 3.0 / (4.0 * 3.14159265358979323846);
    double column = 0.0;
    int sp = 1, np = 0;
    if (lane == 0) S.stack[0] = 0;  // the root's walk slot
    __builtin_amdgcn_wave_barrier();
    while (sp > 0) {
        // 64 elements, or as many as the stack has room for the children of
        const int k = std::min(std::min(sp, 64), (CN_SCAP - sp) / 7);
        if (k < 1) {  // deeper than the stack: the caller makes the targets' own walks
            if (lane == 0) atomicOr(err, 2);
            break;
        }
        const int base = sp - k;
        int e = lane < k ? S.stack[base + lane] : 0;
        const bool ve = lane < k && e >= 0 && e < nslots;
        if (lane < k && !ve) atomicOr(err, 1);  // a corrupt link is reported, never followed
        if (!ve) e = 0;
        __builtin_amdgcn_wave_barrier();
        sp = base;
        const D4 X = xyzm[e], X2 = aux[e];
        const int2 K = kids[e];
        const bool ispart = K.y == 0;
        const double dx = X.x - ox, dy = X.y - oy, dz = X.z - oz;
        const double ea = e1x * dx + e1y * dy + e1z * dz, eb = e2x * dx + e2y * dy + e2z * dz;
        const double ec = rx * dx + ry * dy + rz * dz;
        // the coordinates above and the targets' carry a few 2^-53 of the distances: 1e-14 covers them
        double reach = ispart ? X2.x : X2.x + X2.y * 0.8660254037844386 + X2.z;
        reach += 1e-14 * (fabs(dx) + fabs(dy) + fabs(dz) + tmax);
        const double rr = reach * reach;
        const double ga = box_gap(ea, alo, ahi), gb = box_gap(eb, blo, bhi);
        bool hit = ve & (ga * ga + gb * gb <= rr) & (ec + reach > clo) & (!ispart | (X2.x > 0.0));
        if (ptg_ballot(hit & (side > CN_WIDE * reach))) {
            bool any = !(side > CN_WIDE * reach);
            for (int q = 0; q < 4; q++) {
                const double l0 = __shfl(qalo, 16 * q, 64), l1 = __shfl(qahi, 16 * q, 64);
                const double m0 = __shfl(qblo, 16 * q, 64), m1 = __shfl(qbhi, 16 * q, 64);
                const double a2 = box_gap(ea, l0, l1), b2 = box_gap(eb, m0, m1);
                bool near = hit & !any & (a2 * a2 + b2 * b2 <= rr);
                if (ptg_ballot(near & (fmax(l1 - l0, m1 - m0) > CN_WIDE * reach))) {
                    bool one = !(fmax(l1 - l0, m1 - m0) > CN_WIDE * reach);
                    for (int t = 16 * q; t < 16 * q + 16; t++) {
                        const double da = ea - S.a[t], db = eb - S.b[t];
                        one |= da * da + db * db <= rr;
                    }
                    near &= one;
                }
                any |= near;
            }
            hit &= any;
        }
        const bool list = hit & ispart;
        const uint64_t bl = ptg_ballot(list);
        if (list) {
            const int at = np + lanes_below(bl);
            const double hinv = 1.0 / X2.x;
            S.part[at] = D4{X.x, X.y, X.z, fac_density * X.w * hinv * hinv};
            S.h[at] = X2.x;
            S.hinv[at] = hinv;
        }
        np += (int)__popcll(bl);
        const int cnt = hit & !ispart ? std::min(std::max(K.y, 0), 8) : 0;
        int tot;
        const int below = small_excl_scan(cnt, tot);
        {
            int *dst = &S.stack[sp + below];
#pragma unroll
            for (int c = 0; c < 8; c++)
                if (c < cnt) dst[c] = K.x + c;
        }
        sp += tot;
        __builtin_amdgcn_wave_barrier();
        if (np >= CN_LIST) {
            const int c = np & ~(CN_LIST - 1);
            cn_flush(S, c, px, py, pz, rx, ry, rz, column);
            __builtin_amdgcn_wave_barrier();
            if (lane < np - c) {  // reads [c, np) and writes [0, np - c): disjoint
                S.part[lane] = S.part[c + lane];
                S.h[lane] = S.h[c + lane];
                S.hinv[lane] = S.hinv[c + lane];
            }
            __builtin_amdgcn_wave_barrier();
            np -= c;
        }
    }
    cn_flush(S, np, px, py, pz, rx, ry, rz, column);
    if (live) out[j * nr + i] = column;
}

// angular_bin_scalar (treewalk.py:38-45)
__device__ __forceinline__ int cd_bin(double d0, double d1, double d2)
{
    if (fabs(d0) > fabs(d1) && fabs(d0) > fabs(d2)) return d0 > 0 ? 0 : 1;
    if (fabs(d1) > fabs(d2)) return d1 > 0 ? 2 : 3;
    return d2 > 0 ? 4 : 5;
}

__global__ __launch_bounds__(CD_THREADS) void k_column_binned(const ptg_tree_arrays t, int64_t n, int64_t ne,
                                                              const double *tp, int64_t nt, int64_t gs, double theta,
                                                              double *out, int32_t *err, unsigned long long *ctr)
{
    const int64_t gi = (int64_t)blockIdx.x * CD_THREADS + threadIdx.x;
    const int64_t a = gi * gs;
    if (a >= nt) return;
    const int64_t b = std::min(a + gs, nt);
    const double bin_size = (4.0 * 3.14159265358979323846) / 6.0;
    double bmin0 = tp[3 * a], bmin1 = tp[3 * a + 1], bmin2 = tp[3 * a + 2];
    double bmax0 = bmin0, bmax1 = bmin1, bmax2 = bmin2;
    for (int64_t j = a + 1; j < b; j++) {
        bmin0 = fmin(bmin0, tp[3 * j]);
        bmax0 = fmax(bmax0, tp[3 * j]);
        bmin1 = fmin(bmin1, tp[3 * j + 1]);
        bmax1 = fmax(bmax1, tp[3 * j + 1]);
        bmin2 = fmin(bmin2, tp[3 * j + 2]);
        bmax2 = fmax(bmax2, tp[3 * j + 2]);
    }
    for (int64_t j = a; j < b; j++)
        for (int k = 0; k < 6; k++) out[6 * j + k] = 0.0;
    int64_t no = n, visits = 0, pairs = 0;
    const int64_t stop = t.next_branch[n];
    while (no > -1 && no != stop) {
        if (cd_bad(no, ne, visits)) {
            atomicOr(err, 1);
            break;
        }
        const double cx = t.coordinates[3 * no], cy = t.coordinates[3 * no + 1], cz = t.coordinates[3 * no + 2];
        const double h_no = t.softenings[no], M = t.masses[no];
        if (no < n) {  // a particle contributes to every target of the group, no criterion
            pairs += b - a;
            const double hh = h_no * h_no;
            for (int64_t j = a; j < b; j++) {
                const double d0 = cx - tp[3 * j], d1 = cy - tp[3 * j + 1], d2 = cz - tp[3 * j + 2];
                const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
                const int bin = cd_bin(d0, d1, d2);
                double *o = out + 6 * j;
                if (r2 > hh) {  // no overlap: a point mass at distance sqrt(r2)
                    o[bin] += M / r2 / bin_size;
                } else if (h_no > 0) {  // overlap: blend of the isotropic and directed limits
                    const double col0 = M * (3 / (4 * 3.14159265358979323846 * hh));
                    const double fac = sqrt(r2) / h_no;
                    const double col_iso = (1 - fac) * col0;
                    for (int k = 0; k < 6; k++) o[k] += col_iso;
                    o[bin] += col0 * fac * 2;
                }
            }
            no = t.next_branch[no];
        } else {
            // the reference's opening test (treewalk.py:22-25) at the node's distance to the box
            const double dxm = cx < bmin0 ? bmin0 - cx : (cx > bmax0 ? cx - bmax0 : 0.0);
            const double dym = cy < bmin1 ? bmin1 - cy : (cy > bmax1 ? cy - bmax1 : 0.0);
            const double dzm = cz < bmin2 ? bmin2 - cz : (cz > bmax2 ? cz - bmax2 : 0.0);
            const double r_min = sqrt(dxm * dxm + dym * dym + dzm * dzm);
            const double size = t.sizes[no], delta = t.deltas[no];
            const double c1 = size / theta + delta, c2 = h_no + size * 0.6 + delta;
            if (r_min > (c1 > c2 ? c1 : c2)) {
                pairs += b - a;
                for (int64_t j = a; j < b; j++) {
                    const double d0 = cx - tp[3 * j], d1 = cy - tp[3 * j + 1], d2 = cz - tp[3 * j + 2];
                    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
                    out[6 * j + cd_bin(d0, d1, d2)] += M / r2 / bin_size;
                }
                no = t.next_branch[no];
            } else {
                no = t.first_subnode[no];
            }
        }
    }
    if (ctr) {
        atomicAdd(ctr, (unsigned long long)pairs);
        atomicAdd(ctr + 1, (unsigned long long)visits);
    }
}


// ---- wavefront-per-group binned walk: k_walk64's traversal (walk64.hip) with six sums per target ----
// global spill entries per wave: a step leaves at most 448 a level, so 36 levels of a tree all of whose nodes are
// opened; a tree whose keys collide has up to 84
#define CB_GCAP 16384

static int cb_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    return cus;
}

// workspace: the walk's control block, the spill stacks of three blocks per CU, the deferral pool
extern "C" size_t ptg_column_workspace_bytes(int64_t group_size)
{
    (void)group_size;
    return walk_control_bytes() + (size_t)cb_cus() * 3 * WALK_WAVES * CB_GCAP * sizeof(int) + WALK_POOL;
}

// the walk's flags as ptg_column_binned reports them
__global__ void k_column_err_out(const WalkCtl *ctl, int32_t *err)
{
    if (ctl->err & 1) *err |= 2;  // a traversal stack overflow
    if (ctl->err & 8) *err |= 4;  // the task pass gave up
}
__global__ void k_column_err_init(int32_t *err) { *err = 0; }
static ptg_status column_common(const ptg_tree_arrays *tree, int64_t n, int64_t nnodes, const double *targets,
                                int64_t nt, const char *who)
{
    if (!tree || !tree->coordinates || !tree->masses || !tree->softenings || !tree->sizes || !tree->deltas ||
        !tree->first_subnode || !tree->next_branch || n < 1 || nnodes < 1 || nt < 0 || (nt > 0 && !targets)) {
        ptg_set_error("%s: bad arguments", who);
        return PTG_ERR_ARG;
    }
    return PTG_OK;
}

extern "C" ptg_status ptg_column_rays(const ptg_tree_arrays *tree, int64_t n, int64_t nnodes,
                                      const ptg_walk_tree *wt, const double *targets, int64_t nt, const double *rays,
                                      int64_t nrays, int per_target, const int64_t *order, double *out, int32_t *err,
                                      int64_t *counters, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    ptg_status st = column_common(tree, n, nnodes, targets, nt, "ptg_column_rays");
    if (st) return st;
    if (nrays < 1 || !rays || !out || !err) {
        ptg_set_error("ptg_column_rays: needs nrays >= 1, rays, out and err");
        return PTG_ERR_ARG;
    }
    k_column_err_init<<<1, 1, 0, s>>>(err);
    PTG_LAUNCH_CHECK();
    const int64_t work = nt * nrays;
    if (work == 0) return PTG_OK;
    if (wt) {
        if (wt->prec != PTG_F64 || !wt->xyzm || !wt->aux || !wt->kids || wt->nslots != n + nnodes) {
            ptg_set_error("ptg_column_rays: wt must be the FP64 walk pack of the tree (or NULL)");
            return PTG_ERR_ARG;
        }
        const int64_t tasks = ptg_cdiv(nt, 64) * nrays;
        k_column_rays_wave<<<(unsigned)ptg_cdiv(tasks, CR_WAVES), 64 * CR_WAVES, 0, s>>>(
            (const D4 *)wt->xyzm, (const D4 *)wt->aux, (const int2 *)wt->kids, wt->nslots, targets, nt, rays, nrays,
            per_target != 0, order, out, err, (unsigned long long *)counters);
        PTG_LAUNCH_CHECK();
        return PTG_OK;
    }
    k_column_rays<<<(unsigned)ptg_cdiv(work, CD_THREADS), CD_THREADS, 0, s>>>(*tree, n, n + nnodes, targets, nt, rays,
                                                                              nrays, per_target != 0, out, err,
                                                                              (unsigned long long *)counters);
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

extern "C" ptg_status ptg_column_bundles(const ptg_walk_tree *wt, const double *targets, int64_t nt, const double *rays,
                                         int64_t nrays, const int64_t *order, double *out, int32_t *err, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    if (!wt || wt->prec != PTG_F64 || !wt->xyzm || !wt->aux || !wt->kids || wt->nslots < 1 || nt < 0 || nrays < 1 ||
        !rays || !out || !err || (nt > 0 && !targets)) {
        ptg_set_error("ptg_column_bundles: needs the FP64 walk pack, targets, nrays >= 1, rays, out and err");
        return PTG_ERR_ARG;
    }
    k_column_err_init<<<1, 1, 0, s>>>(err);
    PTG_LAUNCH_CHECK();
    if (nt == 0) return PTG_OK;
    const int64_t blocks = ptg_cdiv(ptg_cdiv(nt, 64) * nrays, CN_WAVES);
    if (blocks > 0x7ffffff8LL) {
        ptg_set_error("ptg_column_bundles: too many (target, ray) pairs for one launch");
        return PTG_ERR_ARG;
    }
    k_column_bundles<<<(unsigned)((blocks + 7) / 8 * 8), 64 * CN_WAVES, 0, s>>>(
        (const D4 *)wt->xyzm, (const D4 *)wt->aux, (const int2 *)wt->kids, wt->nslots, targets, nt, rays, nrays, order,
        out, err);
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

/* Randomized ray grids (treewalk.py:1061-1078 with misc.py:6-54): target k sees the grid rotated by
 * the rotation drawn from a Mersenne-Twister stream seeded with k.  Four doubles are drawn, i.e. the
 * first eight 32-bit outputs of MT19937 after its integer seeding, so a thread needs only state
 * words 0..8 and 397..404 of the seeded table: the first twist combines word i, i+1 and i+397.
 * Each double is the 53-bit (a >> 5, b >> 6) combination of two outputs, as numpy's legacy
 * generator and numba's draw it; uniform(lo, hi) = lo + (hi - lo) * u. */
#define MT_M 397
#define MT_NEED 9 // words 0..8 of the table, and 397..404

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

__global__ void __launch_bounds__(256) k_random_rotations(int64_t first_seed, int64_t nt, const double *__restrict__ rays,
                                                          int nrays, double *__restrict__ out)
{
#pragma clang fp contract(off) // the host's rounding: no fused multiply-adds
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nt) return;
    uint32_t lo[MT_NEED], hi[MT_NEED - 1];
    uint32_t s = (uint32_t)(first_seed + k);
    // integer seeding: word i = 1812433253 * (word(i-1) ^ word(i-1) >> 30) + i
    for (int i = 0; i < MT_M + MT_NEED - 1; ++i) {
        if (i < MT_NEED) lo[i] = s;
        if (i >= MT_M) hi[i - MT_M] = s;
        s = 1812433253u * (s ^ (s >> 30)) + (uint32_t)(i + 1);
    }
    double u[4];
    for (int d = 0; d < 4; ++d) {
        uint32_t w[2];
        for (int q = 0; q < 2; ++q) {
            const int i = 2 * d + q;
            const uint32_t y = (lo[i] & 0x80000000u) | (lo[i + 1] & 0x7fffffffu);
            w[q] = mt_temper(hi[i] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u));
        }
        u[d] = ((double)(w[0] >> 5) * 67108864.0 + (double)(w[1] >> 6)) / 9007199254740992.0;
    }
    double R[3][3];
    for (int row = 0; row < 2; ++row) {
        const double c = -1.0 + 2.0 * u[2 * row];
        const double sn = sqrt(fmax(1.0 - c * c, 0.0));
        const double phi = 2.0 * M_PI * (0.0 + 1.0 * u[2 * row + 1]);
        R[row][0] = sn * cos(phi);
        R[row][1] = sn * sin(phi);
        R[row][2] = c;
    }
    double dot = 0.0;
    for (int c = 0; c < 3; ++c) dot += R[0][c] * R[1][c];
    for (int c = 0; c < 3; ++c) R[1][c] -= dot * R[0][c];
    double nrm = 0.0;
    for (int c = 0; c < 3; ++c) nrm += R[1][c] * R[1][c];
    nrm = sqrt(nrm);
    for (int c = 0; c < 3; ++c) R[1][c] /= nrm;
    for (int c = 0; c < 3; ++c) {
        const int a = (c + 1) % 3, b = (c + 2) % 3;
        R[2][c] = R[0][a] * R[1][b] - R[1][a] * R[0][b];
    }
    double *o = out + k * nrays * 3;
    for (int j = 0; j < nrays; ++j)
        for (int c = 0; c < 3; ++c)
            o[j * 3 + c] = rays[j * 3] * R[0][c] + rays[j * 3 + 1] * R[1][c] + rays[j * 3 + 2] * R[2][c];
}

extern "C" ptg_status ptg_random_rotations(int64_t first_seed, int64_t nt, const double *rays, int64_t nrays,
                                           double *out, void *stream)
{
    if (nt < 0 || nrays < 1 || nrays > (1 << 20) || !rays || (nt > 0 && !out) || first_seed < 0 ||
        first_seed + nt > (1ll << 32)) {
        ptg_set_error("ptg_random_rotations: needs 0 <= first_seed, first_seed + nt <= 2^32, 1 <= nrays <= 2^20, "
                      "rays and out");
        return PTG_ERR_ARG;
    }
    if (nt == 0) return PTG_OK;
    k_random_rotations<<<(unsigned)ptg_cdiv(nt, 256), 256, 0, (hipStream_t)stream>>>(first_seed, nt, rays, (int)nrays,
                                                                                     out);
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

extern "C" ptg_status ptg_column_binned(const ptg_tree_arrays *tree, int64_t n, int64_t nnodes,
                                        const ptg_walk_tree *wt, const double *targets, int64_t nt,
                                        int64_t group_size, double theta, double *out, int32_t *err, void *ws,
                                        size_t ws_bytes, int64_t *counters, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    ptg_status st = column_common(tree, n, nnodes, targets, nt, "ptg_column_binned");
    if (st) return st;
    if (group_size < 1 || !(theta > 0) || !out || !err) {
        ptg_set_error("ptg_column_binned: needs group_size >= 1, theta > 0, out and err");
        return PTG_ERR_ARG;
    }
    k_column_err_init<<<1, 1, 0, s>>>(err);
    PTG_LAUNCH_CHECK();
    if (nt == 0) return PTG_OK;
    if (group_size <= 64) {
        if (!wt || wt->prec != PTG_F64 || !wt->xyzm || !wt->aux || !wt->kids || wt->nslots != n + nnodes || !ws ||
            ws_bytes < ptg_column_workspace_bytes(group_size) || n + nnodes >= (1ll << 28)) {
            ptg_set_error("ptg_column_binned: group_size <= 64 needs the FP64 walk pack of the tree (fewer than "
                          "2^28 elements) and ptg_column_workspace_bytes(group_size) of workspace");
            return PTG_ERR_ARG;
        }
        WalkCtl *ctl = (WalkCtl *)ws;
        st = walk_clear(ctl, ptg_cdiv(nt, group_size), WALK_AGAIN, s);
        if (st) return st;
        const Walk64Args a{(const V4<double> *)wt->xyzm, (const V4<double> *)wt->aux, (const int2 *)wt->kids, nullptr,
                           targets, nullptr, nullptr, 1, wt->nslots, nt, ptg_cdiv(nt, group_size), nullptr, nullptr,
                           (int)group_size, theta, 1.0 / theta, 6.0 / (4.0 * 3.14159265358979323846), 0.0, 0.0, 0.0, 0,
                           nullptr, out, counters, ctl, nullptr};
        st = ptg_walk64_bins(a, cb_cus(), CB_GCAP, WALK_AGAIN, (char *)ws, ws_bytes, s);
        if (st) return st;
        k_column_err_out<<<1, 1, 0, s>>>(ctl, err);
        PTG_LAUNCH_CHECK();
        return PTG_OK;
    }
    const int64_t ngroups = ptg_cdiv(nt, group_size);
    k_column_binned<<<(unsigned)ptg_cdiv(ngroups, CD_THREADS), CD_THREADS, 0, s>>>(*tree, n, n + nnodes, targets, nt,
                                                                                   group_size, theta, out, err,
                                                                                   (unsigned long long *)counters);
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}
