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

#define WALK_ROUNDS 5  // FP64 walk: the group pass and the passes over the subtrees it deferred

struct WalkCtl {
    int32_t ctr[NXCD * CTR_STRIDE];   // per-XCD group counters
    int32_t err;
    int32_t hwm;  // deepest global spill stack (entries) any wave reached in the last walk
    int32_t pad[30];
    // FP64 walk: entries of the task tables (deferred groups, then the tasks of rounds 1, 2, ..), stack
    // entries saved, per-XCD counters of the tasks taken
    int32_t ntask[WALK_ROUNDS], npool, pad2[31 - WALK_ROUNDS];
    int32_t tctr[(WALK_ROUNDS - 1) * NXCD * CTR_STRIDE];
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
