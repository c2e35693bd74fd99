// Direct summation (bruteforce.py).  FP64 is the oracle-grade path used to measure tree errors; FP32 is
// the fast brute-force method.
//
// A block holds P targets (a power of two) and splits the sources over its 16 waves and over the
// 64 / P slices of each wave's lanes: few targets still fill the chip, each lane of a 1000-target call
// summing a few sources.  A wave converts 64 sources at a time into its own LDS tile; its lanes read one
// entry each slice (broadcast).  The common pair, farther than every softening radius, takes one
// reciprocal square root; four pairs are tested together, and only where one lane is closer (or a
// distance is not an ordinary number) are its pairs evaluated by the reference's branches.  Partial sums
// are added in a fixed order, so results do not depend on scheduling.
//
// Bound: VALU (FP32 accelerations: 13 arithmetic instructions a pair of about 18 issue slots; FP64 38 slots).
// One Accel call against one lane per target over scalar-loaded sources with IEEE square roots and divisions:
// FP32 12007 particles 312 -> 85 us (the kernel 73), 1e5 11.0 -> 4.4 ms (2.3e12 pairs/s); FP64 4000 particles
// 124 -> 26 us (host bound), 1e5 17.2 -> 10.0 ms.  Against an extended-precision sum its errors are that kernel's or
// smaller (FP64 1.5e-16 to 5e-13, FP32 6e-8 to 1e-6; FP32 tidal tensors within the summation noise of it).
#include <algorithm>

#include "ptg_common.hpp"

#define DS_WAVES 16
#define DS_TILE 64   // sources per wave tile
#define DS_UNROLL 4  // pairs tested together (<= the smallest P)

template <typename T> __device__ __forceinline__ T d_force_kernel(T r, T h)
{
    if (r > h) return T(1) / (r * r * r);
    T hinv = T(1) / h;
    T q = r * hinv;
    if (q <= T(0.5)) return (T(10.666666666666666666) + q * q * (T(-38.4) + T(32.0) * q)) * hinv * hinv * hinv;
    return (T(21.333333333333) - T(48.0) * q + T(38.4) * q * q - T(10.666666666667) * q * q * q -
            T(0.066666666667) / (q * q * q)) *
           hinv * hinv * hinv;
}

template <typename T> __device__ __forceinline__ T d_tidal_kernel(T r, T h)
{
    if (r > h) {
        T r2 = r * r;
        return T(3) / (r2 * r2 * r);
    }
    T hinv = T(1) / h;
    T hinv2 = hinv * hinv;
    T hinv5 = hinv2 * hinv2 * hinv;
    T q = r * hinv;
    if (q <= T(0.5)) return (T(76.8) - T(96.0) * q) * hinv5;
    T qinv = T(1) / q;
    T qinv3 = qinv * qinv * qinv;
    return (T(48.0) * qinv - T(76.8) + T(32.0) * q - T(0.2) * qinv3 * qinv * qinv) * hinv5;
}

template <typename T> __device__ __forceinline__ T d_potential_kernel(T r, T h)
{
    if (h == T(0)) return T(-1) / r;
    T hinv = T(1) / h;
    T q = r * hinv;
    if (q <= T(0.5)) return (T(-2.8) + q * q * (T(5.33333333333333333) + q * q * (T(6.4) * q - T(9.6)))) * hinv;
    if (q <= T(1))
        return (T(-3.2) + T(0.066666666666666666666) / q +
                q * q * (T(10.666666666666666666666) + q * (T(-16.0) + q * (T(9.6) - T(2.1333333333333333333333) * q)))) *
               hinv;
    return T(-1) / r;
}

template <typename T> struct alignas(4 * sizeof(T)) DV4 {
    T x, y, z, w;
};

// 1/sqrt(x): the hardware's in FP32 (1 ulp)
__device__ __forceinline__ float d_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double d_rsqrt(double x) { return ptg_rsqrt64(x); }

// The plain path takes squared distances from the smallest ordinary number (below, the hardware's
// reciprocal square root may flush them) and, in FP64, up to 1e300 (its step is nan at infinity, where
// the FP32 instruction gives the division's 0).
template <typename T> struct Plain;
template <> struct Plain<float> {
    static constexpr float lo = 1.17549435e-38f;
};
template <> struct Plain<double> {
    static constexpr double lo = 2.2250738585072014e-308;
};

template <typename T, int FIELDS> struct DAcc {
    static constexpr bool P = FIELDS & PTG_POT, A = FIELDS & PTG_ACC, D = FIELDS & PTG_TIDAL;
    static constexpr int W = (P ? 1 : 0) + (A ? 3 : 0) + (D ? 6 : 0);  // sums (tidal: 6 independent)
    T s[W];

    __device__ __forceinline__ void add(T phi, T K, T Q, T dx, T dy, T dz)
    {
        int c = 0;
        if (P) s[c++] += phi;
        if (A) {
            s[c++] += K * dx;
            s[c++] += K * dy;
            s[c++] += K * dz;
        }
        if (D) {
            const T qx = Q * dx, qy = Q * dy;
            s[c++] += qx * dx - K;
            s[c++] += qx * dy;
            s[c++] += qx * dz;
            s[c++] += qy * dy - K;
            s[c++] += qy * dz;
            s[c++] += Q * dz * dz - K;
        }
    }
};

// one pair by the reference's branches (bruteforce.py), unless skip: source and target are the same particle, or the
// entry is past the slice (its 0 mass would make a nan of a singular pair)
template <typename T, int FIELDS, bool SELF>
__device__ __forceinline__ void pair_branches(DAcc<T, FIELDS> &a, T dx, T dy, T dz, T r2, T m, T h, bool skip)
{
    constexpr bool P = DAcc<T, FIELDS>::P, A = DAcc<T, FIELDS>::A, D = DAcc<T, FIELDS>::D;
    if (skip) return;
    const T r = sqrt(r2);
    T phi = 0, K = 0, Q = 0;
    if (P) {
        if (SELF) {  // bruteforce.py:110-115: coincident distinct particles keep the softened term
            if (r < h) phi = m * d_potential_kernel(r, h);
            else if (r > T(0)) phi = -m / r;
        } else if (r != T(0)) {
            phi = r < h ? m * d_potential_kernel(r, h) : -m / r;
        }
    }
    if ((A || D) && r2 != T(0)) {
        if (r < h) {
            K = m * d_force_kernel(r, h);
            if (D) Q = m * d_tidal_kernel(r, h);
        } else {
            K = m / (r2 * r);
            if (D) Q = T(3) * K / r2;
        }
    }
    a.add(phi, K, Q, dx, dy, dz);
}

template <typename T, int FIELDS, bool SELF, int P>
__global__ __launch_bounds__(64 * DS_WAVES) void k_direct(const double *pt, const double *ht, int64_t nt,
                                                          const double *ps, const double *ms, const double *hs,
                                                          int64_t ns, double G, double *out)
{
    constexpr int W = DAcc<T, FIELDS>::W, S = 64 / P;
    struct Tile {
        DV4<T> s[DS_TILE];  // x, y, z, m
        T h2[DS_TILE], h[DS_TILE];
    };
    __shared__ union {
        Tile tile[DS_WAVES];
        T part[DS_WAVES][W][P];
    } lds;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = ptg_lane();
    const int tl = lane & (P - 1), sl = lane / P;
    const int64_t i = (int64_t)blockIdx.x * P + tl;
    const int64_t ic = i < nt ? i : nt - 1;  // lanes past the targets repeat the last one
    const T tx = (T)pt[3 * ic], ty = (T)pt[3 * ic + 1], tz = (T)pt[3 * ic + 2], th = (T)ht[ic];
    const T th2 = std::max(th * th, Plain<T>::lo);
    Tile &L = lds.tile[wave];
    DAcc<T, FIELDS> acc;
#pragma unroll
    for (int c = 0; c < W; c++) acc.s[c] = T(0);
    const int64_t j0 = ns * wave / DS_WAVES, j1 = ns * (wave + 1) / DS_WAVES;
    for (int64_t jt = j0; jt < j1; jt += DS_TILE) {
        {
            // entries past the slice are massless copies of its last source
            const int64_t j = jt + lane < j1 ? jt + lane : j1 - 1;
            L.s[lane] = DV4<T>{(T)ps[3 * j], (T)ps[3 * j + 1], (T)ps[3 * j + 2], jt + lane < j1 ? (T)ms[j] : T(0)};
            const T h = (T)hs[j];
            L.h[lane] = h;
            L.h2[lane] = h * h;
        }
        __builtin_amdgcn_wave_barrier();
        const int cnt = (int)std::min<int64_t>(DS_TILE, j1 - jt);
        for (int k = 0; k < cnt; k += S * DS_UNROLL) {
            T dx[DS_UNROLL], dy[DS_UNROLL], dz[DS_UNROLL], r2[DS_UNROLL], m[DS_UNROLL];
            uint64_t odd = 0;  // lanes with a pair off the plain path (a nan too)
#pragma unroll
            for (int u = 0; u < DS_UNROLL; u++) {
                const int q = k + u * S + sl;
                const DV4<T> s = L.s[q];
                m[u] = s.w;
                dx[u] = s.x - tx;
                dy[u] = s.y - ty;
                dz[u] = s.z - tz;
                r2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
                odd |= ptg_ballot(!(r2[u] >= L.h2[q])) | ptg_ballot(!(r2[u] >= th2));
                if (sizeof(T) == 8) odd |= ptg_ballot(r2[u] > T(1e300));
            }
            if (odd == 0) {
#pragma unroll
                for (int u = 0; u < DS_UNROLL; u++) {
                    const T rinv = d_rsqrt(r2[u]), rinv2 = rinv * rinv;
                    const T mr = m[u] * rinv, K = mr * rinv2;
                    acc.add(-mr, K, T(3) * K * rinv2, dx[u], dy[u], dz[u]);
                }
            } else {
#pragma unroll 1
                for (int u = 0; u < DS_UNROLL; u++) {
                    const int q = k + u * S + sl;
                    const DV4<T> s = L.s[q];
                    const T ex = s.x - tx, ey = s.y - ty, ez = s.z - tz;
                    pair_branches<T, FIELDS, SELF>(acc, ex, ey, ez, ex * ex + ey * ey + ez * ez, s.w,
                                                   L.h[q] > th ? L.h[q] : th, (SELF && jt + q == i) | (q >= cnt));
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // the slices of a wave, then the waves, in order
#pragma unroll
    for (int d = P; d < 64; d <<= 1) {
#pragma unroll
        for (int c = 0; c < W; c++) acc.s[c] += __shfl_xor(acc.s[c], d, 64);
    }
    __syncthreads();
    if (sl == 0) {
#pragma unroll
        for (int c = 0; c < W; c++) lds.part[wave][c][tl] = acc.s[c];
    }
    __syncthreads();
    for (int v = threadIdx.x; v < W * P; v += 64 * DS_WAVES) {
        const int c = v / P, l = v % P;
        const int64_t t = (int64_t)blockIdx.x * P + l;
        if (t >= nt) continue;
        T s = lds.part[0][c][l];
#pragma unroll
        for (int w = 1; w < DS_WAVES; w++) s += lds.part[w][c][l];
        const double o = G * (double)s;
        constexpr int PA = (DAcc<T, FIELDS>::P ? 1 : 0) + (DAcc<T, FIELDS>::A ? 3 : 0);
        constexpr int WO = PA + (DAcc<T, FIELDS>::D ? 9 : 0);
        if (c < PA) {
            out[t * WO + c] = o;
        } else {  // xx xy xz yy yz zz of the symmetric tensor
            const int e = c - PA, a = e < 3 ? 0 : e < 5 ? 1 : 2, b = e < 3 ? e : e < 5 ? e - 2 : 2;
            out[t * WO + PA + 3 * a + b] = o;
            out[t * WO + PA + 3 * b + a] = o;
        }
    }
}

template <typename T, bool SELF, int P>
static ptg_status launch_p(int fields, const double *pt, const double *ht, int64_t nt, const double *ps,
                           const double *ms, const double *hs, int64_t ns, double G, double *out, hipStream_t s)
{
    dim3 grid((unsigned)std::max<int64_t>(1, ptg_cdiv(nt, P)));
#define PTG_D(F)                                                                                    \
    case F:                                                                                         \
        k_direct<T, F, SELF, P><<<grid, 64 * DS_WAVES, 0, s>>>(pt, ht, nt, ps, ms, hs, ns, G, out); \
        break;
    switch (fields) {
        PTG_D(1) PTG_D(2) PTG_D(3) PTG_D(4) PTG_D(5) PTG_D(6) PTG_D(7)
    default:
        ptg_set_error("ptg_direct: fields must be a nonzero combination of PTG_POT|PTG_ACC|PTG_TIDAL");
        return PTG_ERR_ARG;
    }
#undef PTG_D
    PTG_LAUNCH_CHECK();
    return PTG_OK;
}

// Targets per block.  16: many blocks and short sums (12007 targets: 78 us in FP32, 111 with 64).  4 where 16
// makes less than a block per 4 CUs: the kernel takes, with 4 and with 16, FP64 5.2 and 5.5 us for 256 particles,
// 6.6 and 9.3 for 1000, 13.7 and 14.1 for 2000, 35 and 25 for 4000 (FP32 4.5 and 4.7, 5.4 and 7.0, 9.6 and 9.6,
// 20.7 and 16.0); below 4000 the call's 25 us of host and launch hide it.  64 where there are blocks enough and 16
// targets would read the sources four times as often (equal times at 1e5 targets).
template <typename T, bool SELF>
static ptg_status launch_direct(int fields, const double *pt, const double *ht, int64_t nt, const double *ps,
                                const double *ms, const double *hs, int64_t ns, double G, double *out, hipStream_t s)
{
    if (nt <= 1024) return launch_p<T, SELF, 4>(fields, pt, ht, nt, ps, ms, hs, ns, G, out, s);
    if (nt <= 131072) return launch_p<T, SELF, 16>(fields, pt, ht, nt, ps, ms, hs, ns, G, out, s);
    return launch_p<T, SELF, 64>(fields, pt, ht, nt, ps, ms, hs, ns, G, out, s);
}

extern "C" ptg_status ptg_direct(const double *pos_t, const double *soft_t, int64_t nt, const double *pos_s,
                                 const double *m_s, const double *h_s, int64_t ns, int prec, int fields, int self_mode,
                                 double G, double *out, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    if (nt < 0 || ns < 0 || (nt > 0 && (!pos_t || !soft_t || !out)) || (ns > 0 && (!pos_s || !m_s || !h_s))) {
        ptg_set_error("ptg_direct: bad arguments");
        return PTG_ERR_ARG;
    }
    if (self_mode && nt != ns) {
        ptg_set_error("ptg_direct: self_mode needs nt == ns");
        return PTG_ERR_ARG;
    }
    if (nt == 0) return PTG_OK;
    if (prec == PTG_F64)
        return self_mode ? launch_direct<double, true>(fields, pos_t, soft_t, nt, pos_s, m_s, h_s, ns, G, out, s)
                         : launch_direct<double, false>(fields, pos_t, soft_t, nt, pos_s, m_s, h_s, ns, G, out, s);
    if (prec == PTG_F32)
        return self_mode ? launch_direct<float, true>(fields, pos_t, soft_t, nt, pos_s, m_s, h_s, ns, G, out, s)
                         : launch_direct<float, false>(fields, pos_t, soft_t, nt, pos_s, m_s, h_s, ns, G, out, s);
    ptg_set_error("ptg_direct: prec must be PTG_F32 or PTG_F64");
    return PTG_ERR_ARG;
}
