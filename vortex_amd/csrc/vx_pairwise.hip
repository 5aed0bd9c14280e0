// Pairwise O(N^2) stages: Biot-Savart velocity with the nearest-3 distance,
// vortex-vortex diffusive velocity, the birth right-hand side and the probe
// velocities.  Each is templated on the arithmetic type:
//   double  -- the reference formulas in FP64 (VX_PREC_F64);
//   float   -- FP32 pair arithmetic, FP32 partial sums over one 256-source
//              tile, FP64 accumulation of the tile sums (VX_PREC_MIXED).
// The direct kernels read their sources as scalar operands and are cut over
// targets (TPT a thread, spaced one block apart so that loads and stores
// coalesce) and sources; FP64 sums over few sources are added in source order by
// a wave of their own, from terms in LDS.  The probes and the right-hand side
// stage their sources through LDS.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "vx_internal.h"
#include "vx_math.h"
#include "vx_prim.h"
#include "vx_wave.h"

namespace vx {

template <typename T>
struct Src4 {
    T x, y, g, pad;
};

template <typename T>
struct Arith;

template <>
struct Arith<double> {
    static constexpr double kFar = 1e30;  // padding sources: squared distance stays finite
    __device__ static __forceinline__ double div(double a, double b) { return div_pos_exact(a, b); }
    __device__ static __forceinline__ double med3(double a, double b, double c) {
        return fmax(fmin(a, b), fmin(fmax(a, b), c));
    }
    __device__ static __forceinline__ double min_(double a, double b) { return fmin(a, b); }
    __device__ static __forceinline__ double max_(double a, double b) { return fmax(a, b); }
};

template <>
struct Arith<float> {
    static constexpr float kFar = 1e18f;
    __device__ static __forceinline__ float div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
    __device__ static __forceinline__ float med3(float a, float b, float c) {
        return __builtin_amdgcn_fmed3f(a, b, c);
    }
    __device__ static __forceinline__ float min_(float a, float b) { return fminf(a, b); }
    __device__ static __forceinline__ float max_(float a, float b) { return fmaxf(a, b); }
};

constexpr int kTile = 256;

// ---- work split of the direct kernels ---------------------------------------
// A direct launch is cut over targets (kTile * TPT per work-group) and over
// runs of `len` sources, whose partials a second kernel adds in run order.
// One run per work-group would leave most of the chip idle below 64 k
// vortices (10 work-groups at 2.5 k), so the runs are made short enough for
// kDirectWork blocks of kTile targets in all.  The split depends on the
// counts alone, not on TPT or on a launch's bound, so every launch shape,
// stream step and graph replay adds in the same order.
//
// 60001 vortices, FP32: Biot-Savart 2.66 -> 1.02 ms, diffusion 2.66 -> 1.29 ms
// against one work-group per kTile targets over all sources; 20011 in FP64:
// 1.76 -> 0.32 and 3.43 -> 0.64 ms.  With kDirectWork = 1024, 2048 and 8192
// the first pair takes 1.30 and 1.59, 1.09 and 1.40, 1.01 and 1.27 ms; the
// partials grow with it (48 B per target and run), so 4096.
//
// FP32 sums are taken over tiles of kTile sources and added in FP64, so up to
// kOrdered sources a run is one tile and the result is that of one pass over
// the sources in order, bit for bit; a run is several tiles above.  FP64 sums
// up to kOrdered sources go to the ordered kernels below for the same reason:
// a run of many steps multiplies a rounding by 1e6 in 25 steps, so long runs
// at these counts keep the order.
constexpr int64_t kDirectWork = 4096;
constexpr int64_t kOrdered = 16384;

struct DirectSplit {
    int32_t len, runs;
};

template <typename T>
__host__ __device__ __forceinline__ DirectSplit direct_split(int64_t n_tgt, int64_t n_src) {
    constexpr uint32_t unit = sizeof(T) == 4 ? kTile : kTile / 4;
    const uint32_t tb = (uint32_t)((n_tgt + kTile - 1) / kTile), units = (uint32_t)((n_src + unit - 1) / unit);
    if (units == 0 || tb == 0) return DirectSplit{(int32_t)unit, 1};
    uint32_t want = ((uint32_t)kDirectWork + tb - 1) / tb;
    if (want > units || n_src <= kOrdered) want = units;
    const uint32_t per = (units + want - 1) / want;
    return DirectSplit{(int32_t)(per * unit), (int32_t)((units + per - 1) / per)};
}

// Work-groups of kTile * tpt targets times runs, and doubles of partials for q
// values per target and run: exact for host counts.  A device count (the same
// for targets and sources) gets a bound over all counts up to its own; kernels
// leave surplus work-groups at once.  With tb blocks of kTile targets, n
// sources above kOrdered make at most (kDirectWork - 1) / tb + 1 runs, so n
// times runs stays below kTile * kDirectWork + n, and (tb + tpt - 1) / tpt
// times runs below kDirectWork / tpt + tb / tpt + 64 (tb > 64).  Up to kOrdered
// the runs are the units: both products grow with n, to kTile * kDirectWork and
// kDirectWork / tpt in FP32, while FP64 leaves those counts to the ordered kernels.
static_assert(kOrdered == 64 * kTile && kOrdered * 64 == kTile * kDirectWork, "the bounds of both ranges meet");

template <typename T>
static int64_t direct_blocks(Cnt n_tgt, Cnt n_src, int tpt) {
    const int64_t w = kTile * tpt, tb = (n_tgt.ub + w - 1) / w;
    if (!n_tgt.dev || n_src.ub <= kOrdered) return tb * direct_split<T>(n_tgt.ub, n_src.ub).runs;
    return tb + kDirectWork / tpt + 64;
}

template <typename T>
static size_t direct_partials(Cnt n_tgt, Cnt n_src, int q) {
    if (!n_tgt.dev || n_src.ub <= kOrdered)
        return (size_t)(q * n_tgt.ub * direct_split<T>(n_tgt.ub, n_src.ub).runs);
    return (size_t)(q * (n_tgt.ub + kTile * kDirectWork));
}

// The four smallest values seen so far, m0 <= m1 <= m2 <= m3.
template <typename T>
__device__ __forceinline__ void keep4(T &m0, T &m1, T &m2, T &m3, T r) {
    using A = Arith<T>;
    m3 = A::med3(m2, m3, r);
    m2 = A::med3(m1, m2, r);
    m1 = A::med3(m0, m1, r);
    m0 = A::min_(m0, r);
}

// Two values at a time, the same way (6 min/max a value).
__device__ __forceinline__ void keep4x2(double &m0, double &m1, double &m2, double &m3, double a, double b) {
    order2(a, b);
    m2 = fmin(m2, b);
    m3 = fmin(m3, a);
    order2(m0, m2);
    order2(m1, m3);
    order2(m0, m1);
    order2(m2, m3);
}
__device__ __forceinline__ void keep4x4(float &m0, float &m1, float &m2, float &m3, float a, float b, float c, float d) {
    keep4(m0, m1, m2, m3, a);
    keep4(m0, m1, m2, m3, b);
    keep4(m0, m1, m2, m3, c);
    keep4(m0, m1, m2, m3, d);
}

// ---- A6: src/kernel.cu:875-983 -------------------------------------------
// u_i = V_inf + (1/2pi) sum_j g_j (-(y_i-y_j), x_i-x_j) / max(r_ij^2, eps^2), j != i
// d_i = mean of sqrt of the three smallest r_ij^2 over j != i (sentinel 1e5).
// The self pair contributes exactly 0 to the sums (dx = dy = 0); for d the
// four smallest r^2 including the self 0 are kept and the smallest one is
// dropped, which equals the three smallest over j != i.
//
// Bound by VALU issue.  The sources are wave-uniform, so they come through
// scalar loads straight from the arrays: no LDS staging, no barriers, and the
// pair arithmetic takes them as scalar operands.  Partials per run s and
// target: part[(6 s + q) n_tgt + i], q = su, sv, then the four smallest r^2.
template <typename T, int TPT>
__global__ __launch_bounds__(kTile) void k_biot_savart(const T *__restrict__ sx, const T *__restrict__ sy,
                                                       const T *__restrict__ sg, Cnt cn_src, Cnt cn_tgt, T eps2,
                                                       double *__restrict__ part) {
    using A = Arith<T>;
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if (sizeof(T) == 8 && n_src <= kOrdered) return;  // the ordered kernel's
    const DirectSplit sp = direct_split<T>(n_tgt, n_src);
    const uint32_t tb = ((uint32_t)n_tgt + kTile * TPT - 1) / (kTile * TPT);
    if (tb == 0) return;
    const uint32_t s = blockIdx.x / tb, t = blockIdx.x - s * tb;
    if (s >= (uint32_t)sp.runs) return;
    const int32_t lo = (int32_t)s * sp.len, hi = min(n_src, lo + sp.len);
    const int32_t t0 = (int32_t)(t * (kTile * TPT) + threadIdx.x);
    T ax[TPT], ay[TPT], m0[TPT], m1[TPT], m2[TPT], m3[TPT], su[TPT], sv[TPT];
    double au[TPT], av[TPT];
    bool tame = ordinary_eps2(eps2);
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int32_t i = t0 + k * kTile;
        ax[k] = i < n_tgt ? sx[i] : T(0);
        ay[k] = i < n_tgt ? sy[i] : T(0);
        tame = tame && ordinary(ax[k]) && ordinary(ay[k]);
        m0[k] = m1[k] = m2[k] = m3[k] = T(1e5);
        su[k] = sv[k] = T(0);
        au[k] = av[k] = 0.0;
    }
    tame = !__any(!tame);
    auto pair = [&](int k, T x, T y, T g, auto plain) {
        const T dx = ax[k] - x, dy = ay[k] - y;
        const T r2 = dx * dx + dy * dy;
        const T a = A::max_(r2, eps2);
        T w;
        if constexpr (decltype(plain)::value)
            w = g / a;
        else
            w = A::div(g, a);
        sv[k] += w * dx;
        su[k] -= w * dy;
        return r2;
    };
    constexpr std::integral_constant<bool, sizeof(T) == 8> plain64;
    for (int32_t base = lo; base < hi; base += kTile) {
        const int32_t end = min(hi, base + kTile);
        int32_t j = base;
        for (; j + 4 <= end; j += 4) {
            T x[4], y[4], g[4];
            uint32_t odd = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x[q] = sx[j + q];
                y[q] = sy[j + q];
                g[q] = sg[j + q];
                odd |= odd_bit(x[q]) | odd_bit(y[q]) | odd_bit(g[q]);
            }
            if (__builtin_expect(!tame || (int32_t)odd < 0, 0)) break;
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                T r2[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) r2[q] = pair(k, x[q], y[q], g[q], std::false_type());
                keep4x4(m0[k], m1[k], m2[k], m3[k], r2[0], r2[1], r2[2], r2[3]);
            }
        }
        for (; j < end; ++j) {  // the last ones, and the rest of a tile with unordinary values
            const T x = sx[j], y = sy[j], g = sg[j];
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                const T r2 = pair(k, x, y, g, plain64);
                keep4(m0[k], m1[k], m2[k], m3[k], r2);
            }
        }
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                au[k] += (double)su[k];
                av[k] += (double)sv[k];
                su[k] = sv[k] = T(0);
            }
        }
    }
    double *o = part + (int64_t)s * 6 * n_tgt;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int32_t i = t0 + k * kTile;
        if (i >= n_tgt) continue;
        const double q[6] = {sizeof(T) == 8 ? (double)su[k] : au[k], sizeof(T) == 8 ? (double)sv[k] : av[k],
                             (double)m0[k], (double)m1[k], (double)m2[k], (double)m3[k]};
#pragma unroll
        for (int e = 0; e < 6; ++e) o[(int64_t)e * n_tgt + i] = q[e];
    }
}

// Adds the runs' partials in run order: 64 targets per work-group, kSumRuns
// runs at a time read by the four waves, added by the first.
constexpr int kSumRuns = 16;

template <typename T>
__global__ __launch_bounds__(256) void k_bs_sum(const double *__restrict__ part, Cnt cn_src, Cnt cn_tgt,
                                                double vinf_x, double vinf_y, double *__restrict__ u,
                                                double *__restrict__ v, double *__restrict__ d) {
    __shared__ double ls[kSumRuns][2][64];
    __shared__ double lm[3][4][64];
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if ((int32_t)blockIdx.x * 64 >= n_tgt || (sizeof(T) == 8 && n_src <= kOrdered)) return;
    const int32_t runs = direct_split<T>(n_tgt, n_src).runs;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int32_t i = (int32_t)blockIdx.x * 64 + lane, ic = min(i, n_tgt - 1);
    double a = 0.0, b = 0.0, m0 = 1e5, m1 = 1e5, m2 = 1e5, m3 = 1e5;
    for (int32_t s0 = 0; s0 < runs; s0 += kSumRuns) {
#pragma unroll
        for (int q = 0; q < kSumRuns / 4; ++q) {
            const int32_t s = s0 + wv * (kSumRuns / 4) + q;
            if (s >= runs) break;
            const double *o = part + (int64_t)s * 6 * n_tgt + ic;
            ls[s - s0][0][lane] = o[0];
            ls[s - s0][1][lane] = o[(int64_t)n_tgt];
            const double q0 = o[(int64_t)2 * n_tgt], q1 = o[(int64_t)3 * n_tgt], q2 = o[(int64_t)4 * n_tgt],
                         q3 = o[(int64_t)5 * n_tgt];
            keep4x4(m0, m1, m2, m3, q0, q1, q2, q3);
        }
        __syncthreads();
        if (wv == 0) {
            const int32_t c = min(kSumRuns, runs - s0);
            for (int32_t q = 0; q < c; ++q) {
                a += ls[q][0][lane];
                b += ls[q][1][lane];
            }
        }
        __syncthreads();
    }
    if (wv) {
        const double q[4] = {m0, m1, m2, m3};
        for (int e = 0; e < 4; ++e) lm[wv - 1][e][lane] = q[e];
    }
    __syncthreads();
    if (wv || i >= n_tgt) return;
    for (int w = 0; w < 3; ++w) keep4x4(m0, m1, m2, m3, lm[w][0][lane], lm[w][1][lane], lm[w][2][lane], lm[w][3][lane]);
    u[i] = a / (2 * kPi) + vinf_x;
    v[i] = b / (2 * kPi) + vinf_y;
    d[i] = (sqrt(m1) + sqrt(m2) + sqrt(m3)) / 3;
}

// ---- A7: src/kernel.cu:985-1029 -------------------------------------------
// Over j with r_ij > 0.001 ve_size: I2 += -g_j (r_i - r_j)/r e^{-r/d_i},
// I1 += g_j e^{-r/d_i}; if |I1| > 1e-5: V_i += -nu I2 / (I1 d_i).
// Sources and partials as in k_biot_savart: part[(3 s + q) n_tgt + i], q = x
// and y of the weighted separations, then I1.
//
// FP64 takes four sources at a time through expressions for ordinary
// separations; where some lane comes near the threshold (its own source among
// others) or a coordinate or circulation is huge or no number, the four go
// through the plain ones.  Both round alike.
template <typename T>
struct DiffSums {
    T x, y, i1;
};

__device__ __forceinline__ void diff_pair_plain(double dx, double dy, double g, double kd, double thr,
                                                DiffSums<double> &s) {
    const double dist = sqrt(fma(dx, dx, dy * dy));
    if (dist > thr) {
        const double w = g / dist, e = exp(-dist * kd);
        s.x = fma(w * dx, e, s.x);
        s.y = fma(w * dy, e, s.y);
        s.i1 = fma(g, e, s.i1);
    }
}

template <typename T, int TPT>
__global__ __launch_bounds__(kTile) void k_diffusion(const T *__restrict__ sx, const T *__restrict__ sy,
                                                     const T *__restrict__ sg, Cnt cn_src, Cnt cn_tgt,
                                                     const double *__restrict__ dd, T thr,
                                                     double *__restrict__ part) {
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if (sizeof(T) == 8 && n_src <= kOrdered) return;  // the ordered kernel's
    const DirectSplit sp = direct_split<T>(n_tgt, n_src);
    const uint32_t tb = ((uint32_t)n_tgt + kTile * TPT - 1) / (kTile * TPT);
    if (tb == 0) return;
    const uint32_t s = blockIdx.x / tb, t = blockIdx.x - s * tb;
    if (s >= (uint32_t)sp.runs) return;
    const int32_t lo = (int32_t)s * sp.len, hi = min(n_src, lo + sp.len);
    const int32_t t0 = (int32_t)(t * (kTile * TPT) + threadIdx.x);
    T ax[TPT], ay[TPT], kd[TPT];
    DiffSums<T> sum[TPT];
    double a2x[TPT], a2y[TPT], a1[TPT];
    bool tame = true;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int32_t i = t0 + k * kTile;
        ax[k] = i < n_tgt ? sx[i] : T(0);
        ay[k] = i < n_tgt ? sy[i] : T(0);
        const double di = i < n_tgt ? dd[i] : 1.0;
        // FP32: exp(-r/d) = exp2(r * kd)
        kd[k] = (T)((sizeof(T) == 4 ? -1.4426950408889634 : 1.0) / di);
        sum[k] = DiffSums<T>{T(0), T(0), T(0)};
        a2x[k] = a2y[k] = a1[k] = 0.0;
        if constexpr (sizeof(T) == 8) tame = tame && ordinary(ax[k]) && ordinary(ay[k]);
    }
    if constexpr (sizeof(T) == 8) {
        tame = !__any(!tame);
        const double gap2 = fmax(4.0 * thr * thr, 0x1p-900);  // no rounding brings a distance above 2 thr to thr
        int32_t j = lo;
        for (; j + 4 <= hi; j += 4) {
            double x[4], y[4], g[4];
            uint32_t odd = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x[q] = sx[j + q];
                y[q] = sy[j + q];
                g[q] = sg[j + q];
                odd |= odd_bit(x[q]) | odd_bit(y[q]) | odd_bit(g[q]);
            }
            const bool plain = !tame || (int32_t)odd < 0;
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                double r2[4];
                uint64_t near = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double dx = ax[k] - x[q], dy = ay[k] - y[q];
                    r2[q] = fma(dx, dx, dy * dy);
                    near |= __ballot(!(r2[q] > gap2));
                }
                if (__builtin_expect(plain || near != 0, 0)) {
#pragma unroll 1
                    for (int q = 0; q < 4; ++q)
                        diff_pair_plain(ax[k] - sx[j + q], ay[k] - sy[j + q], sg[j + q], kd[k], thr, sum[k]);
                    continue;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double dx = ax[k] - x[q], dy = ay[k] - y[q];
                    double w;
                    const double dist = sqrt_pos_exact(r2[q], g[q], w), e = exp(-dist * kd[k]);
                    sum[k].x = fma(w * dx, e, sum[k].x);
                    sum[k].y = fma(w * dy, e, sum[k].y);
                    sum[k].i1 = fma(g[q], e, sum[k].i1);
                }
            }
        }
        for (; j < hi; ++j)
#pragma unroll
            for (int k = 0; k < TPT; ++k) diff_pair_plain(ax[k] - sx[j], ay[k] - sy[j], sg[j], kd[k], thr, sum[k]);
    } else {
        const T thr2 = thr;  // squared by the caller, in FP64
        for (int32_t base = lo; base < hi; base += kTile) {
            const int32_t end = min(hi, base + kTile);
#pragma unroll 4
            for (int32_t j = base; j < end; ++j) {
                const T x = sx[j], y = sy[j], g = sg[j];
#pragma unroll
                for (int k = 0; k < TPT; ++k) {
                    const T dx = ax[k] - x, dy = ay[k] - y;
                    const T r2 = dx * dx + dy * dy;
                    const T r2c = r2 > thr2 ? r2 : T(1e30f);
                    const T rs = __builtin_amdgcn_rsqf(r2c);
                    const T e = __builtin_amdgcn_exp2f((r2c * rs) * kd[k]);
                    const T ge = g * e;
                    const T w = ge * rs;
                    sum[k].x += w * dx;
                    sum[k].y += w * dy;
                    sum[k].i1 += ge;
                }
            }
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                a2x[k] += (double)sum[k].x;
                a2y[k] += (double)sum[k].y;
                a1[k] += (double)sum[k].i1;
                sum[k] = DiffSums<T>{T(0), T(0), T(0)};
            }
        }
    }
    double *o = part + (int64_t)s * 3 * n_tgt;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int32_t i = t0 + k * kTile;
        if (i >= n_tgt) continue;
        o[i] = sizeof(T) == 8 ? (double)sum[k].x : a2x[k];
        o[(int64_t)n_tgt + i] = sizeof(T) == 8 ? (double)sum[k].y : a2y[k];
        o[(int64_t)2 * n_tgt + i] = sizeof(T) == 8 ? (double)sum[k].i1 : a1[k];
    }
}

// I2 = -sum w (r_i - r_j) e, so -nu I2/(I1 d) = nu a2/(I1 d)
__device__ __forceinline__ void diff_add(int32_t i, double a2x, double a2y, double a1, const double *__restrict__ dd,
                                         double nu, double *__restrict__ u, double *__restrict__ v) {
    if (fabs(a1) > 1e-5) {
        const double di = dd[i];
        u[i] += nu * a2x / (a1 * di);
        v[i] += nu * a2y / (a1 * di);
    }
}

// Adds the runs' partials as k_bs_sum does.
template <typename T>
__global__ __launch_bounds__(256) void k_diff_sum(const double *__restrict__ part, Cnt cn_src, Cnt cn_tgt,
                                                  const double *__restrict__ dd, double nu, double *__restrict__ u,
                                                  double *__restrict__ v) {
    __shared__ double ls[kSumRuns][3][64];
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if ((int32_t)blockIdx.x * 64 >= n_tgt || (sizeof(T) == 8 && n_src <= kOrdered)) return;
    const int32_t runs = direct_split<T>(n_tgt, n_src).runs;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int32_t i = (int32_t)blockIdx.x * 64 + lane, ic = min(i, n_tgt - 1);
    double a2x = 0.0, a2y = 0.0, a1 = 0.0;
    for (int32_t s0 = 0; s0 < runs; s0 += kSumRuns) {
#pragma unroll
        for (int q = 0; q < kSumRuns / 4; ++q) {
            const int32_t s = s0 + wv * (kSumRuns / 4) + q;
            if (s >= runs) break;
            const double *o = part + (int64_t)s * 3 * n_tgt + ic;
            for (int e = 0; e < 3; ++e) ls[s - s0][e][lane] = o[(int64_t)e * n_tgt];
        }
        __syncthreads();
        if (wv == 0) {
            const int32_t c = min(kSumRuns, runs - s0);
            for (int32_t q = 0; q < c; ++q) {
                a2x += ls[q][0][lane];
                a2y += ls[q][1][lane];
                a1 += ls[q][2][lane];
            }
        }
        __syncthreads();
    }
    if (wv || i >= n_tgt) return;
    diff_add(i, a2x, a2y, a1, dd, nu, u, v);
}

// ---- ordered FP64 sums --------------------------------------------------------
// The same sums with one accumulation chain per target over the sources in
// order, for the counts at which the chip is far from full with one lane per
// target.  The pair terms do not depend on the order, only their addition
// does: in a work-group of 16 waves, 15 evaluate terms of TG targets, SL =
// 64 / TG sources per wave and pass, into LDS, and one adds the tile before
// in order, the components of a target on lanes of their own.  The term
// arithmetic is correctly rounded as the plain expressions are, so the
// results are those of the plain loop bit for bit.  Bound by the LDS while
// there is a CU for each work-group: Biot-Savart takes 24 cycles a source, the
// adding wave alone 21 (two 16-byte reads a pair of sources), the evaluating
// ones alone 15; the reads of the next batch stand between the adds (all
// before them: 3 % more).  2500 vortices: Biot-Savart 243 -> 25 us, diffusion
// 475 -> 33 us against one lane per target over all sources.  Above kOrdered the split
// sums are faster: at 17000 0.25 and 0.50 ms against 0.64 and 1.12 ms.
constexpr int kOrdWaves = 15;
constexpr int kAhead = 6;  // pairs of terms per batch: the LDS latency of one is covered by the adds of another

// Sources of a tile, staged three tiles deep (the tile being evaluated, the
// one being added and the next).  A vector load that fetches one or two
// addresses for a wave still costs the load unit a full wave's turns.
template <int TILE>
struct OrdSrc {
    double c[3][3][TILE];  // x, y, g
    __device__ __forceinline__ void put(int b, int e, double3 s) {
        c[b][0][e] = s.x;
        c[b][1][e] = s.y;
        c[b][2][e] = s.z;
    }
};
__device__ __forceinline__ double3 ord_src(const double *__restrict__ sx, const double *__restrict__ sy,
                                           const double *__restrict__ sg, int32_t j, int32_t n) {
    j = min(j, n - 1);  // past the end: the last source, its terms replaced by zeros
    return double3{sx[j], sy[j], sg[j]};
}

template <int TG, int Q>
__global__ __launch_bounds__(1024) void k_biot_savart_ordered(const double *__restrict__ sx,
                                                              const double *__restrict__ sy,
                                                              const double *__restrict__ sg, Cnt cn_src, Cnt cn_tgt,
                                                              double eps2, double vinf_x, double vinf_y,
                                                              double *__restrict__ u, double *__restrict__ v,
                                                              double *__restrict__ d) {
    constexpr int SL = 64 / TG, TILE = kOrdWaves * SL * Q;
    constexpr int kTerms = 2 * TILE * TG, kSmall = 4 * kOrdWaves * 64;
    // terms [2][TILE / 2][TG][2] (a lane reads two sources' at once); at the
    // end the nearest lists
    __shared__ __align__(16) double lw[kTerms > kSmall ? kTerms : kSmall];
    __shared__ __align__(16) OrdSrc<TILE> src;
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if ((int32_t)blockIdx.x * TG >= n_tgt || n_src > kOrdered) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int t = lane & (TG - 1), slot = lane / TG;
    const int32_t i = (int32_t)blockIdx.x * TG + t, ic = min(i, n_tgt - 1);
    const double ax = sx[ic], ay = sy[ic];
    double m0 = 1e5, m1 = 1e5, m2 = 1e5, m3 = 1e5;
    const bool plain = !ordinary_eps2(eps2);
    // the chain of lane (t, slot): sv of dx for even slots, su of -dy for odd
    const bool xr = !(slot & 1);
    const double c1 = xr ? -1.0 : 1.0, c0 = xr ? ax : -ay;
    double acc = 0.0;
    const int32_t tiles = (n_src + TILE - 1) / TILE;
    const bool stager = threadIdx.x < TILE;
    if (stager && tiles) src.put(0, threadIdx.x, ord_src(sx, sy, sg, threadIdx.x, n_src));
    __syncthreads();
    int b0 = 0, b1 = 1, b2 = 2;  // source buffers of tiles k, k + 1 and k - 1
    for (int32_t k = 0; k <= tiles; ++k) {
        double3 next;
        if (stager && k + 1 < tiles) next = ord_src(sx, sy, sg, (k + 1) * TILE + (int32_t)threadIdx.x, n_src);
        if (wv < kOrdWaves) {
            if (k < tiles) {
                double *w_ = lw + (k & 1) * (TILE * TG);
                double r2[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int jj = (q * kOrdWaves + wv) * SL + slot;
                    const double dx = ax - src.c[b0][0][jj], dy = ay - src.c[b0][1][jj], g = src.c[b0][2][jj];
                    r2[q] = fma(dx, dx, dy * dy);
                    const double a = fmax(r2[q], eps2);
                    double w = div_pos_exact(g, a);
                    // (an infinite a or g leaves NaN)
                    if (__builtin_expect(plain || __any(!(fabs(w) < INFINITY)), 0)) {
                        asm volatile("; rare: kept out of the main path");
                        w = g / a;
                    }
                    const bool in = k * TILE + jj < n_src;
                    w_[(jj >> 1) * (2 * TG) + 2 * t + (jj & 1)] = in ? w : 0.0;
                    r2[q] = in ? fmin(r2[q], 1e5) : 1e5;  // no NaN in the lists, which start at 1e5
                }
                if constexpr (Q == 4)
                    keep4x4(m0, m1, m2, m3, r2[0], r2[1], r2[2], r2[3]);
                else
                    keep4x2(m0, m1, m2, m3, r2[0], r2[1]);
            }
        } else if (k > 0 && lane < 2 * TG) {
            __builtin_amdgcn_s_setprio(3);
            const double2 *w_ = (const double2 *)(lw + ((k - 1) & 1) * (TILE * TG)) + t;
            const double2 *s_ = (const double2 *)src.c[b2][xr ? 0 : 1];
            // two batches of kAhead pairs in turn: one is added while the next is read
            double2 w[2][kAhead], p[2][kAhead];
#pragma unroll
            for (int e = 0; e < kAhead; ++e) {
                w[0][e] = w_[e * TG];
                p[0][e] = s_[e];
            }
#pragma unroll
            for (int h = 0; h < TILE / 2 / kAhead; ++h) {
#pragma unroll
                for (int e = 0; e < kAhead; ++e) {
                    if (h + 1 < TILE / 2 / kAhead) {
                        w[(h + 1) & 1][e] = w_[((h + 1) * kAhead + e) * TG];
                        p[(h + 1) & 1][e] = s_[(h + 1) * kAhead + e];
                    }
                    acc = fma(w[h & 1][e].x, fma(p[h & 1][e].x, c1, c0), acc);
                    acc = fma(w[h & 1][e].y, fma(p[h & 1][e].y, c1, c0), acc);
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        if (stager && k + 1 < tiles) src.put(b1, threadIdx.x, next);
        __syncthreads();
        const int r = b2;
        b2 = b0;
        b0 = b1;
        b1 = r;
    }
    // the producers' nearest lists, merged by the adding wave
    if (wv < kOrdWaves) {
        const double q[4] = {m0, m1, m2, m3};
        for (int e = 0; e < 4; ++e) lw[(wv * 4 + e) * 64 + lane] = q[e];
    }
    __syncthreads();
    if (wv < kOrdWaves) return;
    for (int w = 0; w < kOrdWaves; ++w) {
        const double *q = lw + w * 256 + lane;
        keep4x4(m0, m1, m2, m3, q[0], q[64], q[128], q[192]);
    }
#pragma unroll
    for (int o = TG; o < 64; o <<= 1) {
        const double q0 = __shfl_xor(m0, o, 64), q1 = __shfl_xor(m1, o, 64), q2 = __shfl_xor(m2, o, 64),
                     q3 = __shfl_xor(m3, o, 64);
        keep4x4(m0, m1, m2, m3, q0, q1, q2, q3);
    }
    if (i >= n_tgt || slot > 1) return;
    if (xr) {
        v[i] = acc / (2 * kPi) + vinf_y;
        d[i] = (sqrt(m1) + sqrt(m2) + sqrt(m3)) / 3;
    } else {
        u[i] = acc / (2 * kPi) + vinf_x;
    }
}

// The diffusion's three chains: x and y terms (w dx) e, (w dy) e with w = g /
// r on lanes of their own, and I1's g e beside both.  A pair within the
// threshold, or past the end, has e = 0.  A circulation that is no finite
// number is staged as kNoNumber, which leaves such pairs' products zero, and
// far away, where every pair takes the plain expressions: they read its own
// place and value, and the value comes with e.
constexpr double kNoNumber = 0x1p-1074, kNoPlace = 1e300;

template <int TG, int Q>
__global__ __launch_bounds__(1024) void k_diffusion_ordered(const double *__restrict__ sx,
                                                            const double *__restrict__ sy,
                                                            const double *__restrict__ sg, Cnt cn_src, Cnt cn_tgt,
                                                            const double *__restrict__ dd, double nu, double thr,
                                                            double *__restrict__ u, double *__restrict__ v) {
    constexpr int SL = 64 / TG, TILE = kOrdWaves * SL * Q;
    __shared__ __align__(16) double2 lt[2][3][TILE / 2][TG];  // w dx, w dy, e of two sources
    __shared__ __align__(16) OrdSrc<TILE> src;
    const int32_t n_src = (int32_t)cn_src.get(), n_tgt = (int32_t)cn_tgt.get();
    if ((int32_t)blockIdx.x * TG >= n_tgt || n_src > kOrdered) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int t = lane & (TG - 1), slot = lane / TG;
    const int32_t i = (int32_t)blockIdx.x * TG + t, ic = min(i, n_tgt - 1);
    const double ax = sx[ic], ay = sy[ic], kd = 1.0 / dd[ic];
    double acc = 0.0, acc1 = 0.0;
    const int32_t tiles = (n_src + TILE - 1) / TILE;
    const bool stager = threadIdx.x < TILE;
    auto source = [&](int32_t j) {
        double3 q = ord_src(sx, sy, sg, j, n_src);
        return fabs(q.z) < INFINITY ? q : double3{kNoPlace, q.y, kNoNumber};
    };
    if (stager && tiles) src.put(0, threadIdx.x, source(threadIdx.x));
    __syncthreads();
    int b0 = 0, b1 = 1, b2 = 2;
    for (int32_t k = 0; k <= tiles; ++k) {
        const int b = k & 1;
        double3 next;
        if (stager && k + 1 < tiles) next = source((k + 1) * TILE + (int32_t)threadIdx.x);
        if (wv < kOrdWaves) {
            if (k < tiles) {
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int jj = (q * kOrdWaves + wv) * SL + slot;
                    double dx = ax - src.c[b0][0][jj], dy = ay - src.c[b0][1][jj];
                    const double g = src.c[b0][2][jj], r2 = fma(dx, dx, dy * dy);
                    double w, dist = sqrt_pos_exact(r2, g, w), own = 1.0;
                    const bool rare = __any(r2 > 1e300);
                    if (__builtin_expect(rare, 0)) {
                        asm volatile("; rare: kept out of the main path");
                        const double3 q = ord_src(sx, sy, sg, k * TILE + jj, n_src);
                        dx = ax - q.x;
                        dy = ay - q.y;
                        own = fabs(q.z) < INFINITY ? 1.0 : q.z;
                        dist = sqrt(fma(dx, dx, dy * dy));
                        w = q.z / dist;
                    }
                    const bool on = dist > thr && k * TILE + jj < n_src;
                    double e = exp(-dist * kd);
                    if (__builtin_expect(rare, 0)) e *= own;
                    double *o = (double *)&lt[b][0][jj >> 1][t] + (jj & 1);
                    o[0] = on ? w * dx : 0.0;
                    o[TILE * TG] = on ? w * dy : 0.0;
                    o[2 * TILE * TG] = on ? e : 0.0;
                }
            }
        } else if (k > 0 && lane < 2 * TG) {
            __builtin_amdgcn_s_setprio(3);
            const double2 *p_ = &lt[b ^ 1][slot & 1][0][t], *e_ = &lt[b ^ 1][2][0][t];
            const double2 *g_ = (const double2 *)src.c[b2][2];
            constexpr int H = kAhead / 2;
            double2 p[2][H], x[2][H], g[2][H];
#pragma unroll
            for (int q = 0; q < H; ++q) {
                p[0][q] = p_[q * TG];
                x[0][q] = e_[q * TG];
                g[0][q] = g_[q];
            }
#pragma unroll
            for (int h = 0; h < TILE / 2 / H; ++h) {
#pragma unroll
                for (int q = 0; q < H; ++q) {
                    if (h + 1 < TILE / 2 / H) {
                        p[(h + 1) & 1][q] = p_[((h + 1) * H + q) * TG];
                        x[(h + 1) & 1][q] = e_[((h + 1) * H + q) * TG];
                        g[(h + 1) & 1][q] = g_[(h + 1) * H + q];
                    }
                    acc = fma(p[h & 1][q].x, x[h & 1][q].x, acc);
                    acc1 = fma(g[h & 1][q].x, x[h & 1][q].x, acc1);
                    acc = fma(p[h & 1][q].y, x[h & 1][q].y, acc);
                    acc1 = fma(g[h & 1][q].y, x[h & 1][q].y, acc1);
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        if (stager && k + 1 < tiles) src.put(b1, threadIdx.x, next);
        __syncthreads();
        const int r = b2;
        b2 = b0;
        b0 = b1;
        b1 = r;
    }
    if (wv < kOrdWaves) return;
    const double a2y = __shfl(acc, t + TG, 64);
    if (slot == 0 && i < n_tgt) diff_add(i, acc, a2y, acc1, dd, nu, u, v);
}

// atan2 in FP32 for the panel right-hand side: octant reduction to
// t = min(|x|,|y|) / max(|x|,|y|) in [0, 1] and an odd polynomial of degree
// 15 for atan(t), fitted for this library by iteratively reweighted least
// squares on [0, 1] (maximum error 3.8e-8 before FP32 rounding, 1.2e-7 after).
// Signed zeros follow C's atan2 (x = -0 gives +-pi).
__device__ __forceinline__ float vx_atan2f(float y, float x) {
    const float ax = fabsf(x), ay = fabsf(y);
    const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
    const float t = mn == 0.f ? 0.f : fminf(mn * __builtin_amdgcn_rcpf(mx), 1.f);
    const float s = t * t;
    float r = -0.004052795469760895f;
    r = __builtin_fmaf(r, s, 0.021855246275663376f);
    r = __builtin_fmaf(r, s, -0.05589873716235161f);
    r = __builtin_fmaf(r, s, 0.09640958160161972f);
    r = __builtin_fmaf(r, s, -0.13908010721206665f);
    r = __builtin_fmaf(r, s, 0.19946402311325073f);
    r = __builtin_fmaf(r, s, -0.3332984149456024f);
    r = __builtin_fmaf(r, s, 0.9999993443489075f);
    r *= t;
    if (ay > ax) r = 1.57079632679489662f - r;
    if (__builtin_signbit(x)) r = 3.14159265358979324f - r;
    return __builtin_copysignf(r, y);
}

// ---- A3: src/kernel.cu:779-847 --------------------------------------------
// For panel i with end points l, r, d = r - l:
//   y += g_j (alpha d + beta k x d), alpha = atan(s0.d/z) - atan(s1.d/z),
//   beta = 0.5 ln(|s1|^2/|s0|^2), s0 = l - r_j, s1 = r - r_j, z = d x s0.
// In FP32 alpha is evaluated as one atan2(-|d|^2 z, z^2 + (s0.d)(s1.d)),
// the same angle difference.  This is the panel average of the point
// vortices' conjugate velocity g/(2 pi i (z - z_j)), times 2 pi |d|^2.
//
// Sources far from the profile are summed as local expansions instead.
// The panels lie in the profile box, centre c, half-diagonal R_b, and in
// segments of at most 128 consecutive panels, each inside a circle of centre
// c_s and radius R_s.  For sources with |z_j - c| >= 2 R_b (global) and for
// z on a panel,
//   (u - i v)(z) = (i / 2 pi) sum_k S_k (z - c)^k,
//   S_k = sum_j g_j w_j^{k+1},  w_j = 1 / (z_j - c),
// truncated after kLoc terms, which leaves at most 2^{1-kLoc} of the far sum.
// It is shifted exactly to each segment centre (a polynomial of degree
// kLoc - 1 re-expanded: sum_{k>=m} S_k C(k, m) (c_s - c)^{k-m}).  Sources
// nearer than 2 R_b but at least 2 R_s from c_s add their own terms
// g_j w_{s,j}^{m+1} about c_s (the same bound).  The rest, nearer than 2 R_s,
// are summed pair by pair for that segment's panels.  The panel average of
// the segment's expansion is exact:
//   mean over [z_l, z_r] of (z - c_s)^k = Q_k / (k + 1),
//   Q_k = (a^{k+1} - b^{k+1}) / (a - b) = a Q_{k-1} + b^k,  a = z_r - c_s, b = z_l - c_s.
// The sources nearer than 2 R_b (with g != 0) are listed in index order.
constexpr int kLoc = 48;
constexpr int kRhsChunk = 512;

struct RhsNear {
    const double *x, *y, *g;
    double cx, cy, r2;
    __device__ bool operator()(int32_t j) const {
        const double dx = x[j] - cx, dy = y[j] - cy;
        return g[j] != 0 && dx * dx + dy * dy < r2;
    }
};

constexpr int kSegTile = 128;  // panels per segment, threads per pair work-group

// One work-group per (segment, chunk of kRhsChunk listed sources), a thread
// per panel of the segment.  Each tile of sources is staged with a flag for
// |z_j - c_s| < 2 R_s (FP64 positions, as the expansion kernel tests), the
// flagged ones compacted in LDS and summed pair by pair.
template <typename T>
__global__ __launch_bounds__(kSegTile) void k_right_part_partial(
    const T *__restrict__ sx, const T *__restrict__ sy, const T *__restrict__ sg, const double *__restrict__ x,
    const double *__restrict__ y, const int32_t *__restrict__ list, const int32_t *__restrict__ nlist,
    PanelsSoA pan, const RhsSeg *__restrict__ segs, double *__restrict__ part) {
    __shared__ Src4<T> ls[kSegTile];
    __shared__ int wcount[2];
    const RhsSeg S = segs[blockIdx.x];
    const int64_t c = blockIdx.y;
    const int64_t n_src = *nlist;
    const int64_t lo = c * kRhsChunk, hi = min(n_src, lo + kRhsChunk);
    if (lo >= n_src && lo > 0) return;  // a chunk k_right_part_final does not read
    const bool live = (int)threadIdx.x < S.count;
    const int64_t i = S.first + (live ? threadIdx.x : 0);
    // FP32: panel ends and sources relative to the segment centre, the panel
    // vector differenced in FP64 (absolute FP32 coordinates would leave the
    // short panels' vectors with relative errors of ulp(|z|) / length)
    constexpr bool F32 = sizeof(T) == 4;
    const double ox = F32 ? S.cx : 0.0, oy = F32 ? S.cy : 0.0;
    const T l0 = (T)(pan.lx[i] - ox), l1 = (T)(pan.ly[i] - oy);
    const T r0 = (T)(pan.rx[i] - ox), r1 = (T)(pan.ry[i] - oy);
    const T d0 = F32 ? (T)(pan.rx[i] - pan.lx[i]) : r0 - l0, d1 = F32 ? (T)(pan.ry[i] - pan.ly[i]) : r1 - l1;
    const T dd2 = d0 * d0 + d1 * d1;
    const double rn2 = 4.0 * S.r * S.r;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    T y0 = 0, y1 = 0;
    double a0 = 0.0, a1 = 0.0;
    for (int64_t base = lo; base < hi; base += kSegTile) {
        const int64_t j = base + threadIdx.x;
        bool near = false;
        Src4<T> q;
        if (j < hi) {
            const int32_t k = list[j];
            const double ex = x[k] - S.cx, ey = y[k] - S.cy;
            near = ex * ex + ey * ey < rn2;
            q.x = F32 ? (T)ex : sx[k];
            q.y = F32 ? (T)ey : sy[k];
            q.g = sg[k];
            q.pad = T(0);
        }
        const uint64_t m = __ballot(near);
        __syncthreads();  // the previous tile is read
        if (lane == 0) wcount[wv] = __popcll(m);
        __syncthreads();
        const int pos = (wv ? wcount[0] : 0) + __popcll(m & ((1ull << lane) - 1));
        if (near) ls[pos] = q;
        __syncthreads();
        const int cnt = wcount[0] + wcount[1];
        for (int jj = 0; jj < cnt; ++jj) {
            const Src4<T> s_ = ls[jj];
            const T s00 = l0 - s_.x, s01 = l1 - s_.y;
            const T s10 = r0 - s_.x, s11 = r1 - s_.y;
            const T z = d0 * s01 - d1 * s00;
            const T A = s00 * d0 + s01 * d1;
            const T B = s10 * d0 + s11 * d1;
            T alpha, beta;
            if constexpr (sizeof(T) == 4) {
                alpha = vx_atan2f(-dd2 * z, z * z + A * B);
                const T q0 = s00 * s00 + s01 * s01, q1 = s10 * s10 + s11 * s11;
                beta = 0.34657359027997264f * __builtin_amdgcn_logf(q1 * __builtin_amdgcn_rcpf(q0));
            } else {
                alpha = atan(A / z) - atan(B / z);
                beta = 0.5 * log((s10 * s10 + s11 * s11) / (s00 * s00 + s01 * s01));
            }
            y0 += s_.g * (alpha * d0 - beta * d1);
            y1 += s_.g * (alpha * d1 + beta * d0);
        }
        if constexpr (sizeof(T) == 4) {
            a0 += (double)y0;
            a1 += (double)y1;
            y0 = y1 = T(0);
        }
    }
    if constexpr (sizeof(T) == 8) {
        a0 = y0;
        a1 = y1;
    }
    if (live) {
        part[(c * 2 + 0) * pan.P + i] = a0;
        part[(c * 2 + 1) * pan.P + i] = a1;
    }
}

// The pairs with kRhsPG panels per work-group.  An FP64 pair takes two arc
// tangents, a logarithm and five quotients (about 500 instructions; FP32 50), and
// the list is short at the counts where a step is short: one thread per panel
// over a chunk's sources kept 2 work-groups busy for 90 to 200 us.  Here a
// tile's terms are evaluated by all 256 threads, each on one panel and every
// 64th near source, and added in list order by a lane per panel and
// component, with the operations of the loop above (FP32: sums over kSegTile
// listed sources, added in FP64): the same partials, bit for bit.  FP64, 200
// panels, 2785 vortices: 200 -> 12 us; FP32, a batch of plates with up to
// 2040 panels: 35 -> 9.7 us.
constexpr int kRhsPG = 4;
// Larger bounds keep the kernel above: its segments and chunks fill the chip
// by themselves there, and a grid for the bound would be mostly idle groups.
constexpr int64_t kRhsSplitSrc = 32768;

template <typename T>
struct RhsTermsLds {
    T lx[256], ly[256], lg[256];
    T lt[256][kRhsPG][2];
    int wcount[4];
};

template <typename T>
__device__ __forceinline__ void rhs_terms(RhsTermsLds<T> &L, int64_t group, int64_t c, const T *__restrict__ sg,
                                          const double *__restrict__ x, const double *__restrict__ y,
                                          const int32_t *__restrict__ list, int64_t n_src, const PanelsSoA &pan,
                                          const RhsSeg *__restrict__ segs, double *__restrict__ part) {
    constexpr int kPer = kSegTile / kRhsPG;
    constexpr bool F32 = sizeof(T) == 4;
    static_assert(kSegTile == 128, "two tiles of the sums in 256 sources");
    auto &lx = L.lx;
    auto &ly = L.ly;
    auto &lg = L.lg;
    auto &lt = L.lt;
    auto &wcount = L.wcount;
    const RhsSeg S = segs[group / kPer];
    const int p0 = (int)(group % kPer) * kRhsPG;
    const int64_t lo = c * kRhsChunk, hi = min(n_src, lo + kRhsChunk);
    if (p0 >= S.count || (lo >= n_src && lo > 0)) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int pp = tid & (kRhsPG - 1), slot = tid / kRhsPG;
    const int64_t i = S.first + min(p0 + pp, S.count - 1);
    const double ox = F32 ? S.cx : 0.0, oy = F32 ? S.cy : 0.0;
    const T l0 = (T)(pan.lx[i] - ox), l1 = (T)(pan.ly[i] - oy);
    const T r0 = (T)(pan.rx[i] - ox), r1 = (T)(pan.ry[i] - oy);
    const T d0 = F32 ? (T)(pan.rx[i] - pan.lx[i]) : r0 - l0, d1 = F32 ? (T)(pan.ry[i] - pan.ly[i]) : r1 - l1;
    const T dd2 = fma(d0, d0, d1 * d1);
    const double rn2 = 4.0 * S.r * S.r;
    T acc = 0;  // lane (panel, component) of the first wave
    double sum = 0.0;
    auto add_terms = [&](int jj, int end) {
        const T *t = &lt[0][tid >> 1][tid & 1];
        for (; jj + 8 <= end; jj += 8) {
            T v[8], w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = t[(jj + e) * 2 * kRhsPG];
                w[e] = lg[jj + e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = fma(w[e], v[e], acc);
        }
        for (; jj < end; ++jj) acc = fma(lg[jj], t[jj * 2 * kRhsPG], acc);
        if (F32) {
            sum += (double)acc;
            acc = 0;
        }
    };
    for (int64_t base = lo; base < hi; base += 256) {
        const int64_t j = base + tid;
        bool near = false;
        T qx = 0, qy = 0, qg = 0;
        if (j < hi) {
            const int32_t k = list[j];
            const double px = x[k], py = y[k];
            qg = sg[k];
            const double ex = px - S.cx, ey = py - S.cy;
            near = ex * ex + ey * ey < rn2;
            qx = F32 ? (T)ex : (T)px;
            qy = F32 ? (T)ey : (T)py;
        }
        const uint64_t m = __ballot(near);
        if (lane == 0) wcount[wv] = __popcll(m);
        __syncthreads();
        int pos = __popcll(m & ((1ull << lane) - 1)), cnt = 0;
        const int half = wcount[0] + wcount[1];
        for (int q = 0; q < 4; ++q) {
            pos += q < wv ? wcount[q] : 0;
            cnt += wcount[q];
        }
        if (near) {
            lx[pos] = qx;
            ly[pos] = qy;
            lg[pos] = qg;
        }
        __syncthreads();
        for (int jj = slot; jj < cnt; jj += 256 / kRhsPG) {
            const T s00 = l0 - lx[jj], s01 = l1 - ly[jj];
            const T s10 = r0 - lx[jj], s11 = r1 - ly[jj];
            if constexpr (F32) {
                const T z = fma(s01, d0, -(s00 * d1));
                const T A = fma(s00, d0, s01 * d1);
                const T B = fma(s10, d0, s11 * d1);
                const T alpha = vx_atan2f(-dd2 * z, fma(z, z, A * B));
                const T q0 = fma(s00, s00, s01 * s01), q1 = fma(s10, s10, s11 * s11);
                const T beta = 0.34657359027997264f * __builtin_amdgcn_logf(q1 * __builtin_amdgcn_rcpf(q0));
                lt[jj][pp][0] = fma(alpha, d0, -(beta * d1));
                lt[jj][pp][1] = fma(beta, d0, alpha * d1);
            } else {
                const T z = fma(d0, s01, -(d1 * s00));
                const T A = fma(d0, s00, d1 * s01);
                const T B = fma(d0, s10, d1 * s11);
                const T alpha = atan(A / z) - atan(B / z);
                const T beta = 0.5 * log(fma(s10, s10, s11 * s11) / fma(s00, s00, s01 * s01));
                lt[jj][pp][0] = fma(d0, alpha, -(d1 * beta));
                lt[jj][pp][1] = fma(d1, alpha, d0 * beta);
            }
        }
        __syncthreads();
        if (tid < 2 * kRhsPG) {
            if (F32) add_terms(0, half);
            add_terms(F32 ? half : 0, cnt);
        }
        __syncthreads();
    }
    if (tid < 2 * kRhsPG && p0 + (tid >> 1) < S.count)
        part[(c * 2 + (tid & 1)) * pan.P + S.first + p0 + (tid >> 1)] = F32 ? sum : (double)acc;
}

// Sums of g w^{k+1}, w = 1 / (z_j - c), k < kLoc, over a work-group's sources
// (FP64; item(j, g, dx, dy) gives source j, or false to leave it out), in a
// fixed order: each thread its own sources, then the binary tree over the
// 256 threads, strides 128 to 1.  out gets the kLoc complex sums.
//
// Eight terms at a time go through LDS.  The tree used to be walked there,
// eight levels with a barrier and 16 read-add-writes each; now sixteen
// threads take a row, sixteen values each in the tree's order, and the last
// four levels are lane exchanges: the same sums.  A work-group whose threads
// have one source each (all of them, up to 131072 sources and 8192 listed
// ones) runs the terms as a loop with nothing kept in registers: the 48
// unrolled terms are 8 KB of code read once.  Both launches of a step at 2785
// vortices: 41 -> 6.4 us.
constexpr int kRedRow = 256 + 16;  // a row of the LDS stage: 16 doubles of padding split two rows over the banks

__device__ __forceinline__ void rhs_rows_out(const double *red, double *__restrict__ out) {
    const int tid = threadIdx.x, e = tid & 15;
    const double *row = red + (tid >> 4) * kRedRow + e;
    double a[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) a[m] = row[16 * m];
#pragma unroll
    for (int st = 8; st > 0; st >>= 1)
#pragma unroll
        for (int m = 0; m < st; ++m) a[m] += a[m + st];
    double r = a[0];
    for (int st = 8; st > 0; st >>= 1) r += __shfl_xor(r, st, 16);
    if (e == 0) out[tid >> 4] = r;
}

template <class Item>
__device__ __forceinline__ void rhs_expand(Item item, int64_t n, int64_t first, int64_t stride,
                                           double (*red)[16 * kRedRow], double *__restrict__ out) {
    const int tid = threadIdx.x;
    if (n <= stride) {
        double pr = 0.0, pi = 0.0, wr = 0.0, wi = 0.0, gj, dx, dy;
        if (first < n && item(first, gj, dx, dy)) {
            const double q2 = dx * dx + dy * dy;
            wr = dx / q2;
            wi = -dy / q2;
            pr = gj * wr;
            pi = gj * wi;
        }
#pragma unroll 1
        for (int k0 = 0; k0 < kLoc; k0 += 8) {
            double *r = red[(k0 >> 3) & 1];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                r[2 * q * kRedRow + tid] = 0.0 + pr;
                r[(2 * q + 1) * kRedRow + tid] = 0.0 + pi;
                const double npr = fma(wr, pr, -(wi * pi));
                pi = fma(wi, pr, wr * pi);
                pr = npr;
            }
            lds_barrier();  // the other buffer was last read before this one was written
            rhs_rows_out(r, out + 2 * k0);
        }
        return;
    }
    double sr[kLoc], si[kLoc];
#pragma unroll
    for (int k = 0; k < kLoc; ++k) sr[k] = si[k] = 0.0;
    for (int64_t j = first; j < n; j += stride) {
        double gj, dx, dy;
        if (!item(j, gj, dx, dy)) continue;
        const double q2 = dx * dx + dy * dy;
        const double wr = dx / q2, wi = -dy / q2;
        double pr = gj * wr, pi = gj * wi;
#pragma unroll
        for (int k = 0; k < kLoc; ++k) {
            sr[k] += pr;
            si[k] += pi;
            const double npr = fma(wr, pr, -(wi * pi));
            pi = fma(wi, pr, wr * pi);
            pr = npr;
        }
    }
#pragma unroll
    for (int k0 = 0; k0 < kLoc; k0 += 8) {
        double *r = red[(k0 >> 3) & 1];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            r[2 * q * kRedRow + tid] = sr[k0 + q];
            r[(2 * q + 1) * kRedRow + tid] = si[k0 + q];
        }
        lds_barrier();
        rhs_rows_out(r, out + 2 * k0);
    }
}

// The global expansion (far sources, work-groups [0, nfar)) and the segments'
// own (then nseg work-groups for each segment: listed sources at least 2 R_s
// from its centre) in one launch, neither needs the other.  Work-groups
// without a source leave no partial, rhs_groups counts those that do.
constexpr int kFarBlocks = 512;
constexpr int kSegBlocks = 32;

__host__ __device__ __forceinline__ int64_t rhs_groups(int64_t n, int64_t most) {
    const int64_t b = (n + 255) / 256;
    return b < most ? b : most;
}

__device__ __forceinline__ void rhs_expand_group(double (*red)[16 * kRedRow], int64_t group,
                                                 const double *__restrict__ x, const double *__restrict__ y,
                                                 const double *__restrict__ g, int64_t n_src, double cx, double cy,
                                                 double r2, const int32_t *__restrict__ list, int64_t n_list,
                                                 const RhsSeg *__restrict__ segs, int64_t nfar, int64_t nseg,
                                                 double *__restrict__ spart, double *__restrict__ spart_seg) {
    if (group < nfar) {
        const int64_t first = group * 256;
        if (first >= n_src) return;
        rhs_expand(
            [&](int64_t j, double &gj, double &dx, double &dy) {
                gj = g[j];
                dx = x[j] - cx;
                dy = y[j] - cy;
                return !(gj == 0 || !(dx * dx + dy * dy >= r2));
            },
            n_src, first + threadIdx.x, nfar * 256, red, spart + group * kLoc * 2);
    } else {
        const int64_t b = group - nfar, s = b / nseg, first = b % nseg * 256;
        if (first >= n_list) return;
        const RhsSeg S = segs[s];
        const double rn2 = 4.0 * S.r * S.r;
        rhs_expand(
            [&](int64_t t, double &gj, double &dx, double &dy) {
                const int32_t j = list[t];
                gj = g[j];
                dx = x[j] - S.cx;
                dy = y[j] - S.cy;
                return dx * dx + dy * dy >= rn2;
            },
            n_list, first + threadIdx.x, nseg * 256, red, spart_seg + (s * kSegBlocks + first / 256) * kLoc * 2);
    }
}

struct RhsExpand {
    const double *x, *y, *g;
    Cnt cn_src;
    double cx, cy, r2;
    const int32_t *list, *nlist;
    const RhsSeg *segs;
    int64_t nfar, nseg;
    double *spart, *spart_seg;
};

__global__ __launch_bounds__(256) void k_rhs_expand(RhsExpand A) {
    __shared__ double red[2][16 * kRedRow];
    rhs_expand_group(red, blockIdx.x, A.x, A.y, A.g, A.cn_src.get(), A.cx, A.cy, A.r2, A.list, *A.nlist, A.segs, A.nfar,
                     A.nseg, A.spart, A.spart_seg);
}

template <typename T>
__global__ __launch_bounds__(256) void k_right_part_terms(const T *__restrict__ sg, PanelsSoA pan,
                                                          double *__restrict__ part, RhsExpand A) {
    __shared__ RhsTermsLds<T> L;
    rhs_terms<T>(L, blockIdx.x, blockIdx.y, sg, A.x, A.y, A.list, *A.nlist, pan, A.segs, part);
}

// The pairs by terms (work-groups [0, nterm): nx groups of panels for each
// chunk) and the expansions in one launch: up to kRhsOneSrc sources neither
// fills the chip, and the expansions' 6 us pass beside the pairs.  The pairs
// then run with the expansions' registers and LDS, which a longer list would
// feel (a batch with some 20000 sources each: 23 us against 9.4 + 8).
constexpr int64_t kRhsOneSrc = 8192;

template <typename T>
__global__ __launch_bounds__(256) void k_right_part_all(const T *__restrict__ sg, PanelsSoA pan, int64_t nx,
                                                        int64_t nterm, double *__restrict__ part, RhsExpand A) {
    __shared__ __align__(16) union Lds {
        RhsTermsLds<T> terms;
        double red[2][16 * kRedRow];
        __device__ Lds() {}
    } L;
    const int64_t w = blockIdx.x;
    if (w < nterm)
        rhs_terms<T>(L.terms, w % nx, w / nx, sg, A.x, A.y, A.list, *A.nlist, pan, A.segs, part);
    else
        rhs_expand_group(L.red, w - nterm, A.x, A.y, A.g, A.cn_src.get(), A.cx, A.cy, A.r2, A.list, *A.nlist, A.segs,
                         A.nfar, A.nseg, A.spart, A.spart_seg);
}

// S_k over the work-group partials: one work-group per real/imaginary part of
// each term, a strided pass per thread and a tree in LDS (fixed order).
__global__ __launch_bounds__(256) void k_rhs_far_final(const double *__restrict__ spart, Cnt cn_src, int64_t nfar,
                                                       double *__restrict__ S) {
    __shared__ double r[256];
    const int t = blockIdx.x;
    const int64_t nblk = rhs_groups(cn_src.get(), nfar);  // the others would add exact zeros
    double a = 0.0;
    for (int64_t b = threadIdx.x; b < nblk; b += 256) a += spart[b * 2 * kLoc + t];
    r[threadIdx.x] = a;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) r[threadIdx.x] += r[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) S[t] = r[0];
}

// Binomials c[q][m] = C(m + q, m) for m + q < kLoc (below 2^44, so exact),
// else 0; a step of the shift reads a row.
struct Binom {
    double c[kLoc][kLoc];
};
constexpr Binom binomials() {
    Binom b{};
    for (int m = 0; m < kLoc; ++m) b.c[0][m] = 1.0;
    for (int q = 1; q < kLoc; ++q)
        for (int m = 0; m + q < kLoc; ++m) b.c[q][m] = b.c[q - 1][m] + (m > 0 ? b.c[q][m - 1] : 0.0);
    return b;
}
__device__ const Binom kBinom = binomials();

// Each segment's coefficients about c_s: the global S shifted exactly,
//   sum_{k >= m} S_k C(k, m) (c_s - c)^{k - m},
// plus its own sources' partials (fixed order).  Thread m < kLoc.
__device__ __forceinline__ void rhs_seg_coeff(const double *__restrict__ spart, int nb, const double *lS, double er,
                                              double ei, int m, double &ar, double &ai) {
    ar = ai = 0.0;
    double pr = 1.0, pi = 0.0;  // (c_s - c)^{k - m}
#pragma unroll 12
    for (int q = 0; q < kLoc; ++q) {
        const int k = m + q < kLoc ? m + q : kLoc - 1;
        const double bin = kBinom.c[q][m];
        const double tr = pr * bin, ti = pi * bin;
        const double sr = ar + fma(tr, lS[2 * k], -(ti * lS[2 * k + 1]));
        const double si = ai + fma(ti, lS[2 * k], tr * lS[2 * k + 1]);
        ar = m + q < kLoc ? sr : ar;
        ai = m + q < kLoc ? si : ai;
        const double npr = fma(er, pr, -(ei * pi));
        pi = fma(ei, pr, er * pi);
        pr = npr;
    }
#pragma unroll 8
    for (int b = 0; b < nb; ++b) {
        const double *q = spart + ((int64_t)b * kLoc + m) * 2;
        ar += q[0];
        ai += q[1];
    }
}

__global__ __launch_bounds__(64) void k_rhs_seg_final(const double *__restrict__ spart, const double *__restrict__ S,
                                                      double cx, double cy, const RhsSeg *__restrict__ segs,
                                                      const int32_t *__restrict__ nlist, int64_t nseg,
                                                      double *__restrict__ Ss) {
    __shared__ double lS[2 * kLoc];
    for (int t = threadIdx.x; t < 2 * kLoc; t += 64) lS[t] = S[t];
    __syncthreads();
    const int m = threadIdx.x;
    if (m >= kLoc) return;
    const RhsSeg G = segs[blockIdx.x];
    double ar, ai;
    rhs_seg_coeff(spart + (int64_t)blockIdx.x * kSegBlocks * kLoc * 2, (int)rhs_groups(*nlist, nseg), lS, G.cx - cx,
                  G.cy - cy, m, ar, ai);
    Ss[((int64_t)blockIdx.x * kLoc + m) * 2] = ar;
    Ss[((int64_t)blockIdx.x * kLoc + m) * 2 + 1] = ai;
}

// Sum of the chunk partials part[(c * 2 + q) * m + i] for one output i per
// work-group: a strided pass per thread, then a tree in LDS (fixed order).
__device__ __forceinline__ void chunk_sum2(const double *__restrict__ part, int64_t nchunk, int64_t m, int64_t i,
                                           double &a, double &b) {
    __shared__ double r[2][kTile];
    double x0 = 0.0, x1 = 0.0;
    for (int64_t c = threadIdx.x; c < nchunk; c += kTile) {
        x0 += part[(c * 2 + 0) * m + i];
        x1 += part[(c * 2 + 1) * m + i];
    }
    if (nchunk <= 64) {  // the tree's first two levels would add zeros
        if (threadIdx.x < 64) {
            for (int st = 32; st > 0; st >>= 1) {
                x0 += __shfl_xor(x0, st, 64);
                x1 += __shfl_xor(x1, st, 64);
            }
        }
        a = x0;  // of thread 0, the one that goes on
        b = x1;
        return;
    }
    r[0][threadIdx.x] = x0;
    r[1][threadIdx.x] = x1;
    __syncthreads();
    for (int st = kTile / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            r[0][threadIdx.x] += r[0][threadIdx.x + st];
            r[1][threadIdx.x] += r[1][threadIdx.x + st];
        }
        __syncthreads();
    }
    a = r[0][0];
    b = r[1][0];
}

// Panel i's entry from its near sums (y0, y1) and its segment's coefficients
// S about (cx, cy); inv[k] = 1 / (k + 1).
__device__ __forceinline__ double rhs_entry(const PanelsSoA &pan, int64_t i, double cx, double cy, const double *S,
                                            const double *inv, double y0, double y1, double vinf_x, double vinf_y) {
    const double d0 = pan.rx[i] - pan.lx[i], d1 = pan.ry[i] - pan.ly[i];
    const double mnog = 1 / (2 * kPi * fma(d0, d0, d1 * d1));
    // W = sum_k (i S_k / 2 pi) Q_k / (k + 1), u = Re W, v = -Im W
    const double ar = pan.rx[i] - cx, ai = pan.ry[i] - cy;  // a = z_r - c_s
    const double br = pan.lx[i] - cx, bi = pan.ly[i] - cy;  // b = z_l - c_s
    double qr = 1.0, qi = 0.0;                               // Q_0
    double bkr = 1.0, bki = 0.0;                             // b^k
    double wr = 0.0, wi = 0.0;
#pragma unroll 4
    for (int k = 0; k < kLoc; ++k) {
        if (k > 0) {
            const double nbr = fma(br, bkr, -(bi * bki));
            bki = fma(br, bki, bi * bkr);
            bkr = nbr;
            const double nqr = fma(ar, qr, -(ai * qi)) + bkr;
            qi = fma(ar, qi, ai * qr) + bki;
            qr = nqr;
        }
        const double sr = S[2 * k], si = S[2 * k + 1];
        wr = fma(fma(qr, sr, -(qi * si)), inv[k], wr);
        wi = fma(fma(sr, qi, si * qr), inv[k], wi);
    }
    // times i / (2 pi)
    const double uf = -wi / (2 * kPi), vf = -(wr / (2 * kPi));
    const double u = fma(mnog, y0, uf) + vinf_x, v = fma(mnog, y1, vf) + vinf_y;
    return -fma(u, pan.tx[i], v * pan.ty[i]);
}

// One work-group per panel: the near chunk partials, plus the panel average
// of its segment's expansion (thread 0).  Only the chunks of the near list's
// length hold partials (the grid is sized for its bound); the others would
// add exact zeros.
__global__ __launch_bounds__(kTile) void k_right_part_final(const double *__restrict__ part, int64_t nchunk,
                                                            const int32_t *__restrict__ nlist, PanelsSoA pan,
                                                            const double *__restrict__ Ss,
                                                            const RhsSeg *__restrict__ segs,
                                                            const int32_t *__restrict__ seg_of, double vinf_x,
                                                            double vinf_y, double *__restrict__ R) {
    __shared__ double S[2 * kLoc], inv[kLoc];
    const int64_t i = blockIdx.x;
    const int64_t used = ((int64_t)*nlist + kRhsChunk - 1) / kRhsChunk;
    const int32_t sg = seg_of[i];
    if (threadIdx.x < 2 * kLoc) S[threadIdx.x] = Ss[(int64_t)sg * 2 * kLoc + threadIdx.x];
    if (threadIdx.x < kLoc) inv[threadIdx.x] = 1.0 / (double)(threadIdx.x + 1);
    __syncthreads();
    double y0, y1;
    chunk_sum2(part, used < nchunk ? used : nchunk, pan.P, i, y0, y1);
    if (threadIdx.x != 0) return;
    R[i] = rhs_entry(pan, i, segs[sg].cx, segs[sg].cy, S, inv, y0, y1, vinf_x, vinf_y);
}

// The three finals in one launch for at most kFewGroups work-groups of far
// sources: every panel's work-group adds up the global coefficients (32 lanes
// each, the tree of k_rhs_far_final without its levels of zeros), shifts them
// to the panel's segment while another wave adds the near partials, and takes
// the average.  200 panels, 2785 vortices: 4.5 + 5.1 + 5.8 us and two gaps -> 12.3
// us.
constexpr int64_t kFewGroups = 32;

__global__ __launch_bounds__(256) void k_right_part_final_few(
    const double *__restrict__ part, int64_t nchunk, const int32_t *__restrict__ nlist, PanelsSoA pan,
    const double *__restrict__ spart, const double *__restrict__ spart_seg, Cnt cn_src, int64_t nfar, int64_t nseg,
    double cx, double cy, const RhsSeg *__restrict__ segs, const int32_t *__restrict__ seg_of, double vinf_x,
    double vinf_y, double *__restrict__ R) {
    __shared__ double S[2 * kLoc], Ss[2 * kLoc], inv[kLoc], y[2];
    const int64_t i = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int32_t sg = seg_of[i], nl = *nlist;
    const RhsSeg G = segs[sg];
    const int nblk = (int)rhs_groups(cn_src.get(), nfar), b = tid & 31;
    double v[2 * kLoc / 8];
#pragma unroll
    for (int r = 0; r < 2 * kLoc / 8; ++r)
        v[r] = b < nblk ? 0.0 + spart[(int64_t)b * 2 * kLoc + 8 * r + (tid >> 5)] : 0.0;
#pragma unroll
    for (int r = 0; r < 2 * kLoc / 8; ++r) {
        for (int st = 16; st > 0; st >>= 1) v[r] += __shfl_xor(v[r], st, 32);
        if (b == 0) S[8 * r + (tid >> 5)] = v[r];
    }
    __syncthreads();
    if (wv == 0 && lane < kLoc) {
        double ar, ai;
        rhs_seg_coeff(spart_seg + (int64_t)sg * kSegBlocks * kLoc * 2, (int)rhs_groups(nl, nseg), S, G.cx - cx,
                      G.cy - cy, lane, ar, ai);
        Ss[2 * lane] = ar;
        Ss[2 * lane + 1] = ai;
    } else if (wv == 1) {
        const int64_t used = ((int64_t)nl + kRhsChunk - 1) / kRhsChunk;
        const bool on = lane < (used < nchunk ? used : nchunk);
        double x0 = on ? 0.0 + part[((int64_t)lane * 2 + 0) * pan.P + i] : 0.0;
        double x1 = on ? 0.0 + part[((int64_t)lane * 2 + 1) * pan.P + i] : 0.0;
        for (int st = 32; st > 0; st >>= 1) {
            x0 += __shfl_xor(x0, st, 64);
            x1 += __shfl_xor(x1, st, 64);
        }
        if (lane == 0) {
            y[0] = x0;
            y[1] = x1;
        }
    } else if (wv == 2 && lane < kLoc) {
        inv[lane] = 1.0 / (double)(lane + 1);
    }
    __syncthreads();
    if (tid == 0) R[i] = rhs_entry(pan, i, G.cx, G.cy, Ss, inv, y[0], y[1], vinf_x, vinf_y);
}

// ---- A19: src/kernel.cu:1434-1475, split over source chunks ---------------
__global__ __launch_bounds__(kTile) void k_probe_partial(const double *__restrict__ sx, const double *__restrict__ sy,
                                                         const double *__restrict__ sg, Cnt cn_src, int64_t chunk,
                                                         const double *__restrict__ px, const double *__restrict__ py,
                                                         int64_t m, double eps2, double *__restrict__ part) {
    __shared__ Src4<double> ls[kTile];
    using A = Arith<double>;
    const int64_t n_src = cn_src.get();
    const int64_t i = (int64_t)blockIdx.x * kTile + threadIdx.x;
    const int64_t c = blockIdx.y;
    const int64_t lo = c * chunk, hi = min(n_src, lo + chunk);
    const double a0 = i < m ? px[i] : 0.0, a1 = i < m ? py[i] : 0.0;
    const bool tame = ordinary(a0) && ordinary(a1) && ordinary_eps2(eps2);
    double su = 0.0, sv = 0.0;
    for (int64_t base = lo; base < hi; base += kTile) {
        __syncthreads();
        const int64_t j = base + threadIdx.x;
        Src4<double> s;
        s.x = j < hi ? sx[j] : A::kFar;
        s.y = j < hi ? sy[j] : A::kFar;
        s.g = j < hi ? sg[j] : 0.0;
        s.pad = 0.0;
        ls[threadIdx.x] = s;
        const bool plain = __syncthreads_or(!(tame && ordinary(s.x) && ordinary(s.y) && ordinary(s.g)));
        const int cnt = (int)min((int64_t)kTile, hi - base);
        if (plain) {
            for (int jj = 0; jj < cnt; ++jj) {
                const Src4<double> q = ls[jj];
                const double dx = a0 - q.x, dy = a1 - q.y;
                const double w = q.g / A::max_(dx * dx + dy * dy, eps2);
                sv += w * dx;
                su -= w * dy;
            }
            continue;
        }
        for (int jj = 0; jj < cnt; ++jj) {
            const Src4<double> q = ls[jj];
            const double dx = a0 - q.x, dy = a1 - q.y;
            const double w = A::div(q.g, A::max_(dx * dx + dy * dy, eps2));
            sv += w * dx;
            su -= w * dy;
        }
    }
    if (i < m) {
        part[(c * 2 + 0) * m + i] = su;
        part[(c * 2 + 1) * m + i] = sv;
    }
}

// Mixed precision: each pair's separation is taken in FP64 and rounded once,
// so a probe next to a source keeps FP32's relative accuracy in the
// separation (FP32 positions would lose it in the coordinates' magnitude:
// 1e-7 of |x| against separations down to the core radius); kernel and sums
// in FP32 per tile, FP64 across tiles.
__global__ __launch_bounds__(kTile) void k_probe_partial_mixed(
    const double *__restrict__ sx, const double *__restrict__ sy, const double *__restrict__ sg, Cnt cn_src,
    int64_t chunk, const double *__restrict__ px, const double *__restrict__ py, int64_t m, float eps2,
    double *__restrict__ part) {
    __shared__ double lx[kTile], ly[kTile];
    __shared__ float lg[kTile];
    using A = Arith<float>;
    const int64_t n_src = cn_src.get();
    const int64_t i = (int64_t)blockIdx.x * kTile + threadIdx.x;
    const int64_t c = blockIdx.y;
    const int64_t lo = c * chunk, hi = min(n_src, lo + chunk);
    const double a0 = i < m ? px[i] : 0.0, a1 = i < m ? py[i] : 0.0;
    double au = 0.0, av = 0.0;
    for (int64_t base = lo; base < hi; base += kTile) {
        __syncthreads();
        const int64_t j = base + threadIdx.x;
        lx[threadIdx.x] = j < hi ? sx[j] : 0.0;
        ly[threadIdx.x] = j < hi ? sy[j] : 0.0;
        lg[threadIdx.x] = j < hi ? (float)sg[j] : 0.f;
        __syncthreads();
        const int cnt = (int)min((int64_t)kTile, hi - base);
        float su = 0.f, sv = 0.f;
        for (int jj = 0; jj < cnt; ++jj) {
            const float dx = (float)(a0 - lx[jj]), dy = (float)(a1 - ly[jj]);
            const float w = A::div(lg[jj], A::max_(dx * dx + dy * dy, eps2));
            sv += w * dx;
            su -= w * dy;
        }
        au += (double)su;
        av += (double)sv;
    }
    if (i < m) {
        part[(c * 2 + 0) * m + i] = au;
        part[(c * 2 + 1) * m + i] = av;
    }
}

// One work-group per probe.
__global__ __launch_bounds__(kTile) void k_probe_final(const double *__restrict__ part, int64_t nchunk, int64_t m,
                                                       double vinf_x, double vinf_y, double *__restrict__ u,
                                                       double *__restrict__ v) {
    const int64_t i = blockIdx.x;
    double a, b;
    chunk_sum2(part, nchunk, m, i, a, b);
    if (threadIdx.x != 0) return;
    u[i] = a / (2 * kPi) + vinf_x;
    v[i] = b / (2 * kPi) + vinf_y;
}

// ---------------------------------------------------------------------------
static bool mixed(const vx_case *c) { return c->prm.precision == VX_PREC_MIXED; }

// Split [0, n_src) into chunks of whole tiles so that tgt_blocks * chunks
// gives a few thousand work-groups.
static void split(int64_t n_src, int64_t tgt_blocks, int64_t *chunk, int64_t *nchunk) {
    const int64_t tiles = (n_src + kTile - 1) / kTile;
    int64_t want = (4096 + tgt_blocks - 1) / tgt_blocks;
    if (want < 1) want = 1;
    if (want > tiles) want = tiles > 0 ? tiles : 1;
    const int64_t tiles_per = (tiles + want - 1) / want;
    *chunk = (tiles_per > 0 ? tiles_per : 1) * kTile;
    *nchunk = n_src > 0 ? (n_src + *chunk - 1) / *chunk : 1;
}

int launch_biot_savart(vx_case *c, int64_t n_tgt, int64_t n_src, double vinf_x, double vinf_y) {
    return launch_biot_savart(c, host_cnt(n_tgt), host_cnt(n_src), vinf_x, vinf_y);
}

// Targets per thread of the direct kernels: the case's tuning (see
// vx_case_autotune) or one.  Every choice sums each target's sources in the
// same order, so the results do not depend on it.  Sources come as scalar
// operands, so more targets per thread save no loads: 60001 vortices take
// 1.02, 1.11, 1.44 and 1.53 ms (Biot-Savart, FP32) with 1, 2, 4 and 8, and
// 2.39, 2.45, 2.63 and 3.08 ms in FP64 (its diffusion 5.1, 5.4, 5.9, 7.0).
int direct_tpt_default() { return 1; }
bool direct_uses_tpt(bool f32, int64_t n_src) { return f32 || n_src > kOrdered; }

static int tpt_of(int want) {
    if (want == 1 || want == 2 || want == 4 || want == 8) return want;
    return direct_tpt_default();
}

// FP64: the ordered kernels up to kOrdered sources, the split ones above.  A
// device count's bound may lie above it while the count does not: then both
// are queued and the live count decides in the kernels.
static bool takes_ordered(Cnt n_src) { return n_src.dev || n_src.ub <= kOrdered; }
static bool takes_split(Cnt n_src) { return n_src.ub > kOrdered; }
// 16 targets per ordered work-group while that makes no more than one for each
// CU, else 32: at 4000 vortices 40 and 52 us (Biot-Savart, diffusion) against
// 47 and 82 with 32, at 6000 (two rounds of work-groups) 114 and 151 against
// 73 and 126.  A device count goes by the host's last count (a captured step is
// kept for one of the two); the results do not depend on the choice.
constexpr int64_t kOrdNarrow = 4096;
static bool ord_narrow(const vx_case *c, Cnt n_tgt) { return (n_tgt.dev ? c->n : n_tgt.ub) <= kOrdNarrow; }
bool direct_narrow(const vx_case *c) { return !mixed(c) && c->n <= kOrdNarrow; }

template <typename T, int TPT>
static void bs_launch(vx_case *c, const T *sx, const T *sy, const T *sg, Cnt n_src, Cnt n_tgt, T eps2) {
    hipLaunchKernelGGL((k_biot_savart<T, TPT>), dim3((unsigned)direct_blocks<T>(n_tgt, n_src, TPT)), dim3(kTile), 0,
                       c->stream, sx, sy, sg, n_src, n_tgt, eps2, c->partial.p);
}

template <typename T>
static void bs_dispatch(vx_case *c, int tpt, const T *sx, const T *sy, const T *sg, Cnt n_src, Cnt n_tgt, T eps2) {
    switch (tpt) {
        case 1: bs_launch<T, 1>(c, sx, sy, sg, n_src, n_tgt, eps2); break;
        case 2: bs_launch<T, 2>(c, sx, sy, sg, n_src, n_tgt, eps2); break;
        case 4: bs_launch<T, 4>(c, sx, sy, sg, n_src, n_tgt, eps2); break;
        default: bs_launch<T, 8>(c, sx, sy, sg, n_src, n_tgt, eps2); break;
    }
}

int launch_biot_savart(vx_case *c, Cnt n_tgt, Cnt n_src, double vinf_x, double vinf_y) {
    if (n_tgt.ub <= 0) return 0;
    tree_d_changed(c);  // d from direct sums: a tree's sorted copy no longer matches
    const double eps2 = c->prm.ve_size * c->prm.ve_size;
    const dim3 gsum((unsigned)((n_tgt.ub + 63) / 64));
    if (mixed(c)) {
        if (c->partial.ensure(direct_partials<float>(n_tgt, n_src, 6), c->stream) || launch_pack_f32(c, n_src))
            return 1;
        bs_dispatch<float>(c, tpt_of(c->tune.tpt_bs), c->xf.p, c->yf.p, c->gf.p, n_src, n_tgt,
                           (float)eps2);
        hipLaunchKernelGGL(k_bs_sum<float>, gsum, dim3(256), 0, c->stream, c->partial.p, n_src, n_tgt, vinf_x, vinf_y,
                           c->u.p, c->v.p, c->d.p);
    } else {
        if (takes_ordered(n_src)) {
            if (ord_narrow(c, n_tgt))
                hipLaunchKernelGGL((k_biot_savart_ordered<16, 2>), dim3((unsigned)((n_tgt.ub + 15) / 16)), dim3(1024), 0,
                                   c->stream, c->x.p, c->y.p, c->g.p, n_src, n_tgt, eps2, vinf_x, vinf_y, c->u.p,
                                   c->v.p, c->d.p);
            else
                hipLaunchKernelGGL((k_biot_savart_ordered<32, 4>), dim3((unsigned)((n_tgt.ub + 31) / 32)), dim3(1024), 0,
                                   c->stream, c->x.p, c->y.p, c->g.p, n_src, n_tgt, eps2, vinf_x, vinf_y, c->u.p,
                                   c->v.p, c->d.p);
        }
        if (takes_split(n_src)) {
            if (c->partial.ensure(direct_partials<double>(n_tgt, n_src, 6), c->stream)) return 1;
            bs_dispatch<double>(c, tpt_of(c->tune.tpt_bs), c->x.p, c->y.p, c->g.p, n_src, n_tgt,
                                eps2);
            hipLaunchKernelGGL(k_bs_sum<double>, gsum, dim3(256), 0, c->stream, c->partial.p, n_src, n_tgt, vinf_x,
                               vinf_y, c->u.p, c->v.p, c->d.p);
        }
    }
    VX_CHECK(hipGetLastError());
    return 0;
}

int launch_diffusion(vx_case *c, int64_t n_tgt, int64_t n_src) {
    return launch_diffusion(c, host_cnt(n_tgt), host_cnt(n_src));
}

template <typename T, int TPT>
static void diff_launch(vx_case *c, const T *sx, const T *sy, const T *sg, Cnt n_src, Cnt n_tgt, T thr) {
    hipLaunchKernelGGL((k_diffusion<T, TPT>), dim3((unsigned)direct_blocks<T>(n_tgt, n_src, TPT)), dim3(kTile), 0,
                       c->stream, sx, sy, sg, n_src, n_tgt, c->d.p, thr, c->partial.p);
}

template <typename T>
static void diff_dispatch(vx_case *c, int tpt, const T *sx, const T *sy, const T *sg, Cnt n_src, Cnt n_tgt, T thr) {
    switch (tpt) {
        case 1: diff_launch<T, 1>(c, sx, sy, sg, n_src, n_tgt, thr); break;
        case 2: diff_launch<T, 2>(c, sx, sy, sg, n_src, n_tgt, thr); break;
        case 4: diff_launch<T, 4>(c, sx, sy, sg, n_src, n_tgt, thr); break;
        default: diff_launch<T, 8>(c, sx, sy, sg, n_src, n_tgt, thr); break;
    }
}

int launch_diffusion(vx_case *c, Cnt n_tgt, Cnt n_src, bool packed) {
    // No sources (vx_diffusion takes any count below the capacity): nothing to
    // add, and the split and the ordered kernels' staging need one at least.
    if (n_tgt.ub <= 0 || n_src.ub <= 0) return 0;
    const double thr = 0.001 * c->prm.ve_size;
    const dim3 gsum((unsigned)((n_tgt.ub + 63) / 64));
    if (mixed(c)) {
        if (c->partial.ensure(direct_partials<float>(n_tgt, n_src, 3), c->stream) ||
            (!packed && launch_pack_f32(c, n_src)))
            return 1;
        diff_dispatch<float>(c, tpt_of(c->tune.tpt_diff), c->xf.p, c->yf.p, c->gf.p, n_src, n_tgt,
                             (float)(thr * thr));
        hipLaunchKernelGGL(k_diff_sum<float>, gsum, dim3(256), 0, c->stream, c->partial.p, n_src, n_tgt, c->d.p,
                           c->prm.nu, c->u.p, c->v.p);
    } else {
        if (takes_ordered(n_src)) {
            if (ord_narrow(c, n_tgt))
                hipLaunchKernelGGL((k_diffusion_ordered<16, 2>), dim3((unsigned)((n_tgt.ub + 15) / 16)), dim3(1024), 0,
                                   c->stream, c->x.p, c->y.p, c->g.p, n_src, n_tgt, c->d.p, c->prm.nu, thr, c->u.p,
                                   c->v.p);
            else
                hipLaunchKernelGGL((k_diffusion_ordered<32, 2>), dim3((unsigned)((n_tgt.ub + 31) / 32)), dim3(1024), 0,
                                   c->stream, c->x.p, c->y.p, c->g.p, n_src, n_tgt, c->d.p, c->prm.nu, thr, c->u.p,
                                   c->v.p);
        }
        if (takes_split(n_src)) {
            if (c->partial.ensure(direct_partials<double>(n_tgt, n_src, 3), c->stream)) return 1;
            diff_dispatch<double>(c, tpt_of(c->tune.tpt_diff), c->x.p, c->y.p, c->g.p, n_src, n_tgt,
                                  thr);
            hipLaunchKernelGGL(k_diff_sum<double>, gsum, dim3(256), 0, c->stream, c->partial.p, n_src, n_tgt, c->d.p,
                               c->prm.nu, c->u.p, c->v.p);
        }
    }
    VX_CHECK(hipGetLastError());
    return 0;
}

int launch_right_part(vx_case *c, int64_t n_src, double vinf_x, double vinf_y) {
    return launch_right_part(c, host_cnt(n_src), vinf_x, vinf_y);
}

int launch_right_part(vx_case *c, Cnt cn_src, double vinf_x, double vinf_y) {
    const int64_t P = c->P, K = c->nseg;
    hipStream_t st = c->stream;
    const int64_t n_src = cn_src.ub;  // bound: grids, list and partial sizes
    const int64_t nchunk = n_src > 0 ? (n_src + kRhsChunk - 1) / kRhsChunk : 1;
    const size_t ns_far = (size_t)(2 * kLoc * kFarBlocks), ns_glob = 2 * kLoc,
                 ns_seg = (size_t)(2 * kLoc * kSegBlocks * K), ns_segS = (size_t)(2 * kLoc * K);
    if (c->partial.ensure((size_t)(2 * nchunk * P), st) || c->rp.ensure((size_t)P, st) ||
        c->lists.ensure((size_t)(n_src > 0 ? n_src : 1), st) || c->dcount.ensure(16, st) ||
        c->rhs_s.ensure(ns_far + ns_glob + ns_seg + ns_segS, st))
        return 1;
    const vx_params &p = c->prm;
    const double cx = 0.5 * (p.px_min + p.px_max), cy = 0.5 * (p.py_min + p.py_max);
    const double wx = p.px_max - p.px_min, wy = p.py_max - p.py_min;
    const double rnear2 = wx * wx + wy * wy;  // (2 R_b)^2
    int32_t *nlist = (int32_t *)(c->dcount.p + 7);
    double *S = c->rhs_s.p + ns_far, *spart = S + ns_glob, *Ss = spart + ns_seg;
    // sources nearer than 2 R_b, in index order
    {
        const RhsNear pred{c->x.p, c->y.p, c->g.p, cx, cy, rnear2};
        if (c->ptmp.ensure((size_t)prim::tiles_of(n_src) + 1, st)) return 1;
        VX_CHECK(prim::select_flags(prim::pred_flag(pred, cn_src), n_src, prim::WriteIndex{c->lists.p}, c->ptmp.p,
                                    nlist, st));
    }
    // pairs within 2 R_s of each segment
    if (mixed(c) && launch_pack_f32(c, cn_src)) return 1;
    // the global expansion (sources beyond 2 R_b), the segments' own
    // sources, and below each segment's total about c_s
    const int64_t nfar = rhs_groups(n_src, kFarBlocks), nseg = rhs_groups(n_src, kSegBlocks);
    const RhsExpand E{c->x.p, c->y.p, c->g.p, cn_src, cx, cy, rnear2, c->lists.p, nlist, c->segs, nfar, nseg,
                      c->rhs_s.p, spart};
    const int64_t nx = K * (kSegTile / kRhsPG), nterm = nx * nchunk;
    if (n_src <= kRhsOneSrc) {
        const dim3 grid((unsigned)(nterm + nfar + K * nseg));
        if (mixed(c))
            hipLaunchKernelGGL(k_right_part_all<float>, grid, dim3(256), 0, st, c->gf.p, c->pan, nx, nterm,
                               c->partial.p, E);
        else
            hipLaunchKernelGGL(k_right_part_all<double>, grid, dim3(256), 0, st, c->g.p, c->pan, nx, nterm,
                               c->partial.p, E);
    } else {
        const dim3 gterms((unsigned)nx, (unsigned)nchunk), gseg((unsigned)K, (unsigned)nchunk);
        if (n_src <= kRhsSplitSrc && mixed(c))
            hipLaunchKernelGGL(k_right_part_terms<float>, gterms, dim3(256), 0, st, c->gf.p, c->pan, c->partial.p, E);
        else if (n_src <= kRhsSplitSrc)
            hipLaunchKernelGGL(k_right_part_terms<double>, gterms, dim3(256), 0, st, c->g.p, c->pan, c->partial.p, E);
        else if (mixed(c))
            hipLaunchKernelGGL(k_right_part_partial<float>, gseg, dim3(kSegTile), 0, st, c->xf.p, c->yf.p, c->gf.p,
                               c->x.p, c->y.p, c->lists.p, nlist, c->pan, c->segs, c->partial.p);
        else
            hipLaunchKernelGGL(k_right_part_partial<double>, gseg, dim3(kSegTile), 0, st, c->x.p, c->y.p, c->g.p,
                               c->x.p, c->y.p, c->lists.p, nlist, c->pan, c->segs, c->partial.p);
        hipLaunchKernelGGL(k_rhs_expand, dim3((unsigned)(nfar + K * nseg)), dim3(256), 0, st, E);
    }
    VX_CHECK(hipGetLastError());
    if (nfar <= kFewGroups) {
        static_assert(kFewGroups * 256 <= 64 * kRhsChunk, "the near chunks fit a wave");
        hipLaunchKernelGGL(k_right_part_final_few, dim3((unsigned)P), dim3(256), 0, st, c->partial.p, nchunk, nlist,
                           c->pan, c->rhs_s.p, spart, cn_src, nfar, nseg, cx, cy, c->segs, c->seg_of, vinf_x, vinf_y,
                           c->rp.p);
        VX_CHECK(hipGetLastError());
        return 0;
    }
    hipLaunchKernelGGL(k_rhs_far_final, dim3(2 * kLoc), dim3(256), 0, st, c->rhs_s.p, cn_src, nfar, S);
    hipLaunchKernelGGL(k_rhs_seg_final, dim3((unsigned)K), dim3(64), 0, st, spart, S, cx, cy, c->segs, nlist, nseg, Ss);
    VX_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_right_part_final, dim3((unsigned)P), dim3(kTile), 0, st, c->partial.p, nchunk, nlist, c->pan,
                       Ss, c->segs, c->seg_of, vinf_x, vinf_y, c->rp.p);
    VX_CHECK(hipGetLastError());
    return 0;
}

// Probe chunking: at most max_part doubles of split-K partials (2 per probe
// and chunk); max_part <= 0 lets the split choose.
void probe_split(int64_t m, int64_t n_src, int64_t max_part, int64_t *chunk, int64_t *nchunk) {
    const int64_t tb = (m + kTile - 1) / kTile;
    split(n_src, tb, chunk, nchunk);
    if (max_part > 0 && 2 * *nchunk * m > max_part) {
        const int64_t want = max_part / (2 * m) > 1 ? max_part / (2 * m) : 1;
        const int64_t tiles = (n_src + kTile - 1) / kTile;
        const int64_t tiles_per = (tiles + want - 1) / want;
        *chunk = (tiles_per > 0 ? tiles_per : 1) * kTile;
        *nchunk = n_src > 0 ? (n_src + *chunk - 1) / *chunk : 1;
    }
}

int launch_probe_to(vx_case *c, const double *px, const double *py, int64_t m, int64_t n_src, double vinf_x,
                    double vinf_y, double *pu, double *pv, double *part, int64_t max_part) {
    return launch_probe_to(c, px, py, m, host_cnt(n_src), vinf_x, vinf_y, pu, pv, part, max_part);
}

int launch_probe_to(vx_case *c, const double *px, const double *py, int64_t m, Cnt cn_src, double vinf_x,
                    double vinf_y, double *pu, double *pv, double *part, int64_t max_part) {
    if (m <= 0) return 0;
    const int64_t tb = (m + kTile - 1) / kTile;
    const int64_t n_src = cn_src.ub;  // the chunking follows the bound
    int64_t chunk, nchunk;
    probe_split(m, n_src, max_part, &chunk, &nchunk);
    const double eps2 = c->prm.ve_size * c->prm.ve_size;
    const dim3 grid((unsigned)tb, (unsigned)nchunk);
    if (mixed(c)) {
        hipLaunchKernelGGL(k_probe_partial_mixed, grid, dim3(kTile), 0, c->stream, c->x.p, c->y.p, c->g.p, cn_src,
                           chunk, px, py, m, (float)eps2, part);
    } else {
        hipLaunchKernelGGL(k_probe_partial, grid, dim3(kTile), 0, c->stream, c->x.p, c->y.p,
                           c->g.p, cn_src, chunk, px, py, m, eps2, part);
    }
    VX_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_probe_final, dim3((unsigned)m), dim3(kTile), 0, c->stream, part, nchunk, m, vinf_x, vinf_y,
                       pu, pv);
    VX_CHECK(hipGetLastError());
    return 0;
}

int launch_probe(vx_case *c, int64_t m, int64_t n_src, double vinf_x, double vinf_y) {
    if (m <= 0) return 0;
    int64_t chunk, nchunk;
    probe_split(m, n_src, 0, &chunk, &nchunk);
    if (c->partial.ensure((size_t)(2 * nchunk * m), c->stream)) return 1;
    return launch_probe_to(c, c->px.p, c->py.p, m, n_src, vinf_x, vinf_y, c->pu.p, c->pv.p, c->partial.p, 0);
}

// The probes of vx_case_set_probes, sources [0, ceil32(n)) of the current
// state, into c->prb_u / c->prb_v (own partials, so the step's split-K
// buffers are left alone).
int launch_step_probes(vx_case *c, double vinf_x, double vinf_y) {
    const int64_t m = c->prb_m;
    if (m <= 0) return 0;
    const Cnt s = cnt_s(c);
    int64_t chunk, nchunk;
    probe_split(m, s.ub, 0, &chunk, &nchunk);
    if (c->prb_part.ensure((size_t)(2 * nchunk * m), c->stream)) return 1;
    return launch_probe_to(c, c->prb_x.p, c->prb_y.p, m, s, vinf_x, vinf_y, c->prb_u.p, c->prb_v.p, c->prb_part.p,
                           0);
}

// ---- velocity probes without allocation ---------------------------------------
// vx_velocity_probe_noalloc keeps its split-K partials in this file-scope
// device array (one copy per GPU, held until the process ends) instead of
// the case's growable buffer.  Host code never uses the array's name as an
// address: its device address comes from hipGetSymbolAddress, once per
// device, and is kept in scratch_ptr.
constexpr int64_t kProbeScratch = int64_t(1) << 21;  // doubles (16 MiB)
static __device__ __align__(256) double scratch[kProbeScratch];

static std::mutex scratch_mu;
static double *scratch_ptr[256] = {};

static int probe_scratch(int dev, double **out) {
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (dev < 0 || dev >= 256) {
        set_error("bad argument: device index");
        return 2;
    }
    if (!scratch_ptr[dev]) {
        int cur = -1;
        VX_CHECK(hipGetDevice(&cur));
        if (cur != dev) VX_CHECK(hipSetDevice(dev));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) (void)hipSetDevice(cur);
        VX_CHECK(e);
        scratch_ptr[dev] = (double *)p;
    }
    *out = scratch_ptr[dev];
    return 0;
}

int launch_probe_noalloc(vx_case *c, const double *px, const double *py, int64_t m, double vinf_x, double vinf_y,
                         double *pu, double *pv) {
    if (m <= 0) return 0;
    if (2 * m > kProbeScratch) {
        set_error("bad argument: vx_velocity_probe_noalloc takes at most " + std::to_string(kProbeScratch / 2) +
                  " probes");
        return 2;
    }
    double *part = nullptr;
    if (const int rc = probe_scratch(c->device, &part)) return rc;
    const int64_t n_src = std::min<int64_t>((c->n + 31) / 32 * 32, c->cap);
    return launch_probe_to(c, px, py, m, n_src, vinf_x, vinf_y, pu, pv, part, kProbeScratch);
}

}  // namespace vx
