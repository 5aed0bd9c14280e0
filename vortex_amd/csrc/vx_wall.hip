// A8: wall diffusive velocity (src/kernel.cu:1031-1088, quadrature of
// I_0, I_3 at :1300-1346).
//
// For target i with characteristic distance d_i:
//   II0 = 2 pi d^2, II3 = 0; for each panel f in index order, r = |r_i - b_f|
//   with b_f the profile file's birth point:
//     0.1 l_f < r < 5 l_f : II0 -= d * RES0_f, II3 -= RES3_f  (midpoint rule
//                           with n_of_points nodes, normal -n_f)
//     r <= 0.1 l_f        : II0 = pi d^2, II3 = 2 n_f d (1 - e^{-l_f/2d}),
//                           and the panel loop stops there.
//   V_i += nu II3 / II0.
// Targets outside the box of birth points grown by 5 max(l) meet no panel and
// are skipped without touching the panel list.

#include "vx_internal.h"
#include "vx_prim.h"

namespace vx {

// One panel's quadrature I0, (I3_x, I3_y): N midpoints with e = (r_j - r_k) / d,
//   s0 += (e.n) / |e|^2 (|e| + 1) e^{-|e|} dL / N,  s3 += n e^{-|e|} dL / N.
template <typename T>
struct WallPanel {
    T ra0, ra1, dR0, dR1, n0, n1, delt;
};

// One target per wave: the lanes take panels lane, lane + 64, ...  The first panel in
// index order with r <= 0.1 l decides the result alone (the sequential loop
// overwrites II0 and II3 there and stops); without one, the mid-range terms
// are summed, lane partials in FP64 and then across the wave.  FP32 works in
// coordinates relative to the target (differences taken in FP64), so that a
// target a fraction of a short panel away keeps FP32's relative precision.
//
// A target has some ten panels in range, in one or two rounds of 64: a lane
// each for a whole quadrature left the others idle for 20 points of four
// divisions, a square root and an exponential.  The in-range panels of a round
// are listed instead, their points dealt to all lanes, 64 at a time, and each
// panel's terms added in order by a lane of its own: the same sums.  The
// distance test proper (a square root) is taken where a conservative one says
// so, four rounds of panels read at once.  200 panels, 2785 vortices: 23.4 -> 9.9
// us; FP32, 1000 panels, 2^20 vortices, beside the diffusion: 131 -> 106 us.
template <typename T>
struct WallLds {
    WallPanel<T> p[64];
    T prod[64], ex[64];
};

//
// I counts points: 32 bits while a round's 64 N points fit them (kShortPoints),
// whose quotient by N is a few instructions against some hundred in 64 bits.
constexpr int64_t kShortPoints = 1 << 24;

template <typename T, typename I>
__device__ void wave_wall(const PanelsSoA &pan, int lane, double x, double y, T dd, I N, WallLds<T> &L,
                          double &II0, double &II30, double &II31) {
    constexpr bool F32 = sizeof(T) == 4;
    const double ox = F32 ? x : 0.0, oy = F32 ? y : 0.0;
    const T a0 = (T)(x - ox), a1 = (T)(y - oy);
    const uint64_t below = (1ull << lane) - 1ull;
    double c0 = 0.0, c30 = 0.0, c31 = 0.0;
    int64_t fb = pan.P;
    constexpr int kR = 4;
    for (int64_t f0 = 0; f0 < pan.P && fb == pan.P; f0 += 64 * kR) {
        T q2[kR], dL[kR];
        uint64_t maybe[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            const int64_t f = f0 + 64 * r + lane;
            q2[r] = T(1);
            dL[r] = T(0);
            if (f < pan.P) {
                dL[r] = (T)pan.len[f];
                const T q0 = F32 ? (T)(x - pan.bx[f]) : a0 - (T)pan.bx[f];
                const T q1 = F32 ? (T)(y - pan.by[f]) : a1 - (T)pan.by[f];
                q2[r] = fma(q0, q0, q1 * q1);
            }
        }
#pragma unroll
        for (int r = 0; r < kR; ++r)
            maybe[r] = __ballot(f0 + 64 * r + lane < pan.P && !(q2[r] > T(26) * dL[r] * dL[r]));
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            if (maybe[r] == 0 || fb != pan.P) continue;
            const int64_t f = f0 + 64 * r + lane;
            const T d = sqrt(q2[r]);
            const bool in = f < pan.P && d < T(5) * dL[r] && d > T(0.1) * dL[r];
            const uint64_t close = __ballot(f < pan.P && !in && d <= T(0.1) * dL[r]);
            if (close) {
                fb = f0 + 64 * r + __builtin_ctzll(close);
                continue;
            }
            const uint64_t m = __ballot(in);
            const int cnt = (int)__popcll(m), rank = (int)__popcll(m & below);
            if (cnt == 0) continue;
            __builtin_amdgcn_wave_barrier();
            if (in) {
                const T ra0 = (T)(pan.lx[f] - ox), ra1 = (T)(pan.ly[f] - oy);
                const T rb0 = (T)(pan.rx[f] - ox), rb1 = (T)(pan.ry[f] - oy);
                L.p[rank] = WallPanel<T>{ra0,          ra1,          (rb0 - ra0) / (T)N, (rb1 - ra1) / (T)N,
                                         -(T)pan.nx[f], -(T)pan.ny[f], dL[r] / (T)N};
            }
            __builtin_amdgcn_wave_barrier();
            const WallPanel<T> mine = L.p[lane < cnt ? lane : 0];  // the panel whose terms this lane adds
            T s0 = 0, s30 = 0, s31 = 0;
            const I total = cnt * N;
            for (I t0 = 0; t0 < total; t0 += 64) {
                const I t = t0 + lane < total ? t0 + lane : total - 1;
                const I e = t / N, k = t - e * N;
                const WallPanel<T> &q = L.p[e];
                const T rk0 = fma((T)(k + 1), q.dR0, fma((T)k, q.dR0, q.ra0) + q.ra0);
                const T rk1 = fma((T)(k + 1), q.dR1, fma((T)k, q.dR1, q.ra1) + q.ra1);
                const T e0 = (a0 - rk0 / T(2)) / dd, e1 = (a1 - rk1 / T(2)) / dd;
                const T e2 = fma(e0, e0, e1 * e1);
                const T me = sqrt(e2);
                const T ex = exp(-me);
                __builtin_amdgcn_wave_barrier();
                L.prod[lane] = fma(e1, q.n1, e0 * q.n0) / e2 * (me + T(1)) * ex;
                L.ex[lane] = ex;
                __builtin_amdgcn_wave_barrier();
                const I lo = max(lane * N, t0), hi = lane < cnt ? min(lane * N + N, t0 + 64) : 0;
#pragma unroll 4
                for (I u = lo; u < hi; ++u) {
                    const T pr = L.prod[u - t0], xk = L.ex[u - t0];
                    s0 = fma(mine.delt, pr, s0);
                    s30 = fma(mine.delt, mine.n0 * xk, s30);
                    s31 = fma(mine.delt, mine.n1 * xk, s31);
                }
            }
            const T R0 = __shfl(s0, rank & 63, 64), R30 = __shfl(s30, rank & 63, 64), R31 = __shfl(s31, rank & 63, 64);
            if (in) {
                if constexpr (F32)
                    c0 -= (double)(dd * R0);
                else
                    c0 = fma(-dd, R0, c0);
                c30 += (double)R30;
                c31 += (double)R31;
            }
        }
    }
    if (fb < pan.P) {
        const T dL = (T)pan.len[fb];
        const T ex = T(1) - exp(-dL / (T(2) * dd));
        II0 = (double)(T(kPi) * dd * dd);
        II30 = (double)(T(2) * (T)pan.nx[fb] * dd * ex);
        II31 = (double)(T(2) * (T)pan.ny[fb] * dd * ex);
        return;
    }
    for (int o = 32; o > 0; o >>= 1) {
        c0 += __shfl_xor(c0, o, 64);
        c30 += __shfl_xor(c30, o, 64);
        c31 += __shfl_xor(c31, o, 64);
    }
    II0 = (double)(T(2 * kPi) * dd * dd) + c0;
    II30 = -c30;
    II31 = -c31;
}

struct InWallBox {
    const double *x, *y;
    double4 box;
    __device__ bool operator()(int32_t i) const {
        const double xi = x[i], yi = y[i];
        return xi >= box.x && xi <= box.y && yi >= box.z && yi <= box.w;
    }
};

// One wave per target inside the box, selected in index order (grid-stride,
// the count stays on the device).  The velocity terms go to list slot t of
// wst (u term at 2t, v term at 2t + 1) and k_wall_add adds them; with ADD (no
// other stream is writing u and v) the wave adds its own: a launch of 4.7 us less
// in a captured step.
template <typename T, bool ADD, typename I>
__global__ __launch_bounds__(256) void k_diffusion_wall(const double *__restrict__ x,
                                                        const double *__restrict__ y,
                                                        const double *__restrict__ d,
                                                        const int32_t *__restrict__ list,
                                                        const int32_t *__restrict__ cnt, PanelsSoA pan,
                                                        double nu, I npts, double *__restrict__ wst,
                                                        double *__restrict__ u,
                                                        double *__restrict__ v) {
    __shared__ WallLds<T> lds[4];
    const int lane = threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * 4;
    const int64_t total = *cnt;
    for (int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); t < total; t += nw) {
        const int64_t i = list[t];
        double II0, II30, II31;
        wave_wall<T, I>(pan, lane, x[i], y[i], (T)d[i], npts, lds[threadIdx.x >> 6], II0, II30, II31);
        if (lane == 0) {
            if constexpr (ADD) {
                u[i] += nu * II30 / II0;
                v[i] += nu * II31 / II0;
            } else {
                wst[2 * t] = nu * II30 / II0;
                wst[2 * t + 1] = nu * II31 / II0;
            }
        }
    }
}

// The wall pass on the main stream without a list, for bounds up to
// kScanMax: wave w looks at targets w, w + nw, ... (at most 64) and takes those in
// the box in turn.  2785 vortices: 5.1 us for the list and 9.9 for its targets ->
// 10.5 us.
constexpr int64_t kScanMax = 32768;

template <typename T, typename I>
__global__ __launch_bounds__(256) void k_wall_scan(InWallBox pred, Cnt cn, const double *__restrict__ d, PanelsSoA pan,
                                                   double nu, I npts, double *__restrict__ u,
                                                   double *__restrict__ v) {
    __shared__ WallLds<T> lds[4];
    const int lane = threadIdx.x & 63;
    const int64_t n = cn.get(), nw = (int64_t)gridDim.x * 4, w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t mine = w + nw * lane;
    for (uint64_t m = __ballot(mine < n && pred((int32_t)mine)); m; m &= m - 1) {
        const int64_t i = w + nw * __builtin_ctzll(m);
        double II0, II30, II31;
        wave_wall<T, I>(pan, lane, pred.x[i], pred.y[i], (T)d[i], npts, lds[threadIdx.x >> 6], II0, II30, II31);
        if (lane == 0) {
            u[i] += nu * II30 / II0;
            v[i] += nu * II31 / II0;
        }
    }
}

__global__ __launch_bounds__(256) void k_wall_add(const int32_t *__restrict__ list, const int32_t *__restrict__ cnt,
                                                  const double *__restrict__ wst, double *__restrict__ u,
                                                  double *__restrict__ v) {
    const int64_t total = *cnt;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = list[t];
        u[i] += wst[2 * t];
        v[i] += wst[2 * t + 1];
    }
}

template <bool ADD, typename T, typename I>
static int wall_pass_as(vx_case *c, Cnt cn_tgt, hipStream_t st) {
    const int64_t n_tgt = cn_tgt.ub;  // bound: list sizes and the selection's grid
    // buffers grow on the main stream: a reallocation synchronises it, and
    // with it every earlier side-stream pass (joined into it)
    if (c->wlist.ensure((size_t)n_tgt, c->stream) || c->dcount.ensure(16, c->stream) ||
        (!ADD && c->wstage.ensure((size_t)(2 * n_tgt), c->stream)))
        return 1;
    const I npts = (I)c->prm.n_of_points;
    const InWallBox pred{c->x.p, c->y.p, c->wall_box};
    if (ADD && n_tgt <= kScanMax) {
        const dim3 grid((unsigned)std::min<int64_t>(1024, (n_tgt + 3) / 4));
        hipLaunchKernelGGL((k_wall_scan<T, I>), grid, dim3(256), 0, st, pred, cn_tgt, c->d.p, c->pan, c->prm.nu, npts,
                           c->u.p, c->v.p);
        VX_CHECK(hipGetLastError());
        return 0;
    }
    int32_t *cnt = (int32_t *)(c->dcount.p + 5);
    if (c->wtmp.ensure((size_t)prim::tiles_of(n_tgt) + 1, c->stream)) return 1;
    VX_CHECK(prim::select_flags(prim::pred_flag(pred, cn_tgt), n_tgt, prim::WriteIndex{c->wlist.p}, c->wtmp.p, cnt,
                                st));
    hipLaunchKernelGGL((k_diffusion_wall<T, ADD, I>), dim3(1024), dim3(256), 0, st, c->x.p, c->y.p, c->d.p, c->wlist.p,
                       cnt, c->pan, c->prm.nu, npts, c->wstage.p, c->u.p, c->v.p);
    VX_CHECK(hipGetLastError());
    return 0;
}

template <bool ADD>
static int wall_pass(vx_case *c, Cnt cn_tgt, hipStream_t st) {
    if (cn_tgt.ub <= 0 || c->P <= 0) return 0;
    const bool shorts = c->prm.n_of_points <= kShortPoints;
    if (c->prm.precision == VX_PREC_MIXED)
        return shorts ? wall_pass_as<ADD, float, int32_t>(c, cn_tgt, st) : wall_pass_as<ADD, float, int64_t>(c, cn_tgt, st);
    return shorts ? wall_pass_as<ADD, double, int32_t>(c, cn_tgt, st) : wall_pass_as<ADD, double, int64_t>(c, cn_tgt, st);
}

int launch_wall_side(vx_case *c, int64_t n_tgt, hipStream_t st) {
    if (wall_pass<false>(c, host_cnt(n_tgt), st)) return 1;
    c->wall_pending = n_tgt > 0 && c->P > 0;
    return 0;
}

int launch_wall_add(vx_case *c) {
    if (!c->wall_pending) return 0;
    c->wall_pending = false;
    hipLaunchKernelGGL(k_wall_add, dim3(64), dim3(256), 0, c->stream, c->wlist.p, (const int32_t *)(c->dcount.p + 5),
                       c->wstage.p, c->u.p, c->v.p);
    VX_CHECK(hipGetLastError());
    return 0;
}

int launch_diffusion_wall(vx_case *c, Cnt n_tgt) { return wall_pass<true>(c, n_tgt, c->stream); }

int launch_diffusion_wall(vx_case *c, int64_t n_tgt) { return launch_diffusion_wall(c, host_cnt(n_tgt)); }

}  // namespace vx
