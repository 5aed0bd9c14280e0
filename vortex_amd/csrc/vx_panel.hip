// Panel system: influence matrix (A1), its inverse (A2) and the per-step
// birth of vortices from it (A4).  All FP64; multiplies and adds are kept
// separately rounded so the Gauss-Jordan elimination and the newborn
// positions reproduce the FP64 restatement bit for bit.
#pragma clang fp contract(off)

#include "vx_internal.h"
#include "vx_wave.h"

namespace vx {

// ---- A1: src/unit_1.cu:256-373 --------------------------------------------
// L[i][j] = tau_i . vbar_ij, vbar_ij the average over panel i of the velocity
// of a unit sheet on panel j (three atan differences q1_k, three log ratios
// q2_k, vectors c_k); both panels reversed for the right-hand neighbour and
// q1_1 = q2_1 = 0 for either neighbour; L[i][i] = -0.5; row P = lengths,
// column P = 1, L[P][P] = 0.
__device__ __forceinline__ double dot2(double a0, double a1, double b0, double b1) { return a0 * b0 + a1 * b1; }

__global__ void k_panel_matrix(PanelsSoA pan, double *__restrict__ L) {
    const int64_t P = pan.P, m = P + 1;
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j > P || i > P) return;
    if (i == P) {
        L[P * m + j] = j < P ? pan.len[j] : 0.0;
        return;
    }
    if (j == P) {
        L[i * m + P] = 1.0;
        return;
    }
    if (j == i) {
        L[i * m + j] = -0.5;
        return;
    }
    double a00 = pan.lx[i], a01 = pan.ly[i], a10 = pan.rx[i], a11 = pan.ry[i];
    double b00 = pan.lx[j], b01 = pan.ly[j], b10 = pan.rx[j], b11 = pan.ry[j];
    const bool next = (j == i + 1) || (j == 0 && i == P - 1);
    const bool prev = (j == i - 1) || (i == 0 && j == P - 1);
    if (next) {
        a10 = pan.lx[i]; a11 = pan.ly[i]; a00 = pan.rx[i]; a01 = pan.ry[i];
        b10 = pan.lx[j]; b11 = pan.ly[j]; b00 = pan.rx[j]; b01 = pan.ry[j];
    }
    const double dj0 = b10 - b00, dj1 = b11 - b01;
    const double di0 = a10 - a00, di1 = a11 - a01;
    const double p10 = a00 - b10, p11 = a01 - b11;
    const double p20 = a10 - b10, p21 = a11 - b11;
    const double s10 = a00 - b00, s11 = a01 - b01;
    const double s20 = a10 - b00, s21 = a11 - b01;
    const double z1 = p10 * p21 - p11 * p20;
    const double z2 = s10 * s21 - s11 * s20;
    const double z3 = s20 * p21 - s21 * p20;
    double q11 = 0.0, q21 = 0.0;
    if (!(next || prev)) {
        q11 = atan(dot2(di0, di1, p10, p11) / z1) - atan(dot2(di0, di1, p20, p21) / z1);
        q21 = 0.5 * log(dot2(p20, p21, p20, p21) / dot2(p10, p11, p10, p11));
    }
    const double q12 = atan(dot2(di0, di1, s20, s21) / z2) - atan(dot2(di0, di1, s10, s11) / z2);
    const double q13 = atan(dot2(dj0, dj1, p20, p21) / z3) - atan(dot2(dj0, dj1, s20, s21) / z3);
    const double q22 = 0.5 * log(dot2(s10, s11, s10, s11) / dot2(s20, s21, s20, s21));
    const double q23 = 0.5 * log(dot2(p20, p21, p20, p21) / dot2(s20, s21, s20, s21));
    const double djp1 = dot2(dj0, dj1, p10, p11);
    const double dis1 = dot2(di0, di1, s10, s11);
    const double didj = dot2(di0, di1, dj0, dj1);
    const double c10 = djp1 * di0 + dis1 * dj0 - didj * s10;
    const double c11 = djp1 * di1 + dis1 * dj1 - didj * s11;
    const double djj = dot2(dj0, dj1, dj0, dj1);
    const double dii = dot2(di0, di1, di0, di1);
    const double c20 = c10 + djj * di0, c21 = c11 + djj * di1;
    const double c30 = dii * dj0, c31 = dii * dj1;
    const double k = 1.0 / (2 * kPi * sqrt(djj) * dii);
    const double v0 = k * (q11 * c10 + q12 * c20 + q13 * c30 + (q21 * c11 + q22 * c21 + q23 * c31));
    const double v1 = k * (q11 * c11 + q12 * c21 + q13 * c31 - (q21 * c10 + q22 * c20 + q23 * c30));
    L[i * m + j] = dot2(v0, v1, pan.tx[i], pan.ty[i]);
}

int launch_panel_matrix(vx_case *c) {
    const int64_t m = c->P + 1;
    if (c->L.ensure((size_t)(m * m), c->stream)) return 1;
    hipLaunchKernelGGL(k_panel_matrix, dim3((unsigned)((m + 255) / 256), (unsigned)m), dim3(256), 0, c->stream,
                       c->pan, c->L.p);
    VX_CHECK(hipGetLastError());
    return 0;
}

// ---- A2: Gauss-Jordan inverse with partial pivoting ------------------------
// (src/unit_1.cu:115-254 eliminates with a look-ahead pivot choice; the
// standard choice -- largest |A[i][k]| over i >= k once columns < k are
// eliminated, first index on ties -- is used here because the look-ahead rule
// breaks down on the bordered system of thin closed bodies.)
//
// Column by column, step k swaps the pivot row up, takes the factors
// f_k[i] = A[i][k] / A[k][k] and subtracts f_k[i] times row k from every
// other row of A and of the growing inverse.  One column at a time that is
// four launches and 32 m^2 bytes each (109 ms at m = 2577, 15 ms at 1001), so
// it runs in blocks of B columns, with the same operations on every element
// in the same order and the same rounding:
//   k_gj_panel  one work-group takes a block's columns over all rows in
//               registers: pivots and factors of its B steps;
//   k_gj_rows   a thread per other column: the block's row exchanges, and the
//               pivot rows brought to each step in turn (U: their values as
//               the step uses them);
//   k_gj_rank   every other row: a = ((a - f_0 U_0) - f_1 U_1) - ...
// In place: W's columns below the block hold the inverse's columns that are
// not zero yet (in pivot order, the order undone at the end), the others A's.
// The rounding residues that elimination leaves in A's finished columns reach
// the last division through the diagonal, so they are carried along (G: rows
// below the block; D: the diagonal).
// Bound by the panels' latency (one CU, 1.1 to 2.4 us a column) up to about
// 2500 rows and by W's traffic through the caches, 16 m^2 bytes a block, above.
struct GjMoves {
    int32_t src[16];           // the row that the block's r-th pivot step brought to row K + r
    int32_t nq;                // rows below the block that received another row:
    int32_t qdst[16], qsrc[16];
};

// Columns [K, K + nb) of W (column by column in Pt) over all m <= T R rows.
// A thread holds R rows; a row exchange only exchanges the positions of two
// rows.  Each wave offers its largest candidate with its row in LDS and every
// thread picks the winner: one barrier per step.  The step's column is always
// a[.][0]: the update moves the others down, so that the loop stays rolled
// (unrolled, the code is fetched anew on every launch).  Few waves of many
// registers: the reduction is the same work for every wave of a SIMD.
// Results: by the rows' places before the block the factors cf[kk m + i] and
// the columns as each one's own step left them PtG; the places (slot_of), the
// pivots D, the row moves, perm.
template <int NW, int B>
struct GjPanelLds {
    double crow[2][NW][B], ub[B][B], ckey[2][NW], crec[2][NW];
    int cpos[2][NW], nq;
};

// A block's state: a ring of two, one being written by a panel while the
// other is read by the rank update.
struct GjBlock {
    double *Pt, *PtG, *cf;
    int32_t *slot_of;
    GjMoves *mv;
};

// `prev` (null for the first block): the block before, whose rank update the
// panel's own columns still lack; U its pivot rows.
template <int T, int R, int B>
__device__ __forceinline__ void gj_panel(GjPanelLds<T / 64, B> &ls, int32_t m, int32_t K, int32_t nb,
                                         const GjBlock &blk, const GjBlock *prev, const double *__restrict__ U,
                                         double *__restrict__ D, int32_t *__restrict__ perm,
                                         int32_t *__restrict__ bad) {
    constexpr int NW = T / 64;
    static_assert(NW <= 16, "one row of lanes picks the winner");
    const double *__restrict__ Pt = blk.Pt;
    double *__restrict__ cf = blk.cf, *__restrict__ PtG = blk.PtG;
    int32_t *__restrict__ slot_of = blk.slot_of;
    GjMoves *__restrict__ mv = blk.mv;
    auto &ckey = ls.ckey;
    auto &crec = ls.crec;
    auto &cpos = ls.cpos;
    auto &crow = ls.crow;
    int &nq = ls.nq;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double a[R][B];
    int pos[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int s = tid + r * T;
        pos[r] = s < m ? s : -1;
#pragma unroll
        for (int c = 0; c < B; ++c) a[r][c] = s < m && c < nb ? Pt[(int64_t)c * m + s] : 0.0;
    }
    if (tid == 0) nq = 0;
    if (prev) {
        const int64_t ldu = 2 * (int64_t)m;
        for (int e = tid; e < B * B; e += T) ls.ub[e / B][e % B] = e % B < nb ? U[(e / B) * ldu + K + e % B] : 0.0;
        int32_t ps[R];  // where a row's factors are; -1: none (the block's own rows are at their final values)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int s = tid + r * T;
            ps[r] = s < m && !(s >= K - B && s < K) ? prev->slot_of[s] : -1;
        }
        __syncthreads();
#pragma unroll 1
        for (int kk = 0; kk < B; ++kk) {
            double u[B];
#pragma unroll
            for (int c = 0; c < B; ++c) u[c] = ls.ub[kk][c];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const double f = ps[r] >= 0 ? prev->cf[(int64_t)kk * m + ps[r]] : 0.0;
#pragma unroll
                for (int c = 0; c < B; ++c) a[r][c] = a[r][c] - f * u[c];
            }
        }
    }
#pragma unroll 1
    for (int kk = 0; kk < nb; ++kk) {
        const int k = K + kk, par = kk & 1;
        double key = -1.0, cand = 1.0;
        int kp = 0x7fffffff, kr = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double v = fabs(a[r][0]);
            if (pos[r] >= k && (v > key || (v == key && pos[r] < kp))) {
                key = v;
                cand = a[r][0];
                kp = pos[r];
                kr = r;
            }
        }
        const double rec = 1.0 / cand;  // every lane's own, beside the reduction
        const double wm = wave_max(key);
        const uint64_t ties = __ballot(key == wm);
        const int wl = ties ? lowest_lane(ties, kp) : 0;
        const int wr = __builtin_amdgcn_readlane(kr, wl);
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (wr == r) {
                if (lane == wl) {
#pragma unroll
                    for (int c = 0; c < B; ++c) crow[par][wv][c] = a[r][c];
                    ckey[par][wv] = key;
                    cpos[par][wv] = kp;
                    crec[par][wv] = rec;
                }
            }
        lds_barrier();
        const double ck = ckey[par][lane & (NW - 1)];
        const int cp = cpos[par][lane & (NW - 1)];
        const double gm = lane_of(row_max(ck), 15);
        const uint64_t gt = __ballot(ck == gm) & ((1ull << NW) - 1);
        const int gw = gt ? lowest_lane(gt, cp) : 0;
        int p = __builtin_amdgcn_readlane(cp, gw);
        if (!(gm >= kDelt)) {  // no usable pivot: the caller reports it
            if (tid == 0) *bad = 1;
            if (p < k || p >= m) p = k;
        }
        double row[B];
#pragma unroll
        for (int c = 0; c < B; ++c) row[c] = crow[par][gw][c];
        const double y = crec[par][gw];
        if (tid == 0) D[k] = row[0];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            pos[r] = pos[r] == p ? k : pos[r] == k ? p : pos[r];
            // a / pivot correctly rounded from the rounded reciprocal
            double f = a[r][0] * y;
            f = fma(fma(-row[0], f, a[r][0]), y, f);
            f = pos[r] == k ? 0.0 : f;
            const int s = tid + r * T;
            if (s < m) {
                cf[(int64_t)kk * m + s] = f;
                PtG[(int64_t)kk * m + s] = a[r][0] - f * row[0];
            }
#pragma unroll
            for (int c = 1; c < B; ++c) a[r][c - 1] = a[r][c] - f * row[c];
            a[r][B - 1] = 0.0;
        }
    }
    // the moves: slot_of[final position] = the row that is there now
    int mp[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int s = tid + r * T;
        mp[r] = s < m && pos[r] != s ? perm[s] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int s = tid + r * T;
        if (s < m) {
            slot_of[pos[r]] = s;
            if (pos[r] != s) perm[pos[r]] = mp[r];
            if (pos[r] >= K && pos[r] < K + nb) {
                mv->src[pos[r] - K] = s;
            } else if (pos[r] != s) {
                const int q = atomicAdd(&nq, 1);
                mv->qdst[q] = pos[r];
                mv->qsrc[q] = s;
            }
        }
    }
    __syncthreads();
    if (tid == 0) mv->nq = nq;
}

template <int T, int R, int B>
__global__ __launch_bounds__(T) void k_gj_panel(int32_t m, int32_t nb, GjBlock blk, double *__restrict__ D,
                                                int32_t *__restrict__ perm, int32_t *__restrict__ bad) {
    __shared__ __align__(16) GjPanelLds<T / 64, B> ls;
    gj_panel<T, R, B>(ls, m, 0, nb, blk, nullptr, nullptr, D, perm, bad);
}

// A thread per column: of W (q < m) or of G (q - m < K + nb).
// nextPt: the next block's columns, which get the moves and the block's rows
// here and the rest in the next panel; ownPt: those of the block after it,
// which get the block's rows here and the rest from the rank update.
template <int B>
__global__ __launch_bounds__(64) void k_gj_rows(double *__restrict__ W, double *__restrict__ G,
                                                double *__restrict__ D, double *__restrict__ nextPt,
                                                double *__restrict__ ownPt, const double *__restrict__ PtG, int32_t m, int32_t K, int32_t nb,
                                                const double *__restrict__ cf, const GjMoves *__restrict__ mv,
                                                double *__restrict__ U) {
    __shared__ __align__(16) double fb[B][B];  // the factors of the block's own rows
    for (int e = threadIdx.x; e < B * B; e += 64)
        fb[e / B][e % B] = e / B < nb && e % B < nb ? cf[(int64_t)(e / B) * m + mv->src[e % B]] : 0.0;
    __syncthreads();
    const int32_t q = (int32_t)(blockIdx.x * 64 + threadIdx.x);
    if (q >= m + K + nb) return;
    const bool inv = q < m;
    const int32_t j = inv ? q : q - m;
    const bool fresh = j >= K && j < K + nb;  // W: a new column of the inverse; G: one of the block's columns
    double *X = inv ? W : G;
    const int64_t ldu = 2 * (int64_t)m;
    double v[B], t[B];
    const int nq = mv->nq;
#pragma unroll
    for (int r = 0; r < B; ++r) {
        if (r >= nb)
            v[r] = 0.0;
        else if (!fresh)
            v[r] = X[(int64_t)mv->src[r] * m + j];
        else
            v[r] = inv ? (r == j - K ? 1.0 : 0.0) : (r > j - K ? PtG[(int64_t)(j - K) * m + mv->src[r]] : 0.0);
        t[r] = !fresh && r < nq ? X[(int64_t)mv->qsrc[r] * m + j] : 0.0;
    }
    const bool next = inv && j >= K + B && j < K + 2 * B;
    if (!fresh) {
#pragma unroll
        for (int r = 0; r < B; ++r)
            if (r < nq) {
                X[(int64_t)mv->qdst[r] * m + j] = t[r];
                if (next) nextPt[(int64_t)(j - K - B) * m + mv->qdst[r]] = t[r];
            }
    }
    double dj = inv ? 0.0 : D[j];
    const int32_t jrow = !inv && fresh ? mv->src[j - K] : j;  // a finished row stays where it is
#pragma unroll
    for (int kk = 0; kk < B; ++kk) {
        if (kk < nb) {
            const double u = v[kk];
            U[kk * ldu + q] = u;
#pragma unroll
            for (int r = 0; r < B; ++r)
                if (r != kk) v[r] = v[r] - fb[kk][r] * u;
            if (!inv && (!fresh || kk > j - K)) dj = dj - cf[(int64_t)kk * m + jrow] * u;
        }
    }
    if (inv) {
#pragma unroll
        for (int r = 0; r < B; ++r)
            if (r < nb) {
                W[(int64_t)(K + r) * m + j] = v[r];
                if (next) nextPt[(int64_t)(j - K - B) * m + K + r] = v[r];
                if (j >= K + 2 * B && j < K + 3 * B) ownPt[(int64_t)(j - K - 2 * B) * m + K + r] = v[r];
            }
    } else {
        D[j] = dj;
    }
}

// The other rows, and the next block's panel beside them (work-group 0): the
// panel is one CU's work and longer than the update of one below about 2500
// rows.  T / 4 rows x 128 columns per work-group, 4 x 8 per thread; first the
// tiles of W (all rows outside the block), then those of G (rows below it,
// columns below K + nb).  The columns of the block after the next also go to
// its Pt (nextPt).
template <int T, int B>
struct GjRankLds {
    double ff[B][T / 4], uu[B][128];
};
template <int T, int R, int B>
__global__ __launch_bounds__(T) void k_gj_rank(double *__restrict__ W, double *__restrict__ G, int32_t m, int32_t K,
                                               int32_t nb, GjBlock blk, GjBlock next, const double *__restrict__ U,
                                               double *__restrict__ D, int32_t *__restrict__ perm,
                                               int32_t *__restrict__ bad, int32_t tiles_w, int32_t tx_w, int32_t tx_g) {
    constexpr int TR = T / 4;
    __shared__ __align__(16) union Lds {
        GjPanelLds<T / 64, B> panel;
        GjRankLds<T, B> rank;
    } ls;
    if (blockIdx.x == 0) {
        if (K + B < m) gj_panel<T, R, B>(ls.panel, m, K + B, min(B, m - K - B), next, &blk, U, D, perm, bad);
        return;
    }
    auto &ff = ls.rank.ff;
    auto &uu = ls.rank.uu;
    const int32_t w = (int32_t)blockIdx.x - 1;
    const bool inv = w < tiles_w;
    const int32_t q = inv ? w : w - tiles_w, tx_n = inv ? tx_w : tx_g;
    const int32_t i0 = (q / tx_n) * TR + (inv ? 0 : K + nb), j0 = (q % tx_n) * 128;
    const int32_t jn = inv ? m : K + nb;
    if (i0 >= m || j0 >= jn) return;
    const int64_t ldu = 2 * (int64_t)m;
    const int tid = threadIdx.x;
    const int32_t fi = i0 + (tid & (TR - 1)) < m ? blk.slot_of[i0 + (tid & (TR - 1))] : -1;
    for (int e = tid; e < B * TR; e += T)
        ff[e / TR][e & (TR - 1)] = e / TR < nb && fi >= 0 ? blk.cf[(int64_t)(e / TR) * m + fi] : 0.0;
    for (int e = tid; e < B * 128; e += T) {
        const int32_t j = j0 + (e & 127);
        uu[e >> 7][e & 127] = (e >> 7) < nb && j < jn ? U[(e >> 7) * ldu + (inv ? 0 : m) + j] : 0.0;
    }
    // thread (ty, tx): rows 4 ty + r, columns 2 tx + 32 c + {0, 1}
    const int tx = tid & 15, ty = tid >> 4;
    double *X = inv ? W : G;
    double a[4][8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int32_t i = i0 + 4 * ty + r;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int32_t j = j0 + 2 * tx + 32 * (c >> 1) + (c & 1);
            double v = 0.0;
            if (i < m && j < jn) {
                if (j < K || j >= K + nb)
                    v = X[(int64_t)i * m + j];
                else if (!inv)
                    v = blk.PtG[(int64_t)(j - K) * m + blk.slot_of[i]];
            }
            a[r][c] = v;
        }
    }
    __syncthreads();
#pragma unroll 2
    for (int kk = 0; kk < B; ++kk) {
        double f[4], u[8];
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            const double2 v = *reinterpret_cast<const double2 *>(&ff[kk][4 * ty + r]);
            f[r] = v.x;
            f[r + 1] = v.y;
        }
#pragma unroll
        for (int c = 0; c < 8; c += 2) {
            const double2 v = *reinterpret_cast<const double2 *>(&uu[kk][2 * tx + 16 * c]);
            u[c] = v.x;
            u[c + 1] = v.y;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 8; ++c) a[r][c] = a[r][c] - f[r] * u[c];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int32_t i = i0 + 4 * ty + r;
        if (i >= m || (i >= K && i < K + nb)) continue;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int32_t j = j0 + 2 * tx + 32 * (c >> 1) + (c & 1);
            if (j >= jn) continue;
            X[(int64_t)i * m + j] = a[r][c];
            if (inv && j >= K + 2 * B && j < K + 3 * B) blk.Pt[(int64_t)(j - K - 2 * B) * m + i] = a[r][c];
        }
    }
}

// The first two blocks' columns, and the identity permutation.
template <int B>
__global__ void k_gj_first(const double *__restrict__ W, int32_t m, double *__restrict__ Pt0,
                           double *__restrict__ Pt1, int32_t *__restrict__ perm) {
    const int32_t i = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= m) return;
    perm[i] = i;
    for (int c = 0; c < 2 * B && c < m; ++c) (c < B ? Pt0 : Pt1)[(int64_t)(c % B) * m + i] = W[(int64_t)i * m + c];
}

// M[i][perm[p]] = W[i][p] / D[i]: the inverse's columns back in the rows' order.
__global__ void k_gj_finish(const double *__restrict__ W, const double *__restrict__ D,
                            const int32_t *__restrict__ perm, int32_t m, double *__restrict__ M) {
    const int32_t p = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    const int64_t i = blockIdx.y;
    if (p < m) M[i * m + perm[p]] = W[i * m + p] / D[i];
}

// A in W (destroyed), the inverse into M (also G's room); work holds
// gj_work(m) doubles and ints 3 m.
constexpr int kGjMaxB = 16;
static size_t gj_work(int64_t m) { return (size_t)(kGjMaxB * m * 8 + m) + 2 * (sizeof(GjMoves) / sizeof(double) + 2); }

template <int T, int R, int B>
static void gj_blocks(double *W, double *M, int32_t m, double *work, int32_t *ints, int32_t *bad, hipStream_t st) {
    static_assert(B <= kGjMaxB, "work");
    const int64_t bm = (int64_t)B * m;
    GjBlock ring[2];
    double *p = work;
    for (int b = 0; b < 2; ++b) {
        ring[b] = GjBlock{p, p + bm, p + 2 * bm, ints + (int64_t)(1 + b) * m, nullptr};
        p += 3 * bm;
    }
    double *U = p, *D = U + 2 * bm;
    for (int b = 0; b < 2; ++b) ring[b].mv = (GjMoves *)(D + m + (m & 1)) + b;
    int32_t *perm = ints;
    hipLaunchKernelGGL(k_gj_first<B>, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, W, m, ring[0].Pt,
                       ring[1].Pt, perm);
    hipLaunchKernelGGL((k_gj_panel<T, R, B>), dim3(1), dim3(T), 0, st, m, std::min(B, m), ring[0], D, perm, bad);
    for (int32_t K = 0, b = 0; K < m; K += B, b ^= 1) {
        const int32_t nb = std::min(B, m - K);
        const GjBlock &blk = ring[b], &next = ring[b ^ 1];
        hipLaunchKernelGGL(k_gj_rows<B>, dim3((unsigned)((m + K + nb + 63) / 64)), dim3(64), 0, st, W, M, D, next.Pt,
                           blk.Pt, blk.PtG, m, K, nb, blk.cf, blk.mv, U);
        constexpr int TR = T / 4;
        const int32_t tx_w = (m + 127) / 128, ty_w = (m + TR - 1) / TR, tx_g = (K + nb + 127) / 128,
                      ty_g = (m - K - nb + TR - 1) / TR;
        hipLaunchKernelGGL((k_gj_rank<T, R, B>), dim3((unsigned)(1 + tx_w * ty_w + tx_g * ty_g)), dim3(T), 0, st, W, M,
                           m, K, nb, blk, next, U, D, perm, bad, tx_w * ty_w, tx_w, tx_g);
    }
    hipLaunchKernelGGL(k_gj_finish, dim3((unsigned)((m + 255) / 256), (unsigned)m), dim3(256), 0, st, W, D, perm, m,
                       M);
}

// T R rows of a panel in one work-group's registers, R B doubles a thread of
// its 512, 256 or 128 registers (T = 256, 512, 1024).  Measured build times:
// m = 1001: <512, 2> with B = 8, 10, 12, 16: 2.95, 2.95, 2.99, 3.20 ms, <256,
// 4, 16> 3.54; 1501: <1024, 2, 10> 5.38, <512, 4, 12> 5.60, <512, 4, 16> 6.12;
// 2577: <512, 6> with 10, 12, 14: 13.2, 12.6, 13.0; 4001: <512, 8, 10> 36.7,
// <512, 8, 8> 42.4, <512, 12, 7> 48.0, <1024, 4, 9> 73; 5201: <1024, 6, 8>
// 87, <512, 12, 7> 95, <512, 12, 5> 124.  One column at a time took 13.7
// (1001), 28.7, 104, 339 and 913 ms.  Above kGjBlocked rows a panel no longer
// fits: one column at a time there.
constexpr int64_t kGjBlocked = 12288;

static void gj_blocked(double *W, double *M, int64_t m, double *work, int32_t *ints, int32_t *bad, hipStream_t st) {
    const int32_t n = (int32_t)m;
    if (m <= 256) gj_blocks<256, 1, 16>(W, M, n, work, ints, bad, st);
    else if (m <= 512) gj_blocks<256, 2, 16>(W, M, n, work, ints, bad, st);
    else if (m <= 1024) gj_blocks<512, 2, 10>(W, M, n, work, ints, bad, st);
    else if (m <= 2048) gj_blocks<1024, 2, 10>(W, M, n, work, ints, bad, st);
    else if (m <= 3072) gj_blocks<512, 6, 12>(W, M, n, work, ints, bad, st);
    else if (m <= 4096) gj_blocks<512, 8, 10>(W, M, n, work, ints, bad, st);
    else if (m <= 6144) gj_blocks<1024, 6, 8>(W, M, n, work, ints, bad, st);
    else gj_blocks<512, 24, 2>(W, M, n, work, ints, bad, st);
}

__global__ __launch_bounds__(1024) void k_gj_pivot(const double *__restrict__ A, int64_t m, int64_t k,
                                                   int64_t *__restrict__ piv, int32_t *__restrict__ bad) {
    __shared__ double bv[1024];
    __shared__ int64_t bi[1024];
    double best = -1.0;
    int64_t besti = m;
    for (int64_t i = k + threadIdx.x; i < m; i += blockDim.x) {
        const double a = fabs(A[i * m + k]);
        if (a > best) { best = a; besti = i; }
    }
    bv[threadIdx.x] = best;
    bi[threadIdx.x] = besti;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            const double ov = bv[threadIdx.x + s];
            const int64_t oi = bi[threadIdx.x + s];
            if (ov > bv[threadIdx.x] || (ov == bv[threadIdx.x] && oi < bi[threadIdx.x])) {
                bv[threadIdx.x] = ov;
                bi[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *piv = bi[0];
        if (!(bv[0] >= kDelt)) *bad = 1;
    }
}

__global__ void k_gj_swap_factor(double *__restrict__ A, double *__restrict__ I, int64_t m, int64_t k,
                                 const int64_t *__restrict__ piv) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t p = *piv;
    if (j >= m || p == k || p >= m) return;
    double t = A[k * m + j]; A[k * m + j] = A[p * m + j]; A[p * m + j] = t;
    t = I[k * m + j]; I[k * m + j] = I[p * m + j]; I[p * m + j] = t;
}

__global__ void k_gj_colfactor(const double *__restrict__ A, int64_t m, int64_t k, double *__restrict__ cf) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    cf[i] = (i == k) ? 0.0 : A[i * m + k] / A[k * m + k];
}

__global__ void k_gj_update(double *__restrict__ A, double *__restrict__ I, int64_t m, int64_t k,
                            const double *__restrict__ cf) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j >= m || i == k) return;
    const double c = cf[i];
    A[i * m + j] = A[i * m + j] - c * A[k * m + j];
    I[i * m + j] = I[i * m + j] - c * I[k * m + j];
}

__global__ void k_gj_identity(double *__restrict__ I, int64_t m) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j < m) I[i * m + j] = (i == j) ? 1.0 : 0.0;
}

__global__ void k_gj_scale(const double *__restrict__ A, double *__restrict__ I, int64_t m) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j < m) I[i * m + j] = I[i * m + j] / A[i * m + i];
}

int launch_invert(vx_case *c) {
    const int64_t m = c->P + 1;
    const bool blocked = m <= kGjBlocked;
    DBuf<double> A, work;
    DBuf<int32_t> perm;
    int rc = 0;
    if (A.ensure((size_t)(m * m), c->stream) || c->M.ensure((size_t)(m * m), c->stream) ||
        c->dcount.ensure(4, c->stream))
        rc = 1;
    if (!rc && (blocked ? work.ensure(gj_work(m), c->stream) || perm.ensure((size_t)(3 * m), c->stream)
                        : c->red.ensure((size_t)m, c->stream)))
        rc = 1;
    do {
        if (rc) break;
        if (hipMemcpyAsync(A.p, c->L.p, sizeof(double) * m * m, hipMemcpyDeviceToDevice, c->stream) != hipSuccess ||
            hipMemsetAsync(c->dcount.p, 0, sizeof(int64_t) * 4, c->stream) != hipSuccess) {
            set_error("invert: staging failed");
            rc = 1;
            break;
        }
        int64_t *piv = c->dcount.p;
        int32_t *bad = (int32_t *)(c->dcount.p + 1);
        if (blocked) {
            gj_blocked(A.p, c->M.p, m, work.p, perm.p, bad, c->stream);
        } else {
            const dim3 g2((unsigned)((m + 255) / 256), (unsigned)m);
            const unsigned g1 = (unsigned)((m + 255) / 256);
            hipLaunchKernelGGL(k_gj_identity, g2, dim3(256), 0, c->stream, c->M.p, m);
            for (int64_t k = 0; k < m; ++k) {
                hipLaunchKernelGGL(k_gj_pivot, dim3(1), dim3(1024), 0, c->stream, A.p, m, k, piv, bad);
                hipLaunchKernelGGL(k_gj_swap_factor, dim3(g1), dim3(256), 0, c->stream, A.p, c->M.p, m, k, piv);
                hipLaunchKernelGGL(k_gj_colfactor, dim3(g1), dim3(256), 0, c->stream, A.p, m, k, c->red.p);
                hipLaunchKernelGGL(k_gj_update, g2, dim3(256), 0, c->stream, A.p, c->M.p, m, k, c->red.p);
            }
            hipLaunchKernelGGL(k_gj_scale, g2, dim3(256), 0, c->stream, A.p, c->M.p, m);
        }
        if (hipGetLastError() != hipSuccess) {
            set_error("invert: launch failed");
            rc = 1;
            break;
        }
        int32_t hbad = 0;
        if (hipMemcpyAsync(&hbad, bad, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
            hipStreamSynchronize(c->stream) != hipSuccess) {
            set_error("invert: read-back failed");
            rc = 1;
            break;
        }
        if (hbad) {
            set_error("panel matrix is singular (pivot below 1e-12)");
            rc = 1;
        }
    } while (0);
    (void)hipStreamSynchronize(c->stream);
    A.release();
    work.release();
    perm.release();
    return rc;
}

// ---- A4: src/kernel.cu:849-873 ---------------------------------------------
// gsheet_i = sum_{j<P} M[i][j] R_j + M[i][P] d_g  (one wave64 per row,
// coalesced over the row, xor-shuffle reduction), then newborn i at the panel
// midpoint + offset * normal with g = (gsheet_i l_i + gsheet_next l_next)/2.
__global__ __launch_bounds__(256) void k_birth_gemv(const double *__restrict__ M, const double *__restrict__ R,
                                                   double d_g_host, const double *__restrict__ d_g_dev, int64_t P,
                                                   double *__restrict__ gs) {
    const double d_g = d_g_dev ? *d_g_dev : d_g_host;
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= P) return;
    const int64_t m = P + 1;
    const double *Mr = M + row * m;
    double acc = 0.0;
    for (int64_t j = lane; j < P; j += 64) acc += Mr[j] * R[j];
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) gs[row] = acc + Mr[P] * d_g;
}

// Newborn positions, one per panel: the panel midpoint moved off along the
// normal (computed once per case; bp holds x at [0, P), y at [P, 2P)).
__global__ void k_birth_pos(PanelsSoA pan, double off_rel, double *__restrict__ bp) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pan.P) return;
    const double off = off_rel > 0.0 ? off_rel * pan.len[i] : 1e-6;
    bp[i] = (pan.lx[i] + pan.rx[i]) / 2 + off * pan.nx[i];
    bp[pan.P + i] = (pan.ly[i] + pan.ry[i]) / 2 + off * pan.ny[i];
}

int launch_birth_positions(vx_case *c) {
    hipLaunchKernelGGL(k_birth_pos, dim3((unsigned)((c->P + 255) / 256)), dim3(256), 0, c->stream, c->pan,
                       c->prm.birth_offset_rel, c->bpos);
    VX_CHECK(hipGetLastError());
    return 0;
}

// With grow (one work-group then, which has read the count before), the device
// count becomes *grow + P.
__global__ __launch_bounds__(1024) void k_birth_place(const double *__restrict__ gs, PanelsSoA pan,
                                                      const double *__restrict__ bp, Cnt cn, int64_t cap,
                                                      double *__restrict__ x, double *__restrict__ y,
                                                      double *__restrict__ g, int64_t *grow) {
    const int64_t n = cn.get();
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < pan.P; i += (int64_t)gridDim.x * blockDim.x) {
        if (n + i >= cap) break;
        const int64_t nx = pan.rp[i];
        x[n + i] = bp[i];
        y[n + i] = bp[pan.P + i];
        g[n + i] = 0.5 * (gs[i] * pan.len[i] + gs[nx] * pan.len[nx]);
    }
    if (!grow) return;
    __syncthreads();
    if (threadIdx.x == 0) *grow += pan.P;
}

// The sheet strengths of the last birth: the inverse's product, or with the
// FP32 LU the first P entries of the refined solution.
const double *birth_sheet(vx_case *c) { return c->lu ? lu_solution(c) : c->gsheet.p; }

// In device-count mode the absorbed circulation comes from red[0] (the
// previous step's sum) and the newborns go to the device count's slots,
// which then grows by P.
int launch_birth(vx_case *c, double d_g) {
    const int64_t P = c->P;
    const double *dgp = c->devcount ? c->red.p : nullptr;
    if (c->lu) {
        if (launch_lu_solve(c, c->rp.p, d_g, dgp)) return 1;
    } else {
        if (c->gsheet.ensure((size_t)P, c->stream)) return 1;
        hipLaunchKernelGGL(k_birth_gemv, dim3((unsigned)((P + 3) / 4)), dim3(256), 0, c->stream, c->M.p, c->rp.p,
                           d_g, dgp, P, c->gsheet.p);
    }
    const dim3 grid(c->devcount ? 1u : (unsigned)((P + 255) / 256)), wg(c->devcount ? 1024u : 256u);
    hipLaunchKernelGGL(k_birth_place, grid, wg, 0, c->stream, birth_sheet(c), c->pan, c->bpos, cnt_n(c), c->cap, c->x.p,
                       c->y.p, c->g.p, c->devcount ? c->dcount.p + 1 : nullptr);
    VX_CHECK(hipGetLastError());
    return 0;
}

}  // namespace vx
