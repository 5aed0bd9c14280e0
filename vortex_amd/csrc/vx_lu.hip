// Panel system in mixed precision: FP32 LU of the influence matrix with
// partial pivoting (blocked, right-looking; trailing updates as FP32 matrix
// products on MFMA), the triangular factors inverted blockwise (again MFMA
// products), and per birth an FP64-residual iterative refinement:
//
//     x = 0, r = b;  repeat: x += U^-1 L^-1 P r  (FP32 products),
//                            r = b - A x         (FP64, A = the FP64 matrix)
//     until ||r|| <= ||x|| ||A|| eps64 sqrt(n)   (LAPACK dsgesv's test)
//
// The reference inverts the matrix once in FP64 by Gauss-Jordan
// (src/unit_1.cu:115-254) and multiplies by the inverse at every birth
// (src/kernel.cu:849-873); the solution of the same system is what both
// deliver.  Everything stays on the device: the refinement's kernels read a
// convergence flag and return at once after the test passes, so a fixed
// number of them is queued per birth and no host wait is needed.
//
// Layout: the order n = P + 1 is padded to np, a multiple of 64, with an
// identity block (decoupled, never pivoted).  FP32 matrices are np x np
// row-major: F holds L (strict lower, unit diagonal) and U (upper) of P A,
// W the two inverses (strict lower: L^-1 below its unit diagonal; upper
// with diagonal: U^-1).
#include <cmath>
#include <type_traits>

#include "vx_internal.h"
#include "vx_prim.h"
#include "vx_wave.h"

namespace vx {

constexpr int kLuB = 64;       // panel width, block size of the inverses, product tile
constexpr int kLuMaxIt = 6;    // refinement corrections queued per solve

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct LuBufs {
    int64_t n = 0, np = 0;
    DBuf<float> F, W, Wl, Wu, T;
    DBuf<double> A;               // the FP64 matrix (n x n), for the residuals
    DBuf<double> x;               // solution (np)
    DBuf<float> rp, t;            // permuted FP32 residual, L^-1 P r (np)
    DBuf<int32_t> ipiv, perm, pinv;
    DBuf<unsigned long long> st;  // 0 done, 1 corrections, 2 |r| max bits, 3 |x| max bits, 4 singular,
                                  // 5 ||A||_inf bits
    DBuf<double> nrm;             // 1: last ||r|| / (||A|| ||x||)
    int32_t last_iters = 0;
};

// ---- FP32 matrix product on MFMA ---------------------------------------------
// C = alpha A B + beta Cin (Cin may be C) for row-major blocks with M, N
// multiples of 64 and K a multiple of 16.  One work-group of 4 waves per
// 64 x 64 tile of C, each wave a 32 x 32 quarter as 2 x 2 products of
// v_mfma_f32_16x16x4_f32 (A: lane = i + 16 k; B: lane = j + 16 k; C: lane =
// j + 16 (i / 4), register i % 4).
__global__ __launch_bounds__(256) void k_gemm_f32(const float *__restrict__ A, int64_t lda, const float *__restrict__ B,
                                                  int64_t ldb, float *C, int64_t ldc, const float *Cin,
                                                  int64_t ldcin, int64_t K, float alpha, float beta) {
    __shared__ float As[64][17];
    __shared__ float Bs[16][65];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t bm = (int64_t)blockIdx.y * 64, bn = (int64_t)blockIdx.x * 64;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    floatx4 acc[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int ar = tid >> 2, ac = (tid & 3) * 4;     // A tile: 64 rows x 16
    const int br = tid >> 4, bc = (tid & 15) * 4;    // B tile: 16 rows x 64
    for (int64_t k0 = 0; k0 < K; k0 += 16) {
        const float *ap = A + (bm + ar) * lda + k0 + ac;
        const float *bp = B + (k0 + br) * ldb + bn + bc;
        const float4 av = *reinterpret_cast<const float4 *>(ap);
        const float4 bv = *reinterpret_cast<const float4 *>(bp);
        __syncthreads();
        As[ar][ac + 0] = av.x; As[ar][ac + 1] = av.y; As[ar][ac + 2] = av.z; As[ar][ac + 3] = av.w;
        Bs[br][bc + 0] = bv.x; Bs[br][bc + 1] = bv.y; Bs[br][bc + 2] = bv.z; Bs[br][bc + 3] = bv.w;
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) {
            const int kq = kk + (lane >> 4), q = lane & 15;
            const float a0 = As[wm + q][kq], a1 = As[wm + 16 + q][kq];
            const float b0 = Bs[kq][wn + q], b1 = Bs[kq][wn + 16 + q];
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
        }
    }
    for (int si = 0; si < 2; ++si)
        for (int sj = 0; sj < 2; ++sj)
            for (int r = 0; r < 4; ++r) {
                const int64_t i = bm + wm + si * 16 + 4 * (lane >> 4) + r;
                const int64_t j = bn + wn + sj * 16 + (lane & 15);
                const float old = beta != 0.f ? Cin[i * ldcin + j] : 0.f;
                C[i * ldc + j] = alpha * acc[si][sj][r] + beta * old;
            }
}

static int gemm(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int64_t ldc, const float *Cin,
                int64_t ldcin, int64_t M, int64_t N, int64_t K, float alpha, float beta, hipStream_t st) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    if (M % 64 || N % 64 || K % 16) {
        set_error("internal: product sizes must be multiples of 64 (M, N) and 16 (K)");
        return 1;
    }
    hipLaunchKernelGGL(k_gemm_f32, dim3((unsigned)(N / 64), (unsigned)(M / 64)), dim3(256), 0, st, A, lda, B,
                       ldb, C, ldc, Cin, ldcin, K, alpha, beta);
    VX_CHECK(hipGetLastError());
    return 0;
}

// One block column of a triangular factor's inverse, C = -(A B) D with A the
// inverse's finished triangle (TRI 1: lower, 2: upper; A's rows and columns
// start at the same index), B the factor's block column and D its diagonal
// block's inverse (64 x 64).  16 rows of C per work-group, so that the few
// thousand rows there are spread over the chip: 64 x 64 tiles made 52
// work-groups at most (71 us a column at 3392 rows, 14 us now); each wave 16
// columns, K in LDS chunks of 64, the next two loaded while one is
// multiplied.  An element's products are added in the order of k_gemm_f32
// (skipped zeros apart), the second product in the same work-group.
template <int TRI>
__global__ __launch_bounds__(256) void k_lu_inv_col(const float *A, int64_t ld, const float *__restrict__ B,
                                                    const float *D, float *C, int32_t K) {
    __shared__ __align__(16) float As[2][16][68], Bs[2][64][80];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int q = lane & 15, g = lane >> 4, wn = wave * 16;
    const int32_t bm = (int32_t)blockIdx.x * 16;
    const int32_t k_lo = TRI == 2 ? bm / 64 * 64 : 0, k_hi = TRI == 1 ? (bm / 64 + 1) * 64 : K;
    const int32_t chunks = (k_hi - k_lo) / 64;
    const int ar = tid >> 4, ac = (tid & 15) * 4;  // A: a float4 per thread; B: four, 16 rows apart
    const float *ap = A + (int64_t)(bm + ar) * ld + k_lo + ac;
    const float *bp = B + (int64_t)(k_lo + ar) * ld + ac;
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
    struct Chunk {
        floatx4 a, b0, b1, b2, b3;
    } c0, c1;
    auto load = [&](int32_t c, Chunk &v) __attribute__((always_inline)) {
        const int32_t cc = min(c, chunks - 1) * 64;
        const float *bb = bp + (int64_t)cc * ld;
        v.a = *reinterpret_cast<const floatx4 *>(ap + cc);
        v.b0 = *reinterpret_cast<const floatx4 *>(bb);
        v.b1 = *reinterpret_cast<const floatx4 *>(bb + 16 * ld);
        v.b2 = *reinterpret_cast<const floatx4 *>(bb + 32 * ld);
        v.b3 = *reinterpret_cast<const floatx4 *>(bb + 48 * ld);
    };
    auto step = [&](int32_t c, auto half, Chunk &v) __attribute__((always_inline)) {
        constexpr int b = decltype(half)::value;
        *reinterpret_cast<floatx4 *>(&As[b][ar][ac]) = v.a;
        *reinterpret_cast<floatx4 *>(&Bs[b][ar][ac]) = v.b0;
        *reinterpret_cast<floatx4 *>(&Bs[b][ar + 16][ac]) = v.b1;
        *reinterpret_cast<floatx4 *>(&Bs[b][ar + 32][ac]) = v.b2;
        *reinterpret_cast<floatx4 *>(&Bs[b][ar + 48][ac]) = v.b3;
        load(c + 2, v);
        lds_barrier();  // also: every wave is done with chunk c - 1, whose buffer chunk c + 1 takes
        // all operands before the first product: each waits for the one before it alone
        float x[16], y[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            x[s] = As[b][q][4 * s + g];
            y[s] = Bs[b][4 * s + g][wn + q];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 16; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], y[s], acc, 0, 0, 0);
    };
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    load(0, c0);
    load(1, c1);
    int32_t c = 0;
    for (; c + 2 <= chunks; c += 2) {
        step(c, even, c0);
        step(c + 1, odd, c1);
    }
    if (c < chunks) step(c, even, c0);
    lds_barrier();
#pragma unroll
    for (int e = 0; e < 4; ++e)
        *reinterpret_cast<float4 *>(&Bs[0][ar + 16 * e][ac]) =
            *reinterpret_cast<const float4 *>(D + (int64_t)(ar + 16 * e) * ld + ac);
#pragma unroll
    for (int r = 0; r < 4; ++r) As[0][4 * g + r][wn + q] = acc[r];
    lds_barrier();
    acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 16; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(As[0][q][4 * s + g], Bs[0][4 * s + g][wn + q], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) C[(int64_t)(bm + 4 * g + r) * ld + wn + q] = -acc[r];
}

// ---- factorisation ---------------------------------------------------------------
// F = the FP32 matrix padded with an identity block.
__global__ void k_lu_load(const double *__restrict__ L, int64_t n, int64_t np, float *__restrict__ F) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j >= np) return;
    F[i * np + j] = (i < n && j < n) ? (float)L[i * n + j] : (i == j ? 1.f : 0.f);
}

// ||A||_inf (largest row sum of magnitudes), one wave per row, into st[5] as
// the bits of a non-negative double (their integer order is the value order).
__global__ __launch_bounds__(256) void k_lu_norm(const double *__restrict__ L, int64_t n,
                                                 unsigned long long *__restrict__ st) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    double s = 0.0;
    for (int64_t j = lane; j < n; j += 64) s += fabs(L[i * n + j]);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) atomicMax(st + 5, (unsigned long long)__double_as_longlong(s));
}

// One work-group factors the panel of columns [k0, k0 + 64) over rows
// [k0, np): per column, the largest magnitude below the diagonal (ties: the
// first row) is swapped up within the panel, the column is divided by it and
// the rest of the panel is updated.  ipiv[col] = the row swapped with col.
// The panel is factored in a column-major copy Pt (64 x np, column c at
// Pt + c np), so that the pivot search and every column update read and
// write consecutive rows (the row-major matrix would put each thread on its
// own row, 4 np bytes from the next), then copied back.
__global__ __launch_bounds__(1024) void k_lu_panel(float *__restrict__ F, int64_t np, int64_t k0,
                                                   int32_t *__restrict__ ipiv, unsigned long long *__restrict__ st,
                                                   float *__restrict__ Pt) {
    __shared__ float bv[1024];
    __shared__ int bi[1024];
    __shared__ float prow[kLuB];
    const int tid = threadIdx.x;
    const int64_t rows = np - k0;
    for (int64_t e = tid; e < rows * kLuB; e += 1024) {
        const int64_t i = k0 + e / kLuB;
        const int c = (int)(e % kLuB);
        Pt[c * np + i] = F[i * np + k0 + c];
    }
    __syncthreads();
    for (int jj = 0; jj < kLuB; ++jj) {
        const int64_t col = k0 + jj;
        float *pc = Pt + (int64_t)jj * np;
        float best = -1.f;
        int besti = (int)col;
        for (int64_t i = col + tid; i < np; i += 1024) {
            const float v = fabsf(pc[i]);
            if (v > best) { best = v; besti = (int)i; }
        }
        bv[tid] = best;
        bi[tid] = besti;
        __syncthreads();
        for (int s = 512; s > 0; s >>= 1) {
            if (tid < s) {
                const float o = bv[tid + s];
                const int oi = bi[tid + s];
                if (o > bv[tid] || (o == bv[tid] && oi < bi[tid])) { bv[tid] = o; bi[tid] = oi; }
            }
            __syncthreads();
        }
        const int64_t p = bi[0];
        if (tid == 0) ipiv[col] = (int32_t)p;
        if (p != col && tid < kLuB) {
            float *q = Pt + (int64_t)tid * np;
            const float a = q[col], b = q[p];
            q[col] = b;
            q[p] = a;
        }
        __syncthreads();
        if (tid < kLuB) prow[tid] = Pt[(int64_t)tid * np + col];
        __syncthreads();
        const float piv = prow[jj];
        if (piv == 0.f) {
            if (tid == 0) st[4] = 1ull;  // singular: leave the column as it is
            __syncthreads();
            continue;
        }
        for (int64_t i = col + 1 + tid; i < np; i += 1024) {
            const float l = pc[i] / piv;
            pc[i] = l;
            for (int c = jj + 1; c < kLuB; ++c) Pt[(int64_t)c * np + i] -= l * prow[c];
        }
        __syncthreads();
    }
    for (int64_t e = tid; e < rows * kLuB; e += 1024) {
        const int64_t i = k0 + e / kLuB;
        const int c = (int)(e % kLuB);
        F[i * np + k0 + c] = Pt[c * np + i];
    }
}

// The same panel in sub-panels of kLuS columns, bit for bit: the products and
// differences of an element are those of k_lu_panel in the same order, so only
// where they are done changes.  k_lu_panel walks 64 columns of up to np rows
// through memory with one work-group (0.85 ms a panel at 3392 rows).  Here a
// work-group holds a sub-panel's columns of all rows in registers
// (k_lu_sub, one LDS barrier a column), and the panel's other columns take
// the sub-panel's steps on many work-groups (k_lu_sub_apply).  Rows move
// between two column-major copies of the panel (64 x np), so that every
// work-group reads the old places and writes the new.
constexpr int kLuS = 16;

// Panel [k0, k0 + 64) of F, rows from k0 on, column by column into Pt.
__global__ __launch_bounds__(256) void k_lu_in(const float *__restrict__ F, int64_t np, int64_t k0,
                                               float *__restrict__ Pt) {
    __shared__ float t[64][65];
    const int64_t i0 = k0 + (int64_t)blockIdx.x * 64;
    const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
    for (int r = y; r < 64; r += 4) t[r][x] = F[(i0 + r) * np + k0 + x];
    __syncthreads();
    for (int c = y; c < 64; c += 4) Pt[c * np + i0 + x] = t[x][c];
}

// Columns k .. k + 15 (c0 = k - k0 in the panel) over the rows from k on, T R
// of them at most.  A thread holds R rows, a swap exchanges the places of two
// rows; each wave offers its largest candidate with its row in LDS.  The
// step's column is a[.][0], the others move down.  The columns go back to Pt
// by the rows' old places: below the diagonal the factors, on and above it U.
template <int T, int R>
__global__ __launch_bounds__(T) void k_lu_sub(float *__restrict__ Pt, int32_t np, int32_t k0, int32_t k,
                                              int32_t *__restrict__ ipiv, int32_t *__restrict__ slot_of,
                                              unsigned long long *__restrict__ st) {
    constexpr int NW = T / 64, B = kLuS;
    __shared__ __align__(16) float crow[2][NW][B];
    __shared__ float ckey[2][NW];
    __shared__ int cpos[2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int64_t c0 = k - k0;
    float a[R][B];
    int pos[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int s = k + tid + r * T;
        pos[r] = s < np ? s : -1;
#pragma unroll
        for (int c = 0; c < B; ++c) a[r][c] = s < np ? Pt[(c0 + c) * np + s] : 0.f;
    }
#pragma unroll 1
    for (int kk = 0; kk < B; ++kk) {
        const int col = k + kk, par = kk & 1;
        float key = -1.f;
        int kp = 0x7fffffff, kr = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float v = fabsf(a[r][0]);
            if (pos[r] >= col && (v > key || (v == key && pos[r] < kp))) {
                key = v;
                kp = pos[r];
                kr = r;
            }
        }
        const float wm = wave_max(key);
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
                }
            }
        lds_barrier();
        const float ck = ckey[par][lane & (NW - 1)];
        const int cp = cpos[par][lane & (NW - 1)];
        const float gm = lane_of(row_max(ck), 15);
        const uint64_t gt = __ballot(ck == gm) & ((1ull << NW) - 1);
        const int gw = gt ? lowest_lane(gt, cp) : 0;
        int p = __builtin_amdgcn_readlane(cp, gw);
        const bool none = p < col || p >= np;  // no comparable entry (NaN): the diagonal one
        if (none) p = col;
        float row[B];
#pragma unroll
        for (int c = 0; c < B; ++c) row[c] = crow[par][gw][c];
        if (none) row[0] = __builtin_nanf("");
        const bool zero = row[0] == 0.f;  // singular: the column stays as it is
        if (tid == 0) {
            ipiv[col] = p;
            if (zero) st[4] = 1ull;
        }
        // an FP32 quotient is never as near a rounding boundary as the FP64
        // product's error, so this is the correctly rounded quotient
        const double y = 1.0 / (double)row[0];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            pos[r] = pos[r] == p ? col : pos[r] == col ? p : pos[r];
            float f = (float)((double)a[r][0] * y);
            f = zero || pos[r] <= col ? 0.f : f;
            const int s = k + tid + r * T;
            if (s < np) Pt[(c0 + kk) * np + s] = pos[r] > col && !zero ? f : a[r][0];
#pragma unroll
            for (int c = 1; c < B; ++c) a[r][c - 1] = fmaf(-f, row[c], a[r][c]);
            a[r][B - 1] = 0.f;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int s = k + tid + r * T;
        if (s < np) slot_of[pos[r]] = s;
    }
}

// The panel's columns after the sub-panel at k: moved rows in their new places
// (old -> Pt, or -> F for the last), and the columns right of the sub-panel
// through its kLuS steps.  A row per thread, 256 per work-group; each
// work-group solves for U's rows itself.
__global__ __launch_bounds__(256) void k_lu_sub_apply(const float *__restrict__ old, float *__restrict__ Pt,
                                                      float *__restrict__ F, int32_t np, int32_t k0, int32_t k,
                                                      const int32_t *__restrict__ slot_of) {
    constexpr int B = kLuS;
    __shared__ __align__(16) float lb[B][B], ub[B][kLuB];  // the block's factors; U's rows, columns of the panel
    const int32_t c0 = k - k0, c1 = c0 + B;
    const int tid = threadIdx.x;
    lb[tid >> 4][tid & 15] = old[(int64_t)(c0 + (tid & 15)) * np + slot_of[k + (tid >> 4)]];
    __syncthreads();
    if (tid >= c1 && tid < kLuB) {
        float v[B];
#pragma unroll
        for (int r = 0; r < B; ++r) v[r] = old[(int64_t)tid * np + slot_of[k + r]];
#pragma unroll
        for (int q = 0; q < B; ++q) {
            ub[q][tid] = v[q];
#pragma unroll
            for (int r = q + 1; r < B; ++r) v[r] = fmaf(-lb[r][q], v[q], v[r]);
        }
    }
    __syncthreads();
    const int32_t i = k0 + (int32_t)blockIdx.x * 256 + tid;
    if (i >= np) return;
    const int64_t s = i >= k ? slot_of[i] : i;
    float l[B];
#pragma unroll
    for (int q = 0; q < B; ++q) l[q] = old[(c0 + q) * (int64_t)np + s];
    for (int32_t c = 0; c < kLuB; c += 4) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = old[(c + e) * (int64_t)np + s];
        if (c >= c1 && i >= k) {
            if (i < k + B) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ub[i - k][c + e];
            } else {
#pragma unroll
                for (int q = 0; q < B; ++q) {
                    const float4 u = *reinterpret_cast<const float4 *>(&ub[q][c]);
                    v[0] = fmaf(-l[q], u.x, v[0]);
                    v[1] = fmaf(-l[q], u.y, v[1]);
                    v[2] = fmaf(-l[q], u.z, v[2]);
                    v[3] = fmaf(-l[q], u.w, v[3]);
                }
            }
        }
        if (c1 < kLuB) {
#pragma unroll
            for (int e = 0; e < 4; ++e) Pt[(c + e) * (int64_t)np + i] = v[e];
        } else {
            *reinterpret_cast<float4 *>(&F[(int64_t)i * np + k0 + c]) = float4{v[0], v[1], v[2], v[3]};
        }
    }
}

template <int T, int R>
static void lu_sub(float *Pt, int64_t np, int64_t k0, int64_t k, int32_t *ipiv, int32_t *slot_of,
                   unsigned long long *stt, hipStream_t st) {
    hipLaunchKernelGGL((k_lu_sub<T, R>), dim3(1), dim3(T), 0, st, Pt, (int32_t)np, (int32_t)k0, (int32_t)k, ipiv,
                       slot_of, stt);
}

// A panel by sub-panels while its rows fit a work-group's registers (16 floats
// a row, T R rows), else by k_lu_panel.  T: 64 np floats twice.
constexpr int64_t kLuSubRows = 12 * 512;

static void lu_panel(float *F, int64_t np, int64_t k0, int32_t *ipiv, int32_t *slot_of, unsigned long long *stt,
                     float *T, hipStream_t st) {
    if (np - k0 > kLuSubRows) {
        hipLaunchKernelGGL(k_lu_panel, dim3(1), dim3(1024), 0, st, F, np, k0, ipiv, stt, T);
        return;
    }
    float *P[2] = {T, T + kLuB * np};
    hipLaunchKernelGGL(k_lu_in, dim3((unsigned)((np - k0) / 64)), dim3(256), 0, st, F, np, k0, P[0]);
    for (int sub = 0; sub < kLuB / kLuS; ++sub) {
        const int64_t k = k0 + sub * kLuS, rows = np - k;
        float *A = P[sub & 1], *B = P[(sub & 1) ^ 1];
        if (rows <= 256) lu_sub<256, 1>(A, np, k0, k, ipiv, slot_of, stt, st);
        else if (rows <= 512) lu_sub<256, 2>(A, np, k0, k, ipiv, slot_of, stt, st);
        else if (rows <= 1024) lu_sub<512, 2>(A, np, k0, k, ipiv, slot_of, stt, st);
        else if (rows <= 2048) lu_sub<512, 4>(A, np, k0, k, ipiv, slot_of, stt, st);
        else if (rows <= 3072) lu_sub<512, 6>(A, np, k0, k, ipiv, slot_of, stt, st);
        else if (rows <= 4096) lu_sub<512, 8>(A, np, k0, k, ipiv, slot_of, stt, st);
        else lu_sub<512, 12>(A, np, k0, k, ipiv, slot_of, stt, st);
        hipLaunchKernelGGL(k_lu_sub_apply, dim3((unsigned)((np - k0 + 255) / 256)), dim3(256), 0, st, A, B, F,
                           (int32_t)np, (int32_t)k0, (int32_t)k, slot_of);
    }
}

// The panel's row swaps on every other column; block 0 also carries them
// into the row permutation.
__global__ __launch_bounds__(256) void k_lu_swap(float *__restrict__ F, int64_t np, int64_t k0,
                                                 const int32_t *__restrict__ ipiv, int32_t *__restrict__ perm) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        for (int jj = 0; jj < kLuB; ++jj) {
            const int64_t a = k0 + jj, b = ipiv[a];
            const int32_t t = perm[a];
            perm[a] = perm[b];
            perm[b] = t;
        }
    if (c >= np || (c >= k0 && c < k0 + kLuB)) return;
    for (int jj = 0; jj < kLuB; ++jj) {
        const int64_t a = k0 + jj, b = ipiv[a];
        if (b != a) {
            const float u = F[a * np + c], v = F[b * np + c];
            F[a * np + c] = v;
            F[b * np + c] = u;
        }
    }
}

// U12 = L11^-1 A12 for the columns right of the panel, one column per thread
// held in registers, L11 in LDS.
__global__ __launch_bounds__(256) void k_lu_trsm(float *__restrict__ F, int64_t np, int64_t k0) {
    __shared__ float L11[kLuB][kLuB + 1];
    for (int e = threadIdx.x; e < kLuB * kLuB; e += 256) L11[e / kLuB][e % kLuB] = F[(k0 + e / kLuB) * np + k0 + e % kLuB];
    __syncthreads();
    const int64_t c = k0 + kLuB + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= np) return;
    float v[kLuB];
#pragma unroll
    for (int r = 0; r < kLuB; ++r) v[r] = F[(k0 + r) * np + c];
#pragma unroll
    for (int r = 1; r < kLuB; ++r) {
        float s = v[r];
#pragma unroll
        for (int q = 0; q < r; ++q) s -= L11[r][q] * v[q];
        v[r] = s;
    }
#pragma unroll
    for (int r = 1; r < kLuB; ++r) F[(k0 + r) * np + c] = v[r];
}

// Inverses of the diagonal blocks, one work-group of 64 threads per block,
// one column of the inverse per thread: W_l = L_jj^-1 (unit lower, with its
// unit diagonal), W_u = U_jj^-1 (upper).
__global__ __launch_bounds__(kLuB) void k_lu_inv_diag(const float *__restrict__ F, int64_t np,
                                                      float *__restrict__ Wl, float *__restrict__ Wu) {
    __shared__ float D[kLuB][kLuB + 1];
    const int64_t j0 = (int64_t)blockIdx.x * kLuB;
    const int c = threadIdx.x;
    for (int r = 0; r < kLuB; ++r) D[r][c] = F[(j0 + r) * np + j0 + c];
    __syncthreads();
    float x[kLuB];
    // lower, unit diagonal: forward substitution of e_c
#pragma unroll
    for (int r = 0; r < kLuB; ++r) {
        float s = r == c ? 1.f : 0.f;
#pragma unroll
        for (int q = 0; q < r; ++q) s -= D[r][q] * x[q];
        x[r] = r < c ? 0.f : s;
    }
#pragma unroll
    for (int r = 0; r < kLuB; ++r) Wl[(j0 + r) * np + j0 + c] = x[r];
    // upper: backward substitution of e_c
#pragma unroll
    for (int r = kLuB - 1; r >= 0; --r) {
        float s = r == c ? 1.f : 0.f;
#pragma unroll
        for (int q = r + 1; q < kLuB; ++q) s -= D[r][q] * x[q];
        x[r] = r > c ? 0.f : s / D[r][r];
    }
#pragma unroll
    for (int r = 0; r < kLuB; ++r) Wu[(j0 + r) * np + j0 + c] = x[r];
}

// W = strict lower part of Wl, upper part (with the diagonal) of Wu; the
// inverse permutation.
__global__ void k_lu_merge(const float *__restrict__ Wl, const float *__restrict__ Wu, int64_t np,
                           float *__restrict__ W) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = blockIdx.y;
    if (j >= np) return;
    W[i * np + j] = j < i ? Wl[i * np + j] : Wu[i * np + j];
}

__global__ void k_lu_perm_init(int32_t *__restrict__ perm, int64_t np) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) perm[i] = (int32_t)i;
}

__global__ void k_lu_pinv(const int32_t *__restrict__ perm, int64_t np, int32_t *__restrict__ pinv) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) pinv[perm[i]] = (int32_t)i;
}

// ---- per-solve refinement ----------------------------------------------------------
__device__ __forceinline__ unsigned long long dbits(double v) { return (unsigned long long)__double_as_longlong(v); }
__device__ __forceinline__ double bitsd(unsigned long long v) { return __longlong_as_double((long long)v); }

// Convergence test (LAPACK dsgesv): done when ||r|| <= ||x|| ||A|| eps sqrt(n);
// else one more correction is counted.  One thread; r and xm are the maxima
// of |r_i| and |x_i|.
__device__ __forceinline__ void lu_check(unsigned long long *__restrict__ st, double *__restrict__ nrm, int64_t n,
                                         double r, double xm) {
    const double an = bitsd(st[5]);
    const double cte = an * 1.1102230246251565e-16 * sqrt((double)n);
    nrm[1] = (xm > 0.0 && an > 0.0) ? r / (xm * an) : r;
    if (r <= xm * cte) st[0] = 1ull;
    else st[1] += 1ull;
}

// The largest of a value per thread (as bits of a non-negative double), valid
// in thread 0.
template <int W>
__device__ __forceinline__ unsigned long long block_max_bits(unsigned long long v) {
    __shared__ unsigned long long s[W];
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long q = __shfl_xor(v, o, 64);
        v = q > v ? q : v;
    }
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < W; ++w) v = s[w] > v ? s[w] : v;
    return v;
}

// sum_j w[j] v[j] over the lane's j = lo + lane, lo + lane + 64, ... < hi, in
// order, with eight loads of each in flight.
template <typename T>
__device__ __forceinline__ T row_dot(const T *__restrict__ w, const T *__restrict__ v, int64_t lo, int64_t hi,
                                     int lane) {
    T s = T(0);
    int64_t j = lo + lane;
    for (; j + 7 * 64 < hi; j += 8 * 64) {
        T a[8], b[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            a[e] = w[j + 64 * e];
            b[e] = v[j + 64 * e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) s += a[e] * b[e];
    }
    for (; j < hi; j += 64) s += w[j] * v[j];
    return s;
}

// x = 0, so r = b = [R; d_g], permuted and in FP32, and its test, in one
// work-group: no pass over A for it.
__global__ __launch_bounds__(1024) void k_lu_begin(double *__restrict__ x, int64_t n, int64_t np,
                                                   const double *__restrict__ R, double d_g_host,
                                                   const double *__restrict__ d_g_dev,
                                                   const int32_t *__restrict__ pinv, float *__restrict__ rp,
                                                   unsigned long long *__restrict__ st, double *__restrict__ nrm) {
    const double d_g = d_g_dev ? *d_g_dev : d_g_host;
    unsigned long long m = 0ull;
    for (int64_t i = threadIdx.x; i < np; i += 1024) {
        x[i] = 0.0;
        const double b = i < n - 1 ? R[i] : (i < n ? d_g : 0.0);
        rp[pinv[i]] = (float)b;
        const unsigned long long q = dbits(fabs(b));
        m = q > m ? q : m;
    }
    m = block_max_bits<16>(m);
    if (threadIdx.x != 0) return;
    st[0] = st[1] = st[2] = st[3] = st[6] = 0ull;
    lu_check(st, nrm, n, bitsd(m), 0.0);
}

// r = b - A x with b = [R; d_g], one wave per row, written permuted and in
// FP32 (rp[pinv[i]]); the largest |r_i| into st[2].  The last work-group to
// end (st[6] counts them) tests for convergence and clears both for the next
// pass.  Bound by the read of A: with eight loads in flight, without the
// first pass and the test's launches a birth of 1000, 2040 and 3320 panels (three
// corrections) takes 144, 194 and 289 us with its copies, 208, 342 and 517
// before.
__global__ __launch_bounds__(256) void k_lu_resid(const double *__restrict__ A, const double *__restrict__ R,
                                                  double d_g_host, const double *__restrict__ d_g_dev, int64_t n,
                                                  int64_t np, const double *__restrict__ x,
                                                  const int32_t *__restrict__ pinv, float *__restrict__ rp,
                                                  unsigned long long *__restrict__ st, double *__restrict__ nrm) {
    if (st[0]) return;
    const double d_g = d_g_dev ? *d_g_dev : d_g_host;
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    unsigned long long m = 0ull;
    if (i >= n && i < np) {
        if (lane == 0) rp[pinv[i]] = 0.f;
    } else if (i < n) {
        double s = row_dot(A + i * n, x, 0, n, lane);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        const double r = (i < n - 1 ? R[i] : d_g) - s;
        if (lane == 0) rp[pinv[i]] = (float)r;
        m = dbits(fabs(r));
    }
    m = block_max_bits<4>(m);
    if (threadIdx.x != 0) return;
    atomicMax(st + 2, m);
    __threadfence();
    if (atomicAdd(st + 6, 1ull) + 1 != gridDim.x) return;
    __threadfence();
    lu_check(st, nrm, n, bitsd(atomicMax(st + 2, 0ull)), bitsd(atomicMax(st + 3, 0ull)));
    st[2] = 0ull;
    st[6] = 0ull;
}

// t = L^-1 (P r): row i sums W's strict lower part (one wave per row).
__global__ __launch_bounds__(256) void k_lu_apply_l(const float *__restrict__ W, int64_t np,
                                                    const float *__restrict__ rp, float *__restrict__ t,
                                                    const unsigned long long *__restrict__ st) {
    if (st[0]) return;
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= np) return;
    float s = row_dot(W + i * np, rp, 0, i, lane);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) t[i] = s + rp[i];
}

// x += U^-1 t: row i sums W's upper part; the largest |x_i| into st[3].
__global__ __launch_bounds__(256) void k_lu_apply_u(const float *__restrict__ W, int64_t np,
                                                    const float *__restrict__ t, double *__restrict__ x,
                                                    unsigned long long *__restrict__ st) {
    if (st[0]) return;
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    unsigned long long m = 0ull;
    if (i < np) {
        float s = row_dot(W + i * np, t, i, np, lane);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        const double xi = x[i] + (double)s;
        if (lane == 0) x[i] = xi;
        m = dbits(fabs(xi));
    }
    m = block_max_bits<4>(m);
    if (threadIdx.x == 0) atomicMax(st + 3, m);
}

// ---- host side ------------------------------------------------------------------------
static LuBufs &lu_of(vx_case *c) {
    if (!c->lu) c->lu = new LuBufs();
    return *c->lu;
}

void lu_release(vx_case *c) {
    if (!c->lu) return;
    LuBufs &b = *c->lu;
    b.F.release(); b.W.release(); b.Wl.release(); b.Wu.release(); b.T.release(); b.A.release();
    b.x.release(); b.rp.release(); b.t.release(); b.ipiv.release(); b.perm.release(); b.pinv.release();
    b.st.release(); b.nrm.release();
    delete c->lu;
    c->lu = nullptr;
}

// Factor c->L (the FP64 panel matrix, (P+1)^2) and invert the factors.
int launch_lu_setup(vx_case *c) {
    LuBufs &b = lu_of(c);
    hipStream_t st = c->stream;
    const int64_t n = c->P + 1, np = (n + kLuB - 1) / kLuB * kLuB;
    b.n = n;
    b.np = np;
    const size_t nn = (size_t)(np * np);
    if (b.F.ensure(nn, st) || b.Wl.ensure(nn, st) || b.Wu.ensure(nn, st) || b.W.ensure(nn, st) ||
        b.T.ensure((size_t)(2 * np * kLuB), st) || b.A.ensure((size_t)(n * n), st) || b.x.ensure((size_t)np, st) ||
        b.rp.ensure((size_t)np, st) || b.t.ensure((size_t)np, st) || b.ipiv.ensure((size_t)np, st) ||
        b.perm.ensure((size_t)np, st) || b.pinv.ensure((size_t)np, st) || b.st.ensure(8, st) || b.nrm.ensure(2, st))
        return 1;
    VX_CHECK(hipMemcpyAsync(b.A.p, c->L.p, sizeof(double) * n * n, hipMemcpyDeviceToDevice, st));
    VX_CHECK(prim::fill(b.st.p, 8, 0ull, st));
    VX_CHECK(prim::fill(b.Wl.p, (int64_t)nn, 0.f, st));
    VX_CHECK(prim::fill(b.Wu.p, (int64_t)nn, 0.f, st));
    const dim3 g2((unsigned)((np + 255) / 256), (unsigned)np);
    const unsigned g1 = (unsigned)((np + 255) / 256);
    hipLaunchKernelGGL(k_lu_load, g2, dim3(256), 0, st, c->L.p, n, np, b.F.p);
    hipLaunchKernelGGL(k_lu_norm, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, c->L.p, n, b.st.p);
    hipLaunchKernelGGL(k_lu_perm_init, dim3(g1), dim3(256), 0, st, b.perm.p, np);
    // right-looking LU: panel, swaps, block row, trailing product
    for (int64_t k0 = 0; k0 < np; k0 += kLuB) {
        lu_panel(b.F.p, np, k0, b.ipiv.p, b.pinv.p, b.st.p, b.T.p, st);
        hipLaunchKernelGGL(k_lu_swap, dim3(g1), dim3(256), 0, st, b.F.p, np, k0, b.ipiv.p, b.perm.p);
        const int64_t rest = np - k0 - kLuB;
        if (rest > 0) {
            hipLaunchKernelGGL(k_lu_trsm, dim3((unsigned)((rest + 255) / 256)), dim3(256), 0, st, b.F.p, np, k0);
            float *A21 = b.F.p + (k0 + kLuB) * np + k0;
            float *A12 = b.F.p + k0 * np + k0 + kLuB;
            float *A22 = b.F.p + (k0 + kLuB) * np + k0 + kLuB;
            if (gemm(A21, np, A12, np, A22, np, A22, np, rest, rest, kLuB, -1.f, 1.f, st)) return 1;
        }
    }
    VX_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_lu_pinv, dim3(g1), dim3(256), 0, st, b.perm.p, np, b.pinv.p);
    // inverses of the factors: diagonal blocks, then block columns
    //   L: from the last block column back, Wl[j+, j] = -(Wl[j+, j+] L[j+, j]) Wl[j, j]
    //   U: from the first forward,          Wu[:j, j] = -(Wu[:j, :j] U[:j, j]) Wu[j, j]
    hipLaunchKernelGGL(k_lu_inv_diag, dim3((unsigned)(np / kLuB)), dim3(kLuB), 0, st, b.F.p, np, b.Wl.p, b.Wu.p);
    for (int64_t j0 = np - kLuB; j0 >= 0; j0 -= kLuB) {
        const int64_t r0 = j0 + kLuB, m = np - r0;
        if (m <= 0) continue;
        hipLaunchKernelGGL(k_lu_inv_col<1>, dim3((unsigned)(m / 16)), dim3(256), 0, st, b.Wl.p + r0 * np + r0, np,
                           b.F.p + r0 * np + j0, b.Wl.p + j0 * np + j0, b.Wl.p + r0 * np + j0, (int32_t)m);
    }
    for (int64_t j0 = kLuB; j0 < np; j0 += kLuB)
        hipLaunchKernelGGL(k_lu_inv_col<2>, dim3((unsigned)(j0 / 16)), dim3(256), 0, st, b.Wu.p, np, b.F.p + j0,
                           b.Wu.p + j0 * np + j0, b.Wu.p + j0, (int32_t)j0);
    hipLaunchKernelGGL(k_lu_merge, g2, dim3(256), 0, st, b.Wl.p, b.Wu.p, np, b.W.p);
    VX_CHECK(hipGetLastError());
    unsigned long long sing = 0;
    VX_CHECK(hipMemcpyAsync(&sing, b.st.p + 4, sizeof(sing), hipMemcpyDeviceToHost, st));
    VX_CHECK(hipStreamSynchronize(st));
    // the factors' staging is not needed per step
    b.F.release(); b.Wl.release(); b.Wu.release(); b.T.release();
    if (sing) {
        set_error("panel matrix is singular in FP32 (zero pivot)");
        return 1;
    }
    return 0;
}

// Solve A x = [R; d_g] into c->lu->x (first P entries: the sheet strengths);
// d_g from *d_g_dev when that is not null.
int launch_lu_solve(vx_case *c, const double *R, double d_g, const double *d_g_dev) {
    LuBufs &b = *c->lu;
    hipStream_t st = c->stream;
    const int64_t n = b.n, np = b.np;
    const unsigned gw = (unsigned)((np + 3) / 4);
    hipLaunchKernelGGL(k_lu_begin, dim3(1), dim3(1024), 0, st, b.x.p, n, np, R, d_g, d_g_dev, b.pinv.p, b.rp.p,
                       b.st.p, b.nrm.p);
    for (int it = 0; it < kLuMaxIt; ++it) {
        hipLaunchKernelGGL(k_lu_apply_l, dim3(gw), dim3(256), 0, st, b.W.p, np, b.rp.p, b.t.p, b.st.p);
        hipLaunchKernelGGL(k_lu_apply_u, dim3(gw), dim3(256), 0, st, b.W.p, np, b.t.p, b.x.p, b.st.p);
        hipLaunchKernelGGL(k_lu_resid, dim3(gw), dim3(256), 0, st, b.A.p, R, d_g, d_g_dev, n, np, b.x.p, b.pinv.p,
                           b.rp.p, b.st.p, b.nrm.p);
    }
    VX_CHECK(hipGetLastError());
    return 0;
}

const double *lu_solution(vx_case *c) { return c->lu ? c->lu->x.p : nullptr; }

int lu_info(vx_case *c, int32_t *iters, int32_t *converged, double *resid) {
    if (!c->lu) {
        set_error("bad argument: the case has no FP32 LU (VX_FLAG_LU_REFINE)");
        return 2;
    }
    unsigned long long s[2] = {0, 0};
    double r = 0.0;
    VX_CHECK(hipMemcpyAsync(s, c->lu->st.p, sizeof(s), hipMemcpyDeviceToHost, c->stream));
    VX_CHECK(hipMemcpyAsync(&r, c->lu->nrm.p + 1, sizeof(r), hipMemcpyDeviceToHost, c->stream));
    VX_CHECK(hipStreamSynchronize(c->stream));
    if (iters) *iters = (int32_t)s[1];
    if (converged) *converged = (int32_t)s[0];
    if (resid) *resid = r;
    return 0;
}

}  // namespace vx
