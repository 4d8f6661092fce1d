// Small dense factorizations for CholeskyQR on the device.
//
// Reference counterparts: cuda_cusolver_dpotrf (src/cuda_proxy.cu:315-339),
// cuda_cublas_dtrsm (:254-275), and the host LAPACKE_dpotrf / LAPACKE_dtrtri
// calls of examples/example_CholeskyQR.c:120-139.
//
//   hip_dpotrf(U)   blocked right-looking Cholesky A = R^T R over 64-wide
//                   block rows, two launches each: the block row (diagonal
//                   block and R_jj^{-T} A_j,rest) and the FP64 MFMA update of
//                   the trailing upper triangle.  The strictly lower part of
//                   A is not touched.  Returns LAPACK's info (k+1 when the
//                   pivot k is not > 0).
//   hip_dtrtri_upper  R^{-1} for upper-triangular R: up to n = 192 a sweep
//                   per column in one launch, beyond that the 64 x 64 diagonal
//                   blocks in one launch, then pairs of inverted blocks
//                   joined by FP64 MFMA products and corrected once, the
//                   block size doubling.
//   hip_dtrsm(R,U,N,N)  B := alpha * B * R^{-1}: R^{-1} (trtri) followed by
//                   one FP64 MFMA DGEMM per column block of the result, each
//                   reading only the non-zero rows of R^{-1}; blocks are
//                   produced from the last to the first through a workspace,
//                   so B can be overwritten in place.
#include <algorithm>
#include <cfloat>
#include <climits>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "ca3dmm_ext.h"
#include "dgemm_tile.h"
#include "hip_common.h"

namespace {

constexpr int kMaxN = 8192;            // the documented limit of the factorizations

constexpr int kPb = 64;                // block width of the Cholesky and of the inverse

__device__ __forceinline__ double readlane(double v, int lane)
{
    const uint64_t u = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((int) (uint32_t) u, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((int) (uint32_t) (u >> 32), lane);
    return __longlong_as_double((long long) (((uint64_t) hi << 32) | lo));
}

// v of lane I of the row of 16 lanes that the lane is in
template <int I>
__device__ __forceinline__ double row_lane(double v)
{
    return __longlong_as_double(__builtin_amdgcn_update_dpp((long long) 0, __double_as_longlong(v), 0x150 + I, 0xf, 0xf,
                                                            true));                    // row_newbcast:I
}

template <int I, int N, class F>
__device__ __forceinline__ void unrolled(const F &f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<I + 1, N>(f);
    }
}

// 16 steps of the factorization of the 16 x 16 block d, held by every row of
// 16 lanes (lane = column, register = row), and of the columns r; 8 where no
// more than 8 rows are not the identity's.  False if a
// pivot is outside [2^-900, 2^900] (not positive ones among them): r is then
// of no use.  The square root comes from Goldschmidt's iteration, the quotients
// from its reciprocal and one correction, which leaves them as the division
// would round them, and the steps eliminate with these rounded rows: what they
// round off comes back in the rows below.  (Eliminating with d_k / p_k and
// taking all roots at the end leaves up to four times the backward error for
// n <= 32, and is no shorter: 18.3 us a block row, 17.4 so.)
__device__ __forceinline__ bool eliminate16(double (&d)[16], double (&r)[16], int rows, bool first, int col)
{
    bool ok = true;
    auto step = [&](auto K) __attribute__((always_inline)) {
        constexpr int k = decltype(K)::value;
        const double p = row_lane<k>(d[k]), y = __builtin_amdgcn_rsq(p);
        ok = ok && p >= 0x1p-900 && p <= 0x1p900;
        double g = p * y, h = 0.5 * y, e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        const double piv = fma(fma(-g, g, p), h, g), inv = h + h;
        const double qd = d[k] * inv, qr = r[k] * inv;
        const double dk = fma(fma(-qd, piv, d[k]), inv, qd), rk = fma(fma(-qr, piv, r[k]), inv, qr);
        unrolled<k + 1, 16>([&](auto I) {
            constexpr int i = decltype(I)::value;
            const double f = -row_lane<i>(dk);
            d[i] = fma(f, dk, d[i]);
            r[i] = fma(f, rk, r[i]);
        });
        r[k] = first && col == k ? piv : rk;
        // r keeps pace with d: left to itself the compiler runs all of d first
        // and holds 120 multipliers for r
        unrolled<k, 16>([&](auto I) {
            double &ri = r[decltype(I)::value];
            asm volatile("" : "+v"(ri));
        });
        double &dl = d[15];
        asm volatile("" : "+v"(dl));
    };
    unrolled<0, 8>(step);
    if (rows > 8) unrolled<8, 16>(step);
    return ok;
}

// Block row j0 of the factorization: R_jj of the jb x jb diagonal block and
// X = R_jj^{-T} A(j0 : j0 + jb, c) for the columns c right of it, 64 columns
// per workgroup.  Every workgroup factors the diagonal block itself, so that
// the solve needs no second launch behind it; workgroup 0 stores it, to Rjj
// (leading dimension 64) where other workgroups may still read A's.
//
// The block row is a 64 x 128 array in LDS.  16 rows at a time: lane = column,
// the 16 rows in registers of two waves, which both also hold the 16 x 16
// diagonal block, so that no barrier falls between two pivots; then the rows
// below are updated by MFMAs.  The chain of 64 pivots (square root, quotient,
// first update) bounds it.
//
// info: 0 written by the first block row; a later one does nothing once an
// earlier one has set it, and writes j0 + k + 1 when its pivot k is not > 0.
// Workgroup 0 may do so while waves of the same launch still read info: those
// take a value above j0 for none, so that all of them go on alike.  The block
// is then left as LAPACK's: factor rows before the failing pivot, and in the
// others what remains after those; the columns right of it stay as they are.
__global__ __launch_bounds__(256) void potrf_row_kernel(double *A, int64_t lda, int j0, int jb, int n, double *Rjj,
                                                        int *info)
{
    constexpr int LD = 2 * kPb + 1;
    __shared__ double W[kPb][LD];           // W[i][j]: row i; columns j < 64 the diagonal block, then the 64 others
    __shared__ int bad, plain;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int seen = j0 > 0 ? *info : 0;     // looked at once the loads below are under way
    const int c0 = j0 + jb + (int) blockIdx.x * kPb, nc = min(kPb, n - c0);
    double *D = A + (int64_t) j0 * lda + j0, *S = A + (int64_t) c0 * lda + j0;
    if (t == 0) bad = plain = 0;
    // beyond jb the identity, below the diagonal and beyond nc zeros (loaded
    // from clamped places and selected afterwards: a load under a condition
    // would be waited for by itself)
    double dv[kPb / 4], sv[kPb / 4];
    const int ri = min(lane, jb - 1);
#pragma unroll
    for (int q = 0; q < kPb / 4; ++q) {
        const int j = wave + 4 * q;
        dv[q] = D[(int64_t) min(j, jb - 1) * lda + ri];
    }
    if (nc > 0) {
#pragma unroll
        for (int q = 0; q < kPb / 4; ++q) sv[q] = S[(int64_t) min(wave + 4 * q, nc - 1) * lda + ri];
    } else {
#pragma unroll
        for (int q = 0; q < kPb / 4; ++q) sv[q] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < kPb / 4; ++q) {
        const int j = wave + 4 * q;
        W[lane][j] = lane <= j && j < jb ? dv[q] : lane == j ? 1.0 : 0.0;
        W[lane][kPb + j] = lane < jb && j < nc ? sv[q] : 0.0;
    }
    if (seen > 0 && seen <= j0) return;
    __syncthreads();
    for (int s = 0; s < jb; s += 16) {       // (beyond jb the identity)
        double r[16], d[16];
        bool ok = true;
        if (wave < 2) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                r[i] = W[s + i][t];
                d[i] = W[s + i][s + (lane & 15)];
            }
            ok = eliminate16(d, r, jb - s, (t & ~15) == s, lane & 15);
            if (t == 0 && !ok) plain = 1;
        }
        __syncthreads();                   // both waves have read the diagonal block before one stores it
        if (plain) {
            // an extreme pivot in these 16 rows: the same steps in LDS, by
            // square root and division
            for (int k = s; k < s + 16; ++k) {
                const double p = W[k][k];
                __syncthreads();
                if (!(p > 0.0)) {
                    if (t == 0) bad = k + 1;
                    break;
                }
                const double piv = sqrt(p);
                if (t >= k && t < 2 * kPb) W[k][t] = t == k ? piv : W[k][t] / piv;
                __syncthreads();
                if (t > k && t < 2 * kPb)
                    for (int i = k + 1; i < s + 16; ++i) W[i][t] = fma(-W[k][i], W[k][t], W[i][t]);
                __syncthreads();
            }
            __syncthreads();
            if (t == 0) plain = 0;
        } else if (t >= s && wave < 2) {
#pragma unroll
            for (int i = 0; i < 16; ++i) W[s + i][t] = r[i];
        }
        __syncthreads();
        if (bad) {
            // the rows behind these 16 take the steps before the failing one
            if (t < kPb)
                for (int i = s + 16; i < kPb; ++i)
                    for (int k = s; k < bad - 1; ++k) W[i][t] = fma(-W[k][i], W[k][t], W[i][t]);
            __syncthreads();
            break;
        }
        if (s + 16 >= jb) break;
        // rows below: W(i, j) -= W(s : s + 16, i)^T W(s : s + 16, j) for the
        // block rows bi and the blocks bj >= bi of each
        const int s16 = s / 16;
        int e = 0;
        for (int bi = s16 + 1; bi < 4; ++bi)
            for (int bj = bi; bj < 8; ++bj, ++e) {
                if ((e & 3) != wave) continue;
                const int l16 = lane & 15, h = lane >> 4;
                ca3::gemm::f64x4 acc;
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = W[16 * bi + 4 * v + h][16 * bj + l16];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-W[s + 4 * ks + h][16 * bi + l16],
                                                               W[s + 4 * ks + h][16 * bj + l16], acc, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) W[16 * bi + 4 * v + h][16 * bj + l16] = acc[v];
            }
        __syncthreads();
    }
    if (blockIdx.x == 0) {
        const bool last = nc <= 0;
        if (t == 0 && (j0 == 0 || bad)) *info = bad ? j0 + bad : 0;
        for (int j = wave; j < jb; j += 4)
            if (lane <= j) (last ? D : Rjj)[(int64_t) j * (last ? lda : kPb) + lane] = W[lane][j];
    }
    for (int j = wave; !bad && j < nc; j += 4)
        if (lane < jb) S[(int64_t) j * lda + lane] = W[lane][kPb + j];
}

// The trailing update behind a block row of 64: C(i, j) -= X(:, i)^T X(:, j)
// for i <= j < n, X of 64 rows, one 64 x 64 tile per workgroup, tiles of the
// upper triangle only, C loaded under the products.  Workgroup 0 also puts
// the factored diagonal block (up to a failing pivot of its own, info > j0) in
// its place.
template <bool DTL>
__global__ __launch_bounds__(512, 4) void potrf_update_kernel(const double *X, double *C, int64_t lda, int n,
                                                             const double *Rjj, double *D, int j0, const int *info)
{
    using namespace ca3::gemm;
    using TL = Tile64;
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];
    const int failed = *info;                // looked at before the stores
    // tile pairs ti <= tj, column by column of the triangle
    int tj = (int) ((sqrtf(8.0f * (float) blockIdx.x + 1.0f) - 1.0f) * 0.5f);
    while (tj * (tj + 1) / 2 > (int) blockIdx.x) --tj;
    while ((tj + 1) * (tj + 2) / 2 <= (int) blockIdx.x) ++tj;
    const int ti = (int) blockIdx.x - tj * (tj + 1) / 2;
    const int m0 = __builtin_amdgcn_readfirstlane(ti * TL::BM), n0 = __builtin_amdgcn_readfirstlane(tj * TL::BN);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int row0 = m0 + (wave % TL::WM) * (TL::BM / TL::WM) + (lane & 15);
    const int col0 = n0 + (wave / TL::WM) * (TL::BN / TL::WN) + (lane >> 4);
    double c[TL::FI][TL::FJ][4];
#pragma unroll
    for (int i = 0; i < TL::FI; ++i)
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row0 + 16 * i, col = col0 + 16 * j + 4 * r;
                c[i][j][r] = (row <= col && col < n) ? C[(int64_t) col * lda + row] : 0.0;
            }
    f64x4 acc[TL::FI][TL::FJ];
    zero(acc);
    if constexpr (DTL) {
        DtlLoader<0, 4, TL::BM, TL::NW> da, db;
        da.init(X, lda, m0, min(TL::BM, n - m0));
        db.init(X, lda, n0, min(TL::BN, n - n0));
        mainloop_dtl<TL>(da, db, lda, lda, 0, kPb, A0, A1, B0, B1, acc);
    } else {
        TL::OperandLoader<0> la, lb;
        la.init(X, lda, m0, n);
        lb.init(X, lda, n0, n);
        mainloop<TL>(la, lb, 0, kPb, m0 + TL::BM <= n && n0 + TL::BN <= n, LdsPair{A0, A1}, LdsPair{B0, B1}, acc);
    }
    if (!failed) {
#pragma unroll
        for (int i = 0; i < TL::FI; ++i)
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = row0 + 16 * i, col = col0 + 16 * j + 4 * r;
                    if (row <= col && col < n) C[(int64_t) col * lda + row] = ca3::add_rn(c[i][j][r], -acc[i][j][r]);
                }
    }
    if (blockIdx.x == 0 && (!failed || failed > j0))
        for (int e = t; e < kPb * kPb; e += TL::THREADS)
            if (e % kPb <= e / kPb) D[(int64_t) (e / kPb) * lda + e % kPb] = Rjj[e];
}

// X = R^{-1} for n <= kSweepN: one workgroup per column j solves R x = e_j by a
// column sweep in LDS, all columns at once in one launch.  The blocked form
// below has a launch and five more per doubling.  us, sweep / blocked: n = 1
// 11.4 / 37.2, 64 33.2 / 37.6, 129 54.9 / 72.4, 200 80.2 / 78.3, 400 170 / 113.
constexpr int kSweepN = 192;

__global__ __launch_bounds__(256) void trtri_sweep_kernel(const double *R, int64_t ldr, double *X, int64_t ldx, int n)
{
    __shared__ double x[kSweepN];
    const int j = blockIdx.x, t = threadIdx.x;
    for (int p = t; p <= j; p += 256) x[p] = (p == j) ? 1.0 : 0.0;
    __syncthreads();
    for (int i = j; i >= 0; --i) {
        const double xi = x[i] / R[(int64_t) i * ldr + i];
        __syncthreads();
        if (t == 0) x[i] = xi;
        for (int p = t; p < i; p += 256) x[p] = fma(-R[(int64_t) i * ldr + p], xi, x[p]);
        __syncthreads();
    }
    for (int p = t; p < n; p += 256) X[(int64_t) j * ldx + p] = (p <= j) ? x[p] : 0.0;
}

// X = R^{-1} on the 64 x 64 diagonal blocks (the last may be smaller), one
// workgroup each, the zeros below the diagonal included.  A wave sweeps 8
// columns from the bottom row up, lane = row, so that a step is 8 independent
// quotients and updates.  (A column takes no step behind its own row: its zeros
// there would turn an infinity or a zero pivot of a later column into NaN.)
__global__ __launch_bounds__(64 * kPb / 8) void trtri_diag_kernel(const double *R, int64_t ldr, double *X, int64_t ldx, int n)
{
    __shared__ double L[kPb][kPb + 1];     // L[j][i] = R(j0 + i, j0 + j), i <= j
    const int j0 = (int) blockIdx.x * kPb, jb = min(kPb, n - j0);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const double *D = R + (int64_t) j0 * ldr + j0;
    constexpr int NQ = 8;                  // columns per wave, waves 64 / 8
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = D[(int64_t) min(wave + 8 * q, jb - 1) * ldr + min(lane, jb - 1)];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int j = wave + 8 * q;
        L[j][lane] = lane <= j && j < jb ? v[q] : lane == j ? 1.0 : 0.0;
    }
    __syncthreads();
    const int w0 = __builtin_amdgcn_readfirstlane(wave * NQ);
    // quotients from the rounded reciprocal and one correction (the rounded
    // quotient, where nothing leaves the normal range); by division where a
    // diagonal entry is extreme
    const double dl = L[lane][lane], rdiag = 1.0 / dl;
    const bool normal = __all(fabs(dl) > 0x1p-500 && fabs(dl) < 0x1p500);
    double x[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[q] = lane == w0 + q ? 1.0 : 0.0;
    if (normal) {
        auto step = [&](int i, auto own) __attribute__((always_inline)) {       // own: one of the wave's rows
            const double d = L[i][i], rd = readlane(rdiag, i), u = lane < i ? -L[i][lane] : 0.0;
            double t[NQ], xi[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) t[q] = readlane(x[q], i);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const double v0 = t[q] * rd, v1 = fma(fma(-v0, d, t[q]), rd, v0);
                xi[q] = v1 == v1 ? v1 : v0;            // t not finite
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                if (!decltype(own)::value || i <= w0 + q)
                    x[q] = lane < i ? fma(u, xi[q], x[q]) : (lane == i ? xi[q] : x[q]);
        };
        for (int i = w0 + NQ - 1; i > w0; --i) step(i, std::true_type{});
        for (int i = w0; i >= 0; --i) step(i, std::false_type{});
    } else {
        for (int i = w0 + NQ - 1; i >= 0; --i) {
            const double d = L[i][i], u = lane < i ? -L[i][lane] : 0.0;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const double xi = readlane(x[q], i) / d;
                if (i <= w0 + q) x[q] = lane < i ? fma(u, xi, x[q]) : (lane == i ? xi : x[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int j = w0 + q;
        if (j < jb && lane < jb) X[(int64_t) (j0 + j) * ldx + j0 + lane] = lane <= j ? x[q] : 0.0;
    }
}

// A wave's 16 x 16 products of a join again, each over its own k alone (k <= its
// row of X22^T, or, MUL, k >= its row of X11): where R holds an infinity
// or a NaN, the zeros of the triangles that a tile multiplies with it would
// carry it into entries that do not depend on it.  In the order of k, from
// global memory: only waves whose products are not finite come here.
template <bool MUL>
__device__ __forceinline__ void join_one_by_one(const ca3::gemm::GemmArgs &g, int row, int n0, int ct0, int ns,
                                                ca3::gemm::f64x4 &acc)
{
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int ct = ct0 + 4 * r, col = n0 + ct - (ct == ns + 1);
        double v = 0.0;
        if (row < g.M && ct != ns && col < g.N)
            for (int k = MUL ? row : 0; k < (MUL ? g.K : row + 1); ++k)
                v = fma(g.A[MUL ? row + (int64_t) k * g.lda : k + (int64_t) row * g.lda],
                        g.B[col + (int64_t) k * g.ldb], v);
        acc[r] = v;
    }
}

// The products of a tile of X12^T with R11^T for k in [n0, n0 + 32), where R11
// counts as zero below its diagonal: through registers into the LDS images of
// two direct-to-LDS stages.
__device__ __forceinline__ void join_triangle(const ca3::gemm::GemmArgs &g, int m0, int mn, int n0, double *A0,
                                              double *A1, double *B0, double *B1, ca3::gemm::f64x4 (&acc)[1][1])
{
    using namespace ca3::gemm;
    double a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = (int) threadIdx.x + 256 * q, lo = e & 31, hi = e >> 5;
        a[q] = g.A[(int64_t) (m0 + min(hi, mn - 1)) * g.lda + n0 + lo];          // k = lo, x = hi
        b[q] = g.B[(int64_t) (n0 + hi) * g.ldb + n0 + lo];                       // k = hi, x = lo
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = (int) threadIdx.x + 256 * q, lo = e & 31, hi = e >> 5;
        (lo < kBK ? A0 : A1)[dtl_index<0, 32>(lo % kBK, hi)] = a[q];
        (hi < kBK ? B0 : B1)[dtl_index<1, 32>(hi % kBK, lo)] = lo <= hi ? b[q] : 0.0;
    }
    __syncthreads();
    stage_mfma_dtl<0, 1, Tile32, 1, 1>(A0, B0, acc);
    stage_mfma_dtl<0, 1, Tile32, 1, 1>(A1, B1, acc);
}

// Joins pairs of inverted blocks: with R11 (s x s, at o = 2 s blockIdx.y) and
// R22 (w x w) inverted in X, X12 = -X11 (R12 X22).  PART 0 forms the
// transpose of T = R12 X22 in the place of X21 (w x s, zeroed at the end),
// PART 1 the product of X11 with it.  Below the diagonal the 64 x 64 blocks
// hold such products of earlier steps: k starts (ends) at the tile's first
// row (last column), which passes over them and over the zeros.  With fewer
// than 16 k the one stage starts before the block (o + s >= 64, so inside X
// and R) and counts what it reads there as zero.
//
// X11 is a rounded inverse, so that R11 X12 differs from -T by some u |R11|
// |X11| |T|, where a back substitution leaves u |R11| |X12|: at kappa(R) = 1e6
// six times the residual R X - I, and with it 1.3 times that of a solve.  PART
// 2 forms the transpose of what is missing, E = -T - R11 X12, in the place of
// T, and PART 3 adds X11 E to X12, which brings both residuals back to the
// back substitution's.  (Entries that are not finite are left as they are.)
template <int PART, bool DTL>
__global__ __launch_bounds__(256, 4) void trtri_join_kernel(const double *R, int64_t ldr, double *X, int64_t ldx,
                                                           int n, int s)
{
    using namespace ca3::gemm;
    using TL = Tile32;
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];
    const int o = 2 * s * (int) blockIdx.y, w = min(s, n - o - s);
    GemmArgs g;
    constexpr bool MUL = PART & 1;              // by X11
    g.M = MUL ? s : w;
    g.N = MUL ? w : s;
    g.K = PART == 0 ? w : s;
    g.nsrc = 0;
    g.alpha = PART == 1 || PART == 2 ? -1.0 : 1.0;
    g.beta = PART < 2 ? 0.0 : g.alpha;
    double *const X11 = X + (int64_t) o * ldx + o, *const X21 = X11 + s, *const X12 = X11 + (int64_t) s * ldx;
    g.A = MUL ? X11 : PART == 0 ? X12 + s : X12;
    g.lda = ldx;
    g.B = MUL ? X21 : R + (int64_t) (PART == 0 ? o + s : o) * ldr + o;
    g.ldb = MUL ? ldx : ldr;
    g.C = MUL ? X12 : X21;
    g.ldc = ldx;
    const int tiles_m = (g.M + TL::BM - 1) / TL::BM, tiles_n = (g.N + TL::BN - 1) / TL::BN;
    if ((int) blockIdx.x >= tiles_m * tiles_n) return;
    // the tiles with the longest k first
    const int tm = (int) blockIdx.x / tiles_n;
    const int m0 = __builtin_amdgcn_readfirstlane((PART ? tm : tiles_m - 1 - tm) * TL::BM);
    const int n0 = __builtin_amdgcn_readfirstlane(((int) blockIdx.x % tiles_n) * TL::BN);
    const int kbeg = MUL ? m0 : PART == 0 ? 0 : n0 + TL::BN, kend = PART ? s : min(w, m0 + TL::BM);
    const int mn = min(TL::BM, g.M - m0), nn = min(TL::BN, g.N - n0);
    f64x4 acc[TL::FI][TL::FJ];
    zero(acc);
    if constexpr (DTL) {
        DtlLoader<MUL, 4, TL::BM, TL::NW> da;
        DtlLoader<1, 4, TL::BN, TL::NW> db;
        da.init(g.A, g.lda, m0, mn);
        db.init(g.B, g.ldb, n0, nn);
        mainloop_dtl<TL>(da, db, g.lda, g.ldb, kbeg, kend, A0, A1, B0, B1, acc);
    } else {
        TL::OperandLoader<MUL> la;
        TL::OperandLoader<1> lb;
        la.init(g.A, g.lda, m0, g.M);
        lb.init(g.B, g.ldb, n0, g.N);
        mainloop<TL>(la, lb, kbeg, kend, mn == TL::BM && nn == TL::BN, LdsPair{A0, A1}, LdsPair{B0, B1}, acc);
    }
    if constexpr (PART == 2) join_triangle(g, m0, mn, n0, A0, A1, B0, B1, acc);
    const int ns = DTL ? dtl_shift<1, 4>(nn) : -2;              // (rows: contiguous along k, or an even count)
    bool finite = true;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        finite = finite && fabs(acc[0][0][r]) <= DBL_MAX;
        if (PART == 3 && !(fabs(acc[0][0][r]) <= DBL_MAX)) acc[0][0][r] = 0.0;
    }
    if (PART < 2 && !__all(finite)) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        join_one_by_one<MUL>(g, m0 + block_row<TL>(wave % TL::WM, 0) + (lane & 15), n0,
                              block_col<TL>(wave / TL::WM, 0) + (lane >> 4), ns, acc[0][0]);
    }
    epilogue<TL>(g, m0, n0, acc, -2, ns);
}

// The strictly lower 64 x 64 blocks of X := 0, one workgroup per column.
__global__ __launch_bounds__(256) void trtri_zero_kernel(double *X, int64_t ldx, int n)
{
    const int j = blockIdx.x;
    for (int i = (j / kPb + 1) * kPb + (int) threadIdx.x; i < n; i += 256) X[(int64_t) j * ldx + i] = 0.0;
}

// X := B R^{-1} for B of m x n and T = R^{-1}, zero below the diagonal: the
// 128 x 128 tile at column n0 takes k in [0, min(n, n0 + 128)), and a wave
// leaves out the stages behind its own last column.  All column blocks in one
// launch: each by itself leaves part of the chip idle (30011 x 1999: 235 tiles
// each) and reads B again.  Workgroup b runs on XCD b % 8, which works through
// an eighth of the tile rows in groups of 32, the columns with the longest k
// first, so that a group's rows of B stay in that XCD's L2 for all columns.
__global__ __launch_bounds__(512, 4) void trmm_kernel(ca3::gemm::GemmArgs g)
{
    using namespace ca3::gemm;
    using TL = Tile128w8;
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];
    const int tiles_m = (g.M + TL::BM - 1) / TL::BM, tiles_n = (g.N + TL::BN - 1) / TL::BN;
    const int per_xcd = (tiles_m + 7) / 8, first = (int) (blockIdx.x & 7) * per_xcd;
    const int rows = min(per_xcd, tiles_m - first), e = (int) (blockIdx.x >> 3);
    if (e >= rows * tiles_n) return;
    const int grp = e / (32 * tiles_n), r = e - grp * 32 * tiles_n, gsz = min(rows - 32 * grp, 32);
    const int m0 = __builtin_amdgcn_readfirstlane((first + 32 * grp + r % gsz) * TL::BM);
    const int n0 = __builtin_amdgcn_readfirstlane((tiles_n - 1 - r / gsz) * TL::BN);
    const int kend = min(g.K, n0 + TL::BN), mn = min(TL::BM, g.M - m0);
    const int wn = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6) / TL::WM);
    f64x4 acc[TL::FI][TL::FJ];
    zero(acc);
    DtlLoader<1, 4, TL::BM, TL::NW> da;
    DtlLoader<0, 4, TL::BN, TL::NW> db;
    da.init(g.A, g.lda, m0, mn);
    db.init(g.B, g.ldb, n0, min(TL::BN, g.N - n0));
    mainloop_dtl<TL>(da, db, g.lda, g.ldb, 0, kend, A0, A1, B0, B1, acc, n0 + (wn + 1) * (TL::BN / TL::WN));
    epilogue<TL>(g, m0, n0, acc, dtl_shift<1, 4>(mn));
}

// The scratch of the solves, one buffer per device (R_jj and info of a
// factorization, R^{-1} of a right solve).  A call holds the device's mutex
// from before scratch() until its last launch is enqueued (hip_dpotrf until
// info is read back), so that calls of several threads, which share the
// device's stream, neither mix their launches nor free the buffer under each
// other.
struct Ws {
    void *p = nullptr;
    size_t bytes = 0;
    std::mutex mu;
};
Ws g_ws[16];

Ws &device_ws()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    return g_ws[dev & 15];
}

// At least `bytes` of w, whose mutex the caller holds.
void *scratch(Ws &w, size_t bytes, int *rc)
{
    *rc = 0;
    if (w.bytes < bytes) {
        if (w.p) {
            (void) hipStreamSynchronize(ca3::stream());
            (void) hipFree(w.p);
            w.p = nullptr;
            w.bytes = 0;
        }
        hipError_t e = hipMalloc(&w.p, bytes);
        if (e != hipSuccess) { *rc = ca3::fail(e, "solve workspace"); return nullptr; }
        w.bytes = bytes;
    }
    return w.p;
}

}  // namespace

extern "C" {

int hip_dpotrf(const char uplo, const int n, double *A, const int ldA)
{
    if (uplo != 'U' && uplo != 'u')
        return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dpotrf: only uplo = 'U' is implemented");
    if (n < 0 || ldA < std::max(1, n) || (n > 0 && !A)) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dpotrf: bad arguments");
    if (n > kMaxN) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dpotrf: n > %d", kMaxN);
    if (n == 0) return 0;
    int rc = 0;
    Ws &ws = device_ws();
    std::lock_guard<std::mutex> lk(ws.mu);
    int *dinfo = (int *) scratch(ws, 256 + sizeof(double) * kPb * kPb, &rc);
    if (rc) return rc;
    double *Rjj = (double *) ((char *) dinfo + 256);
    const bool dtl = ca3::gemm::dtl_ld_ok(ldA) && ca3::gemm::load_mode() == ca3::gemm::kLoads16;
    for (int j0 = 0; j0 < n && !rc; j0 += kPb) {
        const int jb = std::min(kPb, n - j0), nr = n - j0 - jb;
        potrf_row_kernel<<<std::max(1, (nr + kPb - 1) / kPb), 256, 0, ca3::stream()>>>(A, ldA, j0, jb, n, Rjj, dinfo);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) { rc = ca3::fail(e, "potrf_row_kernel"); break; }
        if (nr == 0) break;
        // trailing upper triangle: A(r, r) -= X^T X, X = A(j0:j0+64, r)
        double *X = A + (int64_t) (j0 + jb) * ldA + j0, *D = A + (int64_t) j0 * ldA + j0;
        const int nt = (nr + kPb - 1) / kPb;
        if (dtl) potrf_update_kernel<true><<<nt * (nt + 1) / 2, 512, 0, ca3::stream()>>>(X, X + jb, ldA, nr, Rjj, D, j0, dinfo);
        else potrf_update_kernel<false><<<nt * (nt + 1) / 2, 512, 0, ca3::stream()>>>(X, X + jb, ldA, nr, Rjj, D, j0, dinfo);
        e = hipGetLastError();
        if (e != hipSuccess) rc = ca3::fail(e, "potrf_update_kernel");
    }
    if (rc) return rc;
    int info = 0;
    CA3_CHECK(hipMemcpyAsync(&info, dinfo, sizeof(int), hipMemcpyDeviceToHost, ca3::stream()));
    CA3_CHECK(hipStreamSynchronize(ca3::stream()));
    return info;
}

int hip_dtrtri_upper(const int n, const double *R, const int ldR, double *X, const int ldX)
{
    if (n < 0 || (n > 0 && (!R || !X)) || ldR < std::max(1, n) || ldX < std::max(1, n))
        return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dtrtri: bad arguments");
    if (n > kMaxN) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dtrtri: n > %d", kMaxN);
    if (n == 0) return HIP_PROXY_OK;
    const bool dtl = ca3::gemm::dtl_ld_ok(ldR) && ca3::gemm::dtl_ld_ok(ldX) &&
                     ca3::gemm::load_mode() == ca3::gemm::kLoads16;
    hipStream_t st = ca3::stream();
    if (n <= kSweepN) {
        trtri_sweep_kernel<<<n, 256, 0, st>>>(R, ldR, X, ldX, n);
        return ca3::finish();
    }
    trtri_diag_kernel<<<(n + kPb - 1) / kPb, 64 * kPb / 8, 0, st>>>(R, ldR, X, ldX, n);
    for (int s = kPb; s < n; s *= 2) {
        // blocks of s joined in pairs; the last block may be alone or short
        const int pairs = (n - s + 2 * s - 1) / (2 * s), tiles = s / 32;
        const dim3 grid((unsigned) (tiles * tiles), (unsigned) pairs);
        auto join = [&](auto PART) {
            constexpr int P = decltype(PART)::value;
            if (dtl) trtri_join_kernel<P, true><<<grid, 256, 0, st>>>(R, ldR, X, ldX, n, s);
            else trtri_join_kernel<P, false><<<grid, 256, 0, st>>>(R, ldR, X, ldX, n, s);
        };
        join(std::integral_constant<int, 0>{});
        join(std::integral_constant<int, 1>{});
        join(std::integral_constant<int, 2>{});
        join(std::integral_constant<int, 3>{});
    }
    trtri_zero_kernel<<<n, 256, 0, st>>>(X, ldX, n);
    return ca3::finish();
}

int hip_dtrsm(hip_proxy_enum_t side, hip_proxy_enum_t uplo, hip_proxy_enum_t trans, hip_proxy_enum_t diag,
              const int m, const int n, const double alpha, const double *A, const int ldA, double *B,
              const int ldB)
{
    if (side != HipRight || uplo != HipUpper || trans != HipNoTrans || diag != HipNonUnit)
        return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dtrsm: only side=Right, uplo=Upper, trans=NoTrans, "
                                                   "diag=NonUnit is implemented");
    if (m < 0 || n < 0 || ldA < std::max(1, n) || ldB < std::max(1, m))
        return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dtrsm: bad arguments");
    if (m == 0 || n == 0) return HIP_PROXY_OK;
    if (n > kMaxN) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dtrsm: n > %d", kMaxN);
    const int nb = 128;
    const int wcols = std::min(n, nb);
    int rc = 0;
    const size_t rinv_bytes = sizeof(double) * (size_t) n * n;
    Ws &ws = device_ws();
    std::unique_lock<std::mutex> lk(ws.mu);
    char *buf = (char *) scratch(ws, rinv_bytes + sizeof(double) * (size_t) m * wcols + 256, &rc);
    if (rc) return rc;
    double *Rinv = (double *) buf;
    double *T = (double *) (buf + ((rinv_bytes + 255) / 256) * 256);
    ca3::Unsynced unsynced;
    rc = hip_dtrtri_upper(n, A, ldA, Rinv, n);
    // column block jb of X = B R^{-1} needs rows 0 .. end(jb) of R^{-1}
    for (int j0 = ((n - 1) / nb) * nb; !rc && j0 >= 0; j0 -= nb) {
        const int w = std::min(nb, n - j0), kk = j0 + w;
        rc = hip_dgemm(HipNoTrans, HipNoTrans, m, w, kk, alpha, B, ldB, Rinv + (size_t) j0 * n, n, 0.0, T, m);
        if (!rc) rc = hip_copy_matrix_block(8, w, m, T, m, B + (size_t) j0 * ldB, ldB);
    }
    unsynced.end();
    lk.unlock();
    if (rc) return rc;
    return ca3::finish();
}

}  // extern "C"

int ca3::trsm_right_upper_out(int m, int n, const double *R, int ldR, const double *B, int ldB, double *X, int ldX)
{
    if (m < 0 || n < 0 || ldR < std::max(1, n) || ldB < std::max(1, m) || ldX < std::max(1, m))
        return ca3::fail_msg(HIP_PROXY_ERR_ARG, "trsm_right_upper_out: bad arguments");
    if (m == 0 || n == 0) return HIP_PROXY_OK;
    if (n > kMaxN) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "trsm_right_upper_out: n > %d", kMaxN);
    int rc = 0;
    Ws &ws = device_ws();
    std::unique_lock<std::mutex> lk(ws.mu);
    double *Rinv = (double *) scratch(ws, sizeof(double) * (size_t) n * n, &rc);
    if (rc) return rc;
    ca3::Unsynced unsynced;
    rc = hip_dtrtri_upper(n, R, ldR, Rinv, n);
    const int64_t tiles = (int64_t) ((m + 127) / 128 + 7) / 8 * 8 * ((n + 127) / 128);
    if (!rc && m > 1 && n >= gemm::kBK && tiles <= INT_MAX && gemm::dtl_ld_ok(ldB) && ((uintptr_t) B % 8) == 0 &&
        gemm::load_mode() == gemm::kLoads16) {
        gemm::GemmArgs g;
        memset(&g, 0, sizeof(g));
        g.M = m; g.N = n; g.K = n;
        g.alpha = 1.0;
        g.A = B; g.lda = ldB; g.B = Rinv; g.ldb = n; g.C = X; g.ldc = ldX;
        trmm_kernel<<<(unsigned) tiles, 512, 0, ca3::stream()>>>(g);
        hipError_t e = hipGetLastError();
        unsynced.end();
        lk.unlock();
        if (e != hipSuccess) return ca3::fail(e, "trmm_kernel");
        return ca3::finish();
    }
    // column block jb of X = B R^{-1} needs rows 0 .. end(jb) of R^{-1}
    const int nb = 128;
    for (int j0 = 0; !rc && j0 < n; j0 += nb) {
        const int w = std::min(nb, n - j0), kk = j0 + w;
        rc = hip_dgemm(HipNoTrans, HipNoTrans, m, w, kk, 1.0, B, ldB, Rinv + (size_t) j0 * n, n, 0.0,
                       X + (size_t) j0 * ldX, ldX);
    }
    unsynced.end();
    lk.unlock();
    if (rc) return rc;
    return ca3::finish();
}
