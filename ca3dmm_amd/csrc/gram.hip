// Upper-triangle Gram product C = A^T A on FP64 MFMA (gfx950).
//
// The reference computes B^T B in full through the general Cannon DGEMM
// (src/ca3dmm.c:1172-1265) and the CholeskyQR driver uses it for
// S = B^T B (examples/example_CholeskyQR.c:109-117, :160-168).  Here only
// tiles (i <= j) of the upper triangle are computed, and in the tiles on the
// diagonal only the 16 x 16 blocks (i <= j): n(n+1)k flops instead of 2n^2 k.
// Tall-skinny inputs (k >> n, e.g. 2e6 x 512) give few tiles, so k is split
// across workgroups; each split writes its partial tile and a second kernel
// adds the partials in split order (deterministic) and writes the upper
// triangle, optionally mirrored into the lower one.  Mirroring copies values,
// so the result is exactly symmetric.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "ca3dmm_ext.h"
#include "dgemm_tile.h"
#include "grouped.h"
#include "hip_common.h"

// Partial tiles of hip_dsyrk_gram_noalloc: a fixed array in device memory,
// 512 tiles of 128 x 128 doubles (64 MiB) per device, held until the process
// ends.  Host code must use the address hipGetSymbolAddress returns for the
// current device, never this name.
static __device__ __align__(256) double scratch[(size_t) 512 * 128 * 128];

namespace {

using namespace ca3::gemm;

// Tile pairs (ti < tj) take k in ranges of step1, s1 of them, the tiles on the
// diagonal ranges of step2, s2 of them.  Partials in P: pair p and range ks at
// (ks noff + p), diagonal tile t at (noff s1 + ks ntile + t), in tiles.
// A workgroup sums its range in chains of at most chain1 (chain2) k and adds
// them up in its partial tile.
struct GramArgs {
    int n, k, ntile, noff, s1, step1, s2, step2, chain1, chain2;
    const double *A;
    int64_t lda;
    double *P;
};

// pair index -> (ti, tj), ti < tj, row-major over the strict upper triangle
__device__ __forceinline__ void pair_of(int p, int nt, int *ti, int *tj)
{
    int i = 0, rem = p;
    while (rem >= nt - 1 - i) { rem -= nt - 1 - i; ++i; }
    *ti = i;
    *tj = i + 1 + rem;
}

// A diagonal tile in direct-to-LDS stages: one panel is both operands, and the
// 16 x 16 blocks on and above the diagonal (36 of 64 in a 128-wide tile) are
// dealt to the 8 waves, which leaves the SIMDs the same number (9 each).  The
// products of an entry and their order are those of mainloop_dtl.
template <class TL>
struct DiagTile {
    static constexpr int NB = TL::BM / 16, BLOCKS = NB * (NB + 1) / 2;
    static constexpr int MOST = (BLOCKS + TL::NW - 1) / TL::NW, LEAST = BLOCKS / TL::NW;
    int bi[MOST], bj[MOST], count;
    f64x4 acc[MOST];

    __device__ __forceinline__ void init()
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        count = (BLOCKS - wave + TL::NW - 1) / TL::NW;
#pragma unroll
        for (int q = 0; q < MOST; ++q) {
            const int p = min(wave + q * TL::NW, BLOCKS - 1);
            int j = 0;
            while ((j + 1) * (j + 2) / 2 <= p) ++j;
            bi[q] = p - j * (j + 1) / 2;
            bj[q] = j;
            acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
    }

    template <bool TAIL = false>
    __device__ __forceinline__ void mfma(const double *S, int lo = 0)
    {
        const int lane = threadIdx.x & 63, li = lane & 15;
#pragma unroll
        for (int ks = 0; ks < kBK / 4; ++ks) {
            const int kk = ks * 4 + (lane >> 4);
            const double *L = S + dtl_index<0, TL::BM>(kk, li);
#pragma unroll
            for (int q = 0; q < MOST; ++q) {
                if (q >= LEAST && q >= count) continue;
                double a = L[bi[q] * 256], b = L[bj[q] * 256];
                if (TAIL) {
                    a = kk >= lo ? a : 0.0;
                    b = kk >= lo ? b : 0.0;
                }
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, acc[q], 0, 0, 0);
            }
        }
    }

    template <class LD>
    __device__ __forceinline__ void run(const LD &ld, int kbeg, int kend, double *S0, double *S1)
    {
        const int nfull = (kend - kbeg) / kBK, rem = (kend - kbeg) % kBK, ns = nfull + (rem > 0);
        auto issue = [&](int z, double *S) __attribute__((always_inline)) {
            ld.issue(min(kbeg + z * kBK, kend - kBK), S);
        };
        if (ns > 0) issue(0, S0);
        for (int z = 0; z < nfull; z += 2) {
            dtl_publish();
            if (z + 1 < ns) issue(z + 1, S1);
            mfma(S0);
            if (z + 1 >= nfull) break;
            dtl_publish();
            if (z + 2 < ns) issue(z + 2, S0);
            mfma(S1);
        }
        if (rem > 0) {
            dtl_publish();
            mfma<true>(nfull & 1 ? S1 : S0, kBK - rem);
        }
        __syncthreads();
    }

    __device__ __forceinline__ void store(double *out, bool add) const
    {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));               // no address is computed before the main loop
#pragma unroll
        for (int q = 0; q < MOST; ++q) {
            if (q >= count) continue;
            double *o = out + (bj[q] * 16 + (lane >> 4)) * TL::BM + bi[q] * 16 + (lane & 15);
            double x[4] = {0.0, 0.0, 0.0, 0.0};      // (acc, from +0 on, is never -0)
            if (add) {
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] = o[4 * r * TL::BM];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) o[4 * r * TL::BM] = ca3::add_rn(x[r], acc[q][r]);
        }
    }
};

// One partial tile per workgroup.  DTL: 16-byte direct-to-LDS stages in 8-wave
// workgroups; otherwise register-staged (both panels are k-contiguous, where
// 4-byte direct-to-LDS loads lose to register staging), the same products in
// the same order.
template <class TL, bool DTL>
__global__ __launch_bounds__(TL::THREADS, DTL ? 4 : 2) void gram_partial_kernel(GramArgs g)
{
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];
    // Workgroups are dealt round-robin over the 8 XCDs; the logical ids are
    // made XCD-contiguous (the grid is a multiple of 8) so that the pairs of
    // one k-range, which share their panels, run behind the same L2.
    const int nb = gridDim.x, off = g.noff * g.s1;
    const int bid = (blockIdx.x & 7) * (nb >> 3) + (blockIdx.x >> 3);
    if (bid >= off + g.ntile * g.s2) return;
    const bool diag = bid >= off;
    int ti, tj, ks;
    if (diag) {
        ks = (bid - off) / g.ntile;
        ti = tj = bid - off - ks * g.ntile;
    } else {
        ks = bid / g.noff;
        pair_of(bid - ks * g.noff, g.ntile, &ti, &tj);
    }
    const int step = diag ? g.step2 : g.step1, chain = diag ? g.chain2 : g.chain1;
    const int kbeg = __builtin_amdgcn_readfirstlane(ks * step);
    const int kend = __builtin_amdgcn_readfirstlane(g.k - kbeg < step ? g.k : kbeg + step);
    const int m0 = __builtin_amdgcn_readfirstlane(ti * TL::BM), n0 = __builtin_amdgcn_readfirstlane(tj * TL::BN);
    // sum(first k, end, whether to add, m0, n0); the tile's origin is opaque in
    // each chain, so that no address is held in registers across the main loop
    auto chains = [&](auto sum) __attribute__((always_inline)) {
        int k0 = kbeg;
        do {
            int sm0 = m0, sn0 = n0;
            asm volatile("" : "+s"(sm0), "+s"(sn0));
            const int k1 = __builtin_amdgcn_readfirstlane(kend - k0 < chain ? kend : k0 + chain);
            sum(k0, k1, k0 > kbeg, sm0, sn0);
            k0 = k1;
        } while (k0 < kend);
    };
    double *out = g.P + (int64_t) bid * (TL::BM * TL::BN);
    // op(A) = A^T and op(B) = A: both panels are contiguous along k.  The
    // splits start at multiples of 16, so the panels keep A's alignment; edge
    // tiles load copies of their last line in place of the missing ones.
    if constexpr (DTL) {
        DtlLoader<0, 4, TL::BM, TL::NW> da;
        if (diag) {
            chains([&](int k0, int k1, bool add, int m0, int) __attribute__((always_inline)) {
                da.init(g.A, g.lda, m0, min(TL::BM, g.n - m0));
                DiagTile<TL> tile;
                tile.init();
                tile.run(da, k0, k1, A0, A1);
                tile.store(out, add);
            });
            return;
        }
        DtlLoader<0, 4, TL::BN, TL::NW> db;
        chains([&](int k0, int k1, bool add, int m0, int n0) __attribute__((always_inline)) {
            da.init(g.A, g.lda, m0, min(TL::BM, g.n - m0));
            db.init(g.A, g.lda, n0, min(TL::BN, g.n - n0));
            f64x4 acc[TL::FI][TL::FJ];
            zero(acc);
            mainloop_dtl<TL>(da, db, g.lda, g.lda, k0, k1, A0, A1, B0, B1, acc);
            store_tile<TL>(out, acc, add);
        });
    } else {
        typename TL::template OperandLoader<0> la, lb;
        chains([&](int k0, int k1, bool add, int m0, int n0) __attribute__((always_inline)) {
            la.init(g.A, g.lda, m0, g.n);
            lb.init(g.A, g.lda, n0, g.n);
            f64x4 acc[TL::FI][TL::FJ];
            zero(acc);
            mainloop<TL>(la, lb, k0, k1, m0 + TL::BM <= g.n && n0 + TL::BN <= g.n, LdsPair{A0, A1}, LdsPair{B0, B1},
                         acc);
            store_tile<TL>(out, acc, add);
        });
    }
}

template <int BM>
__global__ __launch_bounds__(256) void gram_reduce_kernel(GramArgs g, double alpha, double beta, double *C,
                                                          int64_t ldc, int mirror)
{
    const int p = blockIdx.y;
    const bool diag = p >= g.noff;
    int ti = p - g.noff, tj = ti;
    if (!diag) pair_of(p, g.ntile, &ti, &tj);
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int row = e % BM, col = e / BM, gi = ti * BM + row, gj = tj * BM + col;
    if (gi >= g.n || gj >= g.n || gi > gj) return;
    const int ksplit = diag ? g.s2 : g.s1;
    const int64_t step = (int64_t) (diag ? g.ntile : g.noff) * (BM * BM);
    const double *q = g.P + (diag ? (int64_t) g.noff * g.s1 + ti : (int64_t) p) * (BM * BM) + e;
    // sixteen ranges at a time, their loads in flight together: up to a thousand
    // of them in one chain would cost the accuracy that short ranges give
    constexpr int U = 16;
    double s = 0.0;
    int k0 = 0;
    for (; k0 + U <= ksplit; k0 += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = q[(k0 + u) * step];
#pragma unroll
        for (int u = 1; u < U; ++u) v[0] = ca3::add_rn(v[0], v[u]);
        s = ca3::add_rn(s, v[0]);
    }
    if (k0 < ksplit) {
        double t = q[k0 * step];
#pragma unroll 8
        for (int ks = k0 + 1; ks < ksplit; ++ks) t = ca3::add_rn(t, q[ks * step]);
        s = ca3::add_rn(s, t);
    }
    double *c = C + (int64_t) gj * ldc + gi;
    double v = ca3::mul_rn(alpha, s);
    if (beta != 0.0) v = ca3::add_rn(v, ca3::mul_rn(beta, *c));
    *c = v;
    if (mirror && gi != gj) C[(int64_t) gi * ldc + gj] = v;
}

struct Ws {
    void *p = nullptr;
    size_t bytes = 0;
};
Ws g_gram_ws[16];
std::mutex g_gram_mu;

constexpr int kScratchTiles = 512;   // partial 128 x 128 tiles the allocation-free entry can hold
double *g_scratch_ptr[16];          // device address of `scratch` per device (0: not looked up yet)

// Looks it up, once per device, with that device current and g_gram_mu held:
// the host-side name `scratch` is not a device address.  The first lookup
// loads this file's code and the array with it.
hipError_t find_scratch(int dev)
{
    void *q = nullptr;
    const hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
    if (e == hipSuccess) g_scratch_ptr[dev] = (double *) q;
    return e;
}

// Tile width and k ranges for n x n from k, by the cost of a single product's
// rule: a CU that holds w workgroups takes a + b w us per 16-deep stage, a
// diagonal tile f of that b; the second launch and the partials cost what the
// k split of a product does.  Diagonal tiles get longer ranges, so that all
// workgroups end together.  Splits are at least four stages long and the
// partials within the fixed scratch, unless the tiles alone exceed it (one
// range each, then, as 128-wide tiles).
struct Plan {
    GramArgs g;
    int bm, wgs;
};

Plan plan(int n, int k)
{
    static const struct { int bm; double a, b, f; int most; } tiles[] = {
        {128, 0.15, 1.80, 36.0 / 64, 2}, {64, 0.20, 0.47, 12.0 / 16, 4}};
    const int cus = ca3::cu_count(), stages = (k + kBK - 1) / kBK, longest = std::max(1, stages / 4);
    Plan best;
    memset(&best, 0, sizeof(best));
    double cost = 0.0;
    for (const auto &t : tiles) {
        const int ntile = (n + t.bm - 1) / t.bm;
        const int64_t noff = (int64_t) ntile * (ntile - 1) / 2;
        const int64_t cap = (int64_t) kScratchTiles * (128 / t.bm) * (128 / t.bm);
        auto consider = [&](int64_t s1, int64_t s2) {
            const int l1 = (int) ((stages + s1 - 1) / s1), l2 = (int) ((stages + s2 - 1) / s2);
            s1 = l1 ? (stages + l1 - 1) / l1 : 1;
            s2 = l2 ? (stages + l2 - 1) / l2 : 1;
            const int64_t wgs = noff * s1 + ntile * s2;
            const double w = (double) ((wgs + cus - 1) / cus);
            const double us = std::max(noff ? l1 * (t.a + t.b * w) : 0.0, l2 * (t.a + t.b * t.f * w)) +
                              (double) (2 * wgs) * t.bm * t.bm * 8.0 / 4e6;
            if (best.bm && us >= (best.bm == t.bm ? 1.0 : 0.92) * cost) return;
            cost = us;
            best.bm = t.bm;
            best.wgs = (int) wgs;
            best.g.n = n; best.g.k = k; best.g.ntile = ntile; best.g.noff = (int) noff;
            best.g.s1 = (int) s1; best.g.step1 = std::max(1, l1) * kBK;
            best.g.s2 = (int) s2; best.g.step2 = std::max(1, l2) * kBK;
        };
        if (t.bm == 128 || noff + ntile <= cap) consider(1, 1);
        for (int r = 1; r <= t.most; r *= 2) {
            const int64_t slots = std::min((int64_t) r * cus, cap);
            // the split that fills the slots with equally long ranges, and those around it
            const int64_t even = (int64_t) ((double) slots / ((double) noff + t.f * ntile));
            for (int64_t s1 = std::max<int64_t>(1, std::min<int64_t>(even, longest) - 1);
                 s1 <= std::min<int64_t>(even + 1, longest) && noff * s1 + ntile <= slots; ++s1) {
                const int64_t s2 = std::min((slots - noff * s1) / ntile, (int64_t) longest);
                consider(s1, s2);
                consider(s1, std::min(s2, std::max<int64_t>(1, (int64_t) ((double) s1 * t.f + 0.999))));
            }
        }
    }
    // Chains no longer than equal ranges of all 128-wide tiles in one round of
    // the chip (of about 1024 k or more): an entry on the diagonal is a sum of
    // squares, whose error grows with the root of the chain (1000 from 100000,
    // rms of the relative error: in one chain per range 1.0e-15, so 4.2e-16).
    const int64_t nt = (n + 127) / 128, pairs = nt * (nt + 1) / 2;
    const int equal = (int) std::max<int64_t>(1, std::min<int64_t>(2 * cus / pairs, ((int64_t) k + 1023) / 1024));
    const int most = (stages + equal - 1) / equal;
    auto chain = [&](int step) {
        const int len = step / kBK, parts = std::max(1, (len + most - 1) / std::max(1, most));
        return std::max(1, (len + parts - 1) / parts) * kBK;
    };
    best.g.chain1 = chain(best.g.step1);
    best.g.chain2 = chain(best.g.step2);
    return best;
}

int check_args(int n, int k, const double *A, int ldA, const double *C, int ldC)
{
    if (n < 0 || k < 0) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "gram: negative size");
    if (n > 0 && (!C || ldC < n)) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "gram: bad C / ldC");
    if (n > 0 && k > 0 && (!A || ldA < std::max(1, k))) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "gram: bad A / ldA");
    return 0;
}

template <class TL, class TR>
void launch_tile(const Plan &p, bool dtl, double alpha, double beta, double *C, int ldC, int mirror)
{
    hipStream_t st = ca3::stream();
    const int grid = (p.wgs + 7) / 8 * 8;
    if (dtl) gram_partial_kernel<TL, true><<<grid, TL::THREADS, 0, st>>>(p.g);
    else gram_partial_kernel<TR, false><<<grid, TR::THREADS, 0, st>>>(p.g);
    gram_reduce_kernel<TL::BM><<<dim3(TL::BM * TL::BM / 256, p.g.noff + p.g.ntile), 256, 0, st>>>(p.g, alpha, beta, C,
                                                                                               ldC, mirror ? 1 : 0);
}

// Both launches; the caller holds g_gram_mu, so that calls of several threads,
// which share the device's stream and the partials, do not mix theirs.
int launch(const Plan &p, double alpha, double beta, double *C, int ldC, int mirror)
{
    // 16-byte direct-to-LDS loads from any 8-byte aligned A (as the DGEMM;
    // CA3DMM_DGEMM_LOADS=aligned keeps them to 16-byte aligned A with even
    // lda, "reg" and "dword" stage through registers)
    const GramArgs &g = p.g;
    const LoadMode mode = load_mode();
    const bool aligned16 = ((uintptr_t) g.A % 16) == 0 && (g.lda % 2) == 0;
    const bool dtl = g.k >= kBK && dtl_ld_ok(g.lda) && ((uintptr_t) g.A % 8) == 0 &&
                     (mode == kLoads16 || (mode == kLoadsAligned && aligned16));
    if (p.bm == 128) launch_tile<Tile128w8, Tile128>(p, dtl, alpha, beta, C, ldC, mirror);
    else launch_tile<Tile64, Tile64>(p, dtl, alpha, beta, C, ldC, mirror);
    hipError_t e = hipGetLastError();
    return e != hipSuccess ? ca3::fail(e, "gram kernels") : HIP_PROXY_OK;
}

}  // namespace

bool ca3::grouped::gram_ready()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) {
        (void) hipGetLastError();
        return false;
    }
    std::lock_guard<std::mutex> lk(g_gram_mu);
    if (!g_scratch_ptr[dev] && find_scratch(dev) != hipSuccess) (void) hipGetLastError();
    return g_scratch_ptr[dev] != nullptr;
}

extern "C" {

int hip_dsyrk_gram(const int n, const int k, const double alpha, const double *A, const int ldA,
                   const double beta, double *C, const int ldC, int mirror)
{
    int rc = check_args(n, k, A, ldA, C, ldC);
    if (rc || n == 0) return rc;
    Plan p = plan(n, k);
    const size_t bytes = sizeof(double) * (size_t) p.wgs * p.bm * p.bm;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    Ws &w = g_gram_ws[dev & 15];
    {
        std::lock_guard<std::mutex> lk(g_gram_mu);
        if (w.bytes < bytes) {
            if (w.p) {
                (void) hipStreamSynchronize(ca3::stream());
                (void) hipFree(w.p);
                w.p = nullptr;
                w.bytes = 0;
            }
            CA3_CHECK(hipMalloc(&w.p, bytes));
            w.bytes = bytes;
        }
        p.g.A = A; p.g.lda = ldA; p.g.P = (double *) w.p;
        rc = launch(p, alpha, beta, C, ldC, mirror);
    }
    return rc ? rc : ca3::finish();
}

int hip_dsyrk_gram_noalloc(const int n, const int k, const double alpha, const double *A, const int ldA,
                           const double beta, double *C, const int ldC, int mirror)
{
    int rc = check_args(n, k, A, ldA, C, ldC);
    if (rc || n == 0) return rc;
    static_assert(sizeof(scratch) == sizeof(double) * (size_t) kScratchTiles * kBM * kBN, "scratch size");
    const int64_t nt = ((int64_t) n + kBM - 1) / kBM;
    if (nt * (nt + 1) / 2 > kScratchTiles)
        return ca3::fail_msg(HIP_PROXY_ERR_ARG,
                             "gram_noalloc: n = %d, k = %d needs %lld partial 128 x 128 tiles; the fixed scratch "
                             "holds %d (n <= 3968)", n, k, (long long) (nt * (nt + 1) / 2), kScratchTiles);
    Plan p = plan(n, k);
    int dev = 0;
    CA3_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 16) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "gram_noalloc: device %d >= 16", dev);
    {
        std::lock_guard<std::mutex> lk(g_gram_mu);
        if (!g_scratch_ptr[dev]) {
            const hipError_t e = find_scratch(dev);
            if (e != hipSuccess) return ca3::fail(e, "hipGetSymbolAddress");
        }
        p.g.A = A; p.g.lda = ldA; p.g.P = g_scratch_ptr[dev];
        rc = launch(p, alpha, beta, C, ldC, mirror);
    }
    return rc ? rc : ca3::finish();
}

}  // extern "C"
