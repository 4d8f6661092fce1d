// FP64 MFMA DGEMM for gfx950 -- the local DGEMM of CA3DMM's Cannon step.
//
// Replaces cublasDgemm behind cuda_cublas_dgemm (src/cuda_proxy.cu:211-230),
// called at src/cannon.c:418,586,616,665 and src/dev_type.c:212.
//
// Column-major C := alpha*op(A)*op(B) + beta*C, optionally followed by the
// k-layer partial-C fold of the reduce-scatter (src/ca3dmm.c:1311-1324):
// C := ((P0 + P1) + ...) + (alpha*op(A)*op(B) + beta*C).
//
// Design (MI355X / CDNA4):
//  * v_mfma_f64_16x16x4_f64.  A workgroup of 8 wave64s owns a 128x128 tile
//    of C, each wave 64x32 = 4x2 MFMA blocks; smaller products take 64x64 or
//    32x32 tiles (pick_cut).
//  * K advances in stages of 16, loaded direct-to-LDS into a double buffer:
//    the next stage's loads are issued before the current stage's MFMAs, one
//    barrier per stage.  Operands that cannot be loaded so are staged through
//    registers by 4-wave workgroups.
//  * Transposes are fused into the loads: an operand is either contiguous
//    along m/n (A as stored, B^T) or along k (A^T, B as stored); both map to
//    coalesced global reads.
//  * LDS addresses are XOR-swizzled, so that the MFMA operand reads (16
//    consecutive m or n, two k rows per half wave) hit distinct banks.
//  * Tiles are visited XCD-contiguously (workgroup b runs on XCD b % 8) and
//    in groups of 16 tile-rows, so the tiles resident on one XCD share A and
//    B panels in that XCD's L2.
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "ca3dmm_ext.h"
#include "dgemm_tile.h"
#include "grouped.h"
#include "hip_common.h"

namespace {

using namespace ca3::gemm;

// Workgroup -> tile origin, k range and k split.  Workgroup b runs on XCD
// b % 8; logical ids are made XCD-contiguous (gridDim.x is a multiple of 8),
// tiles fastest, so that the workgroups behind one L2 share the panels of
// neighbouring tiles and, split, of one k range.  False for the workgroups
// beyond the last tile.  The results are put in scalar registers: the
// quotients come from the vector ALU, and addresses or loop bounds that stay
// there cost the main loop vector registers and masked branches.
template <class TL>
__device__ __forceinline__ bool locate(const GemmArgs &g, int *m0, int *n0, int *kbeg, int *kend, int *split)
{
    const int tiles = ((g.M + TL::BM - 1) / TL::BM) * ((g.N + TL::BN - 1) / TL::BN);
    const int nb = gridDim.x;
    const int t = (blockIdx.x & 7) * (nb >> 3) + (blockIdx.x >> 3);
    if (t >= tiles * g.ksplit) return false;
    const int s = g.ksplit > 1 ? t / tiles : 0;
    int tm, tn;
    tile_coords<TL>(t - s * tiles, g.M, g.N, &tm, &tn, g.group);
    *m0 = __builtin_amdgcn_readfirstlane(tm * TL::BM);
    *n0 = __builtin_amdgcn_readfirstlane(tn * TL::BN);
    *split = __builtin_amdgcn_readfirstlane(s);
    *kbeg = *split * g.kstep;
    *kend = g.K - *kbeg < g.kstep ? g.K : *kbeg + g.kstep;      // (the sum may pass 2^31)
    return true;
}

// The epilogue of one split: the product itself, or with ksplit > 1 the bare
// sum over the split's k range.  (The arguments are passed one by one: a
// modified copy of g would live in scratch memory, and with it every loop
// bound read from it.)
template <class TL>
__device__ __forceinline__ void store_split(const GemmArgs &g, int split, int m0, int n0,
                                            const f64x4 (&acc)[TL::FI][TL::FJ], int ms = -2, int ns = -2)
{
    const bool whole = g.ksplit == 1;
    epilogue_to<TL>(g, whole ? g.C : g.part + (int64_t) split * g.M * g.N, whole ? g.ldc : (int64_t) g.M,
                    whole ? g.alpha : 1.0, whole ? g.beta : 0.0, whole ? g.nsrc : 0, m0, n0, acc, ms, ns);
}

template <int TA, int TB, class TL>
__global__ __launch_bounds__(TL::THREADS, TL::MIN_BLOCKS) void dgemm_kernel(GemmArgs g)
{
    __shared__ double As[2][kBK * TL::BM];
    __shared__ double Bs[2][kBK * TL::BN];

    int m0, n0, kbeg, kend, split;
    if (!locate<TL>(g, &m0, &n0, &kbeg, &kend, &split)) return;

    // A as stored (TA = 0) is contiguous along m; B as stored (TB = 0) is
    // contiguous along k, B^T along n.
    OperandLoader<!TA, TL::BM, TL::THREADS> la;
    OperandLoader<TB, TL::BN, TL::THREADS> lb;
    la.init(g.A, g.lda, m0, g.M);
    lb.init(g.B, g.ldb, n0, g.N);

    f64x4 acc[TL::FI][TL::FJ];
    zero(acc);
    mainloop<TL>(la, lb, kbeg, kend, m0 + TL::BM <= g.M && n0 + TL::BN <= g.N, As, Bs, acc);
    store_split<TL>(g, split, m0, n0, acc);
}

// The same product with direct-to-LDS stages; needs k >= 16, and 16-byte loads
// of an operand contiguous along m (n) more than one row (column).  WA / WB: 4 for 16-byte loads of an operand,
// 1 for 4-byte loads.  The same products in the same order as dgemm_kernel,
// whatever the tile.  WPE: waves per SIMD to leave registers for.
template <int TA, int TB, int WA, int WB, class TL, int WPE>
__global__ __launch_bounds__(TL::THREADS, WPE) void dgemm_dtl_kernel(GemmArgs g)
{
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];

    int m0, n0, kbeg, kend, split;
    if (!locate<TL>(g, &m0, &n0, &kbeg, &kend, &split)) return;
    const int mn = min(TL::BM, g.M - m0), nn = min(TL::BN, g.N - n0);

    f64x4 acc[TL::FI][TL::FJ];
    zero(acc);
    DtlLoader<!TA, WA, TL::BM, TL::NW> da;
    DtlLoader<TB, WB, TL::BN, TL::NW> db;
    da.init(g.A, g.lda, m0, mn);
    db.init(g.B, g.ldb, n0, nn);
    const int ms = dtl_shift<!TA, WA>(mn), ns = dtl_shift<TB, WB>(nn);
    if constexpr (TL::IL)
        mainloop_edge<TL>(da, db, g.lda, g.ldb, kbeg, kend, A0, A1, B0, B1, acc, blocks_inside<TL>(mn, nn, ms, ns));
    else
        mainloop_dtl<TL>(da, db, g.lda, g.ldb, kbeg, kend, A0, A1, B0, B1, acc);
    store_split<TL>(g, split, m0, n0, acc, ms, ns);
}

// C := fold(P) + (alpha * (sum of the splits' partial products) + beta * C).
// 64 entries per workgroup; wave w adds the splits [w ksplit / 4, (w + 1)
// ksplit / 4) in order and the four sums are added as (0 + 1) + (2 + 3): a
// fixed order, and enough loads in flight for a small C with many splits.
__global__ __launch_bounds__(256) void dgemm_reduce_kernel(GemmArgs g)
{
    __shared__ double part[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t size = (int64_t) g.M * g.N, e = (int64_t) blockIdx.x * 64 + lane;
    const int t0 = w * g.ksplit / 4, t1 = (w + 1) * g.ksplit / 4;
    double s = 0.0;
    if (e < size && t0 < t1) {
        const double *p = g.part + e;
        s = p[t0 * size];
#pragma unroll 4
        for (int t = t0 + 1; t < t1; ++t) s = ca3::add_rn(s, p[t * size]);
    }
    part[w][lane] = s;
    __syncthreads();
    if (w > 0 || e >= size) return;
    s = ca3::add_rn(ca3::add_rn(part[0][lane], part[1][lane]), ca3::add_rn(part[2][lane], part[3][lane]));
    const int64_t col = e / g.M, row = e - col * g.M;
    double *c = g.C + col * g.ldc + row;
    double v = ca3::mul_rn(g.alpha, s);
    if (g.beta != 0.0) v = ca3::add_rn(v, ca3::mul_rn(g.beta, *c));
    if (g.nsrc > 0) {
        double f = g.P[0][col * g.ldp[0] + row];
        for (int t = 1; t < g.nsrc; ++t) f = ca3::add_rn(f, g.P[t][col * g.ldp[t] + row]);
        v = ca3::add_rn(f, v);
    }
    *c = v;
}

// One problem of a batched launch (rank r's product C := sum over its
// Cannon rounds of A_s B_s, every operand as stored, NN): its tiles are
// linear tile indices [base, base + tiles_m tiles_n).
struct BatchProb {
    int M, N, nseg;
    int64_t base;
    double *C;
    int64_t ldc;
    const double *A[ca3::grouped::kMaxSeg];
    const double *B[ca3::grouped::kMaxSeg];
    int64_t lda[ca3::grouped::kMaxSeg], ldb[ca3::grouped::kMaxSeg];
    int k[ca3::grouped::kMaxSeg];
};

// Every problem's tiles in one launch, one workgroup per tile (gridDim.x =
// total tiles rounded up to a multiple of 8).  Linear tile indices are laid
// out XCD-contiguously over the whole batch, so each XCD works through its
// own problems' panels; inside a problem tiles are walked in groups of
// `group` tile-rows.  A tile's segments run in order.
// PER_SEG: each segment is its own product added by the epilogue (beta 0
// on the first, 1 after), the bits of one dgemm_dtl_kernel<0, 0> launch
// per segment.  Otherwise all segments accumulate in registers and the tile
// is stored once (C = the sum), the bits of the persistent grouped kernel.
// DTL: every segment of every problem can take the direct-to-LDS stages;
// otherwise all are register-staged (the two in one kernel spill).
template <bool PER_SEG, bool DTL, class TL, int WPE>
__global__ __launch_bounds__(TL::THREADS, WPE) void dgemm_batch_kernel(const BatchProb *__restrict__ probs, int nprob,
                                                                      int64_t total, int group)
{
    __shared__ __attribute__((aligned(1024))) double A0[kBK * TL::BM], A1[kBK * TL::BM];
    __shared__ __attribute__((aligned(1024))) double B0[kBK * TL::BN], B1[kBK * TL::BN];

    const int64_t nb = gridDim.x;
    int64_t t = blockIdx.x;
    t = (t & 7) * (nb >> 3) + (t >> 3);
    if (t >= total) return;
    int lo = 0, hi = nprob - 1;                // last problem with base <= t
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (probs[mid].base <= t) lo = mid;
        else hi = mid - 1;
    }
    const BatchProb &P = probs[lo];
    int tm, tn;
    tile_coords<TL>((int) (t - P.base), P.M, P.N, &tm, &tn, group);
    const int m0 = __builtin_amdgcn_readfirstlane(tm * TL::BM), n0 = __builtin_amdgcn_readfirstlane(tn * TL::BN);
    const int mn = min(TL::BM, P.M - m0), nn = min(TL::BN, P.N - n0);

    GemmArgs g;
    g.M = P.M; g.N = P.N;
    g.K = 0;                                  // not read by the epilogue
    g.alpha = 1.0;
    g.beta = 0.0;
    g.C = P.C; g.ldc = P.ldc;
    g.nsrc = 0;
    f64x4 acc[TL::FI][TL::FJ];
    for (int s = 0; s < P.nseg; ++s) {
        if (PER_SEG || s == 0) zero(acc);
        const int K = P.k[s];
        int sm0 = m0, sn0 = n0, smn = mn, snn = nn;
        asm volatile("" : "+s"(sm0), "+s"(sn0), "+s"(smn), "+s"(snn));
        if constexpr (DTL) {
            DtlLoader<1, 4, TL::BM, TL::NW> da;
            DtlLoader<0, 4, TL::BN, TL::NW> db;
            da.init(P.A[s], P.lda[s], sm0, smn);
            db.init(P.B[s], P.ldb[s], sn0, snn);
            mainloop_dtl<TL>(da, db, P.lda[s], P.ldb[s], 0, K, A0, A1, B0, B1, acc);
        } else {
            OperandLoader<1, TL::BM, TL::THREADS> la;
            OperandLoader<0, TL::BN, TL::THREADS> lb;
            la.init(P.A[s], P.lda[s], sm0, P.M);
            lb.init(P.B[s], P.ldb[s], sn0, P.N);
            mainloop<TL>(la, lb, 0, K, smn == TL::BM && snn == TL::BN, LdsPair{A0, A1}, LdsPair{B0, B1}, acc);
        }
        if (PER_SEG) {
            // the epilogue's addresses are the same on every segment: keep
            // the compiler from computing them once and holding them (in
            // vector registers) across the main loops
            double *C = P.C;
            int64_t ldc = P.ldc;
            int em0 = m0, en0 = n0;
            asm volatile("" : "+s"(C), "+s"(ldc), "+s"(em0), "+s"(en0));
            g.C = C;
            g.ldc = ldc;
            g.beta = s ? 1.0 : 0.0;
            epilogue<TL>(g, em0, en0, acc, DTL ? dtl_shift<1, 4>(mn) : -2);
        }
    }
    if (!PER_SEG) {
        if (P.nseg == 0) zero(acc);
        epilogue<TL>(g, m0, n0, acc, DTL ? dtl_shift<1, 4>(mn) : -2);       // alpha = 1, beta = 0: C = the sum
    }
}

template <class TL>
int grid_of(const GemmArgs &g)
{
    const int64_t wgs = (int64_t) ((g.M + TL::BM - 1) / TL::BM) * ((g.N + TL::BN - 1) / TL::BN) * g.ksplit;
    return (int) ((wgs + 7) / 8 * 8);
}

template <int TA, int TB, int WA, int WB, class TL, int WPE>
int launch_dtl(const GemmArgs &g)
{
    dgemm_dtl_kernel<TA, TB, WA, WB, TL, WPE><<<grid_of<TL>(g), TL::THREADS, 0, ca3::stream()>>>(g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return ca3::fail(e, "dgemm_dtl_kernel");
    return HIP_PROXY_OK;
}

template <int TA, int TB, class TL>
int launch_tile(const GemmArgs &g)
{
    dgemm_kernel<TA, TB, TL><<<grid_of<TL>(g), TL::THREADS, 0, ca3::stream()>>>(g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return ca3::fail(e, "dgemm_kernel");
    return HIP_PROXY_OK;
}

// CA3DMM_DGEMM_TILE: the workgroup tile, the library's choice unless it names
// one.  CA3DMM_DGEMM_LOADS=reg keeps the register-staged stages throughout;
// =dword takes 4-byte loads for both operands (a test form); =aligned takes
// 16-byte loads only for 16-byte aligned operands with even leading
// dimensions, 4-byte loads for other operands contiguous along m or n, and
// register staging otherwise.  By default whole k-stages are loaded
// direct-to-LDS (6-16 % faster than register staging, same bits) with 16-byte
// loads, whatever the operand's leading dimension and its address modulo 16
// bytes: gfx950 serves 16-byte global loads from 8-byte aligned addresses (the
// compiler itself emits them for such pointers), so a leading dimension of
// 1333 only splits some loads over two cache lines.
enum TileChoice { kTileAuto, kTile128, kTile256x128, kTile128x256, kTile64, kTile32 };

TileChoice tile_choice()
{
    static const struct { const char *name; TileChoice tile; } names[] = {
        {"128x128", kTile128}, {"256x128", kTile256x128}, {"128x256", kTile128x256}, {"64x64", kTile64},
        {"32x32", kTile32}};
    const char *v = getenv("CA3DMM_DGEMM_TILE");
    for (const auto &t : names)
        if (v && !strcmp(v, t.name)) return t.tile;
    return kTileAuto;
}

// How an M x N product from K is cut: the tile, and the number of ranges its k
// is split into.
//
// A CU that holds w workgroups takes about a + b w microseconds per 16-deep
// stage: a is what the stage's latency leaves exposed, b the MFMAs of one tile
// (measured at 64 x 64 x 2000 to 8192^3; the sum is within a few percent of
// the runs below).  A smaller tile spreads a small product over more CUs and
// wastes less on edges and on the last round, but moves more bytes per flop:
// up to 32 workgroups per CU that hardly shows and it is taken where it is 3 %
// better by the sum, beyond that (where it costs up to a fifth) 20 %.
// Microseconds, 128 / 64 / 32 wide:
//   600^3  89 / 36 / 28    1000^3  138 / 50 / 53    1000 x 2000 x 1000
//   138 / 80 / 85    2000^3  267 / 262 / 288    2500^3  598 / 543 / 577
//   3000^3  1070 / 851 / 960    4000^3  1869 / 1951 / 2205    5000 x 5000 x 300
//   276 / 259 / 284    20000 x 300 x 300  91 / 84 / 83    10000 x 10000 x 500
//   1515 / 1737 / 1826    8192^3  15150 / 18830 / 21150
// Register-staged products (below 16 k, single rows) take the same tile: 3 x 12
// from 1 18.6 / - / 13.2, 1 x 1138 from 16 18.4 / - / 14.4.
//
// Splits are tried at 1, 2, 4 and 8 workgroups per CU, each split at least
// four stages long and all partial products within the buffer; one costs a
// second launch (about 6 us) and writing and reading the partials, and has to
// be 10 % better than none.
struct TileCost {
    TileChoice tile;
    int bm, threads;
    double a, b;
};
constexpr TileCost kTileCosts[] = {
    {kTile128, 128, 512, 0.15, 1.80}, {kTile64, 64, 512, 0.20, 0.47}, {kTile32, 32, 256, 0.09, 0.135}};

// A grid has fewer than 2^32 threads (2 x 2^29 from 16 has more 32-wide tiles
// than that holds; beyond 2^23 128-wide ones the 4-wave form runs).
bool grid_fits(int64_t wgs, int threads) { return (wgs + 7) / 8 * 8 * threads < (int64_t) 1 << 32; }

// What a smaller tile's cost has to be below, as a part of the larger one's.
double smaller_tile_margin(int64_t wgs, int64_t cus) { return wgs <= 32 * cus ? 0.97 : 0.8; }

struct Cut {
    TileChoice tile;
    int ksplit, stages;                        // stages: 16-deep k-stages per split
};

constexpr size_t kSplitBytes = (size_t) 64 << 20;

Cut pick_cut(int64_t M, int64_t N, int64_t K, bool may_split)
{
    const int64_t cus = ca3::cu_count(), stages = (K + kBK - 1) / kBK;
    Cut best = {kTile128, 1, (int) stages}, split = best;
    double t = 0.0, ts = 0.0;
    for (const TileCost &c : kTileCosts) {
        const int64_t wgs = ((M + c.bm - 1) / c.bm) * ((N + c.bm - 1) / c.bm);
        if (c.tile != kTile128 && !grid_fits(wgs, c.threads)) continue;
        const double us = (double) stages * (c.a + c.b * (double) ((wgs + cus - 1) / cus));
        if (c.tile == kTile128 || us < smaller_tile_margin(wgs, cus) * t) {
            best.tile = c.tile;
            t = us;
        }
        for (int r = 1; may_split && r <= 8; r *= 2) {
            int64_t s = std::min(r * cus / wgs, std::min(stages / 4, (int64_t) (kSplitBytes / 8) / (M * N)));
            if (s < 2) continue;
            const int64_t len = (stages + s - 1) / s;
            s = (stages + len - 1) / len;
            const double cost = 6.0 + (double) len * (c.a + c.b * (double) ((wgs * s + cus - 1) / cus)) +
                                (double) (2 * s + 1) * M * N * 8.0 / 4e6;
            if (s > 1 && (ts == 0.0 || cost < ts)) {
                split = {c.tile, (int) s, (int) len};
                ts = cost;
            }
        }
    }
    return ts > 0.0 && ts < 0.9 * t ? split : best;
}

// The partial products of split calls: one buffer per device, allocated at the
// first split call and kept.  The mutex is held from before the first to after
// the second launch of a call, so that calls of several threads, which share
// the device's stream, do not use it across each other.
std::mutex g_split_mu;
double *g_split_buf[16];

// The device's buffer; null where there is none to use: the product then runs
// unsplit.  Under stream capture that is always so (the captured launches may
// be replayed beside later calls).
double *split_buffer()
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ca3::stream(), &st) != hipSuccess || st != hipStreamCaptureStatusNone) {
        (void) hipGetLastError();
        return nullptr;
    }
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return nullptr;
    if (!g_split_buf[dev] && hipMalloc((void **) &g_split_buf[dev], kSplitBytes) != hipSuccess) {
        (void) hipGetLastError();              // the failed allocation is not an error of the call
        g_split_buf[dev] = nullptr;
    }
    return g_split_buf[dev];
}

// The direct-to-LDS load width of an operand (4 or 1 words), 0 for none
// (the product is then register-staged).  xc: the operand is contiguous
// along m or n.
int dtl_words(const double *P, int64_t ld, bool xc, LoadMode mode)
{
    if (!dtl_ld_ok(ld) || ((uintptr_t) P % 8) != 0 || mode == kLoadsReg) return 0;
    if (mode == kLoadsDword) return 1;
    if (mode == kLoadsAligned && (((uintptr_t) P % 16) != 0 || (ld % 2) != 0)) return xc ? 1 : 0;
    return 4;
}

// Whether the 128 x 128 tiles take the form that leaves out the 16 x 16 blocks
// outside C: there it can give more than 1.5 % of the MFMAs, over several
// rounds of workgroups (in one round, the whole tiles end last).  us without /
// with it: 120000 x 600 x 600 1398 / 1335, 10000 x 10000 x 500 1519 / 1512;
// without such blocks it is 0.2 % slower.
bool edge_waste(const GemmArgs &g)
{
    const double tiles = (double) ((g.M + 127) / 128) * ((g.N + 127) / 128);
    const double blocks = (double) ((g.M + 15) / 16) * ((g.N + 15) / 16);
    return blocks < 0.985 * 64.0 * tiles && tiles * g.ksplit > 4.0 * ca3::cu_count();
}

template <int TA, int TB>
int launch(const GemmArgs &g, TileChoice best)
{
    const TileChoice tc = tile_choice();
    const LoadMode mode = load_mode();
    const bool reg_tile = tc == kTile256x128 || tc == kTile128x256;
    const int wa = dtl_words(g.A, g.lda, !TA, mode), wb = dtl_words(g.B, g.ldb, TB, mode);
    // a single row (column) contiguous along m (n) has no pair to load
    const bool edges = (TA || wa == 1 || g.M > 1) && (!TB || wb == 1 || g.N > 1);
    if (!reg_tile && wa && wb && edges && g.K >= kBK && grid_fits(grid_of<Tile128w8>(g), Tile128w8::THREADS)) {
        if (wa == 4 && wb == 4) {
            switch (tc == kTileAuto ? best : tc) {
            case kTile64: return launch_dtl<TA, TB, 4, 4, Tile64, 4>(g);
            case kTile32: return launch_dtl<TA, TB, 4, 4, Tile32, 4>(g);
            default:
                return edge_waste(g) ? launch_dtl<TA, TB, 4, 4, Tile128e, 4>(g)
                                     : launch_dtl<TA, TB, 4, 4, Tile128w8, 4>(g);
            }
        }
        if (wa == 4) return launch_dtl<TA, TB, 4, 1, Tile128, 2>(g);
        if (wb == 4) return launch_dtl<TA, TB, 1, 4, Tile128, 2>(g);
        return launch_dtl<TA, TB, 1, 1, Tile128, 2>(g);
    }
    switch (tc == kTileAuto ? best : tc) {
    case kTile256x128: return launch_tile<TA, TB, Tile256x128>(g);
    case kTile128x256: return launch_tile<TA, TB, Tile128x256>(g);
    case kTile64: return launch_tile<TA, TB, Tile64>(g);
    case kTile32: return launch_tile<TA, TB, Tile32>(g);
    default: return launch_tile<TA, TB, Tile128>(g);
    }
}

int run(hip_proxy_enum_t transA, hip_proxy_enum_t transB, int m, int n, int k, double alpha,
        const double *A, int ldA, const double *B, int ldB, double beta, double *C, int ldC,
        int nsrc, const double *const *P, const int *ldp, bool may_split)
{
    const int ta = (transA != HipNoTrans), tb = (transB != HipNoTrans);
    if (m < 0 || n < 0 || k < 0) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: negative size");
    if (m == 0 || n == 0) return HIP_PROXY_OK;
    if (!C || ldC < std::max(1, m)) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: bad C / ldC");
    if (k > 0) {
        if (!A || ldA < std::max(1, ta ? k : m)) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: bad A / ldA");
        if (!B || ldB < std::max(1, tb ? n : k)) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: bad B / ldB");
    }
    if (nsrc < 0 || nsrc > kMaxFoldSrc) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: nsrc %d", nsrc);
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.M = m; g.N = n; g.K = k;
    g.alpha = alpha; g.beta = beta;
    g.A = A; g.lda = ldA; g.B = B; g.ldb = ldB; g.C = C; g.ldc = ldC;
    g.nsrc = nsrc;
    {
        const char *v = getenv("CA3DMM_DGEMM_GROUP");
        const int G = v ? atoi(v) : 16;
        g.group = (G >= 1 && G <= 256) ? G : 16;
    }
    for (int t = 0; t < nsrc; ++t) {
        if (!P || !ldp || !P[t] || ldp[t] < m) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm: partial %d", t);
        g.P[t] = P[t];
        g.ldp[t] = ldp[t];
    }
    std::unique_lock<std::mutex> lk(g_split_mu, std::defer_lock);
    Cut cut = pick_cut(m, n, k, may_split);
    if (cut.ksplit > 1) {
        lk.lock();
        g.part = split_buffer();
        if (!g.part) cut = pick_cut(m, n, k, false);
    }
    g.ksplit = cut.ksplit;
    g.kstep = (int) std::min<int64_t>((int64_t) std::max(1, cut.stages) * kBK, INT_MAX);
    int rc;
    if (!ta && !tb) rc = launch<0, 0>(g, cut.tile);
    else if (!ta && tb) rc = launch<0, 1>(g, cut.tile);
    else if (ta && !tb) rc = launch<1, 0>(g, cut.tile);
    else rc = launch<1, 1>(g, cut.tile);
    if (!rc && g.ksplit > 1) {
        dgemm_reduce_kernel<<<(unsigned) (((int64_t) m * n + 63) / 64), 256, 0, ca3::stream()>>>(g);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = ca3::fail(e, "dgemm_reduce_kernel");
    }
    if (lk.owns_lock()) lk.unlock();
    if (rc) return rc;
    return ca3::finish();
}

}  // namespace

// ---------------------------------------------------------------------
// Batched launch of the simulated grid's per-rank products (grouped.h)
// ---------------------------------------------------------------------
namespace ca3 {
namespace grouped {

struct BatchPlan {
    BatchProb *d = nullptr;
    int nprob = 0;
    int64_t total = 0;
    int group = 16;
    bool per_segment = true, dtl = false;
    TileChoice tile = kTile128;                // register-staged plans: always 128 x 128
};

int build_batch(const std::vector<Problem> &probs, bool per_segment, BatchPlan **out)
{
    *out = nullptr;
    std::vector<BatchProb> h;
    bool all_dtl = true;
    const gemm::LoadMode mode = gemm::load_mode();
    for (const Problem &q : probs) {
        if (q.M <= 0 || q.N <= 0) continue;
        if (q.nseg < 0 || q.nseg > kMaxSeg || !q.C || q.ldc < q.M)
            return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm batch: bad problem");
        BatchProb b;
        memset(&b, 0, sizeof(b));
        b.M = q.M; b.N = q.N; b.nseg = q.nseg;
        b.C = q.C; b.ldc = q.ldc;
        for (int s = 0; s < q.nseg; ++s) {
            const Seg &g = q.seg[s];
            if (g.k < 0 || (g.k > 0 && (!g.A || !g.B || g.lda < q.M || g.ldb < g.k)))
                return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm batch: bad segment %d", s);
            b.A[s] = g.A; b.B[s] = g.B;
            b.lda[s] = g.lda; b.ldb[s] = g.ldb;
            b.k[s] = g.k;
            all_dtl = all_dtl && dtl_words(g.A, g.lda, true, mode) == 4 && dtl_words(g.B, g.ldb, false, mode) == 4 &&
                      g.k >= gemm::kBK && q.M > 1;
        }
        h.push_back(b);
    }
    // (A segment of 1 to 15 k, or a rank of one row, whose neighbours then have
    // two at most, sends the whole plan to the register-staged form: 24 ranks,
    // 8000 x 8000 x 95, rounds of 15 and 16 k: 1.90 ms; a kernel of both forms,
    // in 4 waves, 2.18.)
    // The tile whose rounds of workgroups cost least, by the rule of a single
    // product: a CU takes a + b w per stage for its w workgroups, over the
    // mean number of stages of a tile
    TileChoice tile = kTile128;
    int64_t base = 0;
    double best = 0.0;
    for (const TileCost &c : kTileCosts) {
        int64_t wgs = 0, work = 0;
        for (const BatchProb &b : h) {
            const int64_t n = (int64_t) ((b.M + c.bm - 1) / c.bm) * ((b.N + c.bm - 1) / c.bm);
            int64_t stages = 0;
            for (int s = 0; s < b.nseg; ++s) stages += (b.k[s] + gemm::kBK - 1) / gemm::kBK;
            wgs += n;
            work += n * stages;
        }
        const double us = wgs ? (double) work / (double) wgs *
                                    (c.a + c.b * (double) ((wgs + ca3::cu_count() - 1) / ca3::cu_count()))
                              : 0.0;
        if (c.tile == kTile128) all_dtl = all_dtl && grid_fits(wgs, c.threads);
        else if (!grid_fits(wgs, c.threads)) continue;
        if (c.tile != kTile128 && !(all_dtl && us < smaller_tile_margin(wgs, ca3::cu_count()) * best)) continue;
        tile = c.tile;
        best = us;
        base = 0;
        for (BatchProb &b : h) {
            b.base = base;
            base += (int64_t) ((b.M + c.bm - 1) / c.bm) * ((b.N + c.bm - 1) / c.bm);
        }
    }
    if ((base + 7) / 8 * 8 > INT_MAX) return ca3::fail_msg(HIP_PROXY_ERR_UNSUPP, "dgemm batch: %lld tiles", (long long) base);
    auto *p = new BatchPlan;
    p->per_segment = per_segment;
    p->dtl = all_dtl;
    p->tile = tile;
    p->nprob = (int) h.size();
    p->total = base;
    const char *v = getenv("CA3DMM_DGEMM_GROUP");
    const int G = v ? atoi(v) : 16;
    p->group = (G >= 1 && G <= 256) ? G : 16;
    if (!h.empty()) {
        hipError_t e = hipMalloc(&p->d, h.size() * sizeof(BatchProb));
        if (e == hipSuccess) e = hipMemcpy(p->d, h.data(), h.size() * sizeof(BatchProb), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            destroy_batch(p);
            return ca3::fail(e, "dgemm batch plan");
        }
    }
    *out = p;
    return HIP_PROXY_OK;
}

int run_batch(BatchPlan *p, int group)
{
    if (!p) return ca3::fail_msg(HIP_PROXY_ERR_ARG, "dgemm batch: no plan");
    if (p->total == 0) return HIP_PROXY_OK;
    const int grid = (int) ((p->total + 7) / 8 * 8);
    const int G = (group >= 1 && group <= 256) ? group : p->group;
    auto go = [&](auto per_seg) {
        constexpr bool S = decltype(per_seg)::value;
        hipStream_t st = ca3::stream();
        if (!p->dtl) dgemm_batch_kernel<S, false, Tile128, 2><<<grid, 256, 0, st>>>(p->d, p->nprob, p->total, G);
        else if (p->tile == kTile64)
            dgemm_batch_kernel<S, true, Tile64, 4><<<grid, 512, 0, st>>>(p->d, p->nprob, p->total, G);
        else if (p->tile == kTile32)
            dgemm_batch_kernel<S, true, Tile32, 4><<<grid, 256, 0, st>>>(p->d, p->nprob, p->total, G);
        else dgemm_batch_kernel<S, true, Tile128w8, 4><<<grid, 512, 0, st>>>(p->d, p->nprob, p->total, G);
    };
    if (p->per_segment) go(std::true_type{});
    else go(std::false_type{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return ca3::fail(e, "dgemm_batch_kernel");
    return ca3::finish();
}

int round_product(int m, int n, int k, const double *A, int lda, const double *B, int ldb, double beta, double *C,
                  int ldc)
{
    return ::run(HipNoTrans, HipNoTrans, m, n, k, 1.0, A, lda, B, ldb, beta, C, ldc, 0, nullptr, nullptr, false);
}

void destroy_batch(BatchPlan *p)
{
    if (!p) return;
    if (p->d) (void) hipFree(p->d);
    delete p;
}

}  // namespace grouped
}  // namespace ca3

ca3::gemm::LoadMode ca3::gemm::load_mode()
{
    const char *v = getenv("CA3DMM_DGEMM_LOADS");
    if (!v) return kLoads16;
    if (!strcmp(v, "reg")) return kLoadsReg;
    if (!strcmp(v, "dword")) return kLoadsDword;
    if (!strcmp(v, "aligned")) return kLoadsAligned;
    return kLoads16;
}

extern "C" {

int hip_dgemm(hip_proxy_enum_t transA, hip_proxy_enum_t transB, const int m, const int n,
              const int k, const double alpha, const double *A, const int ldA, const double *B,
              const int ldB, const double beta, double *C, const int ldC)
{
    return run(transA, transB, m, n, k, alpha, A, ldA, B, ldB, beta, C, ldC, 0, nullptr, nullptr, true);
}

int hip_dgemm_fold(hip_proxy_enum_t transA, hip_proxy_enum_t transB, const int m, const int n,
                   const int k, const double alpha, const double *A, const int ldA,
                   const double *B, const int ldB, const double beta, double *C, const int ldC,
                   int nsrc, const double *const *P, const int *ldp)
{
    return run(transA, transB, m, n, k, alpha, A, ldA, B, ldB, beta, C, ldC, nsrc, P, ldp, true);
}

}  // extern "C"
