// Device building blocks of the FP64 MFMA GEMM tile, shared by the plain
// DGEMM, the grouped (simulated-grid) GEMM and the Gram kernel.
//
// MFMA operand / result layout used throughout (v_mfma_f64_16x16x4_f64,
// one wave64):  X(16x4): lane l holds X[l%16][l/16];  Y(4x16): lane l holds
// Y[l/16][l%16];  D = X*Y (16x16): lane l, register r holds D[4*r + l/16][l%16].
// The tile code feeds X = op(B)^T and Y = op(A)^T, so D is a block of C^T:
// lane l, register r holds C[m = l%16][n = 4*r + l/16].  For a fixed r the 16
// lanes of a row group then hold 16 consecutive rows of one column of C,
// which makes the column-major stores 128-byte contiguous.
#pragma once

#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>
#include <type_traits>

#include "hip_common.h"

namespace ca3 {
namespace gemm {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) double gdouble;     // in global memory (a pointer read from a table is generic)

constexpr int kBM = 128, kBN = 128, kBK = 16;
constexpr int kMaxFoldSrc = 8;

template <int XC, int W = 128, int T = 256>
struct OperandLoader;

// Workgroup tile BM x BN of C: WM x WN waves along m and n, each of FI x FJ
// MFMA blocks.  Register-staged kernels: 128 x 128 with 4 waves of 64 x 64
// (two workgroups per CU), 256 x 128 and 128 x 256 with 8 waves (one per CU).
// Direct-to-LDS kernels: Tile128w8, 8 waves of 64 x 32, whose 117 to
// 124 vector registers leave room for four waves per SIMD (8192^3 TN 15.1 ms; the 4
// waves of 64 x 64, two per SIMD, 15.45 ms; 10000 x 10000 x 500 1.52 / 1.59
// ms); Tile64 (8 waves of 32 x 16) and Tile32 (4 waves of 16 x 16) for
// products whose 128 x 128 tiles leave CUs idle.  IL (Tile128e): a wave's
// blocks lie WM (WN) blocks apart instead of side by side, so that the blocks
// inside C of an edge tile are spread over all waves and SIMDs, and blocks
// outside take no MFMAs.
template <int BM_, int BN_, int WM_ = BM_ / 64, int WN_ = BN_ / 64, bool IL_ = false>
struct TileShape {
    static constexpr bool IL = IL_;
    static constexpr int BM = BM_, BN = BN_;
    static constexpr int WM = WM_, WN = WN_;
    static constexpr int FI = BM / WM / 16, FJ = BN / WN / 16;
    static constexpr int NW = WM * WN, THREADS = 64 * NW;
    static constexpr int MIN_BLOCKS = THREADS == 256 ? 2 : 1;     // per CU, for __launch_bounds__
    // the register-staged loader of either operand of a square tile
    template <int XC>
    using OperandLoader = std::enable_if_t<BM_ == BN_, gemm::OperandLoader<XC, BM_, 64 * WM_ * WN_>>;
};
using Tile128 = TileShape<128, 128>;
using Tile256x128 = TileShape<256, 128>;
using Tile128x256 = TileShape<128, 256>;
using Tile128w8 = TileShape<128, 128, 2, 4>;
using Tile128e = TileShape<128, 128, 2, 4, true>;
using Tile64 = TileShape<64, 64, 2, 4>;
using Tile32 = TileShape<32, 32, 2, 2>;

struct GemmArgs {
    int M, N, K;
    double alpha, beta;
    const double *A;
    int64_t lda;
    const double *B;
    int64_t ldb;
    double *C;
    int64_t ldc;
    int group;                      // tile rows walked together (tile_coords)
    int nsrc;                       // partial-C fold in the epilogue
    const double *P[kMaxFoldSrc];
    int64_t ldp[kMaxFoldSrc];
    // ksplit > 1: the workgroups of split s accumulate k in [s kstep, (s + 1)
    // kstep) and store the bare sum to part + s M N (leading dimension M)
    int ksplit, kstep;
    double *part;
};

// First row (column) in the tile of a wave's block i (j).
template <class TL>
__device__ __forceinline__ int block_row(int wm, int i) { return (TL::IL ? i * TL::WM + wm : wm * TL::FI + i) * 16; }
template <class TL>
__device__ __forceinline__ int block_col(int wn, int j) { return (TL::IL ? j * TL::WN + wn : wn * TL::FJ + j) * 16; }

template <int FI, int FJ>
__device__ __forceinline__ void zero(f64x4 (&acc)[FI][FJ])
{
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
}

// XOR swizzle of column x within LDS row kk (see dgemm.hip header).
__device__ __forceinline__ int swz(int kk, int x)
{
    return x ^ (((kk & 1) << 4) | ((kk >> 1) & 7));
}

// Linear tile index -> (tile row, tile col): groups of G tile-rows (16 unless
// CA3DMM_DGEMM_GROUP says otherwise) walked column by column.
template <class TL>
__device__ __forceinline__ void tile_coords(int t, int M, int N, int *tm, int *tn, int G)
{
    const int tiles_m = (M + TL::BM - 1) / TL::BM, tiles_n = (N + TL::BN - 1) / TL::BN;
    const int per = G * tiles_n;
    const int grp = t / per;
    const int first = grp * G;
    const int gsz = min(tiles_m - first, G);
    const int r = t - grp * per;
    *tm = first + r % gsz;
    *tn = r / gsz;
}

// Loads one 16 x W stage of an operand (W = the tile's extent along m or
// n) with T threads into registers and writes it to LDS as [k][x].  XC = 1:
// the operand is contiguous along x (m or n); XC = 0: contiguous along k.
// Out-of-range elements read as 0.  Each thread holds P = 16 W / T elements:
// XC = 1 at k rows kk0, kk0 + T/W, ...; XC = 0 at columns x, x + T/16, ...
template <int XC, int W, int T>
struct OperandLoader {
    static constexpr int P = W * kBK / T;
    static constexpr int KSTEP = T / W;         // XC: k rows per pass of the workgroup
    static constexpr int XSTEP = T / kBK;       // !XC: columns per pass
    static_assert(P >= 1 && P <= 16 && KSTEP * P == kBK && XSTEP * P == W, "loader shape");
    const double *base;   // element (x = this thread's first x, k = 0)
    int64_t ld;
    int kk0;              // XC: first k row of this thread; !XC: its k row
    unsigned xmask;       // bit p: x of element p is in range
    int xcol;             // this thread's (first) x
    double r[P];

    __device__ __forceinline__ void init(const double *M, int64_t ld_, int x0, int xdim)
    {
        const int t = threadIdx.x;
        ld = ld_;
        if (XC) {
            xcol = t % W;
            kk0 = t / W;
            xmask = (x0 + xcol < xdim) ? 0xffffu : 0u;
            base = M + (x0 + xcol);
        } else {
            kk0 = t & 15;
            const int xt = t >> 4;
            xcol = xt;
            xmask = 0;
#pragma unroll
            for (int p = 0; p < P; ++p)
                if (x0 + xt + XSTEP * p < xdim) xmask |= 1u << p;
            base = M + (int64_t) (x0 + xt) * ld;
        }
    }

    __device__ __forceinline__ void load(int k0, int kend)
    {
        if (XC) {
            const double *q = base + (int64_t) (k0 + kk0) * ld;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const bool ok = xmask && (k0 + kk0 + KSTEP * p < kend);
                r[p] = ok ? q[(int64_t) (KSTEP * p) * ld] : 0.0;
            }
        } else {
            const bool kok = (k0 + kk0 < kend);
            const double *q = base + (k0 + kk0);
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const bool ok = kok && ((xmask >> p) & 1u);
                r[p] = ok ? q[(int64_t) (XSTEP * p) * ld] : 0.0;
            }
        }
    }

    // The same stage with every element in range (interior tile, whole
    // k-stage): no predicates, so the loads issue without branches.
    __device__ __forceinline__ void load_full(int k0)
    {
        if (XC) {
            const double *q = base + (int64_t) (k0 + kk0) * ld;
#pragma unroll
            for (int p = 0; p < P; ++p) r[p] = q[(int64_t) (KSTEP * p) * ld];
        } else {
            const double *q = base + (k0 + kk0);
#pragma unroll
            for (int p = 0; p < P; ++p) r[p] = q[(int64_t) (XSTEP * p) * ld];
        }
    }

    __device__ __forceinline__ void store(double *S) const
    {
        if (XC) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int kk = kk0 + KSTEP * p;
                S[kk * W + swz(kk, xcol)] = r[p];
            }
        } else {
#pragma unroll
            for (int p = 0; p < P; ++p) S[kk0 * W + swz(kk0, xcol + XSTEP * p)] = r[p];
        }
    }
};

// k-slices [KS0, KS1) of the 16 k-steps of MFMAs on the LDS stage (4 x
// v_mfma_f64_16x16x4 k-slices in all).
template <class TL = Tile128, int KS0 = 0, int KS1 = kBK / 4>
__device__ __forceinline__ void stage_mfma(const double *As, const double *Bs, f64x4 (&acc)[TL::FI][TL::FJ])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave % TL::WM, wn = wave / TL::WM;
    const int li = lane & 15;
#pragma unroll
    for (int ks = KS0; ks < KS1; ++ks) {
        const int kk = ks * 4 + (lane >> 4);
        double a[TL::FI], b[TL::FJ];
#pragma unroll
        for (int i = 0; i < TL::FI; ++i) a[i] = As[kk * TL::BM + swz(kk, block_row<TL>(wm, i) + li)];
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j) b[j] = Bs[kk * TL::BN + swz(kk, block_col<TL>(wn, j) + li)];
#pragma unroll
        for (int i = 0; i < TL::FI; ++i)
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0);
    }
}

// The two LDS stage buffers of an operand held as two separate arrays (the
// direct-to-LDS loop needs them so); As[i] as for a double[2][...] array.
struct LdsPair {
    double *b0, *b1;
    __device__ __forceinline__ double *operator[](int i) const { return i ? b1 : b0; }
};

// Accumulate op(A)[m0:+BM, kbeg:kend) * op(B)[kbeg:kend, n0:+BN) into acc
// with bounds checks on every element (edge tiles and partial k-stages).
// As / Bs: double[2][16 * BM] (or LdsPair), As[i] = stage buffer i.
template <class TL = Tile128, class LA, class LB, class BA, class BB>
__device__ __forceinline__ void mainloop_checked(LA &la, LB &lb, int kbeg, int kend, BA As, BB Bs,
                                                 f64x4 (&acc)[TL::FI][TL::FJ])
{
    if (kend <= kbeg) return;
    const int nk = (kend - kbeg + kBK - 1) / kBK;
    la.load(kbeg, kend);
    lb.load(kbeg, kend);
    la.store(As[0]);
    lb.store(Bs[0]);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        const bool more = (kt + 1 < nk);
        if (more) {
            la.load(kbeg + (kt + 1) * kBK, kend);
            lb.load(kbeg + (kt + 1) * kBK, kend);
        }
        stage_mfma<TL>(As[cur], Bs[cur], acc);
        if (more) {
            la.store(As[cur ^ 1]);
            lb.store(Bs[cur ^ 1]);
        }
        __syncthreads();
    }
}

// The same accumulation.  A tile that is interior in m and n (interior =
// m0 + BM <= M and n0 + BN <= N) runs its whole k-stages through a loop
// without predicates or data-dependent branches (one register stage in
// flight, the last stage's load repeated in bounds and never consumed);
// edge tiles and the k tail go through mainloop_checked.  Both add the
// k-steps in the same order, so results do not depend on the path.
template <class TL = Tile128, class LA, class LB, class BA, class BB>
__device__ __forceinline__ void mainloop(LA &la, LB &lb, int kbeg, int kend, bool interior, BA As, BB Bs,
                                         f64x4 (&acc)[TL::FI][TL::FJ])
{
    const int nfull = (interior && kend > kbeg) ? (kend - kbeg) / kBK : 0;
    if (nfull > 0) {
        la.load_full(kbeg);
        lb.load_full(kbeg);
        la.store(As[0]);
        lb.store(Bs[0]);
        __syncthreads();
        for (int kt = 0; kt < nfull; ++kt) {
            const int cur = kt & 1;
            const int kn = kbeg + min(kt + 1, nfull - 1) * kBK;
            la.load_full(kn);
            lb.load_full(kn);
            // the next stage goes to the other buffer halfway through this
            // one's MFMAs (its loads have had half a stage to land), so the
            // LDS writes complete under the second half instead of before
            // the barrier
            stage_mfma<TL, 0, kBK / 8>(As[cur], Bs[cur], acc);
            la.store(As[cur ^ 1]);
            lb.store(Bs[cur ^ 1]);
            stage_mfma<TL, kBK / 8, kBK / 4>(As[cur], Bs[cur], acc);
            __syncthreads();
        }
    }
    const int kt0 = kbeg + nfull * kBK;
    if (kt0 < kend) mainloop_checked<TL>(la, lb, kt0, kend, As, Bs, acc);
}

// ---------------------------------------------------------------------
// Direct-to-LDS stages: global_load_lds_dwordx4 writes lane l's 16 bytes
// (two doubles) at M0 + 16 l, so one wave instruction fills a 1 KB LDS
// block; a stage of a W-wide operand is W / 8 blocks (16 k x W), dealt to
// the waves.  No staging registers and no LDS stores.  Layouts (d = one
// double):
//   XC = 1 (contiguous along x): k rows of W x, one after the other; 16-byte
//     chunk c of row k holds x = 2 (c ^ fx(k)), +1 with fx(k) = 8 (k & 1);
//   XC = 0 (contiguous along k): block = 8 x lines of 16 k; chunk c of line
//     x holds k = 2 (c ^ hx(x)), +1 with hx(x) = (x >> 1) & 7.
// Each lane fetches the global chunk its LDS slot holds, so the reads stay
// coalesced, and the MFMA operand reads (16 consecutive x at 4 k) hit 64
// distinct banks per 32 lanes.  The k-slices of the MFMAs are those of
// stage_mfma, so both paths add the same products in the same order.
// ---------------------------------------------------------------------
template <int XC, int W = 128>
__device__ __forceinline__ int dtl_index(int k, int x)
{
    if (XC) return k * W + 2 * ((x >> 1) ^ ((k & 1) << 3)) + (x & 1);
    return x * 16 + 2 * ((k >> 1) ^ ((x >> 1) & 7)) + (k & 1);
}

// Edge tiles: only xn <= W x of the tile exist.  A lane whose slot holds an
// x >= xn loads the last existing x (or x pair) instead, so every load stays
// inside the operand; those LDS rows hold copies whose products land in C
// rows or columns the epilogue never stores.  For XC = 1 and odd xn the
// last chunk holds the pair (xn - 2, xn - 1), one x lower than its slot
// says: the products of x = xn - 1 come out in row (column) xn of the tile,
// and the epilogue stores that one in place of row xn - 1 (dtl_shift).
// Addresses are a wave-uniform base per block (scalar registers) plus a
// 32-bit lane offset, which requires 7 * ld * 8 + 128 < 2^32 bytes
// (dtl_ld_ok).
//
// WORDS = 4: one 16-byte load per lane and block (global_load_lds_dwordx4)
// of a double pair, from an 8-byte aligned address (an odd ld or an
// operand 8 bytes past a 16-byte boundary splits some loads over two
// cache lines); for XC = 1 a lone x (xn = 1) needs the x before it (x0 > 0).
// WORDS = 1 (W = 128 only): four 4-byte loads per lane and block
// (global_load_lds_dword, lane l of load q lands at M0 + 256 q + 4 l), for
// any xn, every x in its own slot; otherwise the same LDS image.
__host__ __device__ constexpr bool dtl_ld_ok(int64_t ld) { return ld >= 0 && ld <= (int64_t) 1 << 26; }

// The x of the tile whose products appear one row (column) further on (see
// above), or -2 for none.
template <int XC, int WORDS>
__device__ __forceinline__ int dtl_shift(int xn)
{
    return (XC && WORDS == 4 && (xn & 1)) ? xn - 1 : -2;
}

// Load forms of the direct-to-LDS stages (CA3DMM_DGEMM_LOADS): 16-byte
// loads from any 8-byte aligned operand (default); "aligned": 16-byte
// loads only for 16-byte aligned operands with even ld, 4-byte loads for
// other operands contiguous along m or n, register staging otherwise;
// "dword": 4-byte loads; "reg": register staging only.
enum LoadMode { kLoads16, kLoadsAligned, kLoadsDword, kLoadsReg };
LoadMode load_mode();

template <int XC_, int WORDS = 4, int W = 128, int NW = 4>
struct DtlLoader;

template <int XC_, int W, int NW>
struct DtlLoader<XC_, 4, W, NW> {
    static constexpr int XC = XC_, WORDS = 4;
    static constexpr int NB = W / (8 * NW);  // blocks per wave
    static constexpr int RPB = 128 / W;      // XC: k rows per block
    const double *base[NB];  // block i of this wave for k0 = 0 (wave-uniform)
    uint32_t off[NB];        // this lane's byte offset from base[i]

    __device__ __forceinline__ void init(const double *M, int64_t ld, int x0, int xn = W)
    {
        const int lane = threadIdx.x & 63;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int b = NB * w + i;
            if (XC) {
                // k rows RPB b .. of the stage; chunk c of a row holds x = 2c, 2c + 1
                const int kr = lane / (W / 2), k = RPB * b + kr;
                const int x = min(2 * ((lane % (W / 2)) ^ ((k & 1) << 3)), xn - 2);
                const int back = xn == 1;           // the pair (x0 - 1, x0)
                base[i] = M + (x0 - back) + (int64_t) (RPB * b) * ld;
                off[i] = (uint32_t) ((int64_t) kr * ld * 8) + 8u * (uint32_t) (x + back);
            } else {
                // lines x = 8b .. 8b + 7 of the tile; the lane's k pair is
                // fixed by its slot (line xl), the line read is x <= xn - 1
                const int xb = min(8 * b, xn - 1), xl = 8 * b + (lane >> 3), x = min(xl, xn - 1);
                base[i] = M + (int64_t) (x0 + xb) * ld;
                off[i] = (uint32_t) ((int64_t) (x - xb) * ld * 8) + 16u * (uint32_t) ((lane & 7) ^ ((xl >> 1) & 7));
            }
        }
    }

    // issue the stage starting at koff (elements) into S (16 x W doubles)
    __device__ __forceinline__ void issue(int64_t koff, double *S) const
    {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const char *g = reinterpret_cast<const char *>(base[i] + koff) + (uint64_t) off[i];
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *) g,
                                             (void __attribute__((address_space(3))) *) (S + (NB * w + i) * 128),
                                             16, 0, 0);
        }
    }
};

// Load q (0..3) of a block fills LDS bytes [256 q, 256 q + 256) of it: lane
// l writes the 4-byte half h = l & 1 of double j = (l >> 1) & 1 of 16-byte
// chunk c = 16 q + (l >> 2).  The offsets are rebuilt per stage from a few
// lane constants (the vector ALU is idle under the MFMAs), so the loader
// holds as many registers as the 16-byte one.
template <int XC_>
struct DtlLoader<XC_, 1, 128, 4> {
    static constexpr int XC = XC_, WORDS = 1;
    const double *M;
    int64_t ld;
    int x0, xn;
    uint32_t t;     // l >> 2: the chunk within the load's 16
    uint32_t jh;    // 8 j + 4 h

    __device__ __forceinline__ void init(const double *M_, int64_t ld_, int x0_, int xn_ = 128)
    {
        const int lane = threadIdx.x & 63;
        M = M_; ld = ld_; x0 = x0_; xn = xn_;
        t = (uint32_t) (lane >> 2);
        jh = 8u * ((lane >> 1) & 1) + 4u * (lane & 1);
    }

    __device__ __forceinline__ void issue(int64_t koff, double *S) const
    {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = 4 * w + i;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double *base;
                uint32_t off;
                if (XC) {
                    // k row b; chunk c = 16 q + t holds x pair p = c ^ 8 (b & 1)
                    base = M + x0 + (int64_t) b * ld + koff;
                    const uint32_t x = 2u * (uint32_t) ((16 * q + (int) t) ^ ((b & 1) << 3)) + (jh >> 3);
                    off = 8u * min(x, (uint32_t) xn - 1u) + (jh & 4u);
                } else {
                    // line xl = 8b + 2q + (t >> 3), k pair (t & 7) ^ ((xl >> 1) & 7)
                    const int xb = min(8 * b + 2 * q, xn - 1);
                    base = M + (int64_t) (x0 + xb) * ld + koff;
                    const int xl = 8 * b + 2 * q + (int) (t >> 3), x = min(xl, xn - 1);
                    off = (uint32_t) ((x - xb) * (int) ld) * 8u +
                          16u * (uint32_t) ((t & 7) ^ (uint32_t) ((xl >> 1) & 7)) + jh;
                }
                auto src = (const void __attribute__((address_space(1))) *) (reinterpret_cast<const char *>(base) +
                                                                             (uint64_t) off);
                auto dst = (void __attribute__((address_space(3))) *) (S + (4 * w + i) * 128 + 32 * q);
                __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
            }
        }
    }
};

// The blocks of this wave that lie inside an mn x nn edge tile (mn and nn with
// the row or column that dtl_shift moves on), in scalar registers.
struct Blocks {
    int fi, fj;
};

template <class TL>
__device__ __forceinline__ Blocks blocks_inside(int mn, int nn, int ms, int ns)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % TL::WM, wn = wave / TL::WM;
    const int rb = (min(mn + (ms >= 0), TL::BM) + 15) >> 4, cb = (min(nn + (ns >= 0), TL::BN) + 15) >> 4;
    return Blocks{__builtin_amdgcn_readfirstlane((rb - wm + TL::WM - 1) / TL::WM),
                  __builtin_amdgcn_readfirstlane((cb - wn + TL::WN - 1) / TL::WN)};
}

// The MFMAs of one stage on the wave's blocks i < FIV, j < FJV.  lo > 0
// (a stage that overlaps the one before it): the k below lo of the stage count
// as zero in both operands.
template <int XCA, int XCB, class TL, int FIV, int FJV, bool TAIL = false>
__device__ __forceinline__ void stage_mfma_dtl(const double *As, const double *Bs, f64x4 (&acc)[TL::FI][TL::FJ],
                                               int lo = 0)
{
    int tid = threadIdx.x;
    if (TAIL) asm volatile("" : "+v"(tid));      // no address of the tail is computed before the main loop
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave % TL::WM, wn = wave / TL::WM;
    const int li = lane & 15;
#pragma unroll
    for (int ks = 0; ks < kBK / 4; ++ks) {
        if (TAIL && ks * 4 + 4 <= lo) continue;
        const int kk = ks * 4 + (lane >> 4);
        double a[TL::FI], b[TL::FJ];
#pragma unroll
        for (int i = 0; i < FIV; ++i) {
            a[i] = As[dtl_index<XCA, TL::BM>(kk, block_row<TL>(wm, i) + li)];
            if (TAIL) a[i] = kk >= lo ? a[i] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < FJV; ++j) {
            b[j] = Bs[dtl_index<XCB, TL::BN>(kk, block_col<TL>(wn, j) + li)];
            if (TAIL) b[j] = kk >= lo ? b[j] : 0.0;
        }
#pragma unroll
        for (int i = 0; i < FIV; ++i)
#pragma unroll
            for (int j = 0; j < FJV; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0);
    }
}

// Own loads of the stage have landed (vmcnt counts the LDS DMA) and own reads
// of the stage before it are done, then every wave's.
__device__ __forceinline__ void dtl_publish()
{
    __builtin_amdgcn_s_waitcnt(0x0070);         // vmcnt(0) lgkmcnt(0); expcnt (6:4) not waited on
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// k in [kbeg, kend) of a TL tile through a double buffer of direct-to-LDS
// stages, one in flight under the MFMAs of the other.  Needs kend >= 16
// (whatever kbeg) and kbeg, kend in scalar registers.  The k left over after
// the whole 16-deep stages are the last ones of a stage that starts at kend -
// 16 and is prefetched like the others: it reads some k a second time, which
// then count as zero.  (A separate bounds-checked stage cost a whole exposed
// load latency.)  The products are added in the order of k either way, so
// results do not depend on the path.  Ends with a barrier after which the
// buffers are free.
//
// A wave takes no part in the products of whole stages that start at kw or
// later (its operand is zero there).
//
// The two buffers of each operand must be distinct __shared__ arrays and
// the loop is unrolled by two so that every access names its array at
// compile time: the compiler then knows the LDS reads of stage z do not
// touch the buffer the DMA of stage z + 1 writes.  With one array indexed
// by the stage's parity it cannot tell, and makes the first LDS read after
// each DMA wait for it, which exposes the whole load latency every stage.
// Rings of three and four stages were slower at every size tried (8192^3
// 16.4 and 16.9 ms against 15.1): their LDS costs the second workgroup per
// CU, and other workgroups' waves hide the latency better than depth does.
template <class TL, int FIV, int FJV, class LA, class LB>
__device__ __forceinline__ void mainloop_blocks(const LA &la, const LB &lb, int64_t lda, int64_t ldb, int kbeg,
                                                int kend, double *A0, double *A1, double *B0, double *B1,
                                                f64x4 (&acc)[TL::FI][TL::FJ], int kw = INT_MAX)
{
    constexpr int XCA = LA::XC, XCB = LB::XC;
    const int nfull = (kend - kbeg) / kBK, rem = (kend - kbeg) % kBK;
    const int ns = nfull + (rem > 0);
    auto issue = [&](int z, double *SA, double *SB) __attribute__((always_inline)) {
        const int64_t k0 = min(kbeg + z * kBK, kend - kBK);
        la.issue(XCA ? k0 * lda : k0, SA);
        lb.issue(XCB ? k0 * ldb : k0, SB);
    };
    if (ns > 0) issue(0, A0, B0);
    for (int z = 0; z < nfull; z += 2) {
        dtl_publish();                              // stage z in buffer 0
        if (z + 1 < ns) issue(z + 1, A1, B1);
        if (kbeg + z * kBK < kw) stage_mfma_dtl<XCA, XCB, TL, FIV, FJV>(A0, B0, acc);
        if (z + 1 >= nfull) break;
        dtl_publish();                              // stage z + 1 in buffer 1
        if (z + 2 < ns) issue(z + 2, A0, B0);
        if (kbeg + (z + 1) * kBK < kw) stage_mfma_dtl<XCA, XCB, TL, FIV, FJV>(A1, B1, acc);
    }
    if (rem > 0) {
        dtl_publish();
        stage_mfma_dtl<XCA, XCB, TL, FIV, FJV, true>(nfull & 1 ? A1 : A0, nfull & 1 ? B1 : B0, acc, kBK - rem);
    }
    __syncthreads();
}

template <class TL, class LA, class LB>
__device__ __forceinline__ void mainloop_dtl(const LA &la, const LB &lb, int64_t lda, int64_t ldb, int kbeg, int kend,
                                             double *A0, double *A1, double *B0, double *B1,
                                             f64x4 (&acc)[TL::FI][TL::FJ], int kw = INT_MAX)
{
    mainloop_blocks<TL, TL::FI, TL::FJ>(la, lb, lda, ldb, kbeg, kend, A0, A1, B0, B1, acc, kw);
}

// The same for a tile whose blocks may lie outside C (IL): one loop per number
// of blocks, a wave's own (a branch around each MFMA would cost copies of the
// accumulators); all loops issue the same loads and barriers.
template <class TL, class LA, class LB>
__device__ __forceinline__ void mainloop_edge(const LA &la, const LB &lb, int64_t lda, int64_t ldb, int kbeg,
                                              int kend, double *A0, double *A1, double *B0, double *B1,
                                              f64x4 (&acc)[TL::FI][TL::FJ], const Blocks &in)
{
    static_assert(TL::FI == 4 && TL::FJ == 2, "the wave shape these loops are for");
    auto run = [&](auto FIV, auto FJV) __attribute__((always_inline)) {
        mainloop_blocks<TL, decltype(FIV)::value, decltype(FJV)::value>(la, lb, lda, ldb, kbeg, kend, A0, A1, B0, B1,
                                                                        acc);
    };
    using std::integral_constant;
    const integral_constant<int, 4> four{};
    const integral_constant<int, 3> three{};
    const integral_constant<int, 2> two{};
    const integral_constant<int, 1> one{};
    if (in.fi <= 0 || in.fj <= 0) run(integral_constant<int, 0>{}, integral_constant<int, 0>{});
    else if (in.fj > 1) {
        if (in.fi > 3) run(four, two);
        else if (in.fi > 2) run(three, two);
        else run(two, two);
    } else if (in.fi > 2) run(four, one);
    else run(two, one);
}

// The whole tile of acc to out, column by column (rows fastest), or added to
// what it stored there before.
template <class TL>
__device__ __forceinline__ void store_tile(double *out, const f64x4 (&acc)[TL::FI][TL::FJ], bool add = false)
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));                // no address is computed before the main loop
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave % TL::WM, wn = wave / TL::WM;
#pragma unroll
    for (int i = 0; i < TL::FI; ++i)
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j) {
            double *o = out + (block_col<TL>(wn, j) + (lane >> 4)) * TL::BM + block_row<TL>(wm, i) + (lane & 15);
            double x[4] = {0.0, 0.0, 0.0, 0.0};  // (acc, from +0 on, is never -0)
            if (add) {
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] = o[4 * r * TL::BM];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) o[4 * r * TL::BM] = ca3::add_rn(x[r], acc[i][j][r]);
        }
}

// C := fold(P) + (alpha*acc + beta*C) for the tile at (m0, n0), with the
// first nsrc partials of g.P.  ms, ns_: dtl_shift of the tile's rows and
// columns.
template <class TL>
__device__ __forceinline__ void epilogue_to(const GemmArgs &g, double *C, int64_t ldc, double alpha, double beta,
                                            int nsrc, int m0, int n0, const f64x4 (&acc)[TL::FI][TL::FJ], int ms,
                                            int ns_)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave % TL::WM, wn = wave / TL::WM;
    // opaque, so that no row, column or address below is computed before the
    // main loop and held in vector registers across it
    m0 = __builtin_amdgcn_readfirstlane(m0);
    n0 = __builtin_amdgcn_readfirstlane(n0);
    ms = __builtin_amdgcn_readfirstlane(ms);
    ns_ = __builtin_amdgcn_readfirstlane(ns_);
    asm volatile("" : "+s"(m0), "+s"(n0), "+s"(ms), "+s"(ns_));
#pragma unroll
    for (int i = 0; i < TL::FI; ++i) {
        int rt = block_row<TL>(wm, i) + (lane & 15);
        const bool rok = rt != ms && m0 + rt - (rt == ms + 1) < g.M;
        rt -= (rt == ms + 1);
        const int row = m0 + rt;
        // a block row at a time, so that its loads of C and of the partials
        // are in flight together (one by one, their latencies add up)
        bool ok[TL::FJ][4];
        int col[TL::FJ][4];
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ct = block_col<TL>(wn, j) + 4 * r + (lane >> 4);
                col[j][r] = n0 + ct - (ct == ns_ + 1);
                ok[j][r] = rok && ct != ns_ && col[j][r] < g.N;
            }
        double v[TL::FJ][4], x[TL::FJ][4];
        auto load = [&](const double *X, int64_t ldx) __attribute__((always_inline)) {
            const gdouble *Xg = (const gdouble *) X;
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) x[j][r] = ok[j][r] ? Xg[(int64_t) col[j][r] * ldx + row] : 0.0;
        };
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[j][r] = ca3::mul_rn(alpha, acc[i][j][r]);
        if (beta != 0.0) {
            load(C, ldc);
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] = ca3::add_rn(v[j][r], ca3::mul_rn(beta, x[j][r]));
        }
        if (nsrc > 0) {
            double s[TL::FJ][4];
            load(g.P[0], g.ldp[0]);
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) s[j][r] = x[j][r];
            for (int t = 1; t < nsrc; ++t) {
                load(g.P[t], g.ldp[t]);
#pragma unroll
                for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[j][r] = ca3::add_rn(s[j][r], x[j][r]);
            }
#pragma unroll
            for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] = ca3::add_rn(s[j][r], v[j][r]);
        }
#pragma unroll
        for (int j = 0; j < TL::FJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (ok[j][r]) ((gdouble *) C)[(int64_t) col[j][r] * ldc + row] = v[j][r];
    }
}

template <class TL = Tile128>
__device__ __forceinline__ void epilogue(const GemmArgs &g, int m0, int n0, const f64x4 (&acc)[TL::FI][TL::FJ],
                                         int ms = -2, int ns_ = -2)
{
    epilogue_to<TL>(g, g.C, g.ldc, g.alpha, g.beta, g.nsrc, m0, n0, acc, ms, ns_);
}

}  // namespace gemm
}  // namespace ca3
