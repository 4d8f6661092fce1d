"""The work a user of this library has it do, as timed cases.

Every case goes through a public entry point, on device matrices that the
caller owns (column-major FP64, here held in torch tensors of the transposed
shape) and with the library's default settings, under which an entry has
finished when it returns.  The kinds of case:

  gemm    one product through hip_dgemm: what a rank's Cannon round calls
  engine  one product through ca3dmm_engine_exec on an engine kept across calls
  btb     C = B^T B through the B^T B engine
  cholqr  A = Q R of a tall-skinny A through hip_cholesky_qr (in place, so A is
          copied first, as a program does that still needs A)
  grid    a whole exec of the simulated p-rank grid from 1D column layouts
  ozaki   one product through the CRT form, the modulus count chosen per
          product from the operands
  move    a redistribution of a matrix into 2D blocks and the sum of kp
          partial blocks of C

The problem classes of the engine cases are those that CA3DMM is built for:
square, large-K, large-M and flat.
"""
import ctypes as C
import math

import numpy as np
import torch

from ca3dmm_amd import device as hip
from ca3dmm_amd import engine as E

F64 = torch.float64


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest local products (a rank's share of a small problem on many ranks): latency
        {"name": "gemm_smallest", "kind": "gemm", "m": 61, "n": 47, "k": 53, "ta": 0, "tb": 0},
        # one rank's product of the 2000^3 example on 4 ranks (grid 2 x 1 x 2)
        {"name": "gemm_rank_share", "kind": "gemm", "m": 1000, "n": 2000, "k": 1000, "ta": 0, "tb": 0},
        # square: the headline product, with A transposed
        {"name": "engine_square", "kind": "engine", "m": 8192, "n": 8192, "k": 8192, "ta": 1, "tb": 0},
        # large-K: a small C summed over a long k (6000 x 6000 x 1.2e6 at a tenth of each size)
        {"name": "engine_large_k", "kind": "engine", "m": 600, "n": 600, "k": 120000, "ta": 0, "tb": 0},
        # large-M: a tall operand times a small one, B transposed
        {"name": "engine_large_m", "kind": "engine", "m": 120000, "n": 600, "k": 600, "ta": 0, "tb": 1},
        # flat: a large C from a short k (1e5 x 1e5 x 5000 at a tenth of each size)
        {"name": "engine_flat", "kind": "engine", "m": 10000, "n": 10000, "k": 500, "ta": 0, "tb": 0},
        # the Gram matrix of a tall-skinny block through the engine the CholeskyQR example uses
        {"name": "btb_tall", "kind": "btb", "n": 1000, "k": 200000},
        # CholeskyQR2 of a very tall block of vectors
        {"name": "cholqr_tall", "kind": "cholqr", "m": 2000000, "n": 512, "variant": 2},
        # CholeskyQR of a wider block with odd sizes, the variant chosen by the library
        {"name": "cholqr_wide", "kind": "cholqr", "m": 30011, "n": 1999, "variant": 0},
        # 8000^3 on 24 ranks (grid 4 x 2 x 3): redistributions, allgathers, Cannon rounds, k-layer sum
        {"name": "grid_24_ranks", "kind": "grid", "m": 8000, "n": 8000, "k": 8000, "p": 24},
        # an FP64-accurate product on the INT8 matrix cores, entries of moderate spread, odd sizes
        {"name": "ozaki_auto", "kind": "ozaki", "m": 5000, "n": 3001, "k": 4001, "ta": 0, "tb": 1, "phi": 2.0},
        # an 8000 x 8000 matrix redistributed into 4 x 6 blocks, and the sum of 3 layers' 2000 x 4000 blocks
        {"name": "move_blocks", "kind": "move", "m": 8000, "n": 8000, "gm": 4, "gn": 6, "kp": 3, "bm": 2000,
         "bn": 4000},
    ]


def _size(rng, lo, hi):
    """A size spread over its logarithm; a quarter of them round, the others as they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.25:
        step = 8 if v < 256 else 64
        v = max(lo, v // step * step)
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "engine", "engine", "engine", "btb", "cholqr", "grid", "ozaki", "move"])
    if kind == "gemm":
        hi = rng.choice([128, 600, 2000])
        return {"kind": kind, "m": _size(rng, 16, hi), "n": _size(rng, 16, hi), "k": _size(rng, 16, hi),
                "ta": rng.randrange(2), "tb": rng.randrange(2)}
    if kind == "engine":
        shape = rng.choice(["square", "large_k", "large_m", "flat"])
        if shape == "square":
            s = _size(rng, 500, 7000)
            m, n, k = (max(400, int(s * rng.uniform(0.8, 1.15))) for _ in range(3))
        elif shape == "large_k":
            m, n, k = _size(rng, 100, 2000), _size(rng, 100, 2000), _size(rng, 10000, 120000)
        elif shape == "large_m":
            m, n, k = _size(rng, 10000, 120000), _size(rng, 100, 2000), _size(rng, 100, 2000)
        else:
            m, n, k = _size(rng, 2000, 10000), _size(rng, 2000, 10000), _size(rng, 100, 1000)
        return {"kind": kind, "m": m, "n": n, "k": k, "ta": rng.randrange(2), "tb": rng.randrange(2)}
    if kind == "btb":
        return {"kind": kind, "n": _size(rng, 64, 2000), "k": _size(rng, 5000, 200000)}
    if kind == "cholqr":
        n = _size(rng, 32, 2048)
        return {"kind": kind, "m": _size(rng, 4 * n, min(2000000, 500000000 // n)), "n": n,
                "variant": rng.choice([0, 2, 3])}
    if kind == "grid":
        s = _size(rng, 600, 7500)
        m, n, k = (int(s * rng.uniform(0.75, 1.05)) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k, "p": rng.choice([2, 4, 6, 8, 12, 16, 24])}
    if kind == "ozaki":
        return {"kind": kind, "m": _size(rng, 128, 6000), "n": _size(rng, 128, 6000), "k": _size(rng, 128, 6000),
                "ta": rng.randrange(2), "tb": rng.randrange(2), "phi": rng.choice([0.5, 2.0, 4.0])}
    return {"kind": kind, "m": _size(rng, 200, 8000), "n": _size(rng, 200, 8000), "gm": rng.randint(1, 6),
            "gn": rng.randint(1, 6), "kp": rng.randint(2, 6), "bm": _size(rng, 100, 4000), "bn": _size(rng, 100, 4000)}


# ---------------------------------------------------------------------------
# device matrices
# ---------------------------------------------------------------------------
class Mat:
    """A column-major nrow x ncol device matrix over a torch tensor of shape (ncol, nrow)."""

    def __init__(self, t):
        self.t = t
        self.shape = (t.shape[1], t.shape[0])
        self.ptr = t.data_ptr()

    def at(self, elems):
        return self.ptr + 8 * int(elems)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, nrow, ncol):
    return Mat(torch.rand((ncol, nrow), generator=g, dtype=F64, device="cuda").mul_(2.0).sub_(1.0))


def _empty(nrow, ncol):
    return Mat(torch.empty((ncol, nrow), dtype=F64, device="cuda"))


def _operands(c, g):
    m, n, k = c["m"], c["n"], c["k"]
    A = _uniform(g, k, m) if c["ta"] else _uniform(g, m, k)
    B = _uniform(g, n, k) if c["tb"] else _uniform(g, k, n)
    return A, B


def _phi_operands(c, g):
    """uniform[-0.5, 0.5] * exp(phi * N(0, 1))"""
    out = []
    for M in _operands(c, g):
        s = torch.randn(M.t.shape, generator=g, dtype=F64, device="cuda").mul_(c["phi"]).exp_()
        out.append(Mat(M.t.mul_(0.5).mul_(s)))
    return out


def _tall(c, g):
    """m x n with singular values from about 1 to 1e-4: Gaussian columns,
    reflected, scaled and reflected again."""
    m, n = c["m"], c["n"]
    t = torch.randn((n, m), generator=g, dtype=F64, device="cuda")
    for r in range(2):
        v = torch.randn((n, 1), generator=g, dtype=F64, device="cuda")
        v /= v.norm()
        t.addmm_(v, v.t() @ t, alpha=-2.0)
        if r == 0:
            t.mul_(torch.logspace(0, -4, n, dtype=F64, device="cuda")[:, None])
    return Mat(t.mul_(m ** -0.5))


def _cuts(length, parts):
    return [length * i // parts for i in range(parts + 1)]


def _columns(nrow, ncol, p):
    """1D column layout over p ranks: {srow, nrow, scol, ncol} blocks."""
    at = _cuts(ncol, p)
    return [(0, nrow, at[r], at[r + 1] - at[r]) for r in range(p)]


class Engine:
    """A ca3dmm engine of the single-process group, freed with this object."""

    def __init__(self, c):
        self.h = E.CA3P()
        if c["kind"] == "btb":
            n, k = c["n"], c["k"]
            E.lib.ca3dmm_engine_init_BTB(n, k, 0, k, 0, n, 0, n, 0, n, None, E.comm_self(), E.DEV_TYPE_HIP,
                                         C.byref(self.h), None)
        else:
            m, n, k = c["m"], c["n"], c["k"]
            ar, ac = (k, m) if c["ta"] else (m, k)
            br, bc = (n, k) if c["tb"] else (k, n)
            E.lib.ca3dmm_engine_init(m, n, k, c["ta"], c["tb"], 0, ar, 0, ac, 0, br, 0, bc, 0, m, 0, n, None,
                                     E.comm_self(), E.DEV_TYPE_HIP, C.byref(self.h), None)
        if not self.h:
            raise RuntimeError("engine init failed")

    def exec(self, A, B, Cm):
        E.lib.ca3dmm_engine_exec(self.h, A.ptr if A else None, A.shape[0] if A else 1, B.ptr, B.shape[0], Cm.ptr,
                                 Cm.shape[0])

    def __del__(self):
        if self.h:
            E.lib.ca3dmm_engine_free(C.byref(self.h))


# ---------------------------------------------------------------------------
# preparation, pass, work, reference values
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, g = dict(case), _gen(seed)
    kind = c["kind"]
    if kind in ("gemm", "engine"):
        c["A"], c["B"] = _operands(c, g)
        c["C"] = _empty(c["m"], c["n"])
        if kind == "engine":
            c["engine"] = Engine(c)
    elif kind == "btb":
        c["B"] = _uniform(g, c["k"], c["n"])
        c["C"] = _empty(c["n"], c["n"])
        c["engine"] = Engine(c)
    elif kind == "cholqr":
        c["A"] = _tall(c, g)
        c["Q"], c["R"] = _empty(c["m"], c["n"]), _empty(c["n"], c["n"])
    elif kind == "grid":
        m, n, k, p = c["m"], c["n"], c["k"], c["p"]
        c["A"], c["B"], c["C"] = _uniform(g, m, k), _uniform(g, k, n), _empty(m, n)
        la, lb, lc = _columns(m, k, p), _columns(k, n, p), _columns(m, n, p)
        c["grid"] = E.SimGrid(p, m, n, k, 0, 0, la, lb, lc)
        c["args"] = ([c["A"].at(r[2] * m) for r in la], [m] * p, [c["B"].at(r[2] * k) for r in lb], [k] * p,
                     [c["C"].at(r[2] * m) for r in lc], [m] * p)
    elif kind == "ozaki":
        c["A"], c["B"] = _phi_operands(c, g)
        c["C"] = _empty(c["m"], c["n"])
    else:
        m, n = c["m"], c["n"]
        c["X"] = _uniform(g, m, n)
        c["Y"] = torch.empty(m * n, dtype=F64, device="cuda")
        rows, cols, blocks, at = _cuts(m, c["gm"]), _cuts(n, c["gn"]), [], 0
        for j in range(c["gn"]):
            for i in range(c["gm"]):
                br, bc = rows[i + 1] - rows[i], cols[j + 1] - cols[j]
                # a block's columns are the rows of the row-major copy
                blocks.append((c["X"].at(cols[j] * m + rows[i]), m, c["Y"].data_ptr() + 8 * at, br, bc, br))
                at += br * bc
        c["blocks"] = blocks
        c["parts"] = [_uniform(g, c["bm"], c["bn"]) for _ in range(c["kp"])]
        c["S"] = _empty(c["bm"], c["bn"])
    return c


def run(state):
    c = state
    kind = c["kind"]
    if kind == "gemm":
        hip.dgemm(c["ta"], c["tb"], c["m"], c["n"], c["k"], 1.0, c["A"], c["B"], 0.0, c["C"])
        return c["C"].t
    if kind in ("engine", "btb"):
        c["engine"].exec(c.get("A"), c["B"], c["C"])
        return c["C"].t
    if kind == "cholqr":
        m, n = c["m"], c["n"]
        hip.copy_matrix_block(8, n, m, c["A"].ptr, m, c["Q"].ptr, m)
        info, passes = hip.cholesky_qr(m, n, c["Q"], c["R"], variant=c["variant"])
        if info:
            raise RuntimeError(f"breakdown at {info} in pass {passes + 1}")
        return {"Q": c["Q"].t, "R": c["R"].t, "passes": passes}
    if kind == "grid":
        c["grid"].exec(*c["args"])
        return c["C"].t
    if kind == "ozaki":
        ta, tb, m, n, k = c["ta"], c["tb"], c["m"], c["n"], c["k"]
        _, moduli = hip.ozaki_choose(ta, tb, m, n, k, c["A"], c["B"])
        hip.ozaki2_dgemm(ta, tb, m, n, k, 1.0, c["A"], c["B"], 0.0, c["C"], moduli)
        return {"C": c["C"].t, "moduli": moduli}
    hip.copy_blocks(8, c["blocks"])
    hip.fold_sum(c["parts"], c["bm"], c["bn"], c["S"])
    return {"Y": c["Y"], "S": c["S"].t}


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("gemm", "engine", "grid", "ozaki"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 8.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    if kind == "btb":
        n, k = c["n"], c["k"]
        return {"bytes": 8.0 * (n * k + n * n), "flops": 1.0 * n * (n + 1) * k}
    if kind == "cholqr":
        # Gram and triangular solve of two passes; A read, Q and R written
        m, n = c["m"], c["n"]
        return {"bytes": 8.0 * (2 * m * n + n * n), "flops": 2.0 * (n * (n + 1.0) * m + 1.0 * m * n * n)}
    mn, bb = c["m"] * c["n"], c["bm"] * c["bn"]
    return {"bytes": 16.0 * mn + 8.0 * (c["kp"] + 1) * bb, "flops": 1.0 * (c["kp"] - 1) * bb}


def _product(c, A, B):
    """(op(A) op(B))^T from the transposed tensors."""
    return (B.t.t() if c.get("tb") else B.t) @ (A.t.t() if c.get("ta") else A.t)


def exact(case, seed):
    c, g = dict(case), _gen(seed)
    kind = c["kind"]
    if kind in ("gemm", "engine"):
        return _product(c, *_operands(c, g))
    if kind == "grid":
        A, B = _uniform(g, c["m"], c["k"]), _uniform(g, c["k"], c["n"])
        return _product(c, A, B)
    if kind == "ozaki":
        return {"C": _product(c, *_phi_operands(c, g)), "moduli": None}
    if kind == "btb":
        B = _uniform(g, c["k"], c["n"]).t
        return B @ B.t()
    if kind == "cholqr":
        Q = _tall(c, g).t
        R = np.eye(c["n"])
        for _ in range(3):
            S = np.linalg.cholesky((Q @ Q.t()).cpu().numpy())      # lower: R_pass^T
            Q = torch.from_numpy(np.linalg.inv(S)).cuda() @ Q
            R = S.T @ R
        # (Q, R) laid out as the column-major results are: transposed
        return {"Q": Q, "R": torch.from_numpy(np.ascontiguousarray(R.T)), "passes": None}
    X = _uniform(g, c["m"], c["n"]).t
    rows, cols = _cuts(c["m"], c["gm"]), _cuts(c["n"], c["gn"])
    Y = torch.cat([X[cols[j]:cols[j + 1], rows[i]:rows[i + 1]].reshape(-1)
                   for j in range(c["gn"]) for i in range(c["gm"])])
    S = None
    for _ in range(c["kp"]):
        P = _uniform(g, c["bm"], c["bn"]).t
        S = P if S is None else S + P
    return {"Y": Y, "S": S}
