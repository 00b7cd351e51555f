"""The work this library is used for, as timed cases.

Every case is a factor-and-solve workload on grid operators (5- and 9-point in
2D, 7- and 27-point in 3D) through the public entry points: resident-factor
solves, numeric factorizations followed by a solve, value updates on a fixed
pattern, many matrices as one batch, and packed solves of uneven column counts
as a server forms them.  Precisions are FP64 (the default) and FP32 factors
refined in FP64 to a backward error of 1e-12.

Matrix values are rounded to multiples of 2^-20 and solutions to multiples of
2^-16, so b = A x holds without rounding and x is the exact solution.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import snusolver_amd as S

IR_TOL = 1e-12  # backward error asked of the FP32 factorizations
DIAG = {5: 4.1, 9: 8.1, 7: 6.1, 27: 0.0}  # the generator's diagonal (27-point: from its row sums)


def listed():
    return [
        # smallest calls: a 400-row system whose factors are resident, then the
        # whole factorize + solve (latency and launch counts)
        dict(name="solve_2d5_20", op="solve", nx=20, ny=20, nz=1, stencil=5, np=4, order="grid",
             precision="fp64", nrhs=1),
        dict(name="factor_2d5_20", op="factor", nx=20, ny=20, nz=1, stencil=5, np=4, order="grid",
             precision="fp64", nrhs=1),
        # ordinary: host arrays in and out, a few columns, a ragged 2D grid
        dict(name="host_2d9_129x115", op="host", nx=129, ny=115, nz=1, stencil=9, np=8, order="grid",
             precision="fp32", nrhs=3),
        # ordinary: time stepping, new values on the same 2D pattern each step
        dict(name="update_2d5_511x389", op="update", nx=511, ny=389, nz=1, stencil=5, np=128, order="grid",
             precision="fp64", nrhs=1),
        # ordinary: a ragged 3D grid factorized and solved
        dict(name="factor_3d7_45x37x29", op="factor", nx=45, ny=37, nz=29, stencil=7, np=32, order="grid",
             precision="fp64", nrhs=1),
        # the benchmark's operator: 64^3, graph nested dissection, 128 leaves;
        # repeated solves with resident factors, and its factorize + solve step
        dict(name="solve_3d7_64", op="solve", nx=64, ny=64, nz=64, stencil=7, np=128, order="nd",
             precision="fp64", nrhs=1),
        dict(name="factor_3d7_64", op="factor", nx=64, ny=64, nz=64, stencil=7, np=128, order="nd",
             precision="fp64", nrhs=1),
        # several right-hand sides at once on a denser stencil
        dict(name="solve16_3d27_48", op="solve", nx=48, ny=48, nz=48, stencil=27, np=64, order="grid",
             precision="fp64", nrhs=16),
        # many right-hand sides on a large 2D grid, FP32 factors refined
        dict(name="solve64_2d5_1000", op="solve", nx=1000, ny=1000, nz=1, stencil=5, np=512, order="grid",
             precision="fp32", nrhs=64),
        # large: anisotropic 27-point operator, FP32 factors refined
        dict(name="factor_3d27_56", op="factor", nx=56, ny=56, nz=56, stencil=27, np=64, order="grid",
             precision="fp32", nrhs=1),
        # many 2D matrices of uneven sizes factorized and solved as one batch
        dict(name="batch_2d9_96", op="batch", count=96, lo=16, hi=192, stencil=9, precision="fp64", nrhs=1),
        # what a server packs: a few resident matrices, 2^k columns each
        dict(name="pack_3d7_2d5_6", op="pack", count=6, lo=30, hi=48, lo2=256, hi2=512, precision="fp32",
             kmax=6),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["solve", "solve", "factor", "factor", "update", "host", "batch", "pack"])
    precision = rng.choice(["fp64", "fp32"])
    if op == "batch":
        return dict(op=op, count=log(4, 96), lo=rng.randint(16, 40), hi=rng.randint(60, 180), stencil=9,
                    precision=precision, nrhs=rng.randint(1, 3))
    if op == "pack":
        return dict(op=op, count=rng.randint(2, 6), lo=rng.randint(12, 24), hi=rng.randint(26, 44),
                    lo2=rng.randint(32, 128), hi2=rng.randint(160, 480), precision=precision,
                    kmax=rng.randint(1, 6))
    stencil = rng.choice([5, 9, 7, 27])
    if stencil in (5, 9):
        n = log(400, 400000)
        nx = max(4, int(math.sqrt(n) * rng.uniform(0.7, 1.4)))
        dims = (nx, max(4, n // nx), 1)
    else:
        n = log(400, 160000 if stencil == 7 else 60000)
        nx = max(4, int(n ** (1 / 3) * rng.uniform(0.8, 1.25)))
        ny = max(4, int(math.sqrt(n / nx) * rng.uniform(0.8, 1.25)))
        dims = (nx, ny, max(4, n // (nx * ny)))
    n = dims[0] * dims[1] * dims[2]
    np_ = max(1 if n < 3000 else 2, S.batch_np(n, rng.choice([1024, 2048])))
    nrhs = log(1, 64) if op == "solve" else rng.choice([1, 1, 2, 7])
    return dict(op=op, nx=dims[0], ny=dims[1], nz=dims[2], stencil=stencil, np=np_,
                order="nd" if n <= 60000 and rng.random() < 0.4 else "grid", precision=precision, nrhs=nrhs)


def _members(case):
    """(nx, ny, nz, stencil, np, nrhs) of every matrix of the case (sizes and
    column counts are the case's alone, values the seed's)."""
    if case["op"] not in ("batch", "pack"):
        return [(case["nx"], case["ny"], case["nz"], case["stencil"], case["np"], case["nrhs"])]
    rng = np.random.default_rng(case["count"])
    out = []
    for i in range(case["count"]):
        if case["op"] == "batch":  # sides log-uniform, one leaf per 2048 rows
            d = int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))))
            out.append((d, d, 1, 9, S.batch_np(d * d), case["nrhs"]))
        else:
            two = i % 2
            d = int(rng.integers(case["lo2" if two else "lo"], case["hi2" if two else "hi"] + 1))
            n = d * d if two else d ** 3
            out.append((d, d, 1 if two else d, 5 if two else 7, S.batch_np(n), 1 << int(rng.integers(0, case["kmax"] + 1))))
    return out


def _solutions(case, seed):
    """The exact solutions, one n x nrhs column-major array per matrix."""
    rng = np.random.default_rng([int(seed), 1])
    out = []
    for nx, ny, nz, _, _, k in _members(case):
        x = rng.integers(-65536, 65536, size=(k, nx * ny * nz)).astype(np.float64) / 65536.0
        out.append(x.T)
    return out


def _matrix(nx, ny, nz, stencil, seed):
    A = S.gen_grid(nx, ny, nz, stencil, 1 if stencil == 27 else 0, DIAG[stencil], seed)
    A.data = np.round(A.data * 1048576.0) / 1048576.0
    return A


@functools.lru_cache(maxsize=32)
def _ordering(nx, ny, nz, stencil, np_, kind):
    """Depends on the pattern alone: a program keeps it over many matrices."""
    if kind == "grid":
        return S.order_grid(nx, ny, nz, np_)
    return S.order_nd(_matrix(nx, ny, nz, stencil, 0), np_, 0)


def prepare(case, seed):
    rng = np.random.default_rng([int(seed), 2])
    mats, bs = [], []
    for (nx, ny, nz, stencil, np_, k), x in zip(_members(case), _solutions(case, seed)):
        A = _matrix(nx, ny, nz, stencil, int(rng.integers(1 << 30)))
        order, sizes = _ordering(nx, ny, nz, stencil, np_, case.get("order", "grid"))
        mats.append(S.SnuMat(A, np_, order=order, sizes=sizes, device=0, precision=case["precision"],
                             ir_tol=IR_TOL))
        bs.append(np.stack([A.matvec(x[:, j]) for j in range(k)]).T)
    s = {"op": case["op"], "mats": mats, "nrhs": [b.shape[1] for b in bs]}
    if case["op"] == "host":
        s["b"] = bs[0]
    else:  # right-hand sides and solutions resident in HBM, matrix after matrix
        s["b"] = torch.from_numpy(np.concatenate([b.T.reshape(-1) for b in bs])).cuda()
        s["x"] = torch.zeros_like(s["b"])
    if case["op"] in ("batch", "pack"):
        m = len(mats)
        s["batch"] = S.Batch(mats)
        off = np.concatenate([[0], np.cumsum([b.size for b in bs])])
        s["pb"] = (ctypes.c_void_p * m)(*[s["b"].data_ptr() + 8 * int(o) for o in off[:-1]])
        s["px"] = (ctypes.c_void_p * m)(*[s["x"].data_ptr() + 8 * int(o) for o in off[:-1]])
        s["cn"] = (ctypes.c_int * m)(*s["nrhs"])
        s["ld"] = (ctypes.c_int * m)(*[b.shape[0] for b in bs])
    if case["op"] in ("solve", "host"):
        mats[0].factorize()
    if case["op"] == "pack":
        s["batch"].factorize()
    if case["op"] == "update":
        s["values"] = mats[0].A.data
    torch.cuda.synchronize()
    return s


def run(state):
    op, mats = state["op"], state["mats"]
    if op == "host":
        return mats[0].solve(state["b"])
    if op in ("batch", "pack"):
        B = state["batch"]
        if op == "batch":
            B.factorize()
        S._check(S.lib().snubatch_solve_device(B._h, state["pb"], state["px"], state["cn"], state["ld"]))
        return state["x"]
    if op == "update":
        mats[0].update_values(state["values"])
    if op in ("factor", "update"):
        mats[0].factorize()
    mats[0].solve_device_ptr(state["b"].data_ptr(), state["x"].data_ptr(), state["nrhs"][0])
    return state["x"]


def exact(case, seed):
    xs = _solutions(case, seed)
    if case["op"] == "host":
        return xs[0]
    return np.concatenate([x.T.reshape(-1) for x in xs])


def work(case):
    """Nested dissection's growth with the unknowns n, in round figures: factor
    entries (L and U) about 4.5 n log2 n in 2D and 12 n^(4/3) in 3D, products of
    the factorization 10 n^1.5 and 10 n^2.  A factorization reads A and writes
    the factors once; a solve reads them once and does two flops per entry and
    column."""
    size = 8 if case["precision"] == "fp64" else 4
    bytes_, flops = 0.0, 0.0
    for nx, ny, nz, stencil, _, k in _members(case):
        n = nx * ny * nz
        entries = 12.0 * n ** (4 / 3) if nz > 1 else 4.5 * n * max(1.0, math.log2(n))
        if case["op"] in ("factor", "update", "batch"):
            bytes_ += 12.0 * stencil * n + size * entries
            flops += 10.0 * (n ** 2 if nz > 1 else n ** 1.5)
        bytes_ += size * entries + 16.0 * n * k
        flops += 2.0 * entries * k
    return {"bytes": bytes_, "flops": flops}
