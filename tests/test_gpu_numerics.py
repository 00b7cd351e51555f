"""Numerics of single steps at the ends of their ranges: pivot divisions near
the largest and smallest values, solves with badly conditioned triangles,
refinement over factors that are not finite."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,power", [("fp64", 1024), ("fp64", -1000), ("fp32", 128), ("fp32", -105)])
@pytest.mark.parametrize("nb", [2, 16, 17, 40, 64])
def test_diagonal_block_quotients_at_the_ends_of_the_range(S, nb, prec, power):
    """Factors of 2^power A are those of A scaled, bit for bit, with dividends
    up to the largest finite value and down to where their remainders would be
    subnormal (all entries of U below 1, those of L up to 1.1)."""
    t = np.float64 if prec == "fp64" else np.float32
    rng = np.random.default_rng(nb)
    off = np.subtract.outer(np.arange(nb), np.arange(nb))
    A = rng.uniform(0.75, 0.95, (nb, nb)) * rng.choice([-1, 1], (nb, nb))
    A = np.tril(A, -1) * np.where(off > 1, 1 / 64, 1) + np.triu(A, 1) / 256 + np.diag(rng.uniform(0.9, 0.95, nb))
    out = []
    for p in (0, power):
        h = p // 2
        D = np.asfortranarray(A.astype(t) * t(2.0 ** h) * t(2.0 ** (p - h)))
        assert np.all(np.isfinite(D))
        Li, Ui = np.zeros(4096, t), np.zeros(4096, t)
        f = S.lib().snu_test_diag_lu if prec == "fp64" else S.lib().snu_test_diag_lu_f32
        ptr = [x.ctypes.data_as(C.c_void_p) for x in (D, Li, Ui)]
        assert f(nb, ptr[0], nb, ptr[1], ptr[2]) == 0
        out.append(D)
    h = power // 2
    want = np.tril(out[0], -1) + np.triu(out[0]) * t(2.0 ** h) * t(2.0 ** (power - h))
    assert np.array_equal(out[1], want)


def _chain(S, n):
    """Diagonal 2, below it -3, above it -0.3, in a full pattern of explicit
    zeros, so that the whole matrix is one front: elimination without pivoting
    is stable (|L||U| is about |A|), but L's inverse grows as 2.3^n."""
    D = 2.0 * np.eye(n) - 3.0 * np.eye(n, k=-1) - 0.3 * np.eye(n, k=1)
    A = S.CSR(n, np.arange(0, n * n + 1, n), np.tile(np.arange(n), n), D.reshape(-1))
    LU = D.copy()
    for k in range(n - 1):
        LU[k + 1, k] /= LU[k, k]
        LU[k + 1, k + 1] -= LU[k + 1, k] * LU[k, k + 1]
    growth = np.max((np.abs(np.tril(LU, -1) + np.eye(n)) @ np.abs(np.triu(LU))).sum(1)) / 5.3
    return D, A, growth


@pytest.mark.parametrize("precision,n", [("fp64", n) for n in (16, 33, 48, 64, 65, 96, 97, 130, 200)]
                         + [("fp32", n) for n in (16, 33, 48, 64, 65, 96, 97)])
def test_solves_through_badly_conditioned_triangles(S, precision, n):
    """The backward error of substitution, 3 (order) u |L||U| / |A| at most,
    whatever the condition of the triangles: one column, one group of columns
    and more than one.  FP32: of the first iterate, A's and b's rounding added
    (ir_max_steps < 0: no step, the scratch solve leaves it in x)."""
    D, A, growth = _chain(S, n)
    u = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    bar = (3 * n * growth + 2) * u
    X = np.asfortranarray(np.random.default_rng(n).uniform(-1, 1, (n, 17)))
    B = np.asfortranarray(D @ X)
    with S.SnuMat(A, 1, order=np.arange(n), sizes=[n], device=0, precision=precision, ir_max_steps=-1) as M:
        M.factorize()
        for k in (1, 2, 17):
            d_b, d_x = S.DeviceBuffer(8 * n * k), S.DeviceBuffer(8 * n * k)
            d_b.upload(B[:, :k])
            rc = S.lib().snumat_solve_device_scratch(M._h, d_b.ptr, d_x.ptr, k, n)
            assert rc == 0 or precision == "fp32"  # (not converged)
            x = np.zeros((n, k), order="F")
            d_x.download(x)
            d_b.free()
            d_x.free()
            for c in range(k):
                assert S.backward_error(A, x[:, c], B[:, c]) <= bar, (k, c)


def test_refinement_of_solutions_that_are_not_finite(S):
    """FP32 factors that overflow give solutions of NaNs: on the device-pointer
    paths too they are answered by FP64 factors, or reported.  A right-hand side
    that is itself not finite is left as it is and does not ask for them."""
    rng = np.random.default_rng(1)
    A = S.gen_grid(20, 19, 1, 5, 0, 4.1, 1)
    A.data = A.data * 1e39  # diagonal beyond FP32
    n = A.n
    for k in (1, 3):
        B = np.asfortranarray(rng.uniform(-1, 1, (n, k)) * 1e39)
        with S.SnuMat(A, 4, grid=(20, 19, 1), device=0, precision="fp32", ir_tol=1e-12) as M:
            M.factorize()
            d_b, d_x = S.DeviceBuffer(8 * n * k), S.DeviceBuffer(8 * n * k)
            d_b.upload(B)
            x = np.zeros((n, k), order="F")

            def check():
                d_x.download(x)
                assert S.backward_error(A, x, B) <= 1e-12

            assert S.lib().snumat_solve_device_scratch(M._h, d_b.ptr, d_x.ptr, k, n) == -10
            M.solve_device_ptr(d_b.ptr.value, d_x.ptr.value, k)
            assert M.timings()["fp64_fallback"] == 1
            check()
            with S.Batch([M]) as batch:
                assert S.backward_error(A, np.asarray(batch.solve([B])[0]).reshape(n, k), B) <= 1e-12
                assert batch.timings()["fp64_fallbacks"] == 1
            d_b.free()
            d_x.free()
    A = S.gen_grid(20, 19, 1, 5, 0, 4.1, 1)
    B = np.asfortranarray(rng.uniform(-1, 1, (n, 3)))
    for bad in (np.nan, np.inf):
        B[5, 1] = bad
        with S.SnuMat(A, 4, grid=(20, 19, 1), device=0, precision="fp32", ir_tol=1e-12) as M:
            M.factorize()
            d_b, d_x = S.DeviceBuffer(8 * n * 3), S.DeviceBuffer(8 * n * 3)
            d_b.upload(B)
            M.solve_device_ptr(d_b.ptr.value, d_x.ptr.value, 3)
            assert M.timings()["fp64_fallback"] == 0
            x = np.zeros((n, 3), order="F")
            d_x.download(x)
            assert not np.all(np.isfinite(x[:, 1]))
            for c in (0, 2):
                assert S.backward_error(A, x[:, c], B[:, c]) <= 1e-12
            d_b.free()
            d_x.free()


def test_introspection_without_an_output(S):
    """A null output is refused, not written to."""
    A = S.gen_grid(12, 11, 1, 5, 0, 4.1, 1)
    for precision in ("fp64", "fp32"):
        with S.SnuMat(A, 2, grid=(12, 11, 1), device=0, precision=precision) as M:
            for stage in (0, 2):
                S._check(S.lib().snumat_factorize_stage(M._h, stage))
                assert S.lib().snumat_leaf_values(M._h, 0, None) == -1
            assert S.lib().snumat_sep_diag(M._h, 1, None) == -1


GRIDS = [((9, 9, 9), 27, 1), ((13, 7, 5), 7, 2), ((31, 23, 1), 9, 4), ((17, 16, 1), 5, 1), ((11, 10, 8), 27, 8),
         ((24, 23, 22), 7, 8)]
DIAG = {5: 4.1, 9: 8.1, 7: 6.1, 27: 0.0}


def test_fp32_sweeps_without_refinement_or_fallback(S):
    """FP32 sweeps on their own, where neither refinement nor the FP64 twin can
    make up for a wrong one: the first iterate within 2 m u of the right-hand
    side (m: the largest order of a dense block, growth at most 2: diagonally
    dominant), then convergence in two steps at most and no fallback, for column
    counts at the edges of the groups; as a batch too."""
    u = 2.0 ** -24
    mats, bs = [], []
    for (dims, st, np_), kb in zip(GRIDS, (1, 17, 2, 16, 33, 3)):
        A = S.gen_grid(*dims, st, 1 if st == 27 else 0, DIAG[st], 3)
        order, sizes = S.order_grid(*dims, np_)
        B = np.asfortranarray(np.random.default_rng(5).standard_normal((A.n, 65)))
        args = dict(order=order, sizes=sizes, device=0, precision="fp32", ir_tol=1e-12)
        m = 0
        with S.SnuMat(A, np_, ir_max_steps=-1, **args) as M:
            M.factorize()
            m = max([int(np.max(F["f"])) for F in (M.leaf_fronts(r) for r in range(np_))] + [int(s) for s in sizes[np_:]])
            d_b, d_x = S.DeviceBuffer(B.nbytes), S.DeviceBuffer(B.nbytes)
            d_b.upload(B)
            for k in (1, 2, 15, 16, 17, 33, 64, 65):
                rc = S.lib().snumat_solve_device_scratch(M._h, d_b.ptr, d_x.ptr, k, A.n)
                assert rc in (0, -10)
                x = np.zeros((A.n, 65), order="F")
                d_x.download(x)
                err = S.backward_error(A, x[:, :k], B[:, :k])
                print("case", dims, st, "columns", k, "order", m, "error / u", err / u, flush=True)
                assert err <= 2 * m * u
            d_b.free()
            d_x.free()
        M = S.SnuMat(A, np_, **args)
        M.factorize()
        for k in (1, 2, 16, 33):
            x = M.solve(B[:, :k])
            t = M.timings()
            assert t["fp64_fallback"] == 0 and t["ir_steps"] <= 2
            assert S.backward_error(A, x, B[:, :k]) <= 1e-12
        mats.append(M)
        bs.append(B[:, :kb])
    with S.Batch(mats) as batch:
        batch.factorize()
        for M, b, x in zip(mats, bs, batch.solve(bs)):
            assert S.backward_error(M.A, np.asarray(x).reshape(b.shape), b) <= 1e-12
        t = batch.timings()
        assert t["fp64_fallbacks"] == 0 and t["ir_steps"] <= 2
    for M in mats:
        M.close()


@pytest.mark.parametrize("precision,n", [("fp64", 20), ("fp64", 64), ("fp32", 20), ("fp32", 96)])
def test_solves_divide_by_pivots_of_any_size(S, precision, n):
    """x = b / d within an ulp for diagonal matrices (in a full pattern: one
    front factored in LDS; larger ones' panels take the inverses of their pivot
    blocks, which overflow for subnormal pivots) whose pivots go from subnormal
    to the largest values, with no clamp; FP32: the first iterate."""
    f64 = precision == "fp64"
    t, lo, hi, u = (np.float64, -1070, 1022, 2.0 ** -52) if f64 else (np.float32, -145, 126, 2.0 ** -23)
    rng = np.random.default_rng(n)
    d = np.ldexp(rng.uniform(0.5, 1, n), np.linspace(lo, hi, n).astype(int)).astype(t) * rng.choice([-1, 1], n).astype(t)
    q = rng.uniform(0.5, 1, (n, 17))
    B = (q * d[:, None].astype(np.float64)).astype(t)  # (representable; subnormal where d is)
    want = B.astype(np.float64) / d[:, None].astype(np.float64)
    A = S.CSR(n, np.arange(0, n * n + 1, n), np.tile(np.arange(n), n), np.diag(d).astype(np.float64).reshape(-1))
    B = np.asfortranarray(B.astype(np.float64))
    with S.SnuMat(A, 1, order=np.arange(n), sizes=[n], device=0, precision=precision, eps=0.0, ir_max_steps=-1) as M:
        M.factorize()
        for k in (1, 2, 17):
            d_b, d_x = S.DeviceBuffer(8 * n * k), S.DeviceBuffer(8 * n * k)
            d_b.upload(B[:, :k])
            rc = S.lib().snumat_solve_device_scratch(M._h, d_b.ptr, d_x.ptr, k, n)
            assert rc == 0 or not f64
            x = np.zeros((n, k), order="F")
            d_x.download(x)
            d_b.free()
            d_x.free()
            assert np.all(np.abs(x - want[:, :k]) <= u * np.abs(want[:, :k]))
