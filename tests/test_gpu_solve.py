"""The solve sweeps over the leaf fronts and the 16-column dense products
against a dense FP64 solve (numpy), through the C-ABI.

Column counts sit at the edges of the column groups (1; 2, 15, 16, 17; 33, 64,
65).  The matrices put fronts on both sides of the LDS order, with pivot counts
around multiples of 16 and 64 (a one-leaf 27-point cube has pivot blocks beyond
64; a one-leaf 2D grid has only small fronts), one leaf and several, and
separators of a few rows.  Bars: those of the path, x within 1e-9 and backward
error <= 1e-12.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [((9, 9, 9), 27, 1), ((13, 7, 5), 7, 2), ((31, 23, 1), 9, 4), ((17, 16, 1), 5, 1), ((11, 10, 8), 27, 8)]
DIAG = {5: 4.1, 9: 8.1, 7: 6.1, 27: 0.0}


def _matrix(S, dims, stencil, seed):
    return S.gen_grid(*dims, stencil, 1 if stencil == 27 else 0, DIAG[stencil], seed)


def _dense(A):
    D = np.zeros((A.n, A.n))
    D[np.repeat(np.arange(A.n), np.diff(A.rowptr)), A.colidx] = A.data
    return D


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,stencil,np_", GRIDS)
def test_column_counts_vs_dense(S, precision, dims, stencil, np_):
    A = _matrix(S, dims, stencil, 3)
    rng = np.random.default_rng(5)
    B = np.asfortranarray(rng.standard_normal((A.n, 65)))
    X = np.linalg.solve(_dense(A), B)
    with S.SnuMat(A, np_, grid=dims, device=0, precision=precision, ir_tol=1e-12) as M:
        M.factorize()
        for k in (1, 2, 15, 16, 17, 33, 64, 65, 1):
            print("case", precision, dims, "columns", k, flush=True)
            x = M.solve(B[:, :k])
            assert np.max(np.abs(x - X[:, :k])) <= 1e-9 * np.max(np.abs(X[:, :k]))
            assert S.backward_error(A, x, B[:, :k]) <= 1e-12


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_of_uneven_columns_bitwise(S, precision):
    """One launch set with one-column, many-column and skipped members: each
    answer equals the member's own solve bit for bit."""
    mats, bs = [], []
    rng = np.random.default_rng(6)
    for (dims, stencil, np_), k in zip(GRIDS, (1, 17, 0, 16, 3)):
        A = _matrix(S, dims, stencil, 4)
        mats.append(S.SnuMat(A, np_, grid=dims, device=0, precision=precision, ir_tol=1e-12))
        bs.append(rng.standard_normal((A.n, k)) if k else None)
    with S.Batch(mats) as batch:
        batch.factorize()
        for M, b, x in zip(mats, bs, batch.solve(bs)):
            if b is not None:
                print("case", precision, M.A.n, "columns", b.shape[1], flush=True)
                assert np.array_equal(x, M.solve(b))
    for M in mats:
        M.close()


def test_scratch_solve_column_by_column(S):
    """A scratch call whose padded column groups do not fit runs its columns
    one at a time: same answers as the allocating solve's single columns, and
    the same size refused as before (16 n nrhs bytes)."""
    A = S.gen_grid(1024, 1024, 1, 5, 0, 4.1, 2)
    k = 2  # two columns pad to 16: 2 x 8 B x 16 n = 256 MiB and the update rows
    rng = np.random.default_rng(7)
    B = np.asfortranarray(rng.standard_normal((A.n, k)))
    with S.SnuMat(A, 512, grid=(1024, 1024, 1), device=0) as M:
        M.factorize()
        d_b, d_x = S.DeviceBuffer(8 * A.n * k), S.DeviceBuffer(8 * A.n * k)
        try:
            d_b.upload(B)
            M.solve_device_scratch_ptr(d_b.ptr.value, d_x.ptr.value, k)
            x = np.zeros((A.n, k), order="F")
            d_x.download(x)
            for c in range(k):
                assert np.array_equal(x[:, c], M.solve(B[:, c]))
            rc = S.lib().snumat_solve_device_scratch(M._h, d_b.ptr, d_x.ptr, 17, A.n)
            assert rc == -1 and b"scratch" in S.lib().snu_last_error()
        finally:
            d_b.free()
            d_x.free()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 96, 97, 128, 129, 200])
def test_dense_leaf_front_orders(S, precision, n):
    """One full matrix as one front, at the orders where the front kernels and
    the 64 x 64 extend-add tiles change: factors against a no-pivot LU in FP64
    (FP32: within n u32 of the largest entry, the diagonally dominant LU's
    rounding bound), solution at the path's bars."""
    rng = np.random.default_rng(n)
    D = rng.uniform(-1, 1, (n, n)) + 2.0 * n * np.eye(n)
    rp = np.arange(0, n * n + 1, n)
    A = S.CSR(n, rp, np.tile(np.arange(n), n), D.reshape(-1))
    LU = D.copy()
    for k in range(n):
        LU[k + 1:, k] /= LU[k, k]
        LU[k + 1:, k + 1:] -= np.outer(LU[k + 1:, k], LU[k, k + 1:])
    tol = 1e-12 if precision == "fp64" else max(n, 8) * 2.0 ** -24
    b = rng.standard_normal((n, 3))
    with S.SnuMat(A, 1, order=np.arange(n), sizes=[n], device=0, precision=precision, ir_tol=1e-12) as M:
        M.factorize()
        v = M.leaf_values(0).reshape(n, n)
        assert np.max(np.abs(v - LU)) <= tol * np.max(np.abs(LU))
        x = np.linalg.solve(D, b)
        for k in (1, 3):
            assert np.max(np.abs(M.solve(b[:, :k]) - x[:, :k])) <= 1e-9 * np.max(np.abs(x))


@pytest.mark.parametrize("prec,power", [("fp64", 600), ("fp64", -600), ("fp32", 60), ("fp32", -60)])
@pytest.mark.parametrize("nb", [1, 15, 16, 31, 33, 48, 49, 63, 64])
def test_diagonal_block_scales_exactly(S, nb, prec, power):
    """Factors of 2^power A are those of A scaled, bit for bit (the pivot
    division keeps its rounding far from 1), and A = L U within the
    elimination's bound nb u |L||U|, elementwise."""
    import ctypes as C
    f64 = prec == "fp64"
    t, u = (np.float64, 2.0 ** -53) if f64 else (np.float32, 2.0 ** -24)
    A = np.random.default_rng(nb).standard_normal((nb, nb)) + 2 * nb * np.eye(nb)
    out = []
    for p in (0, power):
        D = np.asfortranarray((A.astype(t) * t(2.0 ** p)).astype(t))
        Li, Ui = np.zeros(4096, t), np.zeros(4096, t)
        f = S.lib().snu_test_diag_lu if f64 else S.lib().snu_test_diag_lu_f32
        assert f(nb, *(x.ctypes.data_as(C.c_void_p) if i != 1 else nb for i, x in enumerate((D, None, Li, Ui)))) == 0
        out.append((D, Li.reshape(64, 64)[:nb, :nb], Ui.reshape(64, 64)[:nb, :nb]))
    (D, Li, Ui), (Ds, Lis, Uis) = out
    sc = t(2.0 ** power)
    assert np.array_equal(np.tril(D, -1), np.tril(Ds, -1)) and np.array_equal(np.triu(D) * sc, np.triu(Ds))
    assert np.array_equal(Li, Lis) and np.array_equal(Ui, Uis * sc)
    L, U = np.tril(D, -1).astype(np.float64) + np.eye(nb), np.triu(D).astype(np.float64)
    assert np.all(np.abs(L @ U - A.astype(t)) <= (nb + 2) * u * (np.abs(L) @ np.abs(U)))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_diagonal_blocks_beside_schur_updates(S, prec):
    """Diagonal blocks on the second stream beside the Schur updates leave the
    bits of one stream (profiled factorizations run on one), factorization
    after factorization and as replays of a graph."""
    A = S.gen_grid(45, 37, 29, 7, 0, 6.1, 4)
    order, sizes = S.order_grid(45, 37, 29, 32)
    b = S.gen_rhs(A, 1, 1)[1][:, 0]
    with S.SnuMat(A, 32, order=order, sizes=sizes, device=0, precision=prec) as M:
        S._check(S.lib().snumat_set_profiling(M._h, 1))
        x = M.factorize().solve(b)
        S._check(S.lib().snumat_set_profiling(M._h, 0))
        assert S.backward_error(A, x, b) <= 1e-12
        for graph in (0, 0, 1, 1, 0, 1):
            S._check(S.lib().snumat_use_graph(M._h, graph))
            assert np.array_equal(M.factorize().solve(b), x)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [7, 8, 9, 32, 47, 48, 49])
def test_one_wave_front_orders(S, precision, n):
    """The same at the orders around the one-wave front kernel's column chunks
    and its largest order."""
    test_dense_leaf_front_orders(S, precision, n)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_wave_fronts_with_children(S, precision):
    """Chains of fronts of every order up to the one-wave kernel's largest and
    beyond, each with children: banded matrices as one leaf against a dense
    solve."""
    for n, band in ((180, 23), (181, 24), (182, 25), (150, 46), (151, 47), (153, 48)):
        rng = np.random.default_rng(n)
        D = np.where(np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= band, rng.uniform(-1, 1, (n, n)), 0.0)
        D += 2.0 * (band + 1) * np.eye(n)
        r, c = np.nonzero(D)
        A = S.CSR(n, np.searchsorted(r, np.arange(n + 1)), c, D[r, c])
        order = rng.permutation(4).repeat((n + 3) // 4)[:n].argsort(kind="stable")
        b = rng.standard_normal((n, 2))
        x = np.linalg.solve(D, b)
        for o in (np.arange(n), order):
            with S.SnuMat(A, 1, order=o, sizes=[n], device=0, precision=precision, ir_tol=1e-12) as M:
                M.factorize()
                assert np.max(np.abs(M.solve(b) - x)) <= 1e-9 * np.max(np.abs(x))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_split_products_repeat_bitwise(S, prec):
    """One-column products split over K (separators of more than 128 rows) give
    the same bits solve after solve, in a batch, and from the fixed scratch, in
    any order of these: the arrival counters are back at zero after each."""
    A = S.gen_grid(30, 29, 28, 7, 0, 6.1, 2)
    order, sizes = S.order_grid(30, 29, 28, 8)
    b = np.ascontiguousarray(S.gen_rhs(A, 1, 1)[1][:, 0])
    with S.SnuMat(A, 8, order=order, sizes=sizes, device=0, precision=prec) as M:
        x = M.factorize().solve(b)
        assert S.backward_error(A, x, b) <= 1e-12
        db, dx = S.DeviceBuffer(b.nbytes), S.DeviceBuffer(b.nbytes)
        db.upload(b)
        with S.Batch([M]) as B:
            B.factorize()
            for _ in range(3):
                assert np.array_equal(M.solve(b), x)
                M.solve(np.stack([b, b], 1))
                assert np.array_equal(np.asarray(B.solve([b])[0]).reshape(-1), x)
                M.solve_device_scratch_ptr(db.ptr.value, dx.ptr.value, 1)
                xs = np.zeros_like(b)
                dx.download(xs)
                assert np.array_equal(xs, x)
        db.free()
        dx.free()
