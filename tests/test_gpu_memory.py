"""Solves whose working memory cannot be allocated (a limit set from the host:
larger allocations fail as if the device were full)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NO_LIMIT = 2 ** 64 - 1


def _limit(S, M, nbytes):
    S._check(S.lib().snu_test_alloc_limit(M._h, C.c_size_t(nbytes)))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_failed_allocation_leaves_no_buffer_behind(S, precision):
    """A solve that cannot grow its buffers fails, and so does the next one,
    with fewer columns than there were buffers for before; with memory again
    the answers are the same.  Handle and batch."""
    A = S.gen_grid(40, 31, 1, 9, 0, 8.1, 1)
    B = np.asfortranarray(np.random.default_rng(2).standard_normal((A.n, 40)))
    with S.SnuMat(A, 4, grid=(40, 31, 1), device=0, precision=precision, ir_tol=1e-12) as M:
        M.factorize()
        with S.Batch([M]) as batch:
            solves = [lambda k: M.solve(B[:, :k]), lambda k: np.asarray(batch.solve([B[:, :k]])[0])]
            for solve in solves:
                first = {k: solve(k) for k in (1, 3)}
                _limit(S, M, 0)
                for k in (40, 3, 1):
                    with pytest.raises(S.SnuError) as e:
                        solve(k)
                    assert e.value.code == -7
                _limit(S, M, NO_LIMIT)
                for k in (3, 1, 40):
                    x = solve(k)
                    assert k not in first or np.array_equal(x, first[k])
                    assert S.backward_error(A, x, B[:, :k]) <= 1e-12


def test_failed_norms_leave_no_buffer_behind(S):
    """The same where the vectors fit and the norms of the refinement do not
    (4 rows: 816 bytes of norms for 17 columns, 512 of vectors)."""
    D = np.array([[4.0, 1, 0, 0], [1, 4, 1, 0], [0, 1, 4, 1], [0, 0, 1, 4]])
    r, c = np.nonzero(D)
    A = S.CSR(4, np.searchsorted(r, np.arange(5)), c, D[r, c])
    B = np.asfortranarray(np.random.default_rng(3).standard_normal((4, 17)))
    with S.SnuMat(A, 1, order=np.arange(4), sizes=[4], device=0, precision="fp32", ir_tol=1e-12) as M:
        M.factorize()
        d_b, d_x = S.DeviceBuffer(B.nbytes), S.DeviceBuffer(B.nbytes)
        d_b.upload(B)
        with S.Batch([M]) as batch:
            one = lambda v: (C.c_void_p * 1)(v)
            calls = [lambda k: S.lib().snumat_solve_device(M._h, d_b.ptr, d_x.ptr, k, 4),
                     lambda k: S.lib().snubatch_solve_device(batch._h, one(d_b.ptr.value), one(d_x.ptr.value),
                                                             (C.c_int * 1)(k), (C.c_int * 1)(4))]
            for call in calls:
                assert call(3) == 0
                _limit(S, M, 600)
                assert call(17) in (0, -7)
                assert call(3) == 0
                x = np.zeros((4, 17), order="F")
                d_x.download(x)
                assert np.max(np.abs(x[:, :3] - np.linalg.solve(D, B[:, :3]))) <= 1e-12
                _limit(S, M, NO_LIMIT)
                assert call(17) == 0
                d_x.download(x)
                assert np.max(np.abs(x - np.linalg.solve(D, B))) <= 1e-12
        d_b.free()
        d_x.free()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_columns_in_turn_where_groups_do_not_fit(S, precision):
    """Several columns take padded groups of 16; where the memory for those is
    missing but one column's is there, the columns run in turn: the bits of
    single solves, and refinement figures over all columns."""
    A = S.gen_grid(40, 31, 1, 9, 0, 8.1, 1)
    v = 8 if precision == "fp64" else 4
    B = np.asfortranarray(np.random.default_rng(4).standard_normal((A.n, 18)))
    B[:, 4:] = 0.0  # (no step of refinement after the fourth column)
    d_b, d_x = S.DeviceBuffer(B.nbytes), S.DeviceBuffer(B.nbytes)
    d_b.upload(B)
    x = np.zeros((A.n, 18), order="F")
    mats = [S.SnuMat(A, 4, grid=(40, 31, 1), device=0, precision=precision, ir_tol=1e-13) for _ in range(3)]
    for M in mats:
        M.factorize()
    single = np.stack([mats[1].solve(B[:, c]) for c in range(18)], 1)
    steps = []
    for c in range(4):
        mats[1].solve(B[:, c])
        steps.append(mats[1].timings()["ir_steps"])
    assert precision == "fp64" or max(steps) >= 1
    for k in (2, 15, 18):
        M = S.SnuMat(A, 4, grid=(40, 31, 1), device=0, precision=precision, ir_tol=1e-13)
        M.factorize()
        _limit(S, M, 12 * v * A.n)  # (the fronts' update rows of one column: up to 8 A.n)
        M.solve_device_ptr(d_b.ptr.value, d_x.ptr.value, k)
        d_x.download(x)
        assert np.array_equal(x[:, :k], single[:, :k])
        assert M.timings()["ir_steps"] == max(steps[:k])
        _limit(S, M, NO_LIMIT)
        M.solve_device_ptr(d_b.ptr.value, d_x.ptr.value, k)  # as groups again
        d_x.download(x)
        assert S.backward_error(A, x[:, :4], B[:, :4]) <= 1e-12 or k < 4
        M.close()
    ncol = (18, 1, 5)
    with S.Batch(mats) as batch:
        P = lambda q: (C.c_void_p * 3)(q, q, q)
        outs = [S.DeviceBuffer(B.nbytes) for _ in range(3)]
        _limit(S, mats[0], 3 * 12 * v * A.n)
        rc = S.lib().snubatch_solve_device(batch._h, P(d_b.ptr.value), (C.c_void_p * 3)(*[o.ptr.value for o in outs]),
                                           (C.c_int * 3)(*ncol), (C.c_int * 3)(A.n, A.n, A.n))
        assert rc == 0
        for o, k in zip(outs, ncol):
            o.download(x)
            assert np.array_equal(x[:, :k], single[:, :k])
            o.free()
        assert batch.timings()["ir_steps"] == max(steps)
        _limit(S, mats[0], NO_LIMIT)
    for M in mats:
        M.close()
    d_b.free()
    d_x.free()


def test_working_memory_of_column_groups(S):
    """A group of 16 columns takes its right-hand sides, the separators' vectors
    and the update rows alive at once, not every front's side by side."""
    for dims, st, np_ in (((33, 31, 29), 7, 16), ((250, 211, 1), 5, 32)):
        A = S.gen_grid(*dims, st, 0, {7: 6.1, 5: 4.1}[st], 1)
        order, sizes = S.order_grid(*dims, np_)
        with S.SnuMat(A, np_, order=order, sizes=sizes, device=0) as M:
            M.factorize()
            rows = sum(int(np.sum(F["f"] - F["nk"])) for F in (M.leaf_fronts(r) for r in range(np_)))
            seps = A.n - sum(M.leaf_sizes(r)[0] for r in range(np_))
            before = M.info()["device_bytes"]
            d_b, d_x = S.DeviceBuffer(8 * A.n * 2), S.DeviceBuffer(8 * A.n * 2)
            d_b.upload(np.ones((A.n, 2), order="F"))
            M.solve_device_ptr(d_b.ptr.value, d_x.ptr.value, 2)
            d_b.free()
            d_x.free()
            taken = M.info()["device_bytes"] - before
            print("case", dims, "bytes per row and column", taken / (16 * A.n), "rows", rows / A.n, flush=True)
            assert taken <= 16 * 8 * (A.n + seps + 0.8 * rows)
