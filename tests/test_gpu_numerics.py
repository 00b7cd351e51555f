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
    want = np.where(np.tri(nb, k=-1, dtype=bool), out[0], out[0] * t(2.0 ** h) * t(2.0 ** (power - h)))
    assert np.array_equal(out[1], want)
