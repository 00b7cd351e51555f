"""The second stream of a factorization on matrices with a height of empty
separators: grids coupled by a border alone, so that nested dissection leaves
nothing to separate between the border and the grids' own separators, and the
border is updated from two heights below it."""
import ctypes as C

import numpy as np
import pytest

HEIGHT, PANELS, NEXT_D = 10 ** 8, 6 * 10 ** 7, 9 * 10 ** 7
JOIN, FORK, SIDE = 1, 2, 4


def bordered(S, side, border, parts=4):
    """`parts` uncoupled side^3 7-point grids and `border` rows, each coupled to
    a row of every grid and to the next border row."""
    G = S.gen_grid(side, side, side, 7, 0, 8.1, 1)
    n = G.n * parts + border
    gr = np.repeat(np.arange(G.n), np.diff(G.rowptr))
    r = [gr + p * G.n for p in range(parts)]
    c = [G.colidx + p * G.n for p in range(parts)]
    v = [G.data] * parts
    b = G.n * parts + np.arange(border)
    at = np.linspace(0, G.n - 1, border).astype(int)
    for p in range(parts):
        r += [b, at + p * G.n]
        c += [at + p * G.n, b]
        v += [np.full(border, -0.5), np.full(border, -0.25)]
    r += [b, b[:-1], b[1:]]
    c += [b, b[1:], b[:-1]]
    v += [np.full(border, 9.0), np.full(border - 1, -1.0), np.full(border - 1, -0.5)]
    r, c, v = (np.concatenate(x) for x in (r, c, v))
    o = np.lexsort((c, r))
    r, c, v = r[o], c[o], v[o]
    return S.CSR(n, np.searchsorted(r, np.arange(n + 1)), c, v)


def launches(S, M):
    f = S.lib().snu_test_dense_launches
    n = f(M._h, 0, None, None, None)
    assert n >= 0
    key, kind, side = np.zeros(n, np.int64), np.zeros(n, np.int32), np.zeros(n, np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    assert f(M._h, n, p(key), p(kind), p(side)) == n
    return key // HEIGHT, key % HEIGHT, kind, side


def unordered_pairs(height, step, kind, side):
    """Pairs of launches that the streams leave unordered (indices i < j)."""
    n = len(height)
    seen = {0: -1, SIDE: -1}  # last launch of the other stream each waits for
    last = {0: -1, SIDE: -1}
    before = []               # per launch: (its stream, last launch of the other stream before it)
    for i in range(n):
        if side[i] & JOIN:
            seen[0] = last[SIDE]
        if side[i] & FORK:
            seen[SIDE] = last[0]
        s = side[i] & SIDE
        before.append((s, seen[s]))
        last[s] = i
    return [(i, j) for j in range(n) for i in range(j)
            if before[i][0] != before[j][0] and i > before[j][1]]


def independent(height, step, kind, i, j):
    """Launches that may run side by side: the diagonal blocks of a height
    beside the Schur updates, of the height below, of other blocks; the copy of
    a height's panels beside all Schur updates of the height, which read the
    products that it copies."""
    if kind[i] == 3:
        return height[i] == height[j] and step[j] >= NEXT_D
    return height[j] == height[i] + 1 and step[i] == NEXT_D + 1 and step[j] < PANELS


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_launches_ordered_past_a_height_without_panels(S, precision):
    for A, np_ in ((bordered(S, 24, 900), 16), (S.gen_grid(45, 37, 29, 7, 0, 6.1, 4), 32)):
        with S.SnuMat(A, np_, device=-1, precision=precision) as M:
            height, step, kind, side = launches(S, M)
            assert np.any(side & SIDE)  # the matrix is large enough for the second stream
            pairs = unordered_pairs(height, step, kind, side)
            assert pairs
            bad = [(i, j) for i, j in pairs if not independent(height, step, kind, i, j)]
            assert not bad, [(height[i], step[i], kind[i], height[j], step[j], kind[j]) for i, j in bad[:3]]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_height_without_panels_on_two_streams(S, precision):
    """The bits of one stream (profiled factorizations run on one), eager and
    from a graph."""
    A = bordered(S, 24, 900)
    b = S.gen_rhs(A, 1, 1)[1][:, 0]
    with S.SnuMat(A, 16, device=0, precision=precision, ir_tol=1e-12) as M:
        print("case", precision, A.n, flush=True)
        S._check(S.lib().snumat_set_profiling(M._h, 1))
        x = M.factorize().solve(b)
        S._check(S.lib().snumat_set_profiling(M._h, 0))
        assert S.backward_error(A, x, b) <= 1e-12
        for graph in (0, 0, 1, 1, 0, 1):
            S._check(S.lib().snumat_use_graph(M._h, graph))
            assert np.array_equal(M.factorize().solve(b), x)
