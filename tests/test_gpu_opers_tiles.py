"""Operator update at the edges of its tiles (16 rows of a mode, 16 terms of a
state, the wave groups from 65 functions on), against the sums written out in
numpy.

Tolerance: a result is a sum of products of at most (D + 2) n + 2 R roundings
each, so its error is below that many eps of the same sum over absolute values;
the sizes here stay below 1000, and 1000 eps = 2.3e-13.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # nbas, ranks
    ([1], [1, 2]),                              # one mode, one function
    ([16, 17], [16, 17, 1]),                    # a whole tile and one more
    ([32, 48, 64], [15, 33, 2, 16]),
    ([65, 80], [5, 18]),                        # two waves a pair
    ([97, 112, 3], [7, 16, 1]),                 # four waves a pair
    ([128, 96], [70, 3]),                       # the largest mode
]


@pytest.mark.parametrize("nbas,ranks", CASES)
def test_tile_edges(hip, nbas, ranks):
    from mlcp_amd import intertwine as tw
    from mlcp_amd.hoplist import CPBlock
    print("[case] opers", nbas, ranks, flush=True)
    rng = np.random.default_rng(sum(nbas) + sum(ranks))
    D, N, B = len(nbas), sum(ranks), len(ranks)
    fac = [rng.normal(size=(N, n)) / np.sqrt(n) for n in nbas]
    coef = rng.normal(size=N)
    Q = CPBlock(np.array(nbas), np.array(ranks), coef,
                np.concatenate(fac, axis=1), np.zeros(B))
    # five operators on the first mode (a group of four and one), one on the
    # last, none between
    modes = np.array([0] * 5 + [D - 1])
    dense, ops = [], []
    for d in modes:
        a = rng.normal(size=(nbas[d], nbas[d]))
        a = 0.5 * (a + a.T)
        dense.append(a)
        i, j = np.triu_indices(nbas[d])
        order = np.lexsort((i, j))
        ops.append(a[i[order], j[order]])
    out = tw.update_operators(Q, modes, ops)
    off = np.concatenate([[0], np.cumsum(ranks)])
    for o, d in enumerate(modes):
        w = fac[d] @ dense[o] @ fac[d].T
        wa = np.abs(fac[d]) @ np.abs(dense[o]) @ np.abs(fac[d]).T
        for e in range(D):
            if e != d:
                w = w * (fac[e] @ fac[e].T)
                wa = wa * (np.abs(fac[e]) @ np.abs(fac[e]).T)
        w = coef[:, None] * w * coef[None, :]
        wa = np.abs(coef)[:, None] * wa * np.abs(coef)[None, :]
        got = np.asarray(out[o])
        k = 0
        for j in range(B):
            for i in range(j + 1):
                sl = np.s_[off[i]:off[i + 1], off[j]:off[j + 1]]
                assert abs(got[k] - w[sl].sum()) <= 2.3e-13 * wa[sl].sum()
                k += 1
