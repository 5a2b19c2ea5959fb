"""GPU tests of the FCI densities from one-spin matrices: every size at an edge
of its tiles (64 strings, 32 beta strings a stage, 16 columns) against <a+a> and
<a+a+aa> contracted from plain numpy transition densities, with unequal spins,
empty and full shells, the 1-RDM alone, and an unnormalised vector; and of the
ones that go through transition densities in memory (L > 16; the 1-RDM of a space
with many strings of one spin and hardly any of the other)."""
from math import comb

import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


def excitations(L, n):
    """src[p, q, K], sgn[p, q, K]: a+_p a_q takes string src to string K."""
    s = np.array([v for v in range(1 << L) if bin(v).count("1") == n])
    rank = {int(v): i for i, v in enumerate(s)}
    src = np.zeros((L, L, len(s)), dtype=int)
    sgn = np.zeros((L, L, len(s)))
    for K, v in enumerate(s):
        v = int(v)
        for p in range(L):
            if not v >> p & 1:
                continue
            for q in range(L):
                if p == q:
                    src[p, p, K], sgn[p, p, K] = K, 1.0
                elif not v >> q & 1:
                    lo, hi = min(p, q), max(p, q)
                    between = bin((v >> (lo + 1)) & ((1 << (hi - lo - 1)) - 1)).count("1")
                    src[p, q, K] = rank[v ^ (1 << p) ^ (1 << q)]
                    sgn[p, q, K] = -1.0 if between & 1 else 1.0
    return src, sgn


def reference(L, na, nb, c):
    C = c.reshape(comb(L, na), comb(L, nb))
    (sa, ga), (sb, gb) = excitations(L, na), excitations(L, nb)
    X = [(C[sa] * ga[..., None]).reshape(L * L, -1),
         (C[:, sb].transpose(1, 2, 0, 3) * gb[:, :, None, :]).reshape(L * L, -1)]
    g = np.stack([(x @ c).reshape(L, L) for x in X])
    G = []
    for s, t in ((0, 0), (0, 1), (1, 1)):
        M = (X[s] @ X[t].T).reshape(L, L, L, L)   # [r, p, q, u] = <E_pr E_qu>
        B = M.transpose(1, 2, 0, 3).copy()         # [p, q, r, u]
        if s == t:
            for q in range(L):
                B[:, q, q, :] -= g[s]
        G.append(B)
    return g, np.stack(G)


@pytest.mark.parametrize("L,na,nb", [(1, 1, 0), (3, 0, 2), (3, 3, 1), (4, 2, 2), (6, 3, 1), (7, 2, 5), (8, 4, 3),
                                     (9, 2, 4), (10, 1, 5), (11, 3, 2), (12, 2, 3), (13, 2, 2), (16, 1, 2),
                                     (17, 1, 2), (18, 2, 1), (16, 6, 0)])
def test_densities(L, na, nb):
    h, V = CA.gen_integrals(max(L, 2), 3)
    h, V = h[:L, :L].copy(), V[:L, :L, :L, :L].copy()
    ci = CA.FCI(CA.Hamiltonian(h, V, na, nb), build=False)
    c = np.random.default_rng(L).standard_normal(ci.n)   # |c| != 1 on purpose
    g, G = ci.density_dense(c)
    rg, rG = reference(L, na, nb, c)
    # sums of at most n products of two FP64 numbers
    tol = 4e-16 * ci.n ** 0.5 * float(c @ c)
    assert np.max(np.abs(g - rg)) <= tol and np.max(np.abs(G - rG)) <= tol, (np.max(np.abs(G - rG)), tol)
    g1, none = ci.density_dense(c, two=False)
    assert none is None and np.max(np.abs(g1 - rg)) <= tol
