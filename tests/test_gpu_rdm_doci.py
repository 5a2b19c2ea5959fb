"""GPU tests of the DOCI densities over their chunks of rows (16 rows a workgroup,
then 512 workgroups, 1,024 from 100,000 rows on with the 2-RDM), against numpy:
gamma_jj = sum c^2 n_j, Gamma^ab_jkjk = sum c^2 n_j n_k and the pair part
Gamma^ab_jjkk = sum c_I c_J over the pair hops k -> j."""
import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


# n = 3, 15, 28, 924, 8,568, 48,620, 125,970
@pytest.mark.parametrize("L,pairs", [(3, 1), (6, 2), (8, 6), (12, 6), (18, 5), (18, 9), (20, 8)])
def test_doci_densities(L, pairs):
    s = np.arange(1 << L, dtype=np.int64)
    bits = (s[:, None] >> np.arange(L)) & 1
    keep = bits.sum(1) == pairs
    rank = np.cumsum(keep) - 1
    s, bits = s[keep], bits[keep]
    c = np.random.default_rng(L).standard_normal(len(s))
    ci = CA.DOCI(CA.Hamiltonian(*CA.gen_integrals(L, 3), pairs, pairs), build=False)
    assert ci.n == len(s)
    g, G = ci.density_dense(c)
    g1, none = ci.density_dense(c, two=False)
    # sums of at most n products of two FP64 numbers
    tol = 4e-16 * len(s) ** 0.5 * float(c @ c)
    D = (bits * (c * c)[:, None]).T @ bits
    for j in range(L):
        for k in range(L):
            assert abs(G[1, j, k, j, k] - (D[j, k] if j != k else D[j, j])) <= tol
            if j != k:
                sel = (bits[:, k] == 1) & (bits[:, j] == 0)
                P = c[sel] @ c[rank[s[sel] ^ (1 << k) ^ (1 << j)]]
                assert abs(G[1, j, j, k, k] - P) <= tol
                assert abs(G[0, j, k, j, k] - D[j, k]) <= tol and G[0, j, k, k, j] == -G[0, j, k, j, k]
    want = np.diag(np.diag(D))
    for x in (g, g1):
        assert none is None and np.max(np.abs(x - want)) <= tol
