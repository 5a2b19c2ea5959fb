"""GPU tests of the FCI rows written from position-major values: the upper CRS
bit for bit against the oracle at the edges of the tiles (64 strings, 64
positions) and of the chunks (512 strings), with elements that are dropped,
after new integrals, in FP32 copies; and a space whose values take several
passes (more than 2 GiB), against the on-the-fly product; and the rows of a beta
space above 65,535 strings, which are evaluated one by one."""
from math import comb

import numpy as np
import pytest

import ciflow_amd as CA
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def same_upper(cim, h, V, na, nb):
    row, col, val = cim.get_mat().export_upper()
    ref = O.build_crs("FCI", h, V, na, nb)
    assert np.array_equal(row, ref.row) and np.array_equal(col, ref.col) and np.array_equal(val, ref.data)


# d_beta 1, 5, 63 / 64 / 65-ish tiles and 512-string chunks; unequal spins; no alpha or beta singles
@pytest.mark.parametrize("L,na,nb", [(5, 0, 2), (5, 2, 0), (5, 5, 2), (6, 1, 3), (8, 2, 4), (9, 2, 2), (11, 1, 2),
                                     (12, 1, 4), (13, 1, 3), (8, 4, 4), (12, 2, 5)])
def test_rows_bit_exact(L, na, nb):
    h, V = CA.gen_integrals(L, 70 + L + na)
    if (L, na, nb) == (8, 2, 4):   # some elements at the threshold and below
        h[np.abs(h) < 0.03] = 0.0
        V[np.abs(V) < 0.02] = 0.0
    cim = CA.FCI(CA.Hamiltonian(h, V, na, nb), value_prec=CA.CF_F32)
    same_upper(cim, h, V, na, nb)
    x = np.random.default_rng(1).standard_normal(cim.n)
    y = cim.get_mat().mvprod(x)
    if L <= 8:   # the position-major copy on request, then new integrals for everything
        cim.get_mat().set_spmv_kernel(4)
        assert np.linalg.norm(cim.get_mat().mvprod(x) - y) <= 1e-14 * np.linalg.norm(y)
        h, V = CA.gen_integrals(L, 700 + L)
        cim.set_ham(CA.Hamiltonian(h, V, na, nb))
        y4 = cim.get_mat().mvprod(x)
        same_upper(cim, h, V, na, nb)
        cim.get_mat().set_spmv_kernel(1)
        y1 = cim.get_mat().mvprod(x)
        assert np.linalg.norm(y4 - y1) <= 1e-14 * np.linalg.norm(y1)


def test_values_in_several_passes():
    L, na, nb = 12, 3, 6   # 203,280 rows of 1,369 elements: 2.2 GB of values
    h, V = CA.gen_integrals(L, 5)
    ham = CA.Hamiltonian(h, V, na, nb)
    cim = CA.FCI(ham)
    n, nnz, upper = cim.get_mat().info()
    sa, sb = na * (L - na), nb * (L - nb)
    R = (1 + sa) * (1 + sb) + comb(na, 2) * comb(L - na, 2) + comb(nb, 2) * comb(L - nb, 2)
    assert nnz == n * R and 2 * upper == nnz + n
    x = np.random.default_rng(2).standard_normal(n)
    y, z = cim.get_mat().mvprod(x), CA.FCI_Direct(ham).mvprod(x)
    assert np.linalg.norm(y - z) <= 1e-13 * np.linalg.norm(z)
    r0 = n - 924
    row, col, val = cim.get_mat().export_upper(r0, n)
    ref = O.build_crs("FCI", h, V, na, nb, start=219, end=220)
    assert np.array_equal(row, ref.row) and np.array_equal(col, ref.col) and np.array_equal(val, ref.data)


def test_rows_of_a_large_beta_space():
    """77,520 strings of seven electrons: as beta strings (32-bit targets, one evaluation an
    element and pass) and as alpha strings they are the same matrix, bit for bit."""
    L, ne = 20, 7
    h, V = CA.gen_integrals(L, 6)
    beta, alpha = (CA.FCI(CA.Hamiltonian(h, V, *n)) for n in ((0, ne), (ne, 0)))
    n, nnz, upper = beta.get_mat().info()
    row = 1 + ne * (L - ne) + comb(ne, 2) * comb(L - ne, 2)
    assert (n, nnz, upper) == (77520, 77520 * row, 77520 * (row + 1) // 2) == tuple(alpha.get_mat().info())
    for r0 in (0, 31000, n - 500):
        a, b = (m.get_mat().export_upper(r0, r0 + 500) for m in (alpha, beta))
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
    x = np.random.default_rng(3).standard_normal(n)
    y, z = beta.get_mat().mvprod(x), alpha.get_mat().mvprod(x)
    assert np.linalg.norm(y - z) <= 1e-14 * np.linalg.norm(z)
