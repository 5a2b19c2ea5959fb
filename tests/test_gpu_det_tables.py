"""GPU tests of the determinant-list rows built from string tables: the upper
CRS bit for bit against the oracle for lists in (up, down) order, in random
order, with rotated integrals (whose stored values depend on the orientation),
with elements below the threshold, at the density where the tables stop and
just past it, and with repeated determinants (built by lookup); the FP32 copy
and the sliced product of a list whose last chunk and quads are ragged."""
import numpy as np
import pytest

import ciflow_amd as CA
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def full_space(L, na, nb):
    s = lambda n: np.array([v for v in range(1 << L) if bin(v).count("1") == n], dtype=np.uint64)  # noqa: E731
    a, b = s(na), s(nb)
    return np.repeat(a, len(b)), np.tile(b, len(a))


def integrals(L, seed, cut=0.0):
    h, V = CA.gen_integrals(L, seed)
    h, V = CA.rotate_integrals(h, V, CA.expm_skew(CA.gen_rotation(L, seed, 0.2)))
    if cut:
        h[np.abs(h) < cut] = 0.0
        V[np.abs(V) < cut] = 0.0
    return h, V


def check(L, na, nb, up, down, seed, cut=0.0):
    h, V = integrals(L, seed, cut)
    ham = CA.Hamiltonian(h, V, na, nb)
    m = CA.FCI_File(ham, (up, down), value_prec=CA.CF_F32).get_mat()
    row, col, val = m.export_upper()
    ref = O.build_crs_dets(h, V, na, nb, up, down)
    assert np.array_equal(row, ref.row) and np.array_equal(col, ref.col) and np.array_equal(val, ref.data)
    x = np.random.default_rng(seed).standard_normal(len(up))
    m.set_spmv_kernel(1)
    y = m.mvprod(x)
    y32 = m.mvprod(x, CA.CF_F32)
    m.set_spmv_kernel(7)
    assert np.linalg.norm(m.mvprod(x) - y) <= 1e-14 * np.linalg.norm(y)
    assert np.linalg.norm(m.mvprod(x, CA.CF_F32) - y32) <= 1e-14 * np.linalg.norm(y)


@pytest.mark.parametrize("L,na,nb,count", [(4, 2, 2, 1), (5, 2, 3, 37), (6, 3, 1, 64), (6, 3, 3, 65), (8, 4, 3, 700),
                                           (9, 1, 4, 1100)])
@pytest.mark.parametrize("order", ["sorted", "random"])
def test_dense_lists(L, na, nb, count, order):
    up, down = full_space(L, na, nb)
    rng = np.random.default_rng(count)
    pick = rng.permutation(len(up))[:count]
    if order == "sorted":
        pick = np.sort(pick)
    check(L, na, nb, up[pick], down[pick], 10 + L)
    check(L, na, nb, up[pick], down[pick], 20 + L, cut=0.05)


@pytest.mark.parametrize("count", [1900, 7000])   # 1 in 33 and 9 pairs of strings: lookup, tables
def test_sparse_lists(count):
    up, down = full_space(10, 5, 5)
    pick = np.sort(np.random.default_rng(3).permutation(len(up))[:count])
    check(10, 5, 5, up[pick], down[pick], 31)


def test_repeated_determinants():
    up, down = full_space(6, 3, 3)
    pick = np.concatenate([np.arange(100, 300), np.arange(150, 200)])
    check(6, 3, 3, up[pick], down[pick], 41)
    check(6, 3, 3, up[np.sort(pick)], down[np.sort(pick)], 42)
