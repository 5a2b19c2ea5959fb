"""GPU tests of the two-launch Lanczos step of small spaces on each of its
instances (up to 1,024, 2,048, 5,120, 10,240 and 16,384 rows, fewer than a
wavefront included): energies and vectors against dense eigenvalues, or energies
against the Davidson solve (also above 16,384 rows, where the other step takes
over), across restarts, and through a breakdown (a start vector in a small
invariant space)."""
import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


def dense(m, n):
    row, col, val = m.export_full()
    A = np.zeros((n, n))
    for i in range(n):
        A[i, col[row[i]:row[i + 1]]] = val[row[i]:row[i + 1]]
    return A


# FCI dimensions 9, 36, 50, 400, 100, 1225; DOCI 1716, 3432
@pytest.mark.parametrize("kind,L,na,nb", [("FCI", 3, 1, 2), ("FCI", 4, 2, 2), ("FCI", 5, 2, 4), ("FCI", 6, 3, 3),
                                          ("FCI", 5, 2, 2), ("FCI", 7, 3, 4), ("DOCI", 13, 6, 6), ("DOCI", 14, 7, 7)])
@pytest.mark.parametrize("ncv", [42, 12])
def test_against_dense(kind, L, na, nb, ncv):
    h, V = CA.gen_integrals(L, 60 + L)
    ci = (CA.FCI if kind == "FCI" else CA.DOCI)(CA.Hamiltonian(h, V, na, nb))
    w, Y = np.linalg.eigh(dense(ci.get_mat(), ci.n))
    info = ci.solve(ncv=min(ncv, max(2, ci.n)))
    x = ci.get_eigvec()
    assert info.status == 0 and abs(info.eigval - w[0]) <= 1e-11 * max(1.0, abs(w[0]))
    if w[1] - w[0] > 1e-6:
        assert abs(abs(x @ Y[:, 0]) - 1.0) <= 1e-10
    assert abs(x @ x - 1.0) <= 1e-12


# 7,056, 10,584, 15,876 (in range), 25,200 (above)
@pytest.mark.parametrize("L,na,nb", [(9, 3, 3), (9, 4, 3), (9, 4, 4), (10, 4, 3)])
def test_around_the_bound(L, na, nb):
    h, V = CA.gen_integrals(L, 5)
    ci = CA.FCI(CA.Hamiltonian(h, V, na, nb))
    a = ci.solve()
    b = ci.solve(method=CA.CF_DAVIDSON)
    assert a.status == b.status == 0 and abs(a.eigval - b.eigval) <= 1e-10


def test_breakdown_in_an_invariant_space():
    L = 8   # two-body part only between equal orbitals: few distinct eigenvalues, the Krylov space ends early
    h = np.diag(np.repeat([-1.0, 0.5], L // 2))
    V = np.zeros((L,) * 4)
    ci = CA.FCI(CA.Hamiltonian(h, V, 3, 3))
    info = ci.solve()
    assert info.status == 0 and abs(info.eigval + 6.0) <= 1e-10
