"""GPU tests of the alpha-beta sigma as a matrix product: the on-the-fly product
against the stored matrix over every action count and string dimension at an
edge of its tiles (16 strings, 4 actions, 16 pair columns and their
remainders), unequal spins included; integrals that are not symmetric in the
last two orbitals (which keep the other kernel) alone and in one batch with
symmetric ones; batched energies against single solves."""
import numpy as np
import pytest

import ciflow_amd as CA
from oracle.richardson import redbcs_integrals

pytestmark = pytest.mark.gpu


def rotated(L, seed):
    h, V = CA.gen_integrals(L, seed)
    return CA.rotate_integrals(h, V, CA.expm_skew(CA.gen_rotation(L, seed, 0.1)))


# pairs L (L + 1) / 2: 10, 15, 21, 28, 36, 45, 55, 66 (4 tiles + 2), 78, 91, 136; actions up to 40
@pytest.mark.parametrize("L,na,nb", [(4, 1, 2), (5, 2, 2), (6, 3, 2), (7, 3, 4), (8, 4, 4), (8, 2, 5), (9, 4, 3),
                                     (9, 1, 4), (10, 5, 5), (10, 4, 3), (11, 5, 5), (11, 4, 5), (11, 6, 2), (12, 5, 6),
                                     (12, 3, 3), (13, 3, 2), (16, 2, 2), (16, 3, 1), (7, 6, 1), (6, 1, 5)])
def test_product_equals_stored_matrix(L, na, nb):
    h, V = rotated(L, 90 + L)
    ham = CA.Hamiltonian(h, V, na, nb)
    d = CA.FCI_Direct(ham)
    x = np.random.default_rng(L).standard_normal(d.n)
    y, again = d.mvprod(x), d.mvprod(x)
    z = CA.FCI(ham).get_mat().mvprod(x)
    assert np.array_equal(y, again)
    assert np.linalg.norm(y - z) <= 4e-15 * np.linalg.norm(z)


def test_integrals_without_the_symmetry():
    h, V = redbcs_integrals(np.arange(8.0), -0.5)   # V(i,i,j,j) only: not symmetric in q <-> s
    ham = CA.Hamiltonian(h, V, 4, 4)
    d = CA.FCI_Direct(ham)
    x = np.random.default_rng(8).standard_normal(d.n)
    z = CA.FCI(ham).get_mat().mvprod(x)
    assert np.linalg.norm(d.mvprod(x) - z) <= 4e-15 * np.linalg.norm(z)
    reqs = []
    for k in range(5):
        hk, Vk = (h, V) if k in (1, 3) else CA.gen_integrals(8, 300 + k)
        reqs.append({"tag": k, "kind": CA.CF_FCI, "h": hk, "V": Vk, "nup": 4, "ndown": 4, "precision": CA.CF_F64})
    mix = CA.solve_batch(reqs)
    for q, r in zip(reqs, mix):
        alone = CA.solve_batch([q])[0]
        assert r["status"] == 0 and r["solve_status"] == 0
        assert alone["energy"] == r["energy"] and alone["n_matvec"] == r["n_matvec"]
        ci = CA.FCI(CA.Hamiltonian(q["h"], q["V"], 4, 4))
        ci.solve()
        assert abs(ci.get_ci_energy() - r["energy"]) <= 1e-10


@pytest.mark.parametrize("size", [9e-15, 2e-15, 2e-16])
def test_integrals_that_are_nearly_symmetric(size):
    """A Hermitian part that is antisymmetric in q <-> s (the two orders differ by twice its
    size) is used as given unless it is rounding."""
    L = 8
    h, V = CA.gen_integrals(L, 77)
    K = np.triu(np.ones((L, L)), 1)
    K -= K.T
    V = V + size * np.abs(V).max() * np.einsum("pr,qs->pqrs", K, K)
    ham = CA.Hamiltonian(h, V, 4, 4)
    x = np.random.default_rng(8).standard_normal(4900)
    z = CA.FCI(ham).get_mat().mvprod(x)
    y = CA.FCI_Direct(ham).mvprod(x)
    assert np.linalg.norm(y - z) <= 4e-15 * np.linalg.norm(z)
