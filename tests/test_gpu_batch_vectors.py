"""GPU tests of the batched Davidson vector passes: basis sizes on both sides of
the chunks of eight vectors that a thread keeps in registers, dimensions on both
sides of a workgroup, FP64 and FP32-operand phases (the second starts from the
first one's Ritz vector), against the lowest eigenvalue of the stored matrix."""
import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


def lowest(kind, h, V, na, nb):
    ham = CA.Hamiltonian(h, V, na, nb)
    m = (CA.DOCI if kind == CA.CF_DOCI else CA.FCI)(ham).get_mat()
    row, col, val = m.export_upper()
    n = len(row) - 1
    A = np.zeros((n, n))
    A[np.repeat(np.arange(n), np.diff(row.astype(np.int64))), col] = val
    return np.linalg.eigvalsh(A, UPLO="U")[0]


# n = 400, 735, 1960, 252, 462, 924
@pytest.mark.parametrize("kind,L,na,nb", [("fci", 6, 3, 3), ("fci", 7, 3, 2), ("fci", 8, 2, 4),
                                          ("doci", 10, 5, 5), ("doci", 11, 5, 5), ("doci", 12, 6, 6)])
def test_basis_sizes(kind, L, na, nb):
    code = CA.CF_DOCI if kind == "doci" else CA.CF_FCI
    sizes = (3, 8, 9, 16, 17, 24)
    ints = [CA.gen_integrals(L, 500 + k) for k in range(len(sizes))]
    want = [lowest(code, h, V, na, nb) for h, V in ints]
    for prec in (CA.CF_F64, CA.CF_F32):
        # two requests of each basis size: one batch of two lanes each
        reqs = [{"tag": k, "kind": code, "h": ints[k % 6][0], "V": ints[k % 6][1], "nup": na, "ndown": nb,
                 "precision": prec, "ncv": sizes[k % 6], "direct": True} for k in range(12)]
        out = CA.solve_batch(reqs)
        for k, r in enumerate(out):
            assert r["status"] == 0 and r["solve_status"] == 0
            # residual <= 1e-12 |theta| bounds the eigenvalue's error; rounding of the two products on top
            assert abs(r["eigval"] - want[k % 6]) <= 1e-11 * abs(want[k % 6])
            if k < 6:
                alone = CA.solve_batch([reqs[k]])[0]
                assert alone["eigval"] == r["eigval"] and alone["n_matvec"] == r["n_matvec"]
