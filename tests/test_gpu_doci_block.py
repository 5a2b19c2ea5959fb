"""GPU tests of the block-staged DOCI product against the CRS product: every
number of low orbitals (each kernel instance and what it pads) and up to 20 high
ones, on the tabled kernel, and few and many pairs, which run the bit-walking one
(below a third or above two thirds filling; with 12 low orbitals 5/12 and 7/12)."""
import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,pairs,ws", [(2, 1, (1,)), (5, 2, (1, 2, 3, 4)), (13, 6, range(1, 13)), (14, 7, (9, 10, 12)),
                                        (15, 2, (1, 7, 11, 12)), (16, 14, (8, 11, 12)), (24, 3, (4, 5, 9, 12)),
                                        (18, 9, (9, 11, 12)), (13, 1, (3, 12)), (13, 12, (3, 12)),
                                        # tabled with 14 .. 20 high orbitals; 100 hops inside the high part
                                        (21, 7, (1, 3, 5, 7)), (21, 14, (1, 6)), (20, 9, (2, 4)), (21, 10, (1,))])
def test_low_orbitals(L, pairs, ws):
    h, V = CA.gen_integrals(L, 40 + L)
    m = CA.DOCI(CA.Hamiltonian(h, V, pairs, pairs), value_prec=CA.CF_F32).get_mat()
    x = np.random.default_rng(L).standard_normal(m.getn())
    m.set_spmv_kernel(1)
    want = {p: m.mvprod(x, p) for p in (CA.CF_F64, CA.CF_F32)}
    for w in ws:
        m.set_spmv_kernel(6, w)
        for p in (CA.CF_F64, CA.CF_F32):
            y = m.mvprod(x, p)
            assert np.array_equal(y, m.mvprod(x, p))
            # 132 terms a row at most, summed in FP64 in both
            assert np.linalg.norm(y - want[p]) <= 4e-15 * np.linalg.norm(want[p])
