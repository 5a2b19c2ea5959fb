"""GPU test of Context.trim: memory kept for reuse goes back, whichever context
of the device holds it, live handles keep theirs and work on."""
import gc

import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


def test_trim_gives_back_what_is_kept():
    h, V = CA.gen_integrals(9, 1)
    main, other = CA.default_context(), CA.Context()
    live = CA.FCI(CA.Hamiltonian(h, V, 4, 4))
    x = np.random.default_rng(1).standard_normal(live.n)
    y = live.get_mat().mvprod(x)
    nnz = live.get_mat().info()[1]
    main.trim()
    for ctx in (main, other):   # a matrix of 12 bytes an element dropped in either context
        dropped = CA.FCI(CA.Hamiltonian(h, V, 4, 4, ctx=ctx))
        assert np.array_equal(dropped.get_mat().mvprod(x), y)
        del dropped
        gc.collect()
        assert main.trim() >= 12 * nnz
        assert main.trim() == 0
    assert np.array_equal(live.get_mat().mvprod(x), y)
    again = CA.FCI(CA.Hamiltonian(h, V, 4, 4))
    assert np.array_equal(again.get_mat().mvprod(x), y)
