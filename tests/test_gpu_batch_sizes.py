"""GPU tests of cf_solve_doci_batch over its workgroup shapes and splits: spaces
of 2 to 12,870 rows, on either side of the shapes' bounds (1,001 and 1,140 rows;
4,060 and 4,495), more requests than fill the GPU and than a grid dimension, and
requests that stop early, late and at the step limit, against dense eigenvalues
or the stored-matrix solve; the residual estimate against Lanczos in numpy."""
import numpy as np
import pytest

import ciflow_amd as CA

pytestmark = pytest.mark.gpu


def request(L, npair, seed):
    h, V = CA.gen_integrals(L, seed)
    return {"h": h, "V": V, "npair": npair, "U": CA.expm_skew(CA.gen_rotation(L, seed, 0.05))}


def stored_energy(q):
    h, V = CA.rotate_integrals(q["h"], q["V"], q["U"])
    ci = CA.DOCI(CA.Hamiltonian(h, V, q["npair"], q["npair"]))
    if ci.n <= 1001:
        row, col, val = ci.get_mat().export_full()
        A = np.zeros((ci.n, ci.n))
        for i in range(ci.n):
            A[i, col[row[i]:row[i + 1]]] = val[row[i]:row[i + 1]]
        return np.linalg.eigvalsh(A)[0]
    ci.solve()
    return ci.get_ci_energy()


@pytest.mark.parametrize("L,npair", [(2, 1), (4, 2), (8, 4), (12, 6), (14, 4), (13, 8), (14, 7), (15, 6), (16, 8),
                                     (32, 1), (28, 2), (20, 3), (30, 3), (31, 3), (25, 4)])
def test_batch_sizes(L, npair):
    q = request(L, npair, 40 + L + npair)
    res = CA.solve_doci_batch([dict(q), dict(q, tol=1e-9), dict(q, tol_energy=1e-9)])
    E = stored_energy(q)
    for r, tol in zip(res, (1e-10, 1e-9, 1e-8)):
        assert r["status"] == 0 and r["solve_status"] == 0
        assert abs(r["energy"] - E) <= tol, (r["n"], r["n_matvec"], r["energy"], E)


def test_more_requests_than_workgroups_fill_the_gpu():
    qs = [request(10, 5, 500 + k) for k in range(4)]
    alone = [CA.solve_doci_batch([q])[0] for q in qs]
    res = CA.solve_doci_batch([qs[k % 4] for k in range(1100)])   # one workgroup per request
    for k, r in enumerate(res):
        assert r["energy"] == alone[k % 4]["energy"] and r["n_matvec"] == alone[k % 4]["n_matvec"]


def test_requests_that_finish_at_different_steps():
    """An energy stop, the default tolerance and one that no residual meets, in one
    launch sequence: early ones stay as they are alone while the last takes 400 steps."""
    qs = [dict(request(12, 6, 700), tol_energy=1e-3), request(12, 6, 701), dict(request(12, 5, 702), tol=1e-300),
          dict(request(8, 4, 703), tol_energy=1e-9), dict(request(12, 6, 704), tol=1e-6)]
    alone = [CA.solve_doci_batch([q])[0] for q in qs]
    assert [r["solve_status"] for r in alone] == [0, 0, 1, 0, 0] and alone[2]["n_matvec"] == 400
    assert len({r["n_matvec"] for r in alone}) >= 4
    for _ in range(3):
        for a, r in zip(alone, CA.solve_doci_batch(qs)):
            assert all(a[k] == r[k] for k in ("energy", "resid", "n_matvec", "solve_status"))
    assert abs(alone[2]["energy"] - stored_energy(qs[2])) <= 1e-10


def lanczos_residual(q, m):
    """|last residual| of m steps of plain Lanczos on the stored matrix from the solver's start vector."""
    h, V = CA.rotate_integrals(q["h"], q["V"], q["U"])
    mat = CA.DOCI(CA.Hamiltonian(h, V, q["npair"], q["npair"])).get_mat()
    row, col, val = mat.export_full()
    k = np.uint64(20240601) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, len(row), dtype=np.uint64)
    k = (k ^ (k >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    k = (k ^ (k >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    k ^= k >> np.uint64(31)
    v = 1.0 + 0.5 * ((k >> np.uint64(11)) / 2.0 ** 53 - 0.5)
    v, vp, b, al, be = v / np.linalg.norm(v), 0.0 * v, 0.0, [], []
    for _ in range(m):
        w = np.add.reduceat(val * v[col], row[:-1].astype(np.int64))
        al.append(v @ w)
        w = w - al[-1] * v - b * vp
        b = np.linalg.norm(w)
        be.append(b)
        vp, v = v, w / b
    T = np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1)
    return b * abs(np.linalg.eigh(T)[1][-1, 0])


def test_residual_estimates():
    """The estimate that a solve stops on and returns.  At tol 0.02 a solve stops after 10 to 20
    steps, where two Lanczos runs in FP64 agree to about 5e-15; the last component moves by up
    to ten times that (1e-13 allowed; eigenvalues of T taken to 1e-13 gave up to 4.5e-13)."""
    for L, npair in ((9, 4), (10, 5), (12, 6)):
        for seed in range(4):
            q = dict(request(L, npair, 800 + seed), tol=2e-2)
            r = CA.solve_doci_batch([q])[0]
            want = lanczos_residual(q, r["n_matvec"])
            assert abs(r["resid"] - want) <= 1e-13 * want, (L, seed, r["n_matvec"], r["resid"] / want - 1)


def test_more_requests_than_a_grid_dimension():
    q = request(2, 1, 600)
    alone = CA.solve_doci_batch([q])[0]
    res = CA.solve_doci_batch([q] * 70000)
    assert len(res) == 70000
    for r in res:
        assert r["status"] == 0 and r["energy"] == alone["energy"] and r["n_matvec"] == alone["n_matvec"]
