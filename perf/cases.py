"""The work a user of this library has it do, as measured cases.

The library's path is: integrals, rotated by the orbital optimiser -> strings ->
Slater-Condon matrix (stored, or applied on the fly) -> ground state -> density
matrices, one request at a time or in batches of requests.  Every step of it is
a case of its own (a rotation, a build, each kind of product, the density
matrices), and three kinds of whole calls are cases too: one step of an orbital
optimisation, and the two kinds of batched solves that the served stream sends.

  listed()            the measured cases
  draw(rng)           another case of the same ranges
  prepare(case, seed) integrals, vectors and the handles that a program keeps
  run(state)          one pass through the public entry points
  exact(case, seed)   the same results from plain torch / numpy in 64 bits
  work(case), tolerance(case)
"""
import math

import numpy as np
import torch

import ciflow_amd as CA

DEV = "cuda"
SERVED_STOP = 1e-9  # energy stop of the served stream (Eh)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: one step of the DOCI orbital minimiser (rotate, new
        # integrals, solve, 2-RDM) in a minimal basis; latency and launches.
        {"name": "step_doci_L10", "op": "step", "kind": "DOCI", "L": 10, "nup": 5, "ndown": 5},
        # The same step for a small FCI space (4,900 determinants).
        {"name": "step_fci_L8", "op": "step", "kind": "FCI", "L": 8, "nup": 4, "ndown": 4},
        # 48 small DOCI solves of one stream shape: one launch for all.
        {"name": "batch_doci_L14_x48", "op": "batch_small", "L": 14, "npair": 7, "count": 48},
        # Larger DOCI solves of the stream, advanced together (odd L: 9 pairs of 19 orbitals).
        {"name": "batch_doci_L19_x12", "op": "batch", "kind": "DOCI", "L": 19, "nup": 9, "ndown": 9, "count": 12},
        # The largest solves of the stream: FCI of 213,444 determinants, on-the-fly product.
        {"name": "batch_fci_L11_x12", "op": "batch", "kind": "FCI", "L": 11, "nup": 5, "ndown": 5, "count": 12},
        # Build of a stored FCI matrix of ragged shape (462 x 330 strings) and its first product.
        {"name": "build_fci_L11_5a4b", "op": "build", "L": 11, "nup": 5, "ndown": 4, "prec": "f64"},
        # Product with the largest stored matrix (1.55e9 nonzeros): what a stored solve repeats.
        {"name": "product_fci_L12", "op": "product", "kind": "FCI", "L": 12, "nup": 6, "ndown": 6, "prec": "f64"},
        # DOCI product, 11 pairs of 23 orbitals (1,352,078 determinants).
        {"name": "product_doci_L23", "op": "product", "kind": "DOCI", "L": 23, "nup": 11, "ndown": 11, "prec": "f64"},
        # FCI product without a stored matrix.
        {"name": "sigma_fci_L12", "op": "sigma", "L": 12, "nup": 6, "ndown": 6, "prec": "f64"},
        # Selected CI: matrix of a determinant list and its first product, FP32 values.
        {"name": "selected_L12_6a5b", "op": "selected", "L": 12, "nup": 6, "ndown": 5, "list": "block",
         "count": 95040, "prec": "f32"},
        # 1- and 2-RDM of an FCI vector.
        {"name": "rdm_fci_L11", "op": "rdm", "kind": "FCI", "L": 11, "nup": 5, "ndown": 5},
        # Integral rotations of a batch of candidates, arrays on the GPU.
        {"name": "rotate_L18_x16", "op": "rotate", "L": 18, "count": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["step", "step", "batch_small", "batch", "batch", "build", "product", "product", "sigma", "selected",
                     "rdm", "rotate"])
    if op == "rotate":
        L = rng.randint(6, 24)
        return {"op": op, "L": L, "count": _log_int(rng, 1, max(1, min(64, (1 << 21) // L ** 4)))}
    if op == "batch_small":
        L = rng.randint(12, 16)
        return {"op": op, "L": L, "npair": L // 2 - rng.randint(0, 1), "count": _log_int(rng, 4, 64)}
    if op == "batch":
        if rng.random() < 0.5:
            L = rng.randint(17, 20)
            return {"op": op, "kind": "DOCI", "L": L, "nup": L // 2, "ndown": L // 2, "count": _log_int(rng, 2, 12)}
        L = rng.randint(8, 11)
        return {"op": op, "kind": "FCI", "L": L, "nup": L // 2, "ndown": L // 2,
                "count": _log_int(rng, 2, {8: 32, 9: 32, 10: 16, 11: 8}[L])}
    if op == "step":
        if rng.random() < 0.5:
            L = rng.randint(6, 16)
            n = rng.randint(max(2, L // 2 - 2), L // 2)
            return {"op": op, "kind": "DOCI", "L": L, "nup": n, "ndown": n}
        L = rng.randint(5, 9)
        return {"op": op, "kind": "FCI", "L": L, "nup": rng.randint(2, L // 2), "ndown": rng.randint(2, L // 2)}
    if op == "rdm":
        if rng.random() < 0.3:
            L = rng.randint(10, 20)
            n = rng.randint(L // 2 - 2, L // 2)
            return {"op": op, "kind": "DOCI", "L": L, "nup": n, "ndown": n}
        L = rng.randint(7, 11)
        return {"op": op, "kind": "FCI", "L": L, "nup": rng.randint(3, L // 2), "ndown": rng.randint(3, L // 2)}
    prec = rng.choice(["f64", "f32"])
    if op == "product" and rng.random() < 0.5:
        L = rng.randint(18, 23)
        n = rng.randint(L // 2 - 3, L // 2)
        return {"op": op, "kind": "DOCI", "L": L, "nup": n, "ndown": n, "prec": prec}
    if op in ("product", "sigma"):
        L = rng.randint(9, 12)
        c = {"op": op, "L": L, "nup": rng.randint(3, L // 2), "ndown": rng.randint(3, L // 2), "prec": prec}
        return dict(c, kind="FCI") if op == "product" else c
    if op == "build":
        L = rng.randint(8, 11)
        return {"op": op, "L": L, "nup": rng.randint(3, L // 2), "ndown": rng.randint(3, 4), "prec": prec}
    L = rng.randint(10, 13)
    nup, ndown = rng.randint(L // 2 - 1, L // 2), rng.randint(L // 2 - 1, L // 2)
    n = math.comb(L, nup) * math.comb(L, ndown)
    return {"op": op, "L": L, "nup": nup, "ndown": ndown, "list": rng.choice(["block", "random"]),
            "count": _log_int(rng, 2000, min(100000, n // 2)), "prec": prec}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _rng(seed, *key):
    return np.random.default_rng([int(seed), *key])


def _integrals(L, rng):
    """h[L, L] and physics V[L, L, L, L]: an orbital-energy ramp with small
    hoppings, and (ij|kl) = sum_P B^P_ij B^P_kl over 2L symmetric B^P with the
    dominant on-site parts (positive semi-definite, eight-fold symmetric)."""
    h = rng.normal(0.0, 0.05, (L, L))
    h = (h + h.T) / math.sqrt(2.0)
    h[np.arange(L), np.arange(L)] = -2.0 + 3.0 * np.arange(L) / max(L - 1, 1)
    B = rng.normal(0.0, 0.1, (2 * L, L, L))
    B = np.tril(B) + np.tril(B, -1).transpose(0, 2, 1)
    B[np.arange(L), np.arange(L), np.arange(L)] += 0.6
    B = B.reshape(2 * L, L * L)
    V = (B.T @ B).reshape(L, L, L, L).transpose(0, 2, 1, 3)
    return np.ascontiguousarray(h), np.ascontiguousarray(V)


def _rotation(L, rng):
    """U = exp(K), K antisymmetric with N(0, 0.05^2) entries."""
    K = np.triu(rng.normal(0.0, 0.05, (L, L)), 1)
    return torch.linalg.matrix_exp(torch.from_numpy(K - K.T)).numpy()


def _requests(case, seed):
    L = case["L"]
    out = []
    for k in range(case["count"]):
        rng = _rng(seed, 1, k)
        h, V = _integrals(L, rng)
        out.append({"h": h, "V": V, "U": _rotation(L, rng), "tag": k})
    return out


def _dim(case):
    if case.get("kind") == "DOCI":
        return math.comb(case["L"], case["nup"])
    return math.comb(case["L"], case["nup"]) * math.comb(case["L"], case["ndown"])


def _vector(n, seed, unit=False):
    x = torch.from_numpy(_rng(seed, 2).standard_normal(n))
    return x / x.norm() if unit else x


def _strings(L, n):
    """All L-bit strings with n bits set, ascending."""
    s = np.arange(1 << L, dtype=np.uint32)
    c = np.zeros(1 << L, dtype=np.uint8)
    for b in range(L):
        c += ((s >> b) & 1).astype(np.uint8)
    return s[c == n].astype(np.int64)


def _det_list(case, seed):
    """(rank of the alpha string, rank of the beta string) of each determinant:
    the lowest alpha strings times every beta string in order, or a random
    subset of the space in random order (a list sorted by importance)."""
    da, db = math.comb(case["L"], case["nup"]), math.comb(case["L"], case["ndown"])
    if case["list"] == "block":
        i = np.arange(min(case["count"], da * db))
    else:
        i = _rng(seed, 3).permutation(da * db)[: case["count"]]
    return i // db, i % db


PREC = {"f64": CA.CF_F64, "f32": CA.CF_F32}


def prepare(case, seed):
    op, L = case["op"], case["L"]
    st = {"op": op}
    if op == "batch_small":
        st["reqs"] = [dict(q, npair=case["npair"], tol_energy=SERVED_STOP, check_every=2) for q in _requests(case, seed)]
        return st
    if op == "batch":
        kind = CA.CF_DOCI if case["kind"] == "DOCI" else CA.CF_FCI
        st["reqs"] = [dict(q, kind=kind, nup=case["nup"], ndown=case["ndown"], precision=CA.CF_PREC_AUTO,
                           tol_energy=SERVED_STOP) for q in _requests(case, seed)]
        return st
    if op == "rotate":
        q = _requests(case, seed)
        for key in ("h", "V", "U"):
            st[key] = torch.from_numpy(np.stack([r[key] for r in q])).to(DEV)
        st["h_out"], st["V_out"] = torch.empty_like(st["h"]), torch.empty_like(st["V"])
        st.update(L=L, count=case["count"], ctx=CA.default_context())
        return st
    h, V = _integrals(L, _rng(seed, 1, 0))
    if op == "step":
        from ciflow_amd.optimize import OrbitalOptimization
        kind = CA.CF_DOCI if case["kind"] == "DOCI" else CA.CF_FCI
        st["opt"] = OrbitalOptimization(h, V, case["nup"], case["ndown"], 0.0, kind)
        st["U"] = _rotation(L, _rng(seed, 4))
        return st
    st["ham"] = ham = CA.Hamiltonian(h, V, case["nup"], case["ndown"])
    if op == "rdm":
        st["ci"] = (CA.DOCI if case["kind"] == "DOCI" else CA.FCI)(ham, build=False)
        st["c"] = _vector(_dim(case), seed, unit=True).numpy()
        return st
    st["prec"] = prec = PREC[case["prec"]]
    if op == "selected":
        ia, ib = _det_list(case, seed)
        st["dets"] = (_strings(L, case["nup"])[ia].astype(np.uint64), _strings(L, case["ndown"])[ib].astype(np.uint64))
        n = len(ia)
    else:
        n = _dim(case)
    st["x"] = _vector(n, seed).to(DEV)
    st["y"] = torch.empty_like(st["x"])
    if op == "product":
        st["ci"] = (CA.DOCI if case["kind"] == "DOCI" else CA.FCI)(ham, value_prec=prec)
        st["mat"] = st["ci"].get_mat()
    elif op == "sigma":
        st["ci"] = CA.FCI_Direct(ham, value_prec=prec)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _ok(status):
    if status != CA.CF_OK:
        raise CA.CIFlowError(status, (CA.lib().cf_last_error() or b"").decode())


def _product(st, mat):
    _ok(CA.lib().cf_mvprod_dev(mat.ptr, st["prec"], st["x"].data_ptr(), st["y"].data_ptr()))
    return st["y"]


def _energies(results):
    for r in results:
        if r["status"] != CA.CF_OK or r["solve_status"] != 0:
            raise RuntimeError(f"request {r['tag']}: {r['error'] or 'not converged'}")
    return np.array([r["energy"] for r in results])


def run(st):
    op = st["op"]
    if op == "step":
        opt = st["opt"]
        opt.U = st["U"]
        e = opt.update_cim()
        one, two = opt.cim.density_dense()
        return {"energy": e, "one": one, "two": two}
    if op == "batch_small":
        return _energies(CA.solve_doci_batch(st["reqs"]))
    if op == "batch":
        return _energies(CA.solve_batch(st["reqs"]))
    if op == "build":
        ci = CA.FCI(st["ham"], value_prec=st["prec"])
        n, nnz, upper = ci.get_mat().info()
        return {"n": n, "nnz": nnz, "upper": upper, "y": _product(st, ci.get_mat())}
    if op == "selected":
        ci = CA.FCI_File(st["ham"], st["dets"], value_prec=st["prec"])
        n, nnz, upper = ci.get_mat().info()
        return {"n": n, "nnz": nnz, "upper": upper, "y": _product(st, ci.get_mat())}
    if op == "product":
        return _product(st, st["mat"])
    if op == "sigma":
        _ok(CA.lib().cf_sigma_apply_dev(st["ci"].sig.ptr, st["prec"], st["x"].data_ptr(), st["y"].data_ptr()))
        return st["y"]
    if op == "rdm":
        return st["ci"].density_dense(st["c"])
    p = [st[k].data_ptr() for k in ("h", "V", "U", "h_out", "V_out")]
    _ok(CA.lib().cf_rotate_integrals_noalloc(st["ctx"].ptr, st["L"], st["count"], *p))
    return st["h_out"], st["V_out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
NOMINAL_PRODUCTS = 40  # products of one solve to the served energy stop, for scale


def _row(L, na, nb, kind="FCI"):
    if kind == "DOCI":
        return 1 + na * (L - na)
    sa, sb = na * (L - na), nb * (L - nb)
    dd = lambda n: math.comb(n, 2) * math.comb(L - n, 2)  # noqa: E731
    return (1 + sa) * (1 + sb) + dd(na) + dd(nb)


def work(case):
    op, L = case["op"], case["L"]
    ints = 8.0 * (L ** 4 + 2 * L ** 2)
    if op == "rotate":
        return {"bytes": case["count"] * (2 * ints - 8.0 * L ** 2), "flops": case["count"] * (8.0 * L ** 5 + 4.0 * L ** 3)}
    if op == "batch_small":
        row = _row(L, case["npair"], case["npair"], "DOCI")
        return {"bytes": case["count"] * ints,
                "flops": case["count"] * NOMINAL_PRODUCTS * 2.0 * math.comb(L, case["npair"]) * row}
    n = _dim(case)
    row = _row(L, case["nup"], case["ndown"], case.get("kind", "FCI"))
    if op == "batch":
        return {"bytes": case["count"] * ints, "flops": case["count"] * NOMINAL_PRODUCTS * 2.0 * n * row}
    if op == "step":
        return {"bytes": 2 * ints + 8.0 * n + 24.0 * L ** 4, "flops": 8.0 * L ** 5 + NOMINAL_PRODUCTS * 2.0 * n * row}
    if op == "rdm":
        f = n * L ** 2 if case["kind"] == "DOCI" else 6.0 * n * L ** 4
        return {"bytes": 8.0 * n + 24.0 * L ** 4, "flops": float(f)}
    s = 4 if case["prec"] == "f32" else 8
    if op == "selected":
        n = min(case["count"], n)
        # a block of da' x db strings keeps about da'/da of a row's alpha excitations
        keep = n / _dim(case) if case["list"] == "random" else 0.25
        nnz = max(n, n * row * keep)
        return {"bytes": 16.0 * n + nnz * (s + 12 if s == 4 else 12) + 16.0 * n, "flops": 2.0 * nnz}
    if op == "build":
        return {"bytes": ints + n * row * (s + 12 if s == 4 else 12) + 8.0 * n + 16.0 * n, "flops": 2.0 * n * row}
    if op == "product" and case["kind"] == "FCI":
        return {"bytes": n * row * s + 16.0 * n, "flops": 2.0 * n * row}
    if op == "product":
        return {"bytes": 24.0 * n, "flops": 2.0 * n * row}
    return {"bytes": ints + 16.0 * n, "flops": 2.0 * n * row}  # sigma


def tolerance(case):
    op = case["op"]
    if op in ("batch", "batch_small"):
        return {"rel": 1e-10, "max": 1e-10}  # the energy stop, 1e-9 Eh of 10 to 60 Eh
    if op == "step":
        return {"rel": 1e-10, "max": 1e-8}  # densities of a vector with residual 1e-12 |E|, over the gap
    if op == "rdm":
        return {"rel": 4e-14, "max": 4e-12}  # FP64 sums over the determinants, 1e-14 seen
    if op != "rotate" and case["prec"] == "f32":
        return {"rel": 1e-7, "max": 1e-6}  # elements rounded to FP32: 2.3e-8 seen
    return {"rel": 4e-15, "max": 4e-13}  # FP64 sums of at most some thousand terms, 1e-15 seen


# ---------------------------------------------------------------------------
# the same results in plain torch / numpy, 64 bits
# ---------------------------------------------------------------------------
class _Excite:
    """E_pq = a+_p a_q on the n-electron strings of L orbitals: for each pair
    (p, q) and target string K, the source string and the sign (0: none)."""

    def __init__(self, L, n):
        s = _strings(L, n)
        rank = np.full(1 << L, 0, dtype=np.int64)
        rank[s] = np.arange(len(s))
        src = np.zeros((L * L, len(s)), dtype=np.int64)
        sgn = np.zeros((L * L, len(s)))
        bits = ((s[:, None] >> np.arange(L)) & 1).astype(np.int64)
        below = np.concatenate([np.zeros((len(s), 1), dtype=np.int64), np.cumsum(bits, 1)], 1)  # electrons under p
        for p in range(L):
            for q in range(L):
                if p == q:
                    src[p * L + q], sgn[p * L + q] = np.arange(len(s)), bits[:, p]
                    continue
                ok = (bits[:, p] == 1) & (bits[:, q] == 0)  # target holds p, source held q
                lo, hi = min(p, q), max(p, q)
                between = below[:, hi] - below[:, lo + 1]
                src[p * L + q] = np.where(ok, rank[np.where(ok, s ^ (1 << p) ^ (1 << q), s)], 0)
                sgn[p * L + q] = np.where(ok, 1.0 - 2.0 * (between & 1), 0.0)
        self.d = len(s)
        self.src, self.sgn = torch.from_numpy(src).to(DEV), torch.from_numpy(sgn).to(DEV)


class _Fci:
    """sigma = H c of the full space from D_pq = E_pq c: sum_pq E_pq (k_pq c +
    1/2 sum_rs (pq|rs) D_rs), k_pq = h_pq - 1/2 sum_r (pr|rq)."""

    def __init__(self, h, V, L, na, nb):
        self.L = L
        self.a = _Excite(L, na)
        self.b = self.a if na == nb else _Excite(L, nb)
        self.set(h, V)

    def set(self, h, V):
        L = self.L
        k = h - 0.5 * np.einsum("prrq->pq", V)
        self.k = torch.from_numpy(k.reshape(-1)).to(DEV)
        self.G = torch.from_numpy(np.ascontiguousarray(V.transpose(0, 2, 1, 3)).reshape(L * L, L * L)).to(DEV)

    def parts(self, C, spin):
        D = torch.empty(self.L ** 2, self.a.d, self.b.d, dtype=torch.float64, device=DEV)
        for i in range(self.L ** 2):
            if spin == 0:
                D[i] = C[self.a.src[i]] * self.a.sgn[i][:, None]
            else:
                D[i] = C[:, self.b.src[i]] * self.b.sgn[i][None, :]
        return D

    def __call__(self, c):
        C = c.view(self.a.d, self.b.d)
        D = self.parts(C, 0)
        for i in range(self.L ** 2):
            D[i] += C[:, self.b.src[i]] * self.b.sgn[i][None, :]
        X = (0.5 * self.G) @ D.view(self.L ** 2, -1)
        del D
        X += self.k[:, None] * c[None, :]
        X = X.view(self.L ** 2, self.a.d, self.b.d)
        y = torch.zeros_like(C)
        for i in range(self.L ** 2):
            y += X[i][self.a.src[i]] * self.a.sgn[i][:, None]
            y += X[i][:, self.b.src[i]] * self.b.sgn[i][None, :]
        return y.reshape(-1)

    def densities(self, c):
        """gamma[2][p][q] = <E_pq>, Gamma[aa, ab, bb][i][j][k][l] = <a+_i a+_j a_l a_k>."""
        L, C = self.L, c.view(self.a.d, self.b.d)
        D = [self.parts(C, s).view(L * L, -1) for s in (0, 1)]
        g = torch.stack([(d @ c).view(L, L) for d in D])
        blocks = []
        for s, t in ((0, 0), (0, 1), (1, 1)):
            P = (D[s] @ D[t].T).view(L, L, L, L)  # [k, i, j, l] = <E_ik E_jl>
            Q = P.permute(1, 2, 0, 3).clone()
            if s == t:
                for j in range(L):
                    Q[:, j, j, :] -= g[s]
            blocks.append(Q)
        return g, torch.stack(blocks)


class _Doci:
    """Pair hops <ii|jj> between pair strings, 2 h + V on the diagonal."""

    def __init__(self, h, V, L, n):
        s = _strings(L, n)
        rank = np.zeros(1 << L, dtype=np.int32)
        rank[s] = np.arange(len(s))
        self.L, self.s = L, s
        self.occ = torch.from_numpy(((s[:, None] >> np.arange(L)) & 1).astype(np.float64)).to(DEV)
        self.rank = torch.from_numpy(rank).to(DEV)
        self.sd = torch.from_numpy(s).to(DEV)
        self.set(h, V)

    def set(self, h, V):
        i = np.arange(self.L)
        J, K = V[i[:, None], i[None, :], i[:, None], i[None, :]], V[i[:, None], i[None, :], i[None, :], i[:, None]]
        W = 2 * J - K
        W[i, i] = 0.0
        e = torch.from_numpy(2 * h[i, i] + V[i, i, i, i]).to(DEV)
        self.diag = self.occ @ e + ((self.occ @ torch.from_numpy(W).to(DEV)) * self.occ).sum(1)
        self.pair = V[i[:, None], i[:, None], i[None, :], i[None, :]]

    def __call__(self, c):
        y = self.diag * c
        for p in range(self.L):
            for q in range(p + 1, self.L):
                m = (1 << p) | (1 << q)
                t = (self.sd & m)
                hop = (t != 0) & (t != m)
                j = self.rank[torch.where(hop, self.sd ^ m, self.sd)].long()
                y += torch.where(hop, c[j], 0.0) * float(self.pair[p, q])
        return y

    def densities(self, c):
        """gamma and Gamma of the pair state."""
        L = self.L
        n = (self.occ.T @ (c * c)).cpu().numpy()
        nn = (self.occ.T @ (self.occ * (c * c)[:, None])).cpu().numpy()
        g = np.zeros((2, L, L))
        G = np.zeros((3, L, L, L, L))
        for p in range(L):
            g[:, p, p] = n[p]
            G[1, p, p, p, p] = n[p]
            for q in range(L):
                if p == q:
                    continue
                G[0, p, q, p, q] = G[2, p, q, p, q] = G[1, p, q, p, q] = nn[p, q]
                G[0, p, q, q, p] = G[2, p, q, q, p] = -nn[p, q]
                m = (1 << p) | (1 << q)
                t = (self.sd & m)
                hop = t == (1 << q)  # a pair moves from q to p
                j = self.rank[torch.where(hop, self.sd ^ m, self.sd)].long()
                G[1, p, p, q, q] = float((torch.where(hop, c[j] * c, 0.0)).sum())
        return torch.from_numpy(g), torch.from_numpy(G)


def _ground(op, n, steps=90, tol=2e-13, restarts=12):
    """Lowest eigenpair by Lanczos with full re-orthogonalisation, restarted on the Ritz vector."""
    gen = torch.Generator().manual_seed(7)
    v = torch.randn(n, dtype=torch.float64, generator=gen).to(DEV)
    for _ in range(restarts):
        v /= v.norm()
        m = min(steps, n)
        Q = torch.zeros(m, n, dtype=torch.float64, device=DEV)
        T = np.zeros((m, m))
        Q[0] = v
        k = m
        for j in range(m):
            w = op(Q[j])
            for _ in range(2):
                cf = Q[: j + 1] @ w
                w -= Q[: j + 1].T @ cf
                T[j, j] += float(cf[j])
            b = float(w.norm())
            if j + 1 < m:
                if b < 1e-12:
                    k = j + 1
                    break
                T[j, j + 1] = T[j + 1, j] = b
                Q[j + 1] = w / b
        _, Y = np.linalg.eigh(T[:k, :k])
        v = Q[:k].T @ torch.from_numpy(Y[:, 0].copy()).to(DEV)
        v /= v.norm()
        hv = op(v)
        e = float(v @ hv)
        if float((hv - e * v).norm()) <= tol * abs(e) or k == n:
            break
    if v[v.abs().argmax()] < 0:
        v = -v
    return e, v


def _rotate_plain(h, V, U):
    h, V, U = (torch.from_numpy(np.ascontiguousarray(x)).to(DEV) for x in (h, V, U))
    L = h.shape[0]
    for _ in range(4):  # each pass takes the leading index and appends the new one
        V = (V.reshape(L, -1).T.contiguous() @ U.T.contiguous()).reshape(L, L, L, L)
    return (U @ h @ U.T).cpu().numpy(), V.contiguous().cpu().numpy()


def _model(case, h, V):
    if case.get("kind", "FCI") == "DOCI" or case["op"] == "batch_small":
        return _Doci(h, V, case["L"], case.get("npair", case.get("nup")))
    return _Fci(h, V, case["L"], case["nup"], case["ndown"])


def exact(case, seed):
    op, L = case["op"], case["L"]
    if op == "rotate":
        out = [_rotate_plain(q["h"], q["V"], q["U"]) for q in _requests(case, seed)]
        return np.stack([o[0] for o in out]), np.stack([o[1] for o in out])
    if op in ("batch", "batch_small"):
        n = math.comb(L, case["npair"]) if op == "batch_small" else _dim(case)
        if n * case["count"] > 2_600_000:
            return None  # more than a few seconds in plain torch
        model, out = None, []
        for q in _requests(case, seed):
            h, V = _rotate_plain(q["h"], q["V"], q["U"])
            if model is None:
                model = _model(case, h, V)
            else:
                model.set(h, V)
            out.append(_ground(model, n, steps=60, tol=1e-8)[0])
        return np.array(out)
    h, V = _integrals(L, _rng(seed, 1, 0))
    if op == "step":
        model = _model(case, *_rotate_plain(h, V, _rotation(L, _rng(seed, 4))))
        e, v = _ground(model, _dim(case))
        one, two = model.densities(v)
        return {"energy": e, "one": one.cpu(), "two": two.cpu()}
    model = _model(case, h, V)
    if op == "rdm":
        c = _vector(_dim(case), seed, unit=True).to(DEV)
        one, two = model.densities(c)
        return one.cpu(), two.cpu()
    if op == "selected":
        ia, ib = _det_list(case, seed)
        at = torch.from_numpy(ia * model.b.d + ib).to(DEV)
        full = torch.zeros(model.a.d * model.b.d, dtype=torch.float64, device=DEV)
        full[at] = _vector(len(ia), seed).to(DEV)
        return {"n": None, "nnz": None, "upper": None, "y": model(full)[at]}
    y = model(_vector(_dim(case), seed).to(DEV))
    return {"n": None, "nnz": None, "upper": None, "y": y} if op == "build" else y
