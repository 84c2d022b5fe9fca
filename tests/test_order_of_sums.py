"""The order in which fullchem's solvers add their sums (chunks of 32 terms,
backward rows by descending column, Jacobian terms by batch: mechgen/
cell_sched.py) rounds no worse than the plain order (every sum term by term in
ascending order).

One Rodas3 attempt of the 72 cells of the committed fullchem inputs is computed
in both orders in 64 bits and once in 80-bit extended precision (11 more bits,
so its own error is 2,000 times smaller), all cells side by side.  The errors
of a cell's species are averaged; their ratio's geometric mean over the cells
is 0.77, 0.59 and 0.71 for steps of 1, 60 and 1200 s.  (A solution in 64 bits,
pivoted or not, is no reference here: its own error is as large as either's.)
"""
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "geos-chem_amd" / "mechgen"))


@pytest.fixture(scope="module")
def cells(fullchem):
    conc, rct = [], []
    for f in ("fullchem_box", "fullchem_het"):
        d = np.load(ROOT / "tests" / "golden" / (f + ".npz"))
        conc.append(d["conc"])
        rct.append(d["rconst"])
    return np.concatenate(conc, 1), np.concatenate(rct, 1)


@pytest.fixture(scope="module")
def tables(fullchem):
    """The tables in the solvers' order and in the plain one."""
    import cell_sched as C
    from emit_tables import build_tables
    m = fullchem
    raw = {"nvar": m.nvar, "nfix": m.nfix, "nspec": m.nspec, "nreact": m.nreact,
           "lu_nonzero": m.lu_nonzero, "reactions": m.reactions, "lu_irow": m.lu_irow.tolist(),
           "lu_icol": m.lu_icol.tolist(), "lu_crow": m.lu_crow.tolist(), "lu_diag": m.lu_diag.tolist()}
    solver = build_tables(raw)
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(C, "tail_size", lambda m: 0)
        plain = build_tables(raw)
    return raw, solver, plain, C.CHUNK, m.nvar - C.tail_size(raw)


def attempt(raw, t, conc, rct, H, dtype, chunk, s):
    """Ynew of one Rodas3 attempt with step H; chunk 0: the plain order."""
    nv, crow, diag, icol = raw["nvar"], raw["lu_crow"], raw["lu_diag"], raw["lu_icol"]
    Y, R, h = conc.astype(dtype), rct.astype(dtype), dtype(H)

    def total(init, terms, nhead):
        acc, tot = init, None
        for n, (a, b) in enumerate(terms):
            if chunk and n < nhead and n and n % chunk == 0:
                tot, acc = (acc if tot is None else tot + acc), np.zeros_like(init)
            if n == nhead and tot is not None:
                acc, tot = tot + acc, None
            acc = acc + a * b
        return acc if tot is None else tot + acc

    zero = np.zeros(conc.shape[1], dtype)

    def fun(y):
        a = R.copy()
        for r in range(raw["nreact"]):
            for sp in t["rx_s"][3 * r:3 * r + 3]:
                if sp >= 0:
                    a[r] = a[r] * y[sp]
        return np.stack([total(zero, [(dtype(t["fv_c"][x]), a[t["fv_r"][x]])
                                      for x in range(t["fv_ptr"][i], t["fv_ptr"][i + 1])], 1 << 30)
                         for i in range(nv)])

    part = []
    for p, r in enumerate(t["pt_r"]):
        v = dtype(t["pt_m"][p]) * R[r]
        for sp in t["pt_s"][2 * p:2 * p + 2]:
            if sp >= 0:
                v = v * Y[sp]
        part.append(v)
    lu = [-total(zero, [(dtype(t["jv_c"][x]), part[t["jv_b"][x]])
                        for x in range(t["jv_ptr"][q], t["jv_ptr"][q + 1])], 1 << 30)
          for q in range(raw["lu_nonzero"])]
    for i in range(nv):
        lu[diag[i]] = lu[diag[i]] + 1 / (h * dtype(0.5))
    for q in range(raw["lu_nonzero"]):
        v = total(lu[q], [(-lu[t["cr_l"][x]], lu[t["cr_u"][x]])
                          for x in range(t["cr_ptr"][q], t["cr_ptr"][q + 1])], t["cr_hd"][q] - t["cr_ptr"][q])
        lu[q] = v / lu[t["cr_div"][q]] if t["cr_div"][q] >= 0 else v

    def solve(b):
        x = list(b)
        for i in range(nv):
            x[i] = total(x[i], [(-lu[k], x[icol[k]]) for k in range(crow[i], diag[i])], t["fw_hd"][i] - crow[i])
        for i in range(nv - 1, -1, -1):
            ks = list(range(diag[i] + 1, crow[i + 1]))
            if chunk:
                ks.reverse()
            x[i] = total(x[i], [(-lu[k], x[icol[k]]) for k in ks], len(ks) if i < s else 0) / lu[diag[i]]
        return np.stack(x)

    var, fix = Y[:nv], Y[nv:]
    f0 = fun(Y)
    k1 = solve(f0)
    k2 = solve(f0 + dtype(4) / h * k1)
    y = np.concatenate([var + 2 * k1, fix])
    k3 = solve(fun(y) + (k1 - k2) / h)
    y = np.concatenate([var + 2 * k1 + k3, fix])
    k4 = solve(fun(y) + (k1 - k2 - dtype(8) / dtype(3) * k3) / h)
    return var + 2 * k1 + k3 + k4


@pytest.mark.parametrize("H", [1.0, 60.0, 1200.0])
def test_the_solvers_order_rounds_no_worse(H, cells, tables):
    conc, rct = cells
    raw, solver, plain, chunk, s = tables
    ext = attempt(raw, plain, conc, rct, H, np.longdouble, 0, s)
    err = []
    for t, c in ((solver, chunk), (plain, 0)):
        y = attempt(raw, t, conc, rct, H, np.float64, c, s)
        err.append((np.abs(y - ext) / np.maximum(np.abs(ext), 1e-2)).mean(0).astype(float))
    ratio = np.exp(np.log(err[0] / err[1]).mean())
    print("H %g: geometric mean of the error ratio %.3f, median errors %.2e and %.2e"
          % (H, ratio, np.median(err[0]), np.median(err[1])))
    assert ratio <= 1.0
