"""The cell programs (mechgen/cell_sched.py) compute every sum of a Rodas3
attempt in the order the lane-per-cell solvers walk the tables: executed
round by round on the CPU (one IEEE double operation per step, as a lane does
it) they give bit-identical Vdot, Jacobian, LU and substitution results on
random data with the mechanism's pattern; no round reads what a later round,
or one it was not told to wait for, writes; and every word's offsets stay
inside the wave's LDS block and the coefficient table."""
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "geos-chem_amd" / "mechgen"))


@pytest.fixture(scope="module")
def cell(fullchem):
    import cell_sched as C
    from emit_tables import build_tables
    m = fullchem
    raw = {"nvar": m.nvar, "nfix": m.nfix, "nspec": m.nspec, "nreact": m.nreact,
           "lu_nonzero": m.lu_nonzero, "reactions": m.reactions, "lu_irow": m.lu_irow.tolist(),
           "lu_icol": m.lu_icol.tolist(), "lu_crow": m.lu_crow.tolist(), "lu_diag": m.lu_diag.tolist()}
    t = build_tables(raw)
    o = C.build(raw, t)
    code, words, sched = C.emit_code(raw, t, o)
    return C, raw, t, o, code, words, sched


def chunked(C, init, terms, nhead, step):
    """The canonical sum: nhead terms in chunks, the rest one by one."""
    acc, total = init, None
    for n, x in enumerate(terms[:nhead]):
        if n and n % C.CHUNK == 0:
            total = acc if total is None else total + acc
            acc = 0.0
        acc = step(acc, x)
    acc = acc if total is None else total + acc
    for x in terms[nhead:]:
        acc = step(acc, x)
    return acc


def execute(rounds, lds, kind, coef):
    """Runs the rounds; reads of a round happen after the stores of the round
    it depends on and may happen before those of any round in between."""
    snap = [list(lds)]
    for r, rd in enumerate(rounds):
        assert rd.dep < r and len(rd.pieces) <= 64
        old = snap[rd.dep + 1]          # the oldest state its reads may see
        out = {}
        for p in rd.pieces:
            for e in [p.init] + ([p.div] if p.div is not None else []) + \
                    [y for x in p.terms for y in (x if kind == "n" else x[:1])]:
                assert old[e] == lds[e], "a round reads what it does not wait for"
            acc = lds[p.init]
            for a, b in p.terms:
                acc = acc + (-lds[a]) * lds[b] if kind == "n" else \
                    acc + (coef[b] if kind == "c" else -coef[b]) * lds[a]
            assert p.dest not in out
            out[p.dest] = acc if p.div is None else acc / lds[p.div]
        lds = list(lds)
        for e, v in out.items():
            lds[e] = v
        snap.append(lds)
    return lds


def fresh(o, rng):
    L = o["layout"]
    lds = list(rng.uniform(-1.0, 1.0, L["SIZE"]))
    lds[L["ZERO"]], lds[L["ONE"]], lds[L["NEG"]] = 0.0, 1.0, -1.0
    return lds, L


def test_programs_reproduce_the_table_walk(cell, fullchem):
    C, raw, t, o, code, words, sched = cell
    rng = np.random.default_rng(11)
    nv, nz, s = raw["nvar"], raw["lu_nonzero"], o["s"]
    crow, diag, icol = raw["lu_crow"], raw["lu_diag"], raw["lu_icol"]
    coef, lu_of, X = o["coef"], o["lu"], o["layout"]["X"]
    # Vdot
    lds, L = fresh(o, rng)
    A = [lds[L["A"] + o["slot"][r]] for r in range(raw["nreact"])]
    ref = []
    for i in range(nv):
        x = range(t["fv_ptr"][i], t["fv_ptr"][i + 1])
        ref.append(chunked(C, 0.0, list(x), len(x),
                           lambda acc, k: acc + float(t["fv_c"][k]) * A[t["fv_r"][k]]))
    assert execute(sched["fv"], lds, "c", coef)[X:X + nv] == ref
    # Jacobian, batch after batch of partials
    lds, L = fresh(o, rng)
    b = rng.uniform(-1.0, 1.0, len(t["pt_r"]))
    for bt, rounds in enumerate(sched["jv"]):
        for p, (batch, slot) in o["pslot"].items():
            if batch == bt:
                lds[slot] = float(b[p])
        lds = execute(rounds, lds, "d", coef)
    jac = {}
    for q in range(nz):
        x = list(range(t["jv_ptr"][q], t["jv_ptr"][q + 1]))
        jac[q] = chunked(C, 0.0, x, len(x), lambda acc, k: acc + -float(t["jv_c"][k]) * float(b[t["jv_b"][k]]))
        if x:
            assert lds[lu_of[q]] == jac[q]
    # LU: in front of the block by the program, the block by columns
    for i in range(nv):
        lds[lu_of[diag[i]]] += 40.0
        jac[diag[i]] += 40.0
    ref = [0.0] * nz
    for q in range(nz):
        x = list(range(t["cr_ptr"][q], t["cr_ptr"][q + 1]))
        v = chunked(C, jac[q], x, t["cr_hd"][q] - t["cr_ptr"][q],
                    lambda acc, k: acc + (-ref[t["cr_l"][k]]) * ref[t["cr_u"][k]])
        ref[q] = v / ref[t["cr_div"][q]] if t["cr_div"][q] >= 0 else v
    lds = execute(sched["lup"], lds, "n", coef)
    k, pat = o["tail"], o["tailpat"]
    T = [[lds[o["tailslot"][i][j]] for j in range(k)] for i in range(k)]
    for j in range(k):
        for i in range(j + 1, k):
            if pat[i][j]:
                T[i][j] /= T[j][j]
                for c in range(j + 1, k):
                    if pat[j][c]:
                        T[i][c] = T[i][c] + (-T[i][j]) * T[j][c]
    for q in range(nz):
        i, c = raw["lu_irow"][q] - s, icol[q] - s
        assert ref[q] == (T[i][c] if i >= 0 and c >= 0 else lds[lu_of[q]]), q
    # substitutions
    x = [lds[X + i] for i in range(nv)]
    for i in range(nv):
        ks = list(range(crow[i], diag[i]))
        x[i] = chunked(C, x[i], ks, t["fw_hd"][i] - crow[i], lambda acc, q: acc + (-ref[q]) * x[icol[q]])
    for i in range(nv - 1, -1, -1):
        ks = list(range(crow[i + 1] - 1, diag[i], -1))
        x[i] = chunked(C, x[i], ks, len(ks) if i < s else 0,
                       lambda acc, q: acc + (-ref[q]) * x[icol[q]]) / ref[diag[i]]
    lds = execute(sched["sf"], lds, "n", coef)
    y = [lds[X + s + i] for i in range(k)]
    for j in range(k):
        for i in range(j + 1, k):
            if pat[i][j]:
                y[i] = y[i] + (-T[i][j]) * y[j]
    for j in range(k - 1, -1, -1):
        y[j] /= T[j][j]
        for i in range(j):
            if pat[i][j]:
                y[i] = y[i] + (-T[i][j]) * y[j]
    for i in range(k):
        lds[X + s + i] = y[i]
    assert execute(sched["sb"], lds, "n", coef)[X:X + nv] == x


def test_offsets_stay_inside_the_block(cell):
    C, raw, t, o, code, words, sched = cell
    L = o["layout"]
    assert C.KCELLS * 8 * L["SIZE"] + 8 * len(o["coef"]) <= C.LDS_BYTES
    assert len(words) % 256 == 0
    half = [x & 0xFFF8 for x in words] + [x >> 16 for x in words]
    assert all(x % 8 == 0 and x < 8 * L["SIZE"] for x in half)
    for ph, rounds in [("fv", sched["fv"])] + [("jv", r) for r in sched["jv"]]:
        assert all(0 <= b < len(o["coef"]) for r in rounds for p in r.pieces for a, b in p.terms)
    own = [L["A"] + u * 64 + 63 for u in range(len(o["rows"]))] + \
        [L["AB"] + u * 64 + 63 for u in range(C.AB_ROWS)]
    assert max(own) < L["P"]
    # a destination is never a constant or another lane's sink
    for r in [x for k in ("fv", "lup", "sf", "sb") for x in sched[k]] + [x for y in sched["jv"] for x in y]:
        for p in r.pieces:
            assert p.dest < L["ZERO"]


def test_generated_header_holds_the_programs(cell):
    C, raw, t, o, code, words, sched = cell
    hdr = (ROOT / "geos-chem_amd" / "csrc" / "gen" / "cell_fullchem.h").read_text()
    assert code in hdr
    i = hdr.index("unsigned words[%d]" % len(words))
    body = hdr[hdr.index("{", i) + 1:hdr.index("}", i)]
    assert [int(x) for x in body.split(",") if x.strip()] == words
