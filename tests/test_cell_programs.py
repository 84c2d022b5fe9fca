"""The cell programs (mechgen/cell_sched.py) compute every sum of a Rodas3
attempt in the order the lane-per-cell solvers walk the tables: executed
round by round on the CPU (one IEEE double operation per step, as a lane does
it) they give bit-identical Vdot, Jacobian, LU and substitution results on
random data with the mechanism's pattern; no round reads what a later round,
or one it was not told to wait for, writes; and every word's offsets stay
inside the wave's LDS block and the coefficient table."""
import re
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


class Emitted:
    """Runs the emitted code of one program on 64 lanes (one IEEE double
    operation per statement and lane; no fused multiply-add, as in the walk it
    is compared with), idle lanes included."""

    def __init__(self, code, words, lds):
        self.lds, self.words, self.v = lds, np.array(words, dtype=np.uint64).reshape(-1, 64, 4), {}
        self.code, self.lane = code, np.arange(64)

    def function(self, name):
        body = self.code[self.code.index("void %s(" % name):]
        body = body[body.index("{") + 1:body.index("#undef LDW")].split("\n")
        base = int(body[1].split("cell_word(c, ")[1].split(" ")[0])
        return base, [x.strip() for x in body[2:] if x.strip()]

    def expr(self, e):
        """A word, h >> 16, (w & 0xffffu), LD(...), LDL(k), 0.0, a name."""
        e = e.strip()
        if e.startswith("LDL("):
            return self.lds[int(e[4:-1]) // 8 + self.lane]
        if e.startswith("LD"):
            return self.lds[self.expr(e[2:]).astype(np.int64) // 8]
        if e.startswith("(") and e.endswith(")"):
            return self.expr(e[1:-1])
        if e.endswith(">> 16"):
            return self.expr(e[:-5]) >> np.uint64(16)
        if e.endswith("& 0xffffu"):
            return self.expr(e[:-9]) & np.uint64(0xFFFF)
        m = re.fullmatch(r"w(\d+)\.([xyzw])", e)
        if m:
            return self.words[self.base + int(m.group(1)), :, "xyzw".index(m.group(2))]
        return np.zeros(64) if e == "0.0" else self.v[e]

    def run(self, name, tail):
        self.base, lines = self.function(name)
        self.v = {}
        for s in lines:
            m = re.fullmatch(r"const double (a\w+) = (.*), (b\w+) = (.*);", s)
            if m:
                self.v[m.group(1)], self.v[m.group(3)] = self.expr(m.group(2)), self.expr(m.group(4))
                continue
            m = re.fullmatch(r"(c\w+) = fma\(-(\w+), (\w+), (\w+)\);", s)
            if m:
                c, a, b, c0 = (self.v.get(x) for x in m.groups())
                self.v[m.group(1)] = c0 + (-a) * b
                continue
            m = re.fullmatch(r"ST\((h\w+) & 0xffffu, (c\w+)(?: / (d\w+))?\);", s)
            if m:
                v = self.v[m.group(2)] / self.v[m.group(3)] if m.group(3) else self.v[m.group(2)]
                self.lds[(self.v[m.group(1)] & np.uint64(0xFFFF)).astype(np.int64) // 8] = v
                continue
            m = re.fullmatch(r"(?:const )?(?:unsigned|double) (\w+) = (.*);", s)
            if m:
                self.v[m.group(1)] = np.array(self.expr(m.group(2)))
                continue
            if s.startswith("cell_tail("):
                tail(self.lds)
            else:
                assert s.startswith("const u32x4 w"), s


def test_infinite_factors_reach_their_own_rows_only(cell):
    """A lane whose terms have ended reads another row's factor times 0 in
    cell_solve.  With finite factors it gives the walk's result; an infinite
    one makes NaN of rows that have nothing to do with it, but every result
    that differs from the walk's holds a NaN (the solver's sign to take
    cell_solve_apart), and cell_solve_apart's never differs."""
    C, raw, t, o, code, words, sched = cell
    rng = np.random.default_rng(17)
    nv, nz, s, k, L = raw["nvar"], raw["lu_nonzero"], o["s"], o["tail"], o["layout"]
    crow, diag, icol, irow = (raw[x] for x in ("lu_crow", "lu_diag", "lu_icol", "lu_irow"))
    lu0 = rng.uniform(-1.0, 1.0, nz) * 0.1
    lu0[diag[:nv]] = rng.uniform(5.0, 9.0, nv)
    x0 = rng.uniform(-1.0, 1.0, nv)
    head = [q for q in range(nz) if o["lu"][q] < L["LUH"]]
    spoiled = 0
    with np.errstate(all="ignore"):
        for bad in [None] + list(rng.choice(head, 40, replace=False)):
            lu = lu0.copy()
            if bad is not None:
                lu[bad] = rng.choice([np.inf, -np.inf, np.nan])
            x = list(x0)
            sub = lambda acc, q: acc + (-lu[q]) * x[icol[q]]
            for i in range(nv):
                x[i] = chunked(C, x[i], list(range(crow[i], diag[i])), t["fw_hd"][i] - crow[i], sub)
            y = list(x)
            for i in range(nv - 1, -1, -1):
                ks = list(range(crow[i + 1] - 1, diag[i], -1))
                x[i] = chunked(C, x[i], ks, len(ks) if i < s else 0, sub) / lu[diag[i]]

            def tail(lds, ref=(y, x)):   # the block's rows before and after
                X = slice(L["X"] + s, L["X"] + nv)
                z = lds[X].copy()
                for j in range(k):
                    for q in range(crow[s + j], diag[s + j]):
                        if icol[q] >= s:
                            z[j] = z[j] + (-lu[q]) * z[icol[q] - s]
                for j in range(k - 1, -1, -1):
                    for q in range(crow[s + j + 1] - 1, diag[s + j], -1):
                        z[j] = z[j] + (-lu[q]) * z[icol[q] - s]
                    z[j] = z[j] / lu[diag[s + j]]
                lds[X] = z

            got = {}
            for name in ("cell_solve", "cell_solve_apart"):
                lds = np.zeros(L["SIZE"])
                lds[L["ONE"]], lds[L["NEG"]] = 1.0, -1.0
                for q in range(nz):
                    lds[o["lu"][q]] = lu[q]
                lds[L["X"]:L["X"] + nv] = x0
                e = Emitted(code, words, lds)
                e.run(name, tail)
                got[name] = lds[L["X"]:L["X"] + nv].copy()
            assert np.array_equal(got["cell_solve_apart"], x, equal_nan=True)
            if bad is None:
                assert np.array_equal(got["cell_solve"], x) and np.isfinite(x).all()
            elif not np.array_equal(got["cell_solve"], x, equal_nan=True):
                assert np.isnan(got["cell_solve"]).any()
                spoiled += int((np.isfinite(x) & np.isnan(got["cell_solve"])).any())
    assert spoiled > 0    # (the case that cell_solve_apart is there for)
