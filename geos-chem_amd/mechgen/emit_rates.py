"""Mechanism compiler, back end for rate coefficients: writes
  csrc/gen/species_<mech>.h   constexpr 0-based index of every species
  csrc/gen/rates_<mech>.h     the mechanism's rate program: one statement per
                              reaction, rc[r] = <rate law call>, evaluated per
                              cell by the rates kernel (Update_RCONST,
                              KPP/<mech>/gckpp_Rates.F90)
from mech/<mech>.json.  Rate-law calls keep the reference's law names and
argument order (the mechanism's data); their implementations are this
project's (csrc/ratelaws.h, csrc/hetlaws.h).

Run:  python emit_rates.py <mech> [<mech> ...]
"""
import json
import re
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
MATH = {"exp", "log", "log10", "sqrt", "pow", "fmax", "fmin"}


def translate(expr, mech):
    s = expr
    ns = "species_%s" % mech
    s = re.sub(r"CONC\((\w+)\)", lambda m: "E.conc(%s::%s)" % (ns, m.group(1)), s)
    s = re.sub(r"SRMW\((\w+)\)", lambda m: "E.srmw(%s::%s)" % (ns, m.group(1)), s)
    s = re.sub(r"\b(PHOTOL|K_MT|K_CLD)\[(\d+)\]", r"E.\1(\2)", s)
    s = re.sub(r"\bk_(Trop|Strat|TROP|STRAT)\((\d+)(?:\.0)?\)",
               lambda m: "E.K_%s(%d)" % (m.group(1).upper(), int(m.group(2)) - 1), s)
    s = s.replace(",State_Het)", ")").replace("(State_Het)", "()").replace("(State_Het,", "(")

    out, i = [], 0
    for m in re.finditer(r"(?<![\w.])([A-Za-z_]\w*)(\s*\()?", s):
        name, call = m.group(1), m.group(2)
        out.append(s[i:m.start()])
        i = m.end()
        prev = s[:m.start()]
        if prev.endswith("E.") or prev.endswith("::") or re.search(r"\d[eE]$", prev):
            out.append(m.group(0))
            continue
        if name in ("E",) or name.startswith("species_"):
            out.append(m.group(0))
            continue
        if call:
            if name.lower() in MATH:
                out.append(name.lower() + "(")
            else:
                # rate law: the cell environment is its first argument
                rest = s[i:]
                out.append("rl::%s(E%s" % (name, ")" if rest.startswith(")") else ", "))
                if rest.startswith(")"):
                    i += 1
        else:
            out.append("E.%s" % name)
    out.append(s[i:])
    return "".join(out)


# Parts of a rate program, a wave each: short enough for the instruction cache,
# a grid's waves many times what the GPU holds (a call on 238,464 cells: 8 to 20
# parts 1.04 to 1.03 ms).
PARTS = {"fullchem": 8}


def weight(stmt):
    """Rough cost of a statement, in instructions."""
    if re.search(r"[uU]ptk|Brkd|Hyd|hyp|By", stmt):
        return 600
    if "rl::" not in stmt:
        return 12
    return 60 if "GCARR_ac(" in stmt or "ARRPLUS_ade(" in stmt else 400


def parts(mech, stmts):
    """[[(reaction, statement)]]: statements with the same arguments side by
    side (a law's exponentials are evaluated once for all that share them), the
    heterogeneous laws in parts of their own (divergent, many registers), the
    copies of constants and inputs spread evenly (memory beside arithmetic)."""
    n = PARTS.get(mech, 1)
    idx = list(enumerate(stmts))
    if n == 1:
        return [idx]

    def key(x):
        r, s = x
        w = weight(s)
        args = re.findall(r"[-+]?\d[\d.]*e?[-+]?\d*", s.split("(E", 1)[-1])
        if w == 60:  # a0 exp(c0 / T): by c0
            return (2, args[-1], s, r)
        if w == 400:  # by arguments, then law (GC_NIT and GC_ALK share theirs)
            return (1, ",".join(args), s, r)
        return (0 if w == 600 else 3, "", "", r)

    laws = sorted((x for x in idx if weight(x[1]) > 12), key=key)
    copies = [x for x in idx if weight(x[1]) <= 12]
    total, out, acc = sum(weight(s) for r, s in laws), [[]], 0
    for x in laws:
        if acc >= total * len(out) / n:
            out.append([])
        out[-1].append(x)
        acc += weight(x[1])
    # the copies evenly between every part's laws
    for p, xs in enumerate(out):
        cs = copies[len(copies) * p // n:len(copies) * (p + 1) // n]
        m = [((i + 0.5) / len(l), x) for l in (xs, cs) for i, x in enumerate(l)]
        out[p] = [x for _, x in sorted(m)]
    return out


def emit(mech):
    m = json.loads((HERE.parent / "mech" / ("%s.json" % mech)).read_text())
    gen = HERE.parent / "csrc" / "gen"
    gen.mkdir(exist_ok=True)
    L = ["/* Generated by geos-chem_amd/mechgen/emit_rates.py -- do not edit. */",
         "#pragma once", "namespace species_%s {" % mech]
    for i, n in enumerate(m["species"]):
        L.append("constexpr int %s = %d;" % (n, i))
    L.append("constexpr int NSPEC = %d;" % len(m["species"]))
    L.append("}  // namespace species_%s" % mech)
    (gen / ("species_%s.h" % mech)).write_text("\n".join(L) + "\n")

    R = ["/* Generated by geos-chem_amd/mechgen/emit_rates.py from mech/%s.json"
         " -- do not edit. */" % mech, "#pragma once",
         '#include "species_%s.h"' % mech, "",
         "namespace gckpp {",
         "// Update_RCONST of mechanism %s: rc[r*rs] for r = 0..%d, in parts"
         % (mech, m["nreact"] - 1)]
    ps = parts(mech, [translate(rx["rate"], mech) for rx in m["reactions"]])
    R += ["constexpr int RATE_PARTS_%s = %d;" % (mech, len(ps)),
          "template <int P>",
          "__device__ void rates_%s(const rl::RateEnv &E, double *__restrict__ rc, int64_t rs);" % mech]
    for p, xs in enumerate(ps):
        R += ["template <>",
              "__device__ __forceinline__ void rates_%s<%d>(const rl::RateEnv &E, double *__restrict__ rc,"
              % (mech, p), "    int64_t rs) {"]
        R += ["  rc[%d * rs] = %s;" % x for x in xs]
        R += ["}"]
    R += ["}  // namespace gckpp"]
    (gen / ("rates_%s.h" % mech)).write_text("\n".join(R) + "\n")
    print("%s: %d rate statements" % (mech, m["nreact"]))


if __name__ == "__main__":
    for n in sys.argv[1:] or ["fullchem", "Hg", "carbon"]:
        emit(n)
