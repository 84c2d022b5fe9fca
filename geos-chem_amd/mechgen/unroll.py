"""Mechanism compiler, unrolled lane programs: Fun, the Jacobian, the LU and
the substitutions of a small mechanism as straight-line code for one lane
(csrc/lane_unrolled.hip), for mechanisms whose cell fits a lane (`fits`: Hg
with 161 LU entries; fullchem's 5,683 do not, carbon has no LU).

The operations and their order are those of the table walk: reaction r adds
its terms to the rows in increasing r, partial p to the Jacobian entries in
increasing p, an LU position and a substitution row takes its terms in table
order.

Where a lane's values live: the LU's diagonal, the vectors and the stage
vectors in registers; the other LU entries, the fixed species and the first
rate constants in LDS (LDS_FIELDS doubles a lane, two waves a CU); the other
rate constants and the state in the wave's slot block.  Fields in LDS: LU
entries (lds(q)), fixed species, rate constants.
"""
LDS_FIELDS = 160
GROUP = 12   # rate constants requested a group ahead of the reactions that use them


def fits(m):
    return bool(m["lu_irow"]) and m["lu_nonzero"] + m["nspec"] <= LDS_FIELDS + 2 * m["nvar"] \
        and m["nvar"] <= 32


def layout(m):
    """(fields of LU entries, first rate constants in LDS)."""
    ng = m["lu_nonzero"] - m["nvar"]
    return ng, min(m["nreact"], LDS_FIELDS - ng - (m["nspec"] - m["nvar"]))


def code(m, t):
    nv, nz = m["nvar"], m["lu_nonzero"]
    crow, diag, icol = m["lu_crow"], m["lu_diag"], m["lu_icol"]
    row_of = {diag[i]: i for i in range(nv)}
    off = [q for q in range(nz) if q not in row_of]
    pos = {q: k for k, q in enumerate(off)}
    ent = lambda q: "d[%d]" % row_of[q] if q in row_of else "lds(%d)" % pos[q]
    num = lambda c: repr(float(c))
    conc = lambda s: "y[%d]" % s if s < nv else "fix(%d)" % (s - nv)
    out = []
    terms = {}
    for i in range(nv):
        for x in range(t["fv_ptr"][i], t["fv_ptr"][i + 1]):
            terms.setdefault(t["fv_r"][x], []).append((i, t["fv_c"][x]))
    parts = {}
    for p, r in enumerate(t["pt_r"]):
        parts.setdefault(r, []).append(p)
    # Fun, alone and with the partials (the rate constants read once for both)
    for name in ("fun", "fun_partials"):
        jac = name == "fun_partials"
        out += ["template <class R, class F>",
                "__device__ __forceinline__ void %s(const double (&y)[%d], R rate, F fix, double (&v)[%d]%s) {"
                % (name, nv, nv, ", double (&b)[%d]" % len(t["pt_r"]) if jac else "")]
        out += ["  v[%d] = 0.0;" % i for i in range(nv)]
        groups = [list(range(r, min(r + GROUP, m["nreact"]))) for r in range(0, m["nreact"], GROUP)]
        fetch = lambda g: ["  const double k%d = rate(%d);" % (r, r) for r in g] + \
            ["  __builtin_amdgcn_sched_barrier(0);"]
        out += fetch(groups[0])
        for r in range(m["nreact"]):
            if r % GROUP == 0 and r // GROUP + 1 < len(groups):
                out += fetch(groups[r // GROUP + 1])
            s = [x for x in t["rx_s"][3 * r:3 * r + 3] if x >= 0]
            out.append("  { const double k = k%d; double a = k; %s"
                       % (r, " ".join("a *= %s;" % conc(x) for x in s)))
            out += ["    v[%d] = fma(%s, a, v[%d]);" % (i, num(c), i) for i, c in terms.get(r, [])]
            for p in parts.get(r, []) if jac else []:
                o = [x for x in t["pt_s"][2 * p:2 * p + 2] if x >= 0]
                mult = "" if t["pt_m"][p] == 1.0 else "%s * " % num(t["pt_m"][p])
                out.append("    b[%d] = %sk; %s" % (p, mult, " ".join("b[%d] *= %s;" % (p, conc(x)) for x in o)))
            out.append("  }")
        out.append("}")
    # Ghimj = diag - sum c * partial and its LU, a position at a time; true if a
    # diagonal entry was below TINY before its row's elimination
    out += ["template <class LG, class LP>",
            "__device__ __forceinline__ bool lu(const double (&b)[%d], double diag, double (&d)[%d], LG lds, LP put_lds) {"
            % (len(t["pt_r"]), nv), "  bool bad = false;"]
    for q in range(nz):
        out.append("  { double g = 0.0;")
        for x in range(t["jv_ptr"][q], t["jv_ptr"][q + 1]):
            out.append("    g = fma(%s, b[%d], g);" % (num(-t["jv_c"][x]), t["jv_b"][x]))
        if q in row_of:
            out.append("    g = g + diag; bad = bad || fabs(g) < DBL_MIN;")
        for x in range(t["cr_ptr"][q], t["cr_ptr"][q + 1]):
            out.append("    g = fma(-%s, %s, g);" % (ent(t["cr_l"][x]), ent(t["cr_u"][x])))
        if t["cr_div"][q] >= 0:
            out.append("    g = g / %s;" % ent(t["cr_div"][q]))
        out.append("    d[%d] = g; }" % row_of[q] if q in row_of else "    put_lds(%d, g); }" % pos[q])
    out += ["  return bad;", "}"]
    out += ["template <class LG>",
            "__device__ __forceinline__ void solve(const double (&d)[%d], LG lds, double (&x)[%d]) {" % (nv, nv)]
    for i in range(nv):
        for q in range(crow[i], diag[i]):
            out.append("  x[%d] = fma(-lds(%d), x[%d], x[%d]);" % (i, pos[q], icol[q], i))
    for i in range(nv - 1, -1, -1):
        for q in range(diag[i] + 1, crow[i + 1]):
            out.append("  x[%d] = fma(-lds(%d), x[%d], x[%d]);" % (i, pos[q], icol[q], i))
        out.append("  x[%d] = x[%d] / d[%d];" % (i, i, i))
    out.append("}")
    return "\n".join(out)
