"""Mechanism compiler, cell programs: the straight-line programs of the
cell-per-wave Rodas3 solver (csrc/cell_solver.h) for a mechanism whose LU ends
in a block of rows that are eliminated one after the other.

One wavefront integrates one cell.  The last TAIL rows and columns of the
matrix (`tail_size`) are a chain: each pivot needs the one before it, so a
schedule over LDS pays an LDS round trip for every one of them.  Lane i of the
wave holds row s + i of that block in registers (s = NVAR - TAIL); its pivots
and both its substitutions are column steps, one broadcast and one FMA each.
Everything in front of the block is shallow (fullchem: 8 levels forward, 9
backward, 13 in the LU) and is scheduled here: every sum of the solve is cut
into chunks of at most CHUNK terms, a chunk into pieces at the dependency
levels of its operands, and the pieces of a level, sorted by length, are dealt
to the 64 lanes in rounds.  Pieces of one level are independent.

Order of the sums (the lane-per-cell solvers follow it too, see the tables):
  * a sum's terms in table order, in chunks of CHUNK: the first chunk starts
    from the sum's initial value, every other from +0.0, and the chunks' values
    are added in order;
  * an LU position of the tail block first takes the terms of the pivots in
    front of the block (chunked), then those inside it one by one;
  * a substitution row of the tail block likewise; the backward rows take
    their terms in descending column order (inside the block as the pivots'
    solution becomes known, in front of it chunked).

LDS elements (8 bytes each, per wave): LU (the positions outside the tail
block first), AB rows of 64, P partial-sum slots, X (the variable species'
vector, then the fixed species), the constants +0, +1, -1, and 64 sink slots
for idle lanes.  The tail positions' slots hold the block only until it is in
registers; from there on the reaction products A(r) lie over them and AB.

Reactions go to (row u, lane) slots sorted by their number of partial
derivatives (`reaction_rows`), so a lane owns the same reactions' rate
constants, products and partials.  The Jacobian's partials are made and
consumed in batches of AB rows, and the Jacobian's terms are ordered by batch
(build_tables).

A phase's words (one 32-bit word per lane and use, two 16-bit byte offsets
into the wave's LDS): per round a header (destination, initial value), the
divisor in a dividing round, then one word per step (a, b), or half a word (b)
where the lanes' a lie side by side (`solve_order`).  Four words make a block,
64 lanes x 16 bytes.
"""
LANES = 64
CHUNK = 32
KCELLS = 3              # cells (waves) per CU, the most the LU block leaves room for
LDS_BYTES = 163840      # per CU
AB_ROWS = 8             # rows of 64 partials per batch
RING = 12               # word blocks in flight (8: 1 % slower)
DEPTH = 7               # steps whose operands are in flight (lgkmcnt counts 15 reads)


def _pattern(m):
    n, crow, icol = m["nvar"], m["lu_crow"], m["lu_icol"]
    return [[icol[q] for q in range(crow[i], crow[i + 1])] for i in range(n)]


def tail_size(m):
    """Rows of the tail block: the size for which a substitution pair costs
    least at the measured 82 clocks per register column (both ways) and 220
    per level in front of the block; 0 for a mechanism without an LU or with
    one that a lane solves faster (fewer than 128 rows)."""
    n = m["nvar"]
    if not m["lu_irow"] or n < 128:
        return 0
    pat = _pattern(m)
    best = None
    for k in range(16, LANES + 1, 2):
        s = n - k
        lf, lb = [0] * s, [0] * s
        for i in range(s):
            lf[i] = max([lf[c] + 1 for c in pat[i] if c < i], default=0)
        for i in range(s - 1, -1, -1):
            lb[i] = max([lb[c] + 1 for c in pat[i] if i < c < s], default=0)
        cost = 82 * k + 220 * (max(lf) + max(lb) + 2)
        if best is None or cost < best[0]:
            best = (cost, k)
    return best[1]


def reaction_rows(m):
    """slot[r] = u * 64 + lane of reaction r, and per row u the number of its
    reactions' partials: reactions sorted by that number, most first."""
    nv = m["nvar"]
    npart = [sum(1 for s, k in r["reactants"] if s < nv) for r in m["reactions"]]
    order = sorted(range(len(npart)), key=lambda r: (-npart[r], r))
    slot = [0] * len(npart)
    for p, r in enumerate(order):
        slot[r] = p
    rows = [max(npart[r] for r in order[u:u + LANES]) for u in range(0, len(order), LANES)]
    return slot, rows


def partial_batches(m):
    """batch[(row u, index q of the partial in its reaction)] and the list of
    (u, q) rows in order, AB_ROWS to a batch."""
    slot, rows = reaction_rows(m)
    uq = [(u, q) for u, k in enumerate(rows) for q in range(k)]
    return {x: i // AB_ROWS for i, x in enumerate(uq)}, uq


# Phase.schedule's candidates.
POLICIES = ((32, 1, 0.0, 0, 24), (12, 3, 0.0, 48, 24), (24, 1, 0.5, 0, 40), (16, 2, 0.5, 0, 0),
            (8, 1, 0.125, 0, 24), (10, 1, 0.125, 0, 24), (3, 1, 0.0, 0, 24))


class Job:
    """One chunk of a sum: lds[dest] = lds[init] + its terms (/ lds[div]);
    `need`: elements a step or the division reads that another job makes."""
    __slots__ = ("dest", "init", "terms", "div", "final", "pos", "height", "idx")

    def __init__(self, dest, init, terms, div, final):
        self.dest, self.init, self.terms, self.div, self.final = dest, init, terms, div, final
        self.pos = 0


class Piece:
    """One lane's part of a round: terms of one job, the division if div."""
    __slots__ = ("dest", "init", "terms", "div")

    def __init__(self, dest, init, terms, div):
        self.dest, self.init, self.terms, self.div = dest, init, terms, div


class Round:
    __slots__ = ("pieces", "steps", "div", "dep")

    def __init__(self, pieces, dep):
        self.pieces, self.dep = pieces, dep
        self.steps = max(len(p.terms) for p in pieces)
        self.div = any(p.div is not None for p in pieces)


# Clocks of a step, a round, a division and an LDS round trip, the scheduler's
# estimates of what the wave issues and waits for.
T_STEP, T_ROUND, T_DIV, T_LDS = 22, 45, 100, 130


class Phase:
    """Jobs in dependency order, scheduled into rounds.  `kind` 'c': a step is
    acc = fma(coef[b], lds[a], acc), 'd': acc = fma(-coef[b], lds[a], acc),
    'n': acc = fma(-lds[a], lds[b], acc)."""

    def __init__(self, kind, zero, plus, pool):
        self.kind, self.zero, self.plus = kind, zero, plus
        self.jobs, self.pool, self.maker = [], list(pool), {}

    def _job(self, *a):
        j = Job(*a)
        j.idx = len(self.jobs)
        self.jobs.append(j)
        return j

    def add(self, dest, init, terms, div=None):
        """One sum in chunks; later sums may read dest."""
        cuts = list(range(0, max(1, len(terms)), CHUNK))
        if len(cuts) == 1:
            self._job(dest, init, terms, div, True)
        else:
            slots = [dest] + [self.pool.pop(0) for _ in cuts[1:]]
            for n, c in enumerate(cuts):
                self._job(slots[n], init if n == 0 else self.zero, terms[c:c + CHUNK], None, False)
                if n:
                    self.maker[slots[n]] = len(self.jobs) - 1
            # the combining job waits for the first chunk through dest
            self._job(dest, dest, [self.plus(p) for p in slots[1:]], div, True)
            self.jobs[-1].init = ("after", len(self.jobs) - 1 - len(cuts), dest)
        self.maker[dest] = len(self.jobs) - 1

    def reads(self, x):
        """LDS elements of a step that may be made in this phase."""
        return x if self.kind == "n" else x[:1]

    def schedule(self):
        """Rounds by list scheduling: each takes up to 64 jobs with ready
        terms, those with the longest path to the phase's end first, and runs
        the same number of steps of each (fewer where a job has no more)."""
        # (most steps in a round, fewest worth a piece, how far the longest
        # path sets a round's steps, divisions that make a round, jobs apart
        # from the last round that make a round): each the best for one of
        # fullchem's phases (modelled clocks of an attempt's LU 24.7k -> 16.3k,
        # Vdot 3.6k -> 2.6k, Jacobian 10.6k -> 9.1k by the rounds apart)
        best = None
        for policy in POLICIES:
            r = self._try(*policy)
            if best is None or r[0] < best[0]:
                best = r
        self.clocks = best[0]
        return best[1]

    def _try(self, cap, minp, share, divs, apart):
        jobs, maker = self.jobs, self.maker
        nj = len(jobs)
        # producers of every job's steps and division
        prod, divp, users = [], [], [[] for _ in range(nj)]
        for j in jobs:
            pr = []
            first = None
            if isinstance(j.init, tuple):
                first = j.init[1]
            for x in j.terms:
                pr.append([maker[e] for e in self.reads(x) if e in maker and maker[e] < j.idx])
            if first is not None:
                (pr[0] if pr else pr).append(first)
            d = maker.get(j.div, -1) if j.div is not None else -1
            divp.append(d if d < j.idx else -1)
            prod.append(pr)
            for q in pr:
                for k in q:
                    users[k].append(j.idx)
            if divp[-1] >= 0:
                users[divp[-1]].append(j.idx)
        for j in reversed(jobs):
            own = T_STEP * len(j.terms) + T_ROUND + (T_DIV if j.div is not None else 0)
            j.height = own + max([jobs[u].height + T_LDS for u in users[j.idx]], default=0)
            j.pos = 0
        divp_job = lambda k: jobs[k].div is not None
        done = [-1] * nj            # round in which a job ended
        last = [-1] * nj            # round of a job's latest piece
        todo = set(range(nj))
        left = sum(len(j.terms) for j in jobs)
        rounds, clk, costs = [], 0, []
        order = sorted(range(nj), key=lambda k: -jobs[k].height)
        while todo:
            cand = []
            for k in order:
                if k not in todo:
                    continue
                j = jobs[k]
                n = 0
                for x in range(j.pos, len(j.terms)):
                    if any(done[q] < 0 for q in prod[k][x]):
                        break
                    n += 1
                ends = j.pos + n == len(j.terms)
                fin = ends and (divp[k] < 0 or done[divp[k]] >= 0)
                if not n and not fin:
                    continue
                cand.append((k, n, fin))
                if len(cand) >= 6 * LANES:
                    break
            if apart and rounds:
                # jobs that need nothing of the last round do not wait for it:
                # they make the round when they nearly fill it
                r1 = len(rounds) - 1

                def free(c):
                    j = jobs[c[0]]
                    return last[c[0]] < r1 and \
                        all(done[q] < r1 for x in range(j.pos, j.pos + c[1]) for q in prod[c[0]][x]) and \
                        not (c[2] and divp[c[0]] >= 0 and done[divp[c[0]]] >= r1)
                sub = [c for c in cand if free(c)]
                if len(sub) >= apart:
                    cand = sub
            crit = jobs[cand[0][0]].height > 1.2 * T_STEP * left / LANES
            keep = [c for c in cand if c[2] or c[1] >= minp] or cand[:1]
            # divs: divisions have rounds of their own, begun when that many
            # wait, the job with the longest path waits, or nothing else can run
            only = None
            if divs:
                wait = [c for c in cand if not c[1] and c[2] and divp_job(c[0])]
                rest = [c for c in keep if c[1] or (c[2] and not divp_job(c[0]))]
                only = bool(wait) and (not rest or len(wait) >= divs or
                                       (crit and wait[0][0] == cand[0][0]))
                keep = wait if only else rest or cand[:1]
            sel = keep[:LANES]
            if only:
                ln = 0
            elif crit and share:
                ln = max(1, min(cap, max(c[1] for c in sel[:max(1, int(share * 8))])))
            else:
                ln, top = 1, -1.0
                for l in range(1, cap + 1):
                    v = sum(min(c[1], l) for c in sel) / (T_ROUND + T_STEP * l)
                    if v > top:
                        ln, top = l, v
                if not any(c[1] for c in sel):
                    ln = 0
            ps, dep, r = [], -1, len(rounds)
            for k, n, fin in sel:
                j = jobs[k]
                n2 = min(n, ln)
                fin2 = fin and n2 == n and (only is None or only or not divp_job(k))
                if not n2 and not fin2:
                    continue
                for x in range(j.pos, j.pos + n2):
                    for q in prod[k][x]:
                        dep = max(dep, done[q])
                if fin2 and divp[k] >= 0:
                    dep = max(dep, done[divp[k]])
                dep = max(dep, last[k])
                init = j.init[2] if isinstance(j.init, tuple) else j.init
                ps.append((k, Piece(j.dest, init if last[k] < 0 else j.dest,
                                    j.terms[j.pos:j.pos + n2], j.div if fin2 else None), fin2, n2))
            for k, p, fin2, n2 in ps:
                jobs[k].pos += n2
                left -= n2
                last[k] = r
                if fin2:
                    done[k] = r
                    todo.discard(k)
            ps.sort(key=lambda z: -len(z[1].terms))
            rd = Round([z[1] for z in ps], dep)
            c = T_ROUND + T_STEP * rd.steps + (T_DIV if rd.div else 0)
            if dep >= 0:
                c += max(0, T_LDS - sum(costs[dep + 1:]))
            costs.append(c)
            clk += c
            rounds.append(rd)
        return clk, rounds


def build(m, t):
    """The cell program of mechanism m (tables t), or None without a tail."""
    k = tail_size(m)
    if not k:
        return None
    return _build(m, t, k, solve_order(_build(m, t, k, [])))


def solve_order(o):
    """LU positions in front of the tail block in the order in which the
    substitutions' steps read them, a step's lanes side by side: a lane then
    reads its factor at a fixed offset from its own slot (no address, no bank
    conflict), and the word of the step names the other operand only."""
    pos = {p: q for q, p in o["lu"].items() if p < o["layout"]["LUH"]}
    order, seen = [], set()
    for rd in o["sf"].schedule() + o["sb"].schedule():
        for x in range(rd.steps):
            es = [p.terms[x][0] for p in rd.pieces if x < len(p.terms)]
            if all(e in pos and e not in seen for e in es):
                order += [pos[e] for e in es]
                seen.update(es)
    return order


def _build(m, t, k, order):
    """`order`: LU positions that lie first, in this order."""
    n, nspec, nz = m["nvar"], m["nspec"], m["lu_nonzero"]
    s = n - k
    crow, diag, icol, irow = m["lu_crow"], m["lu_diag"], m["lu_icol"], m["lu_irow"]
    head = [q for q in range(nz) if not (irow[q] >= s and icol[q] >= s)]
    tail = [q for q in range(nz) if irow[q] >= s and icol[q] >= s]
    first = set(order)
    lu = {q: p for p, q in enumerate(order + [q for q in head if q not in first] + tail)}
    slot, rows = reaction_rows(m)
    batch, uq = partial_batches(m)
    coefs, cidx = [-0.0], {}
    for c in list(t["fv_c"]) + list(t["jv_c"]):
        if float(c) not in cidx:
            cidx[float(c)] = len(coefs)
            coefs.append(float(c))
    for c in (1.0, -1.0):
        if c not in cidx:
            cidx[c] = len(coefs)
            coefs.append(c)
    size = (LDS_BYTES // 8 - len(coefs)) // KCELLS
    L = {"LUH": len(head), "AB": nz, "A": len(head)}
    fixed = AB_ROWS * LANES + nspec + 3 + LANES
    L["P"] = nz + AB_ROWS * LANES
    L["NP"] = size - nz - fixed
    assert L["NP"] > 0
    L["X"] = L["P"] + L["NP"]
    L["ZERO"] = L["X"] + nspec
    L["ONE"], L["NEG"], L["SINK"] = L["ZERO"] + 1, L["ZERO"] + 2, L["ZERO"] + 3
    L["SIZE"] = L["SINK"] + LANES
    assert L["SIZE"] <= size and 8 * L["SIZE"] < 65536
    na = len(rows) * LANES
    assert L["A"] + na <= L["P"]
    X, ZERO, ONE, NEG = L["X"], L["ZERO"], L["ONE"], L["NEG"]
    ppool = list(range(L["P"], L["P"] + L["NP"]))
    plus_c = lambda p: (p, cidx[1.0])
    plus_d = lambda p: (p, cidx[-1.0])
    plus_n = lambda p: (p, NEG)
    out = {"tail": k, "s": s, "layout": L, "coef": coefs, "lu": lu, "rows": rows, "slot": slot,
           "uq": uq, "na": na}
    # Vdot into X (the products' operands have been read by then)
    fv = Phase("c", ZERO, plus_c, list(range(L["A"] + na, L["P"])) + ppool)
    for i in range(n):
        tt = [(L["A"] + slot[t["fv_r"][x]], cidx[float(t["fv_c"][x])])
              for x in range(t["fv_ptr"][i], t["fv_ptr"][i + 1])]
        fv.add(X + i, ZERO, tt)
    out["fv"] = fv
    # Ghimj's off-diagonal part, -sum c*partial; batch b of the partials is
    # there at level b only
    first, pslot = {}, {}
    for p, r in enumerate(t["pt_r"]):
        first.setdefault(r, p)
        u, lane = divmod(slot[r], LANES)
        row = uq.index((u, p - first[r]))
        pslot[p] = (row // AB_ROWS, L["AB"] + (row % AB_ROWS) * LANES + lane)
    out["pslot"] = pslot
    nb = (len(uq) + AB_ROWS - 1) // AB_ROWS
    jv = [Phase("d", ZERO, plus_d, []) for _ in range(nb)]
    jpool = list(ppool)
    diags = set(diag[:n])
    written = set()
    for q in range(nz):
        xs = range(t["jv_ptr"][q], t["jv_ptr"][q + 1])
        if not len(xs) and q not in diags:
            continue
        written.add(q)
        chunks = [list(xs[c:c + CHUNK]) for c in range(0, len(xs), CHUNK)] or [[]]
        slots = [lu[q]] + [jpool.pop(0) for _ in chunks[1:]]
        for dst, ch in zip(slots, chunks):
            by, bs = {}, [pslot[t["jv_b"][x]][0] for x in ch]
            assert bs == sorted(bs)
            for x, bt in zip(ch, bs):
                by.setdefault(bt, []).append((pslot[t["jv_b"][x]][1], cidx[float(t["jv_c"][x])]))
            for k_, bt in enumerate(sorted(by) or [0]):
                jv[bt]._job(dst, ZERO if k_ == 0 else dst, by.get(bt, []), None, True)
                jv[bt].maker[dst] = len(jv[bt].jobs) - 1
        if len(chunks) > 1:
            last = jv[-1]
            first = last.maker.get(lu[q])
            last._job(lu[q], lu[q] if first is None else ("after", first, lu[q]),
                      [plus_d(p) for p in slots[1:]], None, True)
            last.maker[lu[q]] = len(last.jobs) - 1
    out["jv"] = jv
    # LU in front of the tail block, and its pivots' terms of the block
    ph = Phase("n", ZERO, plus_n, list(range(L["AB"], L["P"])) + ppool)
    for q in range(nz):
        xs = [x for x in range(t["cr_ptr"][q], t["cr_ptr"][q + 1]) if icol[t["cr_l"][x]] < s]
        dv = t["cr_div"][q]
        inblock = irow[q] >= s and icol[q] >= s
        div = lu[dv] if dv >= 0 and not inblock else None
        if not xs and div is None:
            continue
        tt = [(lu[t["cr_l"][x]], lu[t["cr_u"][x]]) for x in xs]
        ph.add(lu[q], lu[q] if q in written else ZERO, tt, div)
        written.add(q)
    # a step's idle lanes read what lies after its factors, times 0
    assert written.issuperset(head) and len(head) - len(order) >= LANES
    out["lup"] = ph
    # the tail block: slot of (row, column), ZERO where the pattern has none
    out["tailslot"] = [[ZERO] * k for _ in range(k)]
    out["tailpat"] = [[False] * k for _ in range(k)]
    for q in tail:
        out["tailpat"][irow[q] - s][icol[q] - s] = True
        if q in written:
            out["tailslot"][irow[q] - s][icol[q] - s] = lu[q]
    # forward rows, then (after the block) backward rows
    sf = Phase("n", ZERO, plus_n, list(range(L["AB"], L["P"])) + ppool)
    for i in range(n):
        qs = [q for q in range(crow[i], diag[i]) if icol[q] < s]
        if qs:
            tt = [(lu[q], X + icol[q]) for q in qs]
            sf.add(X + i, X + i, tt)
    out["sf"] = sf
    sb = Phase("n", ZERO, plus_n, list(range(L["AB"], L["P"])) + ppool)
    for i in range(s - 1, -1, -1):
        tt = [(lu[q], X + icol[q]) for q in range(crow[i + 1] - 1, diag[i], -1)]
        sb.add(X + i, X + i, tt, lu[diag[i]])
    out["sb"] = sb
    out["diagslot"] = [lu[diag[i]] for i in range(n)]
    return out




# ---------------------------------------------------------------------------
# Emission.  A program is straight-line code over one stream of words.
class Stream:
    """Words of one program and its code lines.  word() appends a word (64
    lane values) and returns the expression that holds it; a block's loads
    are issued RING blocks ahead."""

    def __init__(self, name):
        self.name, self.words, self.code, self.open = name, [], [], None

    def line(self, s):
        self.code.append(s)

    def word(self, lanes):
        assert len(lanes) == LANES and all(0 <= w < (1 << 32) for w in lanes)
        i = len(self.words)
        if i % 4 == 0:
            self.line("@%d" % (i // 4))
        self.words.append(list(lanes))
        return "w%d.%s" % (i // 4, "xyzw"[i % 4])

    def half(self, lanes):
        """The expression of a 16-bit value per lane, two to a word."""
        if self.open is None:
            self.open = (len(self.words), self.word(lanes))
            return "(%s & 0xffffu)" % self.open[1]
        (i, e), self.open = self.open, None
        self.words[i] = [w | x << 16 for w, x in zip(self.words[i], lanes)]
        return "(%s >> 16)" % e

    def finish(self):
        """Code lines with the block loads in place, and the words as uint4
        blocks [block][lane][4]."""
        while len(self.words) % 4:
            self.words.append([0] * LANES)
        nb = len(self.words) // 4
        out = ["const u32x4 w%d = LDW(%d);" % (b, b) for b in range(min(RING, nb))]
        for c in self.code:
            if c[0] != "@":
                out.append(c)
                continue
            b = int(c[1:]) + RING - 1
            if b >= RING and b < nb:
                out.append("const u32x4 w%d = LDW(%d);" % (b, b))
        flat = []
        for b in range(nb):
            for ln in range(LANES):
                flat += [self.words[4 * b + k][ln] for k in range(4)]
        return out, flat


def side_by_side(rd, x, L):
    """The first LU position of step x of a round of kind 'n' when the step's
    factors lie side by side, lane by lane (see solve_order); else None."""
    fs = [p.terms[x][0] for p in rd.pieces if x < len(p.terms)]
    if fs[-1] < L["LUH"] and fs == list(range(fs[0], fs[0] + len(fs))) and \
            all(x < len(p.terms) for p in rd.pieces[:len(fs)]):
        return fs[0]
    return None


def emit_rounds(st, rounds, kind, L, tag, own=True):
    """A phase's rounds: the operands of up to DEPTH steps are requested ahead,
    across round ends too, but never before the stores of the round they wait
    for (LDS operations of a wave execute in order, so no wait is needed).
    own: steps whose factors lie side by side read them at a fixed offset from
    the lane's own slot.  A lane whose terms have ended then reads the LU
    position after the step's factors, times 0: harmless unless that position
    is infinite or NaN, which makes the lane's sum NaN.  Without own every idle
    lane reads the zero slot."""
    zero, one, sink = L["ZERO"], L["ONE"], L["SINK"]
    pad = (zero, 0 if kind != "n" else zero)
    seq = []
    for r, rd in enumerate(rounds):
        seq.append(("I", r, 0))
        seq += [("T", r, k) for k in range(rd.steps)]
        seq.append(("E", r, 0))
    load_b = "LD" if kind == "n" else "CF"
    fma = {"n": "fma(-%s, %s, %s)", "c": "fma(%s, %s, %s)", "d": "fma(-%s, %s, %s)"}[kind]
    name = lambda r: "%s%d" % (tag, r)
    ended, nxt, flight = -1, 0, 0

    def issue(op):
        k, r, x = op
        rd, n = rounds[r], name(r)
        if k == "I":
            ps = rd.pieces + [None] * (LANES - len(rd.pieces))
            h = [8 * (p.dest if p else sink + ln) | (8 * (p.init if p else zero)) << 16
                 for ln, p in enumerate(ps)]
            st.line("const unsigned h%s = %s;" % (n, st.word(h)))
            if all(p.init == zero for p in rd.pieces):
                st.line("double c%s = 0.0;" % n)
            else:
                st.line("double c%s = LD(h%s >> 16);" % (n, n))
            if rd.div:
                d = [8 * (p.div if p and p.div is not None else one) for p in ps]
                st.line("const double d%s = LD(%s);" % (n, st.word(d)))
        elif k == "T":
            w = []
            f = side_by_side(rd, x, L) if own and kind == "n" else None
            if f is not None:
                for ln in range(LANES):
                    t = rd.pieces[ln].terms if ln < len(rd.pieces) else []
                    w.append(8 * (t[x][1] if x < len(t) else zero))
                st.line("const double a%s_%d = LDL(%d), b%s_%d = LD%s;"
                        % (n, x, 8 * f, n, x, st.half(w)))
                return
            for ln in range(LANES):
                t = rd.pieces[ln].terms if ln < len(rd.pieces) else []
                a, b = t[x] if x < len(t) else pad
                w.append(8 * a | (8 * b) << 16)
            e = st.word(w)
            st.line("const double a%s_%d = LD(%s & 0xffffu), b%s_%d = %s(%s >> 16);"
                    % (n, x, e, n, x, load_b, e))

    for i, (k, r, x) in enumerate(seq):
        while nxt < len(seq):
            kk, rr, xx = seq[nxt]
            if rounds[rr].dep > ended or (kk == "T" and flight >= DEPTH):
                break
            if kk != "E":
                issue(seq[nxt])
                flight += kk == "T"
            nxt += 1
        assert nxt > i or k == "E"
        n = name(r)
        if k == "T":
            a, b = "a%s_%d" % (n, x), "b%s_%d" % (n, x)
            x0, x1 = (a, b) if kind == "n" else (b, a)
            st.line("c%s = %s;" % (n, fma % (x0, x1, "c" + n)))
            flight -= 1
        elif k == "E":
            st.line("ST(h%s & 0xffffu, c%s%s);" % (n, n, " / d" + n if rounds[r].div else ""))
            ended = r


def emit_code(m, t, o):
    """(C++ text of the generated header's functions, the words of all its
    programs, the phases' rounds)."""
    L, k, s, rows, uq = o["layout"], o["tail"], o["s"], o["rows"], o["uq"]
    n, nv = m["nvar"], m["nvar"]
    one = L["ONE"]
    rx = [[sp for sp, c in r["reactants"] for _ in range(c)] for r in m["reactions"]]
    at = [None] * (len(rows) * LANES)
    for r, p in enumerate(o["slot"]):
        at[p] = r
    out, all_words, sched = [], [], {}

    def func(name, args, st):
        code, words = st.finish()
        out.append("__device__ __forceinline__ void %s(const CellLds &c%s) {" % (name, args))
        out.append("#define LDW(k) cell_word(c, %d + (k))" % (len(all_words) // (4 * LANES)))
        out.extend("  " + x for x in code)
        out.append("#undef LDW\n}")
        all_words.extend(words)

    # Fun: products into A, then Vdot into X
    st = Stream("fun")
    for u in range(len(rows)):
        ls = [rx[at[u * LANES + ln]] if at[u * LANES + ln] is not None else [] for ln in range(LANES)]
        el = lambda ln, q: 8 * (L["X"] + ls[ln][q] if q < len(ls[ln]) else one)
        e = st.word([el(ln, 0) | el(ln, 1) << 16 for ln in range(LANES)])
        more = any(len(x) > 2 for x in ls)
        st.line("const double p%d = LD(%s & 0xffffu), q%d = LD(%s >> 16);" % (u, e, u, e))
        if more:
            st.line("const double r%d = LD(%s);" % (u, st.word([el(ln, 2) for ln in range(LANES)])))
        st.line("double v%d = R[%d]; v%d *= p%d; v%d *= q%d;%s" %
                (u, u, u, u, u, u, " v%d *= r%d;" % (u, u) if more else ""))
        st.line("STL(%d, v%d);" % (8 * (L["A"] + u * LANES), u))
    sched["fv"] = o["fv"].schedule()
    emit_rounds(st, sched["fv"], "c", L, "f")
    func("cell_fun", ", const double (&R)[%d]" % len(rows), st)
    # Ghimj: per batch the partials, then its terms; the diagonal last
    st = Stream("jac")
    first = {}
    for p, r in enumerate(t["pt_r"]):
        first.setdefault(r, p)
    sched["jv"] = []
    for b, ph in enumerate(o["jv"]):
        for i in range(b * AB_ROWS, min(len(uq), (b + 1) * AB_ROWS)):
            u, q = uq[i]
            oth, dbl = [], []
            for ln in range(LANES):
                r = at[u * LANES + ln]
                p = first.get(r, -1) + q if r is not None else -1
                ok = r is not None and r in first and p < len(t["pt_r"]) and t["pt_r"][p] == r
                oth.append([x for x in t["pt_s"][2 * p:2 * p + 2] if x >= 0] if ok else [])
                dbl.append(bool(ok and t["pt_m"][p] == 2.0))
                assert not ok or t["pt_m"][p] in (1.0, 2.0)
            el = lambda ln, j: 8 * (L["X"] + oth[ln][j] if j < len(oth[ln]) else one)
            e = st.word([el(ln, 0) | el(ln, 1) << 16 | int(dbl[ln]) for ln in range(LANES)])
            v = "R[%d]" % u
            if any(dbl):
                v = "((%s & 1u) ? 2.0 * %s : %s)" % (e, v, v)
            st.line("double g%d = %s; g%d *= LD(%s & 0xfff8u);" % (i, v, i, e))
            if any(len(x) > 1 for x in oth):
                st.line("g%d *= LD(%s >> 16);" % (i, e))
            st.line("STL(%d, g%d);" % (8 * (L["AB"] + (i % AB_ROWS) * LANES), i))
        rs = ph.schedule()
        sched["jv"].append(rs)
        emit_rounds(st, rs, "d", L, "j%d_" % b)
    for j in range((n + LANES - 1) // LANES):
        e = st.word([8 * (o["diagslot"][ln + LANES * j] if ln + LANES * j < n else L["SINK"] + ln)
                     for ln in range(LANES)])
        st.line("const double z%d = LD(%s) + diag;" % (j, e))
        live = "" if LANES * (j + 1) <= n else "c.lane < %d && " % (n - LANES * j)
        st.line("bad = bad || (%sfabs(z%d) < DBL_MIN);" % (live, j))
        st.line("ST(%s, z%d);" % (e, j))
    func("cell_jac", ", const double (&R)[%d], double diag, bool &bad" % len(rows), st)
    # LU in front of the block, then the block's rows to the lanes' registers
    st = Stream("lu")
    sched["lup"] = o["lup"].schedule()
    emit_rounds(st, sched["lup"], "n", L, "u")
    ts, pat = o["tailslot"], o["tailpat"]
    for j in range(0, k, 2):
        sl = lambda ln, c: 8 * (ts[ln][c] if ln < k and c < k else L["ZERO"])
        e = st.word([sl(ln, j) | sl(ln, j + 1) << 16 for ln in range(LANES)])
        st.line("T[%d] = LD(%s & 0xffffu);" % (j, e))
        if j + 1 < k:
            st.line("T[%d] = LD(%s >> 16);" % (j + 1, e))
    mask = lambda rs: "0x%xu, 0x%xu" % (sum(1 << i for i in rs if i < 32),
                                        sum(1 << i - 32 for i in rs if i >= 32))
    st.line("ud = 1.0;")
    for j in range(k):
        below = [i for i in range(j + 1, k) if pat[i][j]]
        st.line("if (c.lane == %d) ud = T[%d];" % (j, j))
        if not below:
            continue
        cols = [x for x in range(j + 1, k) if pat[j][x]]
        st.line("{ const double u = bcast(T[%d], %d);" % (j, j))
        for x in cols:
            st.line("const double s%d = bcast(T[%d], %d);" % (x, x, j))
        st.line("if (lanes_of<%s>()) {" % mask(below))
        st.line("T[%d] = T[%d] / u;" % (j, j))
        for x in cols:
            st.line("T[%d] = fma(-T[%d], s%d, T[%d]);" % (x, j, x, x))
        st.line("} }")
    st.line("yd = 1.0 / ud;")
    func("cell_lu", ", double (&T)[%d], double &ud, double &yd" % k, st)
    # substitutions of the block: x of the lane's row, in X before and after
    st = Stream("tail")
    st.line("wave_sync();")
    st.line("double x = LDL(%d);" % (8 * (L["X"] + s)))
    st.line("x = c.lane < %d ? x : 0.0;" % k)
    for j in range(k):
        below = [i for i in range(j + 1, k) if pat[i][j]]
        if below:
            st.line("fma_on<%s>(x, T[%d], bcast(x, %d));" % (mask(below), j, j))
    st.line("const double x0 = x;")
    above = [[i for i in range(j) if pat[i][j]] for j in range(k)]
    for j in range(k - 1, -1, -1):
        if above[j]:
            st.line("fma_on<%s>(x, T[%d], bcast(cell_div(x, ud, yd), %d));" % (mask(above[j]), j, j))
    st.line("double q = cell_div(x, ud, yd);")
    st.line("if (__any(q != q)) {  // infinities and NaN: as the division has them")
    st.line("x = x0;")
    for j in range(k - 1, -1, -1):
        if above[j]:
            st.line("fma_on<%s>(x, T[%d], bcast(x / ud, %d));" % (mask(above[j]), j, j))
    st.line("q = x / ud;")
    st.line("}")
    st.line("if (c.lane < %d) STL(%d, q);" % (k, 8 * (L["X"] + s)))
    st.line("wave_sync();")
    args = ", const double (&T)[%d], double ud, double yd" % k
    func("cell_tail", args, st)
    # substitutions: forward in front of the block, the block, backward; and
    # the same without a read of an unrelated LU position
    sched["sf"], sched["sb"] = o["sf"].schedule(), o["sb"].schedule()
    for name, own in (("cell_solve", True), ("cell_solve_apart", False)):
        st = Stream("solve")
        emit_rounds(st, sched["sf"], "n", L, "f", own)
        st.line("cell_tail(c, T, ud, yd);")
        emit_rounds(st, sched["sb"], "n", L, "b", own)
        func(name, args, st)
    return "\n".join(out), all_words, sched
