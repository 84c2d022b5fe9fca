"""Edges of the dispatch between the solvers' kernels, bit by bit.

fullchem solves start on the cell-per-wave kernel, one wave to a workgroup up
to 512 cells and three above; Hg solves on the unrolled lane kernel, 64 cells
a wave and two waves a CU.  Every kernel does the same operations in the same
order, so the tolerance is zero.  The rate program runs in parts of 64 cells:
a cell's rates do not depend on the call's size.
"""
import numpy as np
import pytest

from gckpp_amd import options

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def _t(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype=torch.float64)


@pytest.fixture(scope="module")
def inputs(torch_dev, fullchem, hg):
    """(workload, rates of all its cells) per mechanism."""
    from gckpp_amd import hip, synth
    from pathlib import Path
    w = synth.box_cells(fullchem, 1024, 7)
    ctx = hip.Context(fullchem, 1024)
    rct = ctx.rates(*(_t(torch_dev, x) for x in (w.met, w.photol, w.het, w.conc))).cpu().numpy()
    ctx.close()
    g = dict(np.load(Path(__file__).resolve().parent / "golden" / "Hg_box.npz"))
    return {"fullchem": (w, w.conc, rct), "Hg": (None, g["conc"], g["rconst"])}


@pytest.mark.parametrize("name,variant,n", [("fullchem", 4, n) for n in (1, 2, 511, 512, 513, 515, 769)] +
                         [("Hg", 7, n) for n in (1, 63, 64, 65, 1000)])
def test_default_kernel_equals_the_other(name, variant, n, inputs, mech_of, torch_dev):
    print("case: %s, %d cells, default kernel against variant %d" % (name, n, variant), flush=True)
    from gckpp_amd import hip
    m = mech_of(name)
    _, conc, rct = inputs[name]
    cells = (np.arange(n) * 37) % conc.shape[1]
    scale = 1.0 + 1.0e-3 * (np.arange(n) // conc.shape[1])
    ic, rc = options.fullchem_icntrl()
    out = []
    for v in (None, variant):
        ctx = hip.Context(m, max(n, 64))
        ctx.set_solver(hip.SOLVER_PERSISTENT)
        if v is not None:
            ctx.set_persistent_config(v, 1)
        c = _t(torch_dev, conc[:, cells] * scale)
        ist, rst, ierr = ctx.integrate(c, _t(torch_dev, rct[:, cells]), _t(torch_dev, np.zeros(n)), 0.0, 1200.0, ic, rc)
        out.append([x.cpu().numpy() for x in (c, ist, rst, ierr)])
        ctx.close()
    assert (out[0][3] == 1).mean() > 0.9
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 769])
def test_rates_do_not_depend_on_the_number_of_cells(n, inputs, fullchem, torch_dev):
    from gckpp_amd import hip
    w, _, rct = inputs["fullchem"]
    het = w.het if w.het.ndim == 1 or w.het.shape[1] == 1 else w.het[:, :n]
    ctx = hip.Context(fullchem, 1024)
    r = ctx.rates(_t(torch_dev, w.met[:, :n]), _t(torch_dev, w.photol[:, :n]), _t(torch_dev, het),
                  _t(torch_dev, w.conc[:, :n])).cpu().numpy()
    ctx.close()
    assert np.array_equal(r, rct[:, :n])


def test_handoff_count_is_the_last_steps(inputs, fullchem, hg, torch_dev):
    """gckpp_batch_handoff_count after a step that handed cells over, then after
    steps that did not: eager, and replayed from a graph."""
    from gckpp_amd import hip, synth
    print("case: hand-off count of a batch", flush=True)
    T = torch_dev
    mechs = [fullchem, hg]
    ws = [synth.box_cells(m, 256, 3) for m in mechs]
    ctxs = [hip.Context(m, w.ncell) for m, w in zip(mechs, ws)]
    B = hip.Batch(*ctxs)
    st = [dict(met=_t(T, w.met), photol=_t(T, w.photol), het=_t(T, w.het), conc=_t(T, w.conc),
               hstart=_t(T, np.zeros(w.ncell)), icntrl=options.icntrl_for(m.name)[0],
               rcntrl=options.icntrl_for(m.name)[1],
               istatus=T.zeros((20, w.ncell), dtype=T.int32, device="cuda"),
               ierr=T.zeros(w.ncell, dtype=T.int32, device="cuda")) for m, w in zip(mechs, ws)]
    parts = [B.part(**d) for d in st]

    def count(variant, replay):
        # (a cold step each time: a settled cell takes one integration step, and
        # so never stands at the boundary where it could be handed over)
        for d, w in zip(st, ws):
            d["conc"].copy_(_t(T, w.conc))
            d["hstart"].zero_()
        B.set_config(variant, 1)
        if replay:
            B.capture(parts, 1200.0)
            B.replay()
        else:
            B.step(parts, 1200.0)
        T.cuda.synchronize()
        return B.handoff_count()

    B.set_handoff(100)
    assert B.handoff_count() == 0            # no step yet
    assert count(4, False) > 0
    assert count(hip.WAVE_VARIANT, False) == 0
    assert count(4, True) > 0
    assert count(hip.WAVE_VARIANT, True) == 0
    assert count(4, False) > 0
    B.set_handoff(0)
    assert count(4, False) == 0
    B.close()
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("counts,handoff,lanes", [((100, 60000, 10), 2000, True),      # Hg is the work
                                                  ((100, 60000, 10), 0, False),        # ... no hand-off
                                                  ((100, 60000, 10), 70000, False),    # ... of every cell
                                                  ((5000, 60000, 10), 2000, False),    # fullchem over the cap
                                                  ((700, 200, 100), 500, False)])
def test_batch_picks_its_kernel_by_its_cells(counts, handoff, lanes, inputs, fullchem, hg, mech_of, torch_dev):
    """A batch without a configuration: the lane kernel (then cells are handed
    off) where many Hg cells stand beside few fullchem ones, the cell-per-wave
    kernel otherwise; the results are those of the configured cell-per-wave
    kernel, bit by bit, also replayed from a graph."""
    from gckpp_amd import hip, synth
    print("case: batch of %s cells, hand-off %d" % (counts, handoff), flush=True)
    T = torch_dev
    mechs = [fullchem, hg, mech_of("carbon")]
    ws = [synth.box_cells(m, 1024, 3) for m in mechs]
    ctxs = [hip.Context(m, n) for m, n in zip(mechs, counts)]
    B = hip.Batch(*ctxs)

    def state():
        st = []
        for m, w, n in zip(mechs, ws, counts):
            ic, rc = options.icntrl_for(m.name)
            i = np.arange(n) % w.ncell
            het = w.het if w.het.shape[1] == 1 else w.het[:, i]
            st.append(dict(met=_t(T, w.met[:, i]), photol=_t(T, w.photol[:, i]), het=_t(T, het),
                           conc=_t(T, w.conc[:, i]), hstart=_t(T, np.zeros(n)), icntrl=ic, rcntrl=rc,
                           istatus=T.zeros((20, n), dtype=T.int32, device="cuda"),
                           ierr=T.zeros(n, dtype=T.int32, device="cuda")))
        return st

    def result(st):
        T.cuda.synchronize()
        return [d[k].cpu().numpy() for d in st for k in ("conc", "hstart", "istatus", "ierr")]

    B.set_handoff(handoff)
    st = state()
    B.step([B.part(**d) for d in st], 1200.0)
    a = result(st)
    if handoff:
        assert (B.handoff_count() > 0) == lanes
    else:
        assert B.handoff_count() == 0 and not lanes
    sg = state()
    pg = [B.part(**d) for d in sg]
    B.capture(pg, 1200.0)
    B.replay()
    g = result(sg)
    B.set_config(hip.WAVE_VARIANT, 1)
    sw = state()
    B.step([B.part(**d) for d in sw], 1200.0)
    for x, y, z in zip(a, g, result(sw)):
        assert np.array_equal(x, y) and np.array_equal(x, z)
    B.close()
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("factor", [np.inf, 1.0e300])
def test_infinite_entries_spoil_the_same_rows_in_every_kernel(factor, inputs, fullchem, torch_dev):
    """One reaction a cell with a rate whose Jacobian entries overflow, for each
    of the mechanism's reactions, and reactants at zero in every other cell: at
    most two attempts, after which the cell-per-wave kernel holds NaN and
    infinities exactly where the lane kernel does.  (Where unrelated rows of
    the factorisation meet, a row that stays finite has to stay the same.)"""
    from gckpp_amd import hip
    print("case: one overflowing reaction a cell, rate times %g" % factor, flush=True)
    m, n = fullchem, fullchem.nreact
    _, conc, rct = inputs["fullchem"]
    cells = (np.arange(n) * 37) % conc.shape[1]
    c0, r = conc[:, cells].copy(), rct[:, cells].copy()
    for k, rx in enumerate(m.reactions):
        r[k, k] = max(r[k, k], 1.0e-20) * factor
        if k % 2:
            for sp, mult in rx["reactants"]:
                if sp < m.nvar:
                    c0[sp, k] = 0.0
    ic, rc = options.fullchem_icntrl()
    ic = ic.copy()
    ic[3] = 1
    out = []
    for v in (7, 4):
        ctx = hip.Context(m, n)
        ctx.set_solver(hip.SOLVER_PERSISTENT)
        ctx.set_persistent_config(v, 1)
        c = _t(torch_dev, c0)
        ist, rst, ierr = ctx.integrate(c, _t(torch_dev, r), _t(torch_dev, np.full(n, 1.0)), 0.0, 1200.0, ic, rc)
        out.append([x.cpu().numpy() for x in (c, ist, rst, ierr)])
        ctx.close()
    some = np.isnan(out[0][0]).any(0) & np.isfinite(out[0][0][:m.nvar]).any(0)
    print("cells with NaN and finite species: %d of %d" % (some.sum(), n))
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f")
    assert some.sum() > 20


@pytest.mark.parametrize("variant", [0, 1, 4, 6, 8, 9, None])
@pytest.mark.parametrize("n", [1, 65, 200])
def test_every_lane_solver_adds_in_the_same_order(n, variant, inputs, fullchem, torch_dev):
    """fullchem's lane kernels and the plain solver (None), whose gathers load
    one to sixteen terms at a time, against the default kernel, bit by bit."""
    from gckpp_amd import hip
    print("case: fullchem, %d cells, lane variant %s" % (n, variant), flush=True)
    _, conc, rct = inputs["fullchem"]
    cells = (np.arange(n) * 37) % conc.shape[1]
    ic, rc = options.fullchem_icntrl()
    out = []
    for v in (7, variant):
        ctx = hip.Context(fullchem, max(n, 64))
        if v is not None:
            ctx.set_solver(hip.SOLVER_PERSISTENT)
            ctx.set_persistent_config(v, 1)
        c = _t(torch_dev, conc[:, cells])
        ist, rst, ierr = ctx.integrate(c, _t(torch_dev, rct[:, cells]), _t(torch_dev, np.zeros(n)), 0.0, 1200.0, ic, rc)
        out.append([x.cpu().numpy() for x in (c, ist, rst, ierr)])
        ctx.close()
    assert (out[0][3] == 1).all()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
