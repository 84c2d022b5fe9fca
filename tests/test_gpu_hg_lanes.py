"""The unrolled Hg lane kernel's refill and retry paths, and when the hand-off
applies to it.

A wave of it integrates 64 cells at a time and takes new ones when 16 of its
lanes are idle, so more cells than lanes (a wave cap of one or two waves) run
the refill between attempts, and Hstart = 1e-13 s with ICNTRL(4) at the median
number of cold steps the cold restart of failed cells.  The plain solver and the cell-per-wave kernel do the
same operations in the same order, so the tolerance is zero.
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


def _step(torch, hg, w, n, limit, setup):
    from gckpp_amd import hip
    ic, rc = options.hg_icntrl()
    hs = np.zeros(n)
    if limit:
        ic = ic.copy()
        ic[3] = limit
        hs = np.full(n, 1e-13)
    ctx = hip.Context(hg, 1024)
    setup(ctx)
    het = w.het if w.het.ndim == 1 or w.het.shape[1] == 1 else w.het[:, :n]
    conc = _t(torch, w.conc[:, :n])
    hnew, ist, ierr, _ = ctx.fullchem_step(_t(torch, w.met[:, :n]), _t(torch, w.photol[:, :n]), _t(torch, het),
                                           conc, _t(torch, hs), 1200.0, ic, rc)
    out = [x.cpu().numpy() for x in (conc, hnew, ist, ierr)]
    ctx.close()
    return out


@pytest.mark.parametrize("forced", [False, True])
@pytest.mark.parametrize("n,waves", [(1000, 1), (997, 2), (79, 1)])
def test_refill_and_retry_bitwise(n, waves, forced, hg, torch_dev):
    from gckpp_amd import hip, synth
    print("case: Hg, %d cells on %d wave(s), forced retries %s" % (n, waves, forced), flush=True)
    w = synth.box_cells(hg, 1024, 5)

    def lanes(ctx):
        ctx.set_solver(hip.SOLVER_PERSISTENT)
        ctx.set_persistent_waves(waves)
        cfg = ctx.persistent_config()
        assert cfg["wave_per_cell"] == 0 and cfg["waves"] == waves

    def cell_per_wave(ctx):
        ctx.set_solver(hip.SOLVER_PERSISTENT)
        ctx.set_persistent_config(hip.WAVE_VARIANT, 1)

    limit = 0
    if forced:
        limit = int(np.median(_step(torch_dev, hg, w, n, 0, lanes)[2][2]))
    a = _step(torch_dev, hg, w, n, limit, lanes)
    if forced:
        assert (a[3] < 0).sum() > 8 and (a[3] == 1).sum() > 8
    else:
        assert (a[3] == 1).all()
    for x, y in zip(a, _step(torch_dev, hg, w, n, limit, cell_per_wave)):
        assert np.array_equal(x, y)
    if not forced:  # (the plain solver's retry counts both integrations)
        for x, y in zip(a, _step(torch_dev, hg, w, n, limit, lambda ctx: ctx.set_solver(hip.SOLVER_PLAIN))):
            assert np.array_equal(x, y)


def test_autotuner_leaves_the_launch_it_timed(hg, torch_dev):
    """A hand-off set on an unconfigured Hg context does not apply to it; after
    the autotuner, whose trials ran so, it still does not."""
    from gckpp_amd import hip
    from pathlib import Path
    g = dict(np.load(Path(__file__).resolve().parent / "golden" / "Hg_box.npz"))
    n = 8192
    print("case: Hg autotuner with a hand-off set, %d cells" % n, flush=True)
    cells = np.arange(n) % g["conc"].shape[1]
    conc, rct = _t(torch_dev, g["conc"][:, cells]), _t(torch_dev, g["rconst"][:, cells])
    zero = _t(torch_dev, np.zeros(n))
    ic, rc = options.hg_icntrl()
    ctx = hip.Context(hg, n)
    ctx.set_solver(hip.SOLVER_PERSISTENT)
    ctx.set_persistent_handoff(4096)

    def handed_off():
        c = conc.clone()
        ist, rst, ierr = ctx.integrate(c, rct, zero, 0.0, 1200.0, ic, rc)
        return [x.cpu().numpy() for x in (c, ist, rst, ierr)], ctx.handoff_stats()[0]

    a, before = handed_off()
    ms = ctx.autotune(conc, rct, zero, 0.0, 1200.0, ic, rc)
    lane = np.delete(ms, hip.WAVE_VARIANT, 0)
    b, after = handed_off()
    assert before == 0 and after == 0
    assert (lane == lane.flat[0]).all() and lane.flat[0] > 0     # one kernel, timed once
    ctx.set_persistent_config(4, 1)                                # the caller's own choice
    c, chosen = handed_off()
    assert chosen > 0
    for x, y, z in zip(a, b, c):
        assert np.array_equal(x, y) and np.array_equal(x, z)
    ctx.close()
