"""The separate sweeps (st_kernels.hip), which the solves outside the one-pass
stage run: the launch shapes, the compacted WENO lists, the mixed form and the
batched launches of a default channel's tests, on channels stretched in x, with
the Rusanov split or with KEEP(2).  And the launch shapes of the one-pass stage
where it has any: without bulk sums.

Tolerance: the trajectory bars of the parity tests, 1e-10 relative L2 per
conserved variable in FP64 and 1e-5 in the mixed form; everything else bit for
bit."""
import numpy as np
import pytest

from helpers import interior, rel_l2
from oracle import Oracle
from streams_mi355x import PREC_MIXED, capi, make_channel
from streams_mi355x.cases import make_bl_box
from streams_mi355x.params import params_copy
from streams_mi355x.serve import Request, run_sequential, run_serving
from streams_mi355x.solver import ChannelSolver

pytestmark = pytest.mark.gpu

TRAJ_TOL = 1e-10
MIXED_TOL = 1e-5
KINDS = ["stretched", "rusanov", "keep2"]


def _channel(kind, nx=32, ny=24, nz=16, **kw):
    if kind == "keep2":
        kw["nkeep"] = 2
    c = make_channel(nx=nx, ny=ny, nz=nz, **kw)
    if kind == "rusanov":
        c.params.flux_splitting = 1
    if kind == "stretched":
        f = 1.0 + 0.05 * np.sin(2.0 * np.pi * np.arange(nx) / nx)
        c.grid.dcsidx[:] *= f
        c.grid.dcsidxs[:] *= f * f
    return c


def _advance(c, nsteps, precision=0, tuning=(0, 0)):
    p = params_copy(c.params)
    p.precision = precision
    with ChannelSolver(p, c.grid) as g:
        capi.check(g.L.st_set_tuning(g.h, *tuning))
        g.copy_from_field(c.w0)
        g.init_run()
        g.advance(nsteps)
        return g.copy_to_field(), g.count_weno()


def _oracle(c, nsteps):
    o = Oracle(c.params, c.grid)
    o.w[:] = c.w0
    o.init_run()
    o.advance(nsteps)
    return o


def _errors(w, o):
    return [rel_l2(interior(w)[m], interior(o.w)[m]) for m in range(5)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("tuning", [(8, 8), (1, 3), (16, 32), (3, 5)])
def test_results_independent_of_launch_shape(kind, tuning):
    c = _channel(kind, mach=0.8, retau=150.0, sensor_threshold=0.5)
    a, b = (_advance(c, 12, tuning=t)[0] for t in ((0, 0), tuning))
    assert np.array_equal(interior(a), interior(b))


@pytest.mark.parametrize("precision", [0, PREC_MIXED])
@pytest.mark.parametrize("visc_chunk", [1, 3, 8, 32, 33, 1024])
def test_one_pass_without_bulk_sums_independent_of_launch_shape(visc_chunk, precision):
    """48 planes: chunks of one plane, with a remainder, and above the 32 of the
    kernel's tables, to which they are clamped."""
    c = make_bl_box(nx=40, ny=17, nz=48, seed=2, sensor_threshold=0.5)
    a, b = (_advance(c, 6, precision, t)[0] for t in ((0, 0), (visc_chunk, 0)))
    assert np.array_equal(interior(a), interior(b))


@pytest.mark.parametrize("kind", KINDS)
def test_trajectory_ragged_cell_count(kind):
    """29 x 21 x 11 cells, not a multiple of 8: the last word of the per-cell
    WENO flags also holds the sweeps' any-dirty bytes."""
    c = _channel(kind, nx=29, ny=21, nz=11, sensor_threshold=0.2, seed=2)
    o = _oracle(c, 10)
    w, count = _advance(c, 10)
    assert min(o.count_weno()) > 0.005 and np.array_equal(count, o.count_weno())
    errs = _errors(w, o)
    assert max(errs) <= TRAJ_TOL, errs


@pytest.mark.parametrize("kind", KINDS)
def test_bitwise_reproducible_all_weno(kind):
    """Every face WENO: several segments of the compacted lists."""
    c = _channel(kind, nx=64, ny=48, nz=32, sensor_threshold=0.0, seed=3)
    a, b = (_advance(c, 4)[0] for _ in range(2))
    assert np.array_equal(interior(a), interior(b))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("kw", [{}, {"sensor_threshold": -1.0}, {"conservative_viscous": 1, "visc_model": 2},
                                {"theta_wall": 1.0}], ids=["default", "all-weno", "conservative", "bulk-temperature"])
def test_mixed_trajectory(kind, kw):
    c = _channel(kind, nx=40, ny=32, nz=24, **kw)
    errs = _errors(_advance(c, 20, PREC_MIXED)[0], _oracle(c, 20))
    assert max(errs) <= MIXED_TOL, errs


@pytest.mark.parametrize("precision", [0, PREC_MIXED])
@pytest.mark.parametrize("autotune", [False, True])
def test_served_and_batched(precision, autotune):
    """The sweeps' kernels over a table of solves, and their nine launch shapes
    timed on the first chunks of a class."""
    reqs = [Request(_channel(KINDS[n % 2], nx=32 + 8 * (n % 2), sensor_threshold=0.5, seed=n, precision=precision), 40, 0.0)
            for n in range(6)]
    seq = run_sequential(reqs, want_fields=True)
    srv = run_serving(reqs, hbm_bytes=8 << 30, max_slots=6, steps_per_graph=4, autotune=autotune, want_fields=True,
                      timeout=60.0, batch=1)
    assert srv["stats"]["batched_chunks"] > 0
    for n, (a, b) in enumerate(zip(seq["results"], srv["results"])):
        assert b["error"] is None, (n, b["error"])
        assert np.array_equal(interior(a["w"]), interior(b["w"])), n
