"""The one-pass stage (st_stage.hip) at the sizes where it can go wrong,
against the oracle: extents around its 32 x 8 tiles, 32-cell masks, 64-cell
records and plane chunks, boundary cells of lowered stencil order on every
kind of face, and work-item lists from empty over scattered (cells flagged in
one, two and three directions, sensors in the ghost points included) to full.

Tolerance: the trajectory bar of the parity tests, 1e-10 relative L2 per
conserved variable over a few steps, which leaves four decades over the
round-off the two orders of summation differ by; mixed precision 1e-5, its
bar there.
"""
import numpy as np
import pytest

from helpers import interior, rel_l2
from oracle import Oracle
from streams_mi355x import PREC_MIXED, make_channel
from streams_mi355x.cases import make_bl_box
from streams_mi355x.params import params_copy
from streams_mi355x.solver import ChannelSolver

pytestmark = pytest.mark.gpu

TOL = 1e-10
MIXED_TOL = 1e-5


def _errors(params, grid, w0, steps, sensor_seed=None, precision=None, twin=None):
    o = Oracle(params, grid)
    o.w[:] = w0
    o.init_run()
    p = params
    if precision is not None:
        p = params_copy(params)
        p.precision = precision
    with ChannelSolver(p, twin or grid) as g:
        g.copy_from_field(w0)
        g.init_run()
        if sensor_seed is not None:
            s = np.random.default_rng(sensor_seed).uniform(0.0, 1.0, size=o.w_aux[7].shape)
            o.w_aux[7][:] = s
            g.set_aux(8, s)
        o.advance(steps)
        g.advance(steps)
        w = g.copy_to_field()
        assert np.array_equal(g.count_weno(), o.count_weno())
    return [rel_l2(interior(w)[m], interior(o.w)[m]) for m in range(5)]


@pytest.mark.parametrize("size", [(3, 3, 3), (31, 8, 5), (32, 9, 3), (33, 7, 34), (63, 16, 7), (64, 17, 8), (65, 24, 4),
                                  (130, 3, 33)])
@pytest.mark.parametrize("threshold", [1.01, 0.97, 0.5, -1.0])
def test_channel_sizes_and_item_lists(size, threshold):
    nx, ny, nz = size
    c = make_channel(nx=nx, ny=ny, nz=nz, sensor_threshold=threshold, uniform_y=True, seed=nx)
    if not np.isfinite(c.params.mu0):
        c.params.mu0 = 1e-3  # three rows: the Re_tau relation has no half channel to integrate
    seed = None if threshold < 0 else 5
    errs = _errors(c.params, c.grid, c.w0, 2, sensor_seed=seed)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("kw", [{"ep_order": 2}, {"ep_order": 4, "weno_scheme": 2}, {"weno_scheme": 1},
                                {"correct_bound_ord": 0}, {"weno_version": 1}, {"theta_wall": 1.0},
                                {"conservative_viscous": 1, "visc_model": 2}])
def test_channel_schemes(kw):
    c = make_channel(nx=45, ny=21, nz=10, sensor_threshold=0.9, uniform_y=True, seed=3, **kw)
    errs = _errors(c.params, c.grid, c.w0, 3, sensor_seed=9)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("size", [(40, 24, 16), (33, 9, 5), (67, 19, 6)])
@pytest.mark.parametrize("conservative", [0, 1])
@pytest.mark.parametrize("nr", [(0, 1, 0, 1, 0, 0), (0, 0, 0, 0, 0, 0), (2, 1, 6, 3, 0, 0)])
def test_boundary_layer_faces(size, conservative, nr):
    nx, ny, nz = size
    c = make_bl_box(nx=nx, ny=ny, nz=nz, seed=2, conservative_viscous=conservative, bctags_nr=nr,
                    sensor_threshold=0.95)
    errs = _errors(c.params, c.grid, c.w0, 2, sensor_seed=4)
    assert max(errs[:3] + errs[4:]) <= TOL, errs
    assert errs[3] <= TOL, errs


@pytest.mark.parametrize("size", [(31, 8, 5), (65, 17, 12)])
@pytest.mark.parametrize("conservative", [0, 1])
def test_mixed_sizes(size, conservative):
    nx, ny, nz = size
    c = make_channel(nx=nx, ny=ny, nz=nz, uniform_y=True, seed=1, conservative_viscous=conservative)
    errs = _errors(c.params, c.grid, c.w0, 3, precision=PREC_MIXED)
    assert max(errs) <= MIXED_TOL, errs


@pytest.mark.parametrize("theta_wall", [-2.0, 1.0])
def test_non_uniform_x_takes_the_separate_sweeps(theta_wall):
    """The bulk sums by parts need one x metric; other grids keep the pass of
    their own."""
    c = make_channel(nx=36, ny=20, nz=8, seed=6, theta_wall=theta_wall)
    f = 1.0 + 0.1 * np.sin(2.0 * np.pi * np.arange(36) / 36.0)
    c.grid.dcsidx[:] *= f
    c.grid.dcsidxs[:] *= f * f
    errs = _errors(c.params, c.grid, c.w0, 3)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("make", [lambda: make_channel(nx=34, ny=11, nz=7, seed=8),
                                  lambda: make_channel(nx=34, ny=11, nz=7, seed=8, theta_wall=1.0),
                                  lambda: make_bl_box(nx=40, ny=17, nz=6, seed=2)])
@pytest.mark.parametrize("precision", [0, PREC_MIXED])
def test_one_call_leaves_what_single_steps_leave(make, precision):
    """Within a call, what no later stage reads is not stored; the arrays a
    caller can read afterwards are those of step-by-step calls, bit for bit."""
    c = make()
    c.params.precision = precision
    got = []
    for calls in ([3], [1, 1, 1]):
        with ChannelSolver(c.params, c.grid) as g:
            g.copy_from_field(c.w0)
            g.init_run()
            for n in calls:
                g.advance(n)
            got.append([g.copy_to_field(), g.get_fl()] + [g.get_aux(v) for v in range(1, 11)])
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("size", [(20, 7, 6), (20, 8, 6), (131, 9, 5)])
@pytest.mark.parametrize("tags", [(2, 2, 6, 7, 0, 0), (4, 2, 6, 2, 2, 2), (1, 4, 5, 7, 2, 2), (3, 4, 6, 4, 0, 0)])
def test_faces_of_one_launch(size, tags):
    """All faces at once, where a node wall or a shock changes the row an x
    face or a z face reads, down to rows that the y faces read from each other
    (they then launch one by one).  The bar of the face tests, 1e-14."""
    nx, ny, nz = size
    c = make_bl_box(nx=nx, ny=ny, nz=nz, seed=4, bctags=tags, bctags_nr=(0,) * 6, mach=0.5 if 3 in tags else 2.0,
                    **(dict(shock_angle_deg=35.0, xshock_imp=5.0, tanhfacs=0.5) if 7 in tags else {}))
    rng = np.random.default_rng(nx + ny)
    w0 = c.w0 * (1.0 + 0.01 * rng.standard_normal(c.w0.shape))
    o = Oracle(c.params, c.grid)
    o.w[:] = w0
    with ChannelSolver(c.params, c.grid) as g:
        g.copy_from_field(w0)
        o.update_ghost(0)
        g.update_ghost(0)
        w = g.copy_to_field()
    n = 3
    for m in range(5):
        a, b = w[m], o.w[m]
        assert rel_l2(a[n:-n, n:-n, :], b[n:-n, n:-n, :]) <= 1e-14, m
        assert rel_l2(a[n:-n, :, n:-n], b[n:-n, :, n:-n]) <= 1e-14, m
        assert rel_l2(a[:, n:-n, n:-n], b[:, n:-n, n:-n]) <= 1e-14, m


def test_unequal_nodes_in_x_take_the_separate_sweeps():
    """The conservative viscous form works from the node coordinates: with one
    x metric but unequal nodes the sums by parts do not hold either, which the
    pressure gradient they give shows."""
    c = make_channel(nx=36, ny=20, nz=8, seed=6, conservative_viscous=1)
    x = c.grid.x
    lx = 36 * (x[4] - x[3])
    x += 0.02 * lx * np.sin(2.0 * np.pi * (x - x[3]) / lx)
    o = Oracle(c.params, c.grid)
    o.w[:] = c.w0
    o.init_run()
    o.advance(1)
    with ChannelSolver(c.params, c.grid) as g:
        g.copy_from_field(c.w0)
        g.init_run()
        g.advance(1)
        dpdx = g.scalars()["dpdx"]
    assert abs(dpdx / o.scalars()["dpdx"] - 1.0) <= TOL
