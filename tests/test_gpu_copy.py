"""Field copies through the staged path (st_copy.hip): every ghosted value in
and out unchanged, for fields of one thread, of some and of all, rows that do
not divide a buffer, rows longer than one, both precisions of w_aux, and two
solvers that copy at once.  Copies are exact."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from streams_mi355x import PREC_MIXED, make_channel
from streams_mi355x.solver import ChannelSolver

pytestmark = pytest.mark.gpu


def _case(size, precision=0):
    nx, ny, nz = size
    c = make_channel(nx=nx, ny=ny, nz=nz, uniform_y=True, seed=1)
    if not np.isfinite(c.params.mu0):
        c.params.mu0 = 1e-3  # three rows: the Re_tau relation has no half channel to integrate
    c.params.precision = precision
    return c


def _round_trip(size, seed):
    c = _case(size)
    with ChannelSolver(c.params, c.grid) as g:
        w = np.random.default_rng(seed).standard_normal((5,) + g.shape_g)
        for _ in range(2):
            g.copy_from_field(w)
            assert np.array_equal(g.copy_to_field(), w)
            w = w[:, ::-1].copy()


@pytest.mark.parametrize("size", [(3, 3, 3), (32, 24, 16), (61, 33, 47), (62, 66, 64), (131, 97, 90), (263000, 3, 3)])
def test_field_round_trip(size):
    _round_trip(size, seed=size[0])


@pytest.mark.parametrize("precision", [0, PREC_MIXED])
def test_aux_round_trip(precision):
    c = _case((131, 97, 90), precision)
    with ChannelSolver(c.params, c.grid) as g:
        a = np.random.default_rng(2).standard_normal(g.shape_g).astype(np.float32).astype(np.float64)
        g.set_aux(3, a)
        assert np.array_equal(g.get_aux(3), a)


def test_two_solvers_copy_at_once():
    with ThreadPoolExecutor(2) as ex:
        for f in [ex.submit(_round_trip, (96, 80, 70), s) for s in (3, 4)]:
            f.result()


def test_one_handle_read_by_two_threads():
    c = _case((96, 80, 70))
    with ChannelSolver(c.params, c.grid) as g:
        w = np.random.default_rng(5).standard_normal((5,) + g.shape_g)
        g.copy_from_field(w)
        with ThreadPoolExecutor(2) as ex:
            for f in [ex.submit(g.copy_to_field) for _ in range(4)]:
                assert np.array_equal(f.result(), w)
