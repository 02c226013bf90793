"""GPU: every part of an output array that reaches the caller is the run's own.
A context keeps the device blocks of earlier runs for later ones, so each test
makes a run that fills a block and then one of the same sizes that fills less
of it: what the second does not write must be zero, as in a fresh context.
"""
import sys

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import munk_env
from bellhopcuda_amd.env3d import c3_env

pytestmark = pytest.mark.gpu

NARR = 12


def _announce(name):
    print("\n[gpu-case]", name, flush=True)
    sys.stdout.flush()


def _raw(array, shape):
    """A ctypes array's records as bytes, so that every field is compared."""
    a = np.ctypeslib.as_array(array)
    return a.view(np.uint8).reshape(shape + (a.dtype.itemsize,))


def _shelf(run, dense):
    return c3_env(nalpha=61 if dense else 5, nbeta=4, ntheta=4, nrz=7, nrr=21, nxy=41, run_type=run)


ARRIVALS = {
    "2d": (lambda dense: munk_env(nbeams=801 if dense else 21, nrz=7, nrr=41, run_type="AB" if dense else "AG"),
           bh.field_run),
    "2d_first_ones": (lambda dense: munk_env(nbeams=801 if dense else 21, nrz=7, nrr=41,
                                             run_type="aB" if dense else "aG"), bh.field_run),
    "3d": (lambda dense: _shelf("AB   3" if dense else "AG   3", dense), bh.field_run3d),
    "nx2d": (lambda dense: _shelf("AB   2" if dense else "AG   2", dense), bh.field_run3d),
}


@pytest.mark.parametrize("name", list(ARRIVALS))
def test_arrival_slots_past_the_count_are_zero(name):
    _announce("arrival_slots_" + name)
    make, run = ARRIVALS[name]
    merging = 0 if name == "2d_first_ones" else 1
    ctx = bh.Context(0)
    try:
        dense = run(make(True), ctx=ctx, max_narr=NARR, allow_merging=merging)
        sparse = run(make(False), ctx=ctx, max_narr=NARR, allow_merging=merging)
    finally:
        ctx.close()
    n = len(sparse.narr)
    assert np.any(np.minimum(dense.narr, NARR) > sparse.narr)     # the first run filled slots the second does not
    tail = _raw(sparse.arr, (n, NARR))[np.arange(NARR) >= sparse.narr[:, None]]
    assert tail.size and not tail.any()


@pytest.mark.parametrize("dim", [2, 3])
def test_ray_points_past_the_last_step_are_zero(dim):
    _announce("ray_points_%dd" % dim)
    M = 2500
    ctx = bh.Context(0)
    try:
        if dim == 2:
            long, short = [munk_env(nbeams=9, run_type="RG", r_max_km=r) for r in (100.0, 5.0)]
            bh.ray_run(long, ctx=ctx, max_points=M)
            pts, nsteps, _ = bh.ray_run(short, ctx=ctx, max_points=M)
            raw = np.ascontiguousarray(pts).view(np.uint8).reshape(len(nsteps), M, pts.dtype.itemsize)
        else:
            long, short = _shelf("R    3", False), _shelf("R    3", False)
            short.box_x_km = short.box_y_km = 2.0
            n_long = bh.ray_run3d(long, ctx=ctx, max_points=M)[2]
            _, pts, nsteps = bh.ray_run3d(short, ctx=ctx, max_points=M)
            assert np.any(n_long > nsteps)
            raw = _raw(pts, (len(nsteps), M))
    finally:
        ctx.close()
    tail = raw[np.arange(M) >= nsteps[:, None]]
    assert tail.size and not tail.any()


def test_download_before_a_launch_gives_zeros():
    _announce("download_before_launch")
    env = munk_env(nbeams=301, nrz=21, nrr=51)
    ctx = bh.Context(0)
    try:
        first = bh.field_run(env, ctx=ctx, stats=True)
        assert np.any(first.field) and np.all(first.nsteps > 0)
        dev = bh.Resident(bh.Problem(env), ctx, stats=True)
        g = dev.download()
        assert not g.field.any() and not g.nsteps.any() and not g.xend.any()
        assert (g.err, g.warn, g.total_steps, g.total_contrib) == (0, 0, 0, 0)
        dev.launch()
        g = dev.download()
        assert np.array_equal(g.nsteps, first.nsteps) and g.total_contrib == first.total_contrib
        dev.release()
    finally:
        ctx.close()
