"""Beams whose width grows past the largest number: a ray that reflects on and
on along a rough bottom multiplies its q at every bounce. The reference's
arithmetic turns p, and with the next step q, into NaN there (its zero second
derivatives multiply an infinite q), so the product's must, step for step."""
import ctypes as C

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd import _abi
from bellhopcuda_amd.env import Boundary, Halfspace, munk_env
from bellhopcuda_amd.env3d import c3_env
import oracle
from test_host import harness  # noqa: F401  (fixture)


def _duct():
    """A wavy channel of 135 to 165 m, 20 km long, rigid bottom, FP32."""
    e = munk_env(nbeams=24, run_type="RG", precision=32, r_max_km=20.0, alpha=(-40.0, 40.0), sd=50.0)
    x = np.linspace(0.0, 21.2, 500)
    e.bty = Boundary("CS", r_km=x, z=150.0 + 15.0 * np.sin(12.0 * x))
    e.bot = Halfspace("R", depth=5000.0)
    return e


def _shelf(precision):
    return c3_env(seed=33, nalpha=3, nbeta=2, ntheta=2, nrz=3, nrr=5, nxy=22, precision=precision, run_type="R    3")


def _overflows(q, n):
    return [k for k in range(len(n)) if not np.isfinite(q[k, :n[k]]).all()]


def test_2d_rays_equal_the_oracle(harness):  # noqa: F811
    e, M = _duct(), 4000
    po, no, _ = oracle.ray_run(e, max_points=M)
    rays = _overflows(po["q"], no)
    assert rays
    p = bh.Problem(e)
    harness.core_ray_run2d.argtypes = [C.POINTER(_abi.Problem2D), C.c_int, C.c_int, C.c_int, C.POINTER(_abi.RayPt2D),
                                       C.POINTER(C.c_int)]
    for k in rays:
        pts, n = (_abi.RayPt2D * M)(), C.c_int()
        assert harness.core_ray_run2d(C.byref(p.view), 0, k, M, pts, C.byref(n)) == 0
        g = np.ctypeslib.as_array(pts)
        assert n.value == no[k]
        for f in ("x", "t", "p", "q"):
            assert np.array_equal(g[:no[k]][f], po[k, :no[k]][f], equal_nan=True), (k, f)


@pytest.mark.parametrize("precision", [32, 64])
def test_3d_rays_equal_the_oracle(precision, harness):  # noqa: F811
    e, M = _shelf(precision), 2500
    po, no = oracle.ray_run3d(e, max_points=M)
    ao = np.ctypeslib.as_array(po).reshape(len(no), M)
    assert _overflows(ao["q"], no)
    harness.core_ray_run3d.restype = C.c_int
    harness.core_ray_run3d.argtypes = [C.POINTER(_abi.Problem3D), C.POINTER(_abi.RayPt3D), _abi.c_int32_p, C.c_int]
    p = bh.Problem3D(e)
    pts, n = (_abi.RayPt3D * (len(no) * M))(), np.zeros(len(no), np.int32)
    assert harness.core_ray_run3d(C.byref(p.view), pts, n.ctypes.data_as(_abi.c_int32_p), M) == 0
    assert np.array_equal(n, no)
    g = np.ctypeslib.as_array(pts).reshape(len(no), M)
    for k in range(len(no)):
        for f in ("x", "t", "p", "q", "phi"):
            assert np.array_equal(g[k, :no[k]][f], ao[k, :no[k]][f], equal_nan=True), (k, f)


@pytest.mark.gpu
def test_gpu_2d_rays_equal_the_oracle(gpu_ctx):
    print("\n[gpu-case] overflow_2d", flush=True)
    e, M = _duct(), 4000
    po, no, _ = oracle.ray_run(e, max_points=M)
    pg, ng, _ = bh.ray_run(e, ctx=gpu_ctx, max_points=M)
    assert np.array_equal(no, ng) and _overflows(po["q"], no)
    for k in range(len(no)):
        for f in ("x", "t", "p", "q"):
            assert np.array_equal(pg[k, :no[k]][f], po[k, :no[k]][f], equal_nan=True), (k, f)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
def test_gpu_3d_p_is_nan_after_an_infinite_q(precision, gpu_ctx):
    """(The torsion's device functions differ from the host's by an ulp, so the
    step at which q overflows may, too; what follows it may not.)"""
    print("\n[gpu-case] overflow_3d_f%d" % precision, flush=True)
    e, M = _shelf(precision), 2500
    _, pts, n = bh.ray_run3d(e, ctx=gpu_ctx, max_points=M)
    g = np.ctypeslib.as_array(pts).reshape(len(n), M)
    rays = _overflows(g["q"], n)
    assert rays
    for k in rays:
        first = int(np.argmax(~np.isfinite(g[k, :n[k]]["q"]).all(axis=1)))
        # one more point may be a reflection, which leaves p to the next step
        assert np.isnan(g[k, first + 2:n[k]]["p"]).any(axis=1).all(), k
