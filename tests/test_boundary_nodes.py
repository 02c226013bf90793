"""CPU: a boundary node packed as position and normal (straight segments whose
tangent follows from the normal, no curvature) gives the rays of the node with
its tangent and curvature written out."""
import ctypes as C

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import c2_env, munk_env
import cases
from test_host import harness  # noqa: F401  (fixture)

CASES = {
    "flat": lambda b: munk_env(nbeams=65, nrz=11, nrr=21, precision=b),
    "seamount": lambda b: c2_env(nbeams=65, nrz=11, nrr=21, precision=b),
    "altimetry": lambda b: cases.altimetry(b),
    "beam_shift": lambda b: cases.beam_shift(b),
}


def _run(p, harness):  # noqa: F811
    res = bh.FieldResult()
    out = bh._make_out(p, res, True, 0, 1, 0)
    assert harness.core_field_run2d(C.byref(p.view), C.byref(out)) == 0
    return res, out


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("name", list(CASES))
def test_short_and_full_straight_nodes_agree(name, bits, harness):  # noqa: F811
    p = bh.Problem(CASES[name](bits))
    a, oa = _run(p, harness)
    # a curvature far below the last place of every sum it enters
    p.view.bty[0].kappa = 1e-300
    b, ob = _run(p, harness)
    assert (oa.err, oa.warn) == (ob.err, ob.warn)
    assert oa.total_steps == ob.total_steps and oa.total_contrib == ob.total_contrib
    assert np.array_equal(a.nsteps, b.nsteps) and np.array_equal(a.xend, b.xend)
    assert np.sum(a.nbot) > 0 and np.array_equal(a.nbot, b.nbot)
    # the sums' order may differ between runs on several threads
    assert np.allclose(a.field, b.field, rtol=2e-5, atol=2e-6 * np.abs(a.field).max())
