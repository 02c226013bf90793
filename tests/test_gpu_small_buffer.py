"""GPU: fans on small segment buffers. A fan is spread over as many wavefronts
as the buffer has room for, so that a run takes the passes that its segments
need and not one for every few slot blocks that the wavefronts reserve."""
import sys

import numpy as np
import pytest

import bellhopcuda_amd as bh
import oracle
from bellhopcuda_amd.env import munk_env
from parity import env_context, tl_err

pytestmark = pytest.mark.gpu


def _announce(name):
    print("\n[gpu-case]", name, flush=True)
    sys.stdout.flush()


def _check(env, g):
    o = oracle.field_run(env, nthreads=0)
    assert (g.err, g.warn, g.total_steps, g.total_contrib) == (o.err, o.warn, o.total_steps, o.total_contrib)
    assert np.array_equal(g.nsteps, o.nsteps) and np.array_equal(g.xend, o.xend)
    assert tl_err(g.problem.scale_pressure(g.field), oracle.scale_pressure(env, o.field)) <= 0.1


# A step that is handed to the scatter crosses a receiver range, so a ray has
# at most as many segments as there are ranges (here they increase along it):
# rays x ranges slots at most, beside the partly used blocks' eighth.
@pytest.mark.parametrize("nbeams,nrr,precision", [(1025, 101, 64), (2001, 101, 64), (2001, 101, 32), (4097, 41, 64)])
def test_noalloc_launch_takes_one_pass(nbeams, nrr, precision, gpu_ctx):
    _announce("noalloc_one_pass_%d_%d_f%d" % (nbeams, nrr, precision))
    env = munk_env(nbeams=nbeams, nrz=11, nrr=nrr, r_max_km=5.0, precision=precision)
    dev = bh.Resident(bh.Problem(env), gpu_ctx, stats=True)
    try:
        rc = bh.lib().bhc_field_launch_noalloc(gpu_ctx._h, dev._h)
        assert rc == 0, bh.lib().bhc_last_error().decode()
        g = dev.download()
        assert gpu_ctx.last_phase()[2] == 1
        if precision == 64:
            g.problem = dev.prob
            _check(env, g)
    finally:
        dev.release()


@pytest.mark.parametrize("nbeams", [2, 500, 1025])
def test_smallest_segment_buffer_takes_one_pass(nbeams):
    _announce("smallest_buffer_%d" % nbeams)
    env = munk_env(nbeams=nbeams, nrz=11, nrr=41, r_max_km=5.0)
    ctx = env_context(BHC_SEG_BUFFER_MB=16)
    try:
        g = bh.field_run(env, ctx=ctx, stats=True)
        assert ctx.last_phase()[2] == 1
        _check(env, g)
    finally:
        ctx.close()
