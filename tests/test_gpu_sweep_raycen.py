"""GPU: ray-centred beams in a sweep. Their depth window is searched for every
step, in the problem's staged copy of the receiver depths where it has one, else
in memory, with the other tables staged or not: all give the single runs' rays
and fields."""
import sys

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import Boundary, c2_env
from parity import tl_err

pytestmark = pytest.mark.gpu


def _env(k, nodes, nrz, precision):
    e = c2_env(seed=20260002 + k, nbeams=17, nrz=nrz, nrr=31, run_type="Cb" if k % 2 else "Cg", precision=precision,
               r_max_km=10.0)
    r = np.linspace(0.0, 11.0, nodes)
    e.bty = Boundary("LS", r_km=r, z=2900.0 - 300.0 * np.sin(r / 3.0))
    return e


@pytest.mark.parametrize("precision", [64, 32])
def test_depths_staged_and_in_memory(precision, gpu_ctx):
    print("\n[gpu-case] sweep_raycen_f%d" % precision, flush=True)
    sys.stdout.flush()
    # nodes and depths: all tables staged; the depths one time too many (FP64:
    # 3.3 KB of profile, 32 bytes per node, 8 per depth against 20480); tables
    # over the default budget, and over the largest
    sizes = [(2, 11), (2, 501), (500, 11), (500, 501), (1200, 31), (3000, 31)]
    probs = [bh.Problem(_env(k, n, z, precision)) for k, (n, z) in enumerate(sizes)]
    single = [bh.field_run(p, ctx=gpu_ctx, stats=True) for p in probs]
    sw = bh.Sweep(probs, gpu_ctx, stats=True)
    try:
        for lds, mode in ((None, 1), (None, 3), (40960, 1), (40960, 3), (0, 1)):
            if lds is not None:
                sw.set_launch(1024, lds)
            sw.set_scatter(mode)
            sw.launch()
            assert sw.stats()["contrib"] == sum(s.total_contrib for s in single), (lds, mode)
            for i, (p, s) in enumerate(zip(probs, single)):
                g = sw.download(i)
                assert (g.err, g.warn) == (s.err, s.warn), (lds, mode, i)
                assert np.array_equal(g.nsteps, s.nsteps) and np.array_equal(g.xend, s.xend), (lds, mode, i)
                # n FP32 terms in another order: n * 2^-24 of their absolute sum
                assert tl_err(p.scale_pressure(g.field), p.scale_pressure(s.field)) <= 0.01, (lds, mode, i)
    finally:
        sw.release()
