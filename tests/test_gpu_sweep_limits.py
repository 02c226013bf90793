"""GPU: the staging budgets that bhc_sweep_set_launch takes: multiples of a
real up to the largest problem's whole tables, or 40960 bytes."""
import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import Boundary, munk_env

pytestmark = pytest.mark.gpu


def _env(ssp, nodes, precision):
    e = munk_env(nbeams=65, nrz=17, nrr=21, r_max_km=8.0, ssp_type=ssp, precision=precision)
    e.bty = Boundary("LS", r_km=np.linspace(0.0, 9.0, nodes), z=np.linspace(4900.0, 4700.0, nodes))
    return e


def _table_reals(p):
    """Depth, density, sound speed and its gradient (complex) and the spline's
    four complex coefficients per knot; 8 reals per node; the receiver depths."""
    v = p.view
    n = v.ssp_npts
    return (2 + 2 + 2 + (8 if p.env.ssp_type == "S" else 0)) * n + 8 * (v.ati_npts + v.bty_npts) + v.NRz


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("ssp,nodes", [("C", 2), ("S", 2), ("C", 300), ("C", 3000)])
def test_budgets_up_to_the_largest_table(ssp, nodes, precision, gpu_ctx):
    print("\n[gpu-case] sweep_budget_%s_%d_f%d" % (ssp, nodes, precision), flush=True)
    probs = [bh.Problem(_env("C", 2, precision)), bh.Problem(_env(ssp, nodes, precision))]
    size = precision // 8
    limit = min(40960, size * max(_table_reals(p) for p in probs))
    sw = bh.Sweep(probs, gpu_ctx)
    try:
        sw.launch()
        contrib = sw.stats()["contrib"]
        for refused in (limit + size, limit + 4096, limit - 1, -size):
            with pytest.raises(bh.BhcError):
                sw.set_launch(1024, refused)
        for budget in (limit, limit // 2 // size * size, 0):
            sw.set_launch(1024, budget)
            sw.launch()
            assert sw.stats()["contrib"] == contrib > 0
    finally:
        sw.release()
