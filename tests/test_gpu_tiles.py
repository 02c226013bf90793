"""GPU: which fields have LDS tiles for their scatter, at the edges of the rule:
the depths that a 64 KiB tile of six range columns still holds, and sources
that get range bins of their own while 16384 bins last."""
import sys

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import munk_env
from parity import tl_db, tl_err

pytestmark = pytest.mark.gpu


def _announce(name):
    print("\n[gpu-case]", name, flush=True)
    sys.stdout.flush()


def _mappings_agree(env, ctx):
    """The sums differ by the order of their FP32 atomics: n terms in another
    order move a sum by at most n * 2^-24 of the terms' absolute sum, 0.01 dB for
    the at most ~100 terms per receiver here, wherever they do not cancel by more
    than two orders."""
    p = bh.Problem(env)
    dev = bh.Resident(p, ctx)
    try:
        ref = None
        for mode in (2, 1, 3, 0):
            dev.set_scatter(mode)
            dev.launch()
            g = dev.download()
            field = p.scale_pressure(g.field)
            if ref is None:
                ref, contrib = field, g.total_contrib
                assert contrib > 0 and all(np.any(tl_db(f) < 120) for f in field)     # every source has a field
                continue
            assert g.total_contrib == contrib, mode
            assert tl_err(field, ref) <= 0.01, mode
    finally:
        dev.release()


@pytest.mark.parametrize("run", ["CB", "Cb"])
@pytest.mark.parametrize("nrz", [1317, 1318, 1365, 1366])
def test_depths_of_the_narrowest_tile(nrz, run, gpu_ctx):
    _announce("tile_depths_%d_%s" % (nrz, run))
    _mappings_agree(munk_env(nbeams=65, nrz=nrz, nrr=41, run_type=run), gpu_ctx)


def test_narrowest_tile_is_used(gpu_ctx):
    """The mapping search finds the tiles, four times as fast here as the others."""
    _announce("narrowest_tile_used")
    dev = bh.Resident(bh.Problem(munk_env(nbeams=1001, nrz=1365, nrr=501, run_type="CB")), gpu_ctx)
    try:
        assert dev.autotune() == 1
    finally:
        dev.release()


# steps of 500 m and ranges 2 m apart: one range per bin
@pytest.mark.parametrize("sources,nrr", [(1, 16384), (1, 16385), (2, 9001), (3, 6001), (5, 6001)])
def test_sources_beyond_the_bins(sources, nrr, gpu_ctx):
    _announce("tile_sources_%d_%d" % (sources, nrr))
    env = munk_env(nbeams=33, nrz=51, nrr=nrr, r_max_km=0.002 * (nrr - 1), run_type="CB")
    env.Sz = np.linspace(400.0, 3000.0, sources).astype(np.float32)
    _mappings_agree(env, gpu_ctx)
