"""GPU: the edges of the launch rules -- how a fan is spread over wavefronts,
where a problem's tables lie, which scatter mapping a pass takes, how a sweep
orders and splits its problems, kept device blocks and the surrogate network's
tiles -- each against the oracle, a single-problem run or the FP64 restatement.
"""
import sys

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import Boundary, c2_env, munk_env
import cases
import mlp_ref
import oracle
from parity import env_context, tl_err

pytestmark = pytest.mark.gpu


def _announce(name):
    print("\n[gpu-case]", name, flush=True)
    sys.stdout.flush()


def _same_as_oracle(env, ctx):
    o = oracle.field_run(env, nthreads=0)
    g = bh.field_run(env, ctx=ctx, stats=True)
    assert (g.err, g.warn) == (o.err, o.warn)
    assert np.array_equal(g.nsteps, o.nsteps) and np.array_equal(g.xend, o.xend)
    assert np.array_equal(g.ntop, o.ntop) and np.array_equal(g.nbot, o.nbot)
    assert g.total_steps == o.total_steps and g.total_contrib == o.total_contrib
    # the parity bar for TL: FP32 atomics in another order
    assert tl_err(g.problem.scale_pressure(g.field), oracle.scale_pressure(env, o.field)) <= 0.1


@pytest.mark.parametrize("nbeams", [2, 63, 64, 65, 1023, 1025, 4097])
def test_fan_spread_over_wavefronts(nbeams, gpu_ctx):
    """One ray per wavefront up to the number of SIMDs, then more, up to 64."""
    _announce("fan_%d" % nbeams)
    _same_as_oracle(munk_env(nbeams=nbeams, nrz=11, nrr=21), gpu_ctx)


@pytest.mark.parametrize("nodes", [2, 600, 1300, 3000])
@pytest.mark.parametrize("node_kind", ["LS", "CS"])
def test_tables_staged_and_in_memory(nodes, node_kind, gpu_ctx):
    """Tables within a wavefront's share of the LDS, over it, and over the
    largest budget; four reals per node for straight segments, more else."""
    _announce("tables_%d_%s" % (nodes, node_kind))
    e = munk_env(nbeams=129, nrz=11, nrr=21, r_max_km=30.0)
    r = np.linspace(0.0, 31.0, nodes)
    e.bty = Boundary(node_kind, r_km=r, z=4600.0 - 300.0 * np.sin(r / 3.0))
    e.box_r_km = 31.0
    _same_as_oracle(e, gpu_ctx)


MAPPED = {
    "hat_sparse": lambda: munk_env(nbeams=301, nrz=11, nrr=201),
    "hat_dense": lambda: munk_env(nbeams=65, nrz=201, nrr=201),
    "gauss_sparse": lambda: munk_env(nbeams=301, nrz=5, nrr=201, run_type="CB"),
    "gauss_dense": lambda: munk_env(nbeams=65, nrz=201, nrr=201, run_type="CB"),
    "raycen_short_rows": lambda: c2_env(nbeams=101, nrz=61, nrr=101),
    "raycen_long_rows": lambda: c2_env(nbeams=65, nrz=31, nrr=2001, run_type="Cg"),
    "several_sources": lambda: cases.several_sources(),
    "irregular_grid": lambda: cases.irregular_grid(),
}


@pytest.mark.parametrize("name", list(MAPPED))
def test_chosen_scatter_mapping_equals_each_one(name, gpu_ctx):
    """The mapping that a pass chooses for itself, and each that can be asked
    for, hand out the same contributions. The sums differ by the order of their
    FP32 atomics: n terms in another order move a sum by at most n * 2^-24 of
    the terms' absolute sum, 0.01 dB for the at most ~100 terms per receiver
    here, wherever they do not cancel by more than two orders."""
    _announce("mapping_" + name)
    env = MAPPED[name]()
    p = bh.Problem(env)
    ref = bh.field_run(p, ctx=gpu_ctx)
    o = oracle.field_run(env, nthreads=0)
    assert ref.total_contrib == o.total_contrib
    assert tl_err(p.scale_pressure(ref.field), oracle.scale_pressure(env, o.field)) <= 0.1
    dev = bh.Resident(p, gpu_ctx)
    for mode in (1, 2, 3):
        dev.set_scatter(mode)
        dev.launch()
        g = dev.download()
        assert g.total_contrib == ref.total_contrib, mode
        assert tl_err(p.scale_pressure(g.field), p.scale_pressure(ref.field)) <= 0.01, mode
    dev.release()


def _mixed_lengths(precision):
    """Problems whose rays differ in length by an order of magnitude, short
    ones first, with tables from a few hundred bytes to over a wavefront's
    share of the LDS."""
    envs = [munk_env(nbeams=100 + 7 * k, nrz=11, nrr=31, r_max_km=8.0, precision=precision) for k in range(9)]
    wide = munk_env(nbeams=65, nrz=11, nrr=31, r_max_km=8.0, precision=precision)
    wide.bty = Boundary("LS", r_km=np.linspace(0.0, 9.0, 1500), z=np.linspace(4900.0, 4600.0, 1500))
    envs.append(wide)
    envs += [munk_env(nbeams=n, nrz=21, nrr=41, r_max_km=100.0, ssp_type=t, precision=precision)
             for n, t in ((17, "C"), (130, "P"), (33, "S"))]
    return envs


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("segment_mb", [None, 3000])
def test_sweep_order_long_rays_and_wavefronts(precision, segment_mb, gpu_ctx):
    """Long problems go first and a few rays per wavefront; two wavefronts per
    SIMD with the default LDS share, one where the segment buffer is small or
    the budget is the largest table's, and no staging: the same rays."""
    _announce("sweep_order_f%d_%s" % (precision, segment_mb))
    ctx = gpu_ctx if segment_mb is None else env_context(BHC_SEG_BUFFER_MB=segment_mb)
    probs = [bh.Problem(e) for e in _mixed_lengths(precision)]
    single = [bh.field_run(p, ctx=gpu_ctx, stats=True) for p in probs]
    sw = bh.Sweep(probs, ctx, stats=True)
    for lds in (None, 40960, 0):
        if lds is not None:
            sw.set_launch(1024, lds)
        sw.launch()
        assert sw.stats()["contrib"] == sum(s.total_contrib for s in single)
        for i, (p, s) in enumerate(zip(probs, single)):
            g = sw.download(i)
            assert (g.err, g.warn) == (s.err, s.warn), (lds, i)
            assert np.array_equal(g.nsteps, s.nsteps) and np.array_equal(g.xend, s.xend), (lds, i)
            assert tl_err(p.scale_pressure(g.field), p.scale_pressure(s.field)) <= 0.01, (lds, i)
    sw.release()
    if segment_mb is not None:
        ctx.close()


def test_kept_blocks_hold_no_earlier_run(gpu_ctx):
    """Blocks that one run gave back serve the next, of another size and kind:
    arrivals (every byte, the slots past the counts among them), eigenray hits
    (in any order) and fields are those of a fresh context."""
    _announce("kept_blocks")
    # the Gaussian beams fill slots of the arrivals array that the hat beams leave
    envs = [munk_env(nbeams=301, nrz=21, nrr=41, run_type="AB"), munk_env(nbeams=101, nrz=51, nrr=101),
            munk_env(nbeams=101, nrz=11, nrr=21, run_type="EG"), munk_env(nbeams=301, nrz=21, nrr=41, run_type="AG")]
    fresh = []
    for e in envs:
        c = bh.Context(0)
        fresh.append(bh.field_run(e, ctx=c, max_narr=20, eigen_memsize=100000))
        c.close()
    for e, f in zip(envs, fresh):
        g = bh.field_run(e, ctx=gpu_ctx, max_narr=20, eigen_memsize=100000)
        assert g.total_contrib == f.total_contrib and (g.err, g.warn) == (f.err, f.warn)
        if "A" in e.run_type:
            assert f.narr.sum() > 0 and np.array_equal(g.narr, f.narr) and bytes(g.arr) == bytes(f.arr)
        elif "E" in e.run_type:
            n = int(f.neigen[0])
            assert 0 < n <= 100000 and g.neigen[0] == n
            hits = [np.ctypeslib.as_array(r.hits)[:n] for r in (g, f)]
            assert np.array_equal(*[np.sort(h, order=h.dtype.names) for h in hits])
        else:
            assert tl_err(g.problem.scale_pressure(g.field), f.problem.scale_pressure(f.field)) <= 0.01


@pytest.mark.parametrize("n,n_out,front", [(32, 1, 1), (160, 1, 0), (32, 32, 0), (160, 256, 1), (992, 96, 0)])
def test_network_tiles(n, n_out, front):
    """Batches of an odd number of row tiles and output widths from one tile to
    the hidden width: gradients against the FP64 restatement (bounds of the
    existing gradient test: BF16 operands, FP32 sums)."""
    _announce("network_tiles_%d_%d_%d" % (n, n_out, front))
    from bellhopcuda_amd import surrogate
    m = surrogate.Mlp(members=3, max_batch=1024, seed=5, n_out=n_out, front=front)
    try:
        rng = np.random.default_rng(n + n_out)
        x = rng.random((n, 16), dtype=np.float32)
        y = rng.normal(size=(n, n_out) if n_out > 1 else n).astype(np.float32)
        P, Bf = m.params()
        o, nw = mlp_ref.layout(n_out)[0]["Wout"][0], 256 * n_out + n_out
        P[:, o:o + nw] = rng.normal(scale=0.1, size=(3, nw)).astype(np.float32)
        m.set_params(P)
        g, loss = m.gradients(x, y)
        for e in range(3):
            _, loss_r, g_r = mlp_ref.forward_backward(P[e], Bf, x, y.astype(np.float64), n_out, front)
            assert loss[e] == pytest.approx(loss_r, rel=2e-4)
            assert np.max(np.abs(g[e] - g_r)) < 2e-3 * np.max(np.abs(g_r))
        whole = m.predict(x)
        for k in (1, 31, n - 1):   # part of a tile: each row is its own
            assert np.array_equal(m.predict(x[:k]), whole[:, :k])
    finally:
        m.close()


@pytest.mark.parametrize("nodes", [2, 3000])
@pytest.mark.parametrize("ssp_type", ["C", "N", "S", "P"])
@pytest.mark.parametrize("nbeams", [2, 65, 1100])
def test_ray_paths_spread_over_wavefronts(nbeams, ssp_type, nodes, gpu_ctx):
    """Every point of every ray, bit for bit, for fans below and above one ray
    per SIMD and tables in the LDS and in memory."""
    _announce("ray_paths_%d_%s_%d" % (nbeams, ssp_type, nodes))
    e = munk_env(nbeams=nbeams, run_type="RG", ssp_type=ssp_type, r_max_km=20.0)
    r = np.linspace(0.0, 21.0, nodes)
    e.bty = Boundary("LS", r_km=r, z=4600.0 - 300.0 * np.sin(r / 3.0))
    e.box_r_km = 21.0
    po, no, _ = oracle.ray_run(e, max_points=600)
    pg, ng, _ = bh.ray_run(e, ctx=gpu_ctx, max_points=600)
    assert np.array_equal(no, ng)
    for k in range(len(no)):
        for f in ("x", "t", "NumTopBnc", "NumBotBnc"):
            assert np.array_equal(po[k, :no[k]][f], pg[k, :no[k]][f]), (k, f)
