"""Forward steps of one launch each against steps of two launches: a context
that also records pressure keeps the two.  The sums and updates of a point are
the same operations in the same order, so fields and seismograms are equal.

Cases: calls of one to a few steps and around one and two replayed pieces of
odd and even length; tiles of 64, 16 and 3 elements (shared points of two to
four tiles); sampled every step and every third; 4- and 9-node elements.  The
kernel launches of each run say which form it took: a chain of n steps is n
launches, one for the predictor, one for the counters, one for the seismograms
of its last step and one that closes it."""

import ctypes
import dataclasses

import numpy as np
import pytest

from specfempp_amd import _lib
from specfempp_amd.config import Config2D, Receivers2D, Sources2D
from specfempp_amd.mesh import Mesh2D, box_mesh, elastic_moduli
from specfempp_amd.solver import Context
from tests._cases import acoustic_box, adjoint_small, rel_l2, warped

pytestmark = pytest.mark.gpu


DVA = ("displacement", "velocity", "acceleration")


def _kernels(ctx):
    n = ctypes.c_int()
    _lib.check(ctx.lib.smx_last_run_kernels(ctx.h, ctypes.byref(n)))
    return n.value


def _run(cfg, types, nsbs, options, precision, calls):
    """Seismograms and fields, and the kernel launches of each call."""
    ctx = Context(cfg.mesh, cfg.sources, cfg.receivers, cfg.dt, cfg.nstep, nsbs=nsbs,
                  seismo_types=types, precision=precision, options=options)
    ctx.initialize()
    at, launches = 0, []
    for n in calls:
        ctx.run_forward(at, n)
        launches.append(_kernels(ctx))
        at += n
    ctx.synchronize()
    out = [ctx.seismograms()] + [ctx.get_field(f) for f in ("u", "v", "a")]
    ctx.close()
    return out, launches


@pytest.mark.parametrize("ngnod,precision", [(4, 4), (9, 4), (4, 8)])
@pytest.mark.parametrize("tile,graph,nsbs,calls", [
    (64, 8, 1, (1, 2, 3, 9, 10, 17)), (64, 7, 3, (8, 15, 16, 3)), (16, 1, 1, (2, 5, 1)),
    (3, 5, 1, (11, 12)), (3, 8, 3, (25,))])
def test_one_launch_equals_two(tile, graph, nsbs, calls, ngnod, precision):
    cfg = adjoint_small(nx=13, nz=10, nstep=sum(calls))
    if ngnod == 9:
        m = box_mesh(0.0, 650.0, 0.0, 500.0, 13, 10, ngnod=9,
                     absorbing=("bottom", "right", "left"))
        cfg = dataclasses.replace(cfg, mesh=dataclasses.replace(
            m, kappa=cfg.mesh.kappa, mu=cfg.mesh.mu, rho=cfg.mesh.rho))
    cfg = warped(cfg)
    print(f"one-launch steps: tile {tile}, graph {graph}, calls {calls}, ngnod {ngnod}, "
          f"precision {precision}", flush=True)
    opt = {"tile_elems": tile, "graph_steps": graph}
    one, k_one = _run(cfg, DVA, nsbs, opt, precision, calls)
    two, k_two = _run(cfg, ("pressure", *DVA), nsbs, opt, precision, calls)
    only, k_only = _run(cfg, ("displacement",), nsbs, opt, precision, calls)
    assert k_one == k_only == [n + 4 for n in calls]
    assert k_two == [4 * n + 2 for n in calls]  # pressure, tiles, sums, shared points
    assert np.abs(one[0]).max() > 0 and np.isfinite(one[0]).all()
    assert np.array_equal(one[0], two[0][:, 1:])
    assert np.array_equal(only[0][:, 0], one[0][:, 0])
    for a, b, c in zip(one[1:], two[1:], only[1:]):
        assert np.array_equal(a, b) and np.array_equal(c, b)


@pytest.mark.parametrize("types", [("displacement",), DVA])
def test_checkpoint_segments(types):
    """Checkpointed runs by segment length: seismograms and the final state of
    the plain run, and never more launches than steps in pairs take."""
    nstep = 22
    cfg = warped(adjoint_small(nx=13, nz=10, nstep=nstep))
    opt = {"tile_elems": 16, "graph_steps": 3}
    want, _ = _run(cfg, types, 1, opt, 4, (nstep,))
    pair = 2 if types == ("displacement",) else 3  # tiles, shared points, sums
    for every in (1, 2, 3, 4, 7, 21, 22):
        print(f"checkpoints every {every} of {nstep}, {types}", flush=True)
        ctx = Context(cfg.mesh, cfg.sources, cfg.receivers, cfg.dt, nstep, seismo_types=types,
                      options=opt)
        ctx.initialize()
        ctx.run_forward_checkpointed(every)
        # predictor and counter; the sums of the last step are a launch of their own
        assert _kernels(ctx) <= 2 + pair * nstep + 1
        got = [ctx.seismograms()] + [ctx.get_field(f) for f in ("u", "v", "a")]
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
        ctx.close()


def _fan(n=6, radius=60.0):
    """n elements around one vertex: with one element to a tile the vertex is
    shared by n tiles."""
    t = 2 * np.pi / n * np.arange(n)
    ring = radius * np.stack([np.cos(t), np.sin(t)], axis=1)
    outer = 1.3 * radius * np.stack([np.cos(t + np.pi / n), np.sin(t + np.pi / n)], axis=1)
    k = np.arange(n)
    knods = np.stack([0 * k, 1 + k, 1 + n + k, 1 + (k + 1) % n], axis=1).astype(np.int32)
    m = [np.full((n, 5, 5), v, np.float32) for v in elastic_moduli(2700.0, 3000.0, 1732.0)]
    none = np.zeros(0, np.int32)
    return Mesh2D(coord=np.concatenate([[[0.0, 0.0]], ring, outer]), knods=knods, kappa=m[0],
                  mu=m[1], rho=m[2], abs_ispec=none, abs_type=none)


def test_point_of_many_tiles(oracle_lib):
    """The table of a chain holds four tiles to a point: a mesh with a vertex of
    six keeps the two launches, against the oracle.  Bound: twice the FP32 floor
    (oracle FP32 against FP64), at least 1e-5."""
    print("fan of six elements, one to a tile", flush=True)
    src = Sources2D.ricker(np.array([31.0]), np.array([9.0]), f0=40.0, factor=1e10, angle=20.0)
    rec = Receivers2D(x=np.array([-25.0, 0.0, 12.0]), z=np.array([11.0, 0.0, -30.0]))
    cfg = Config2D("fan", _fan(), src, rec, 5e-4, 200, seismo_types=DVA)
    got, launches = _run(cfg, DVA, 1, {"tile_elems": 1}, 4, (cfg.nstep,))
    assert launches == [3 * cfg.nstep + 2]
    ref = [oracle_lib.Oracle2D(cfg.mesh, src, rec, cfg.dt, cfg.nstep, precision=p).run(types=DVA)
           for p in (4, 8)]
    for k in range(3):
        bound = max(1e-5, 2.0 * rel_l2(ref[0][:, k], ref[1][:, k]))
        assert rel_l2(got[0][:, k], ref[0][:, k]) <= bound


def test_launch_count_of_other_contexts():
    print("kernel launches are counted for 2D elastic contexts only", flush=True)
    cfg = acoustic_box(nx=5, nz=4, nstep=3)
    ctx = Context(cfg.mesh, cfg.sources, cfg.receivers, cfg.dt, cfg.nstep)
    n = ctypes.c_int()
    assert ctx.lib.smx_last_run_kernels(ctx.h, ctypes.byref(n)) == _lib.SMX_ERR_STATE
    assert ctx.lib.smx_last_run_kernels(None, ctypes.byref(n)) == _lib.SMX_ERR_ARG
    assert ctx.lib.smx_last_run_kernels(ctx.h, None) == _lib.SMX_ERR_ARG
    ctx.close()
