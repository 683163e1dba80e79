"""Geometry of 4-node elements re-formed in the step kernels against the
stored terms: a batch that also holds a 9-node shot reads every shot's stored
terms, a context of the 4-node shot alone forms them from the control nodes.

Both take the same FP32 operations except the quotients, which the kernels
round from one correction of a shared reciprocal: they differ only where a
quotient lies within 2^-46 of a rounding tie, so results are compared for
equality.
"""

import ctypes
import dataclasses

import numpy as np
import pytest

from specfempp_amd import _lib
from specfempp_amd.solver import Context, simulate, simulate_batch
from tests._cases import acoustic_box, adjoint_small, coupled_box, nine_node_shot, warped

pytestmark = pytest.mark.gpu

TYPES = ("displacement", "velocity", "acceleration")


def _shifted(cfg, dx):
    m, s, r = cfg.mesh, cfg.sources, cfg.receivers
    return dataclasses.replace(
        cfg, mesh=dataclasses.replace(m, coord=m.coord + np.array([dx, 0.0])),
        sources=dataclasses.replace(s, x=s.x + dx), receivers=dataclasses.replace(r, x=r.x + dx))


def _shot(kind):
    # 11 x 7 elements: a full tile and one of 13; 4 x 3: part of one tile
    n = (4, 3) if kind == "regular" else (11, 7)
    cfg = dataclasses.replace(adjoint_small(nx=n[0], nz=n[1], nstep=60), seismo_types=TYPES)
    return {"regular": lambda: cfg, "warped": lambda: warped(cfg),
            "far": lambda: _shifted(warped(cfg), 36864.0)}[kind]()


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("kind", ["regular", "warped", "far"])
def test_nodes_equal_stored_terms(kind, precision):
    cfg = _shot(kind)
    print(f"geometry: {kind} 4-node shot, precision {precision}", flush=True)
    alone, _ = simulate(cfg, precision=precision)
    both, _ = simulate_batch([cfg, nine_node_shot(cfg)], precision=precision)
    assert np.isfinite(alone).all() and np.abs(alone).max() > 0
    assert np.array_equal(both[0], alone)


def test_gradient_of_nodes_equals_stored_terms():
    cfg = _shot("warped")
    print("geometry: gradient of a warped 4-node shot", flush=True)
    out = []
    for shots in ([cfg], [cfg, nine_node_shot(cfg)]):
        ctx = Context.batch(shots)
        ctx.initialize()
        ctx.run_forward_checkpointed(every=25)
        rng = np.random.default_rng(1)
        g = np.zeros((ctx.nstep, ctx.nrec, 2), np.float32)
        n = len(cfg.receivers.x)
        g[:, :n] = 1e-9 * rng.standard_normal((ctx.nstep, n, 2))
        ctx.run_adjoint(g)
        out.append(ctx.gradient()[:, :cfg.mesh.nspec])
        ctx.close()
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])


def _report(cfg, precision=4, **options):
    ctx = Context(cfg.mesh, cfg.sources, cfg.receivers, cfg.dt, cfg.nstep, precision=precision,
                  seismo_types=cfg.seismo_types, options=options)
    gm, mis = ctypes.c_int(), ctypes.c_longlong()
    _lib.check(ctx.lib.smx_ctx_geometry(ctx.h, ctypes.byref(gm), ctypes.byref(mis)))
    ctx.close()
    return gm.value, mis.value


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("kind", ["regular", "warped", "far"])
def test_check_of_formed_terms(kind, precision):
    """The terms the steps form are the stored ones at every point (at the
    centre in the affine elements of the regular mesh)."""
    print(f"geometry check: {kind}, precision {precision}", flush=True)
    assert _report(_shot(kind), precision, geometry_from_nodes=True) == (2, 0)


def test_geometry_source_reported():
    """What the steps read, with and without the check."""
    print("geometry source of 4- and 9-node, acoustic and coupled contexts", flush=True)
    cfg = _shot("warped")
    assert _report(cfg) == (2, 0)
    for check in (False, True):
        assert _report(nine_node_shot(cfg), geometry_from_nodes=check) == (0, 0)
    assert _report(acoustic_box(nx=9, nz=7, nstep=4)) == (2, 0)
    assert _report(coupled_box(nx=9, nz=8, nstep=4)) == (2, 0)
