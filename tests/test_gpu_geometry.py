"""Geometry of 4-node elements re-formed in the step kernels against the
stored terms: a batch that also holds a 9-node shot reads every shot's stored
terms, a context of the 4-node shot alone forms them from the control nodes.

Both take the same FP32 operations except the quotients, which the kernels
round from one correction of a shared reciprocal: they differ only where a
quotient lies within 2^-46 of a rounding tie, so results are compared for
equality.
"""

import dataclasses

import numpy as np
import pytest

from specfempp_amd.mesh import box_mesh
from specfempp_amd.solver import Context, simulate, simulate_batch
from tests._cases import adjoint_small, warped

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


def _nine(nstep):
    cfg = dataclasses.replace(adjoint_small(nx=5, nz=4, nstep=nstep), seismo_types=TYPES)
    m = box_mesh(0.0, 250.0, 0.0, 200.0, 5, 4, ngnod=9, absorbing=("bottom", "right", "left"))
    return warped(dataclasses.replace(cfg, mesh=dataclasses.replace(
        m, kappa=cfg.mesh.kappa, mu=cfg.mesh.mu, rho=cfg.mesh.rho)))


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("kind", ["regular", "warped", "far"])
def test_nodes_equal_stored_terms(kind, precision):
    cfg = _shot(kind)
    print(f"geometry: {kind} 4-node shot, precision {precision}", flush=True)
    alone, _ = simulate(cfg, precision=precision)
    both, _ = simulate_batch([cfg, _nine(cfg.nstep)], precision=precision)
    assert np.isfinite(alone).all() and np.abs(alone).max() > 0
    assert np.array_equal(both[0], alone)


def test_gradient_of_nodes_equals_stored_terms():
    cfg = _shot("warped")
    print("geometry: gradient of a warped 4-node shot", flush=True)
    out = []
    for shots in ([cfg], [cfg, _nine(cfg.nstep)]):
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
