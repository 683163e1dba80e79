"""Forward steps of one launch each against steps of two launches: a context
that also records pressure keeps the two.  The sums and updates of a point are
the same operations in the same order, so fields and seismograms are equal.

Cases: calls of one to a few steps and around one and two replayed pieces of
odd and even length; tiles of 64, 16 and 3 elements (shared points of two to
four tiles); sampled every step and every third; 4- and 9-node elements."""

import dataclasses

import numpy as np
import pytest

from specfempp_amd.mesh import box_mesh
from specfempp_amd.solver import Context
from tests._cases import adjoint_small, warped

pytestmark = pytest.mark.gpu


def _run(cfg, types, nsbs, options, precision, calls):
    ctx = Context(cfg.mesh, cfg.sources, cfg.receivers, cfg.dt, cfg.nstep, nsbs=nsbs,
                  seismo_types=types, precision=precision, options=options)
    ctx.initialize()
    at = 0
    for n in calls:
        ctx.run_forward(at, n)
        at += n
    ctx.synchronize()
    out = [ctx.seismograms()] + [ctx.get_field(f) for f in ("u", "v", "a")]
    ctx.close()
    return out


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
    one = _run(cfg, ("displacement", "velocity", "acceleration"), nsbs, opt, precision, calls)
    two = _run(cfg, ("pressure", "displacement", "velocity", "acceleration"), nsbs, opt,
               precision, calls)
    only = _run(cfg, ("displacement",), nsbs, opt, precision, calls)
    assert np.abs(one[0]).max() > 0 and np.isfinite(one[0]).all()
    assert np.array_equal(one[0], two[0][:, 1:])
    assert np.array_equal(only[0][:, 0], one[0][:, 0])
    for a, b, c in zip(one[1:], two[1:], only[1:]):
        assert np.array_equal(a, b) and np.array_equal(c, b)
