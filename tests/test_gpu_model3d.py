"""A new model of a 3D context against a context assembled with it: mass,
moduli, impedances and boundary matrices are the same operations in the same
order, so seismograms, inverse mass and gradients are equal.  Models constant
in every element and models that vary inside them, changed one into the other;
a rejected model changes nothing."""

import dataclasses

import numpy as np
import pytest

from specfempp_amd import _lib
from specfempp_amd.solver3d import Context3D
from tests._cases import adjoint_small3d

pytestmark = pytest.mark.gpu


def _context(cfg, model, precision):
    mesh = dataclasses.replace(cfg.mesh, kappa=model[0], mu=model[1], rho=model[2])
    ctx = Context3D(mesh, cfg.sources, cfg.receivers, cfg.dt, cfg.nstep, precision=precision)
    ctx.initialize()
    return ctx


def _results(ctx):
    rng = np.random.default_rng(4)
    ctx.run_forward_checkpointed(11)
    ctx.synchronize()
    s = ctx.seismograms().copy()
    ctx.run_adjoint(1e-9 * rng.standard_normal((ctx.nstep, ctx.nrec, 3)))
    return s, ctx.get_field("minv"), ctx.gradient()


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 5)])
def test_new_model_equals_fresh_context(n, precision):
    cfg = adjoint_small3d(n=n, nstep=24)
    print(f"3D model change: {n} elements, precision {precision}", flush=True)
    varying = (cfg.mesh.kappa, cfg.mesh.mu, cfg.mesh.rho)
    flat = tuple(np.ascontiguousarray(np.broadcast_to(
        a.reshape(a.shape[0], -1)[:, :1, None, None], a.shape)).astype(np.float32)
        for a in varying)
    scaled = tuple((c * a).astype(np.float32) for c, a in zip((1.03, 0.96, 1.02), varying))
    ctx = _context(cfg, varying, precision)
    for model in (flat, scaled, flat, varying):
        ctx.set_model(*model)
        fresh = _context(cfg, model, precision)
        for a, b in zip(_results(ctx), _results(fresh)):
            assert np.abs(b).max() > 0
            assert np.array_equal(a, b)
        fresh.close()


def test_rejected_model_changes_nothing():
    cfg = adjoint_small3d(n=(3, 2, 2), nstep=24)
    model = (cfg.mesh.kappa, cfg.mesh.mu, cfg.mesh.rho)
    ctx = _context(cfg, model, 4)
    ctx.set_model(*model)
    before = _results(ctx)
    for which, value in ((0, 0.0), (1, -1.0), (2, np.nan)):
        bad = [a.copy() for a in model]
        bad[which][7, 4, 2, 1] = value
        bad[which][9, 0, 0, 0] = value
        with pytest.raises(_lib.SmxError, match="element 7"):
            ctx.set_model(*bad)
    for a, b in zip(before, _results(ctx)):
        assert np.array_equal(a, b)


def test_gradient_memory():
    """A gradient holds the point maps (16 B per element point) and a bounded
    output buffer (25 MB), not what a model change needs; a mesh of more than
    one output piece, against the gradient of a context that made the maps of
    a model change first."""
    import torch
    cfg = adjoint_small3d(n=(32, 24, 22), nstep=32)
    model = (cfg.mesh.kappa, cfg.mesh.mu, cfg.mesh.rho)
    print("3D gradient memory: 32x24x22 elements", flush=True)
    rng = np.random.default_rng(8)
    gsrc = 1e-9 * rng.standard_normal((cfg.nstep, len(cfg.receivers.x), 3))
    grads = []
    for change in (False, True):
        ctx = _context(cfg, model, 4)
        if change:
            ctx.set_model(*model)
        ctx.run_forward_checkpointed(8)
        ctx.run_adjoint(gsrc)
        ctx.synchronize()
        before = torch.cuda.mem_get_info()[0]
        grads.append(ctx.gradient())
        held = before - torch.cuda.mem_get_info()[0]
        # three allocations of 2 MiB granularity beside the sizes
        assert held <= 16 * 125 * cfg.mesh.nspec + 3 * 8 * 125 * 8192 + (8 << 20), held
        ctx.close()
    assert np.abs(grads[0]).max() > 0
    assert np.array_equal(*grads)
