"""Acoustic seismograms summed in the shared-point pass (displacement and
pressure only) against those of a launch of their own (velocity recorded too):
the same terms summed in the same order, so they are equal.  Tiles of 64 and 3
elements, FP32 and FP64, every step and every third, coupled meshes."""

import dataclasses

import numpy as np
import pytest

from specfempp_amd.solver import simulate
from tests._cases import acoustic_box, coupled_box, warped

pytestmark = pytest.mark.gpu


def _types(cfg, types, **kw):
    return simulate(dataclasses.replace(cfg, seismo_types=types), **kw)[0]


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("tile,nsbs,nstep", [(64, 1, 27), (64, 3, 26), (3, 1, 10), (3, 3, 31)])
def test_shared_pass_sums(tile, nsbs, nstep, precision):
    cfg = dataclasses.replace(warped(acoustic_box(nx=13, nz=10, nstep=nstep, nrec=11)), nsbs=nsbs)
    print(f"acoustic seismograms: tile {tile}, nsbs {nsbs}, precision {precision}", flush=True)
    kw = {"precision": precision, "options": {"tile_elems": tile, "graph_steps": 5}}
    full = _types(cfg, ("displacement", "velocity", "pressure"), **kw)
    assert np.isfinite(full).all() and np.abs(full).max() > 0
    assert np.array_equal(_types(cfg, ("displacement",), **kw)[:, 0], full[:, 0])
    assert np.array_equal(_types(cfg, ("pressure", "displacement"), **kw), full[:, [2, 0]])


def test_coupled_shared_pass_sums():
    cfg = coupled_box(nx=14, nz=12, nstep=60)
    print("coupled seismograms: displacement alone and with velocity", flush=True)
    full = _types(cfg, ("displacement", "velocity"))
    assert np.abs(full[:, 0]).max() > 0
    assert np.array_equal(_types(cfg, ("displacement",))[:, 0], full[:, 0])
