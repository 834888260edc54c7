"""Batches of many small objects and a large one, whose small objects share tiles,
against the colour launches (variant "quad"): the same bits, with contacts and
without, and every object where it belongs."""
import numpy as np
import pytest

import workloads as W
import xpbd_amd as X

pytestmark = pytest.mark.gpu


def _batch(sizes, faces):
    return [W.grid_object(*d, 0.01, E=5e3, nu=0.45, noise=0.02, seed=i, faces=faces) for i, d in enumerate(sizes)]


BATCHES = {
    "cells": [(1, 1, 1)] * 700 + [(8, 8, 8)] + [(1, 1, 1)] * 300,
    "small ones of three sizes": ([(1, 2, 1), (2, 2, 2), (3, 1, 2)] * 120) + [(7, 8, 9)],
}


@pytest.mark.parametrize("faces", [False, True], ids=["free", "contacts"])
@pytest.mark.parametrize("kind", list(BATCHES))
def test_small_objects_share_tiles(kind, faces):
    meshes = _batch(BATCHES[kind], faces)
    a, b = (X.Solver(meshes, solver="gs", iters=3, collision_every=1, **v) for v in ({}, {"variant": "quad"}))
    assert a.launch_config() == ("quad", 4000, True)
    if faces:
        for s in (a, b):
            s.set_sdf(X.SDF_BOX, (0.0, 0.0, 0.03), params=(0.05, 0.05, 0.05))
    for n in (1, 4):
        a.step(n)
        b.step(n)
        for f in ("positions", "velocities", "lambdas"):
            np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f)
    assert not faces or len(a.contacts()[0]) > 0
    big = max(range(len(meshes)), key=lambda i: meshes[i].nv)
    x, at = a.positions(), np.cumsum([0] + [m.nv for m in meshes])
    for i in (0, big, len(meshes) - 1):
        np.testing.assert_array_equal(a.instance_positions(i), x[at[i]:at[i + 1]])
