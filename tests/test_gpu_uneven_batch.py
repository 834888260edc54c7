"""Batches of more objects than compute units, whose small objects share tiles, against
the colour launches (variant "quad") and the patch launches: the same bits, with
contacts and without, and every object where it belongs."""
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
    "cells alone": [(1, 1, 1)] * 3001,
    "alike": [(3, 3, 3)] * 1100,
    "no two share": [(5, 5, 5)] * 300,
}


@pytest.mark.parametrize("faces", [False, True], ids=["free", "contacts"])
@pytest.mark.parametrize("kind", list(BATCHES))
@pytest.mark.parametrize("solver,variant,tile", [("gs", "quad", 4000), ("jacobi", "patch", 2)])
def test_small_objects_share_tiles(solver, variant, tile, kind, faces):
    meshes = _batch(BATCHES[kind], faces)
    a, b = (X.Solver(meshes, solver=solver, g=1.0, iters=3, collision_every=1, **v) for v in ({}, {"variant": variant}))
    assert a.launch_config() == (variant, tile, True) and b.launch_config()[1] != tile
    if faces:
        for s in (a, b):
            s.set_sdf(X.SDF_BOX, (0.0, 0.0, 0.03), params=(0.05, 0.05, 0.05))
            s.detect()
            assert len(s.contacts()[0]) > 0
    for n in (1, 4):
        a.step(n)
        b.step(n)
        for f in ("positions", "velocities", "lambdas"):
            np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f)
    big = max(range(len(meshes)), key=lambda i: meshes[i].nv)
    x, at = a.positions(), np.cumsum([0] + [m.nv for m in meshes])
    for i in (0, big, len(meshes) - 1):
        np.testing.assert_array_equal(a.instance_positions(i), x[at[i]:at[i + 1]])
