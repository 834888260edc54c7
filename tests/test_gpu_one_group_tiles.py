"""Plans with all colours in one launch whose tiles share clusters (plates and bars, of
four and two colours): the motions change between two arrays from iteration to
iteration, and contacts are applied in whichever holds them.  Odd and even counts of
iterations against the colour launches (variant "quad"), the same bits."""
import numpy as np
import pytest

import workloads as W
import xpbd_amd as X

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("contacts", [False, True], ids=["free", "contacts"])
@pytest.mark.parametrize("iters", [1, 2, 3, 4])
@pytest.mark.parametrize("dims", [(60, 60, 1), (600, 1, 1), (43, 71, 1)], ids=lambda d: "x".join(map(str, d)))
def test_two_arrays_in_turn(dims, iters, contacts):
    mesh = W.grid_object(*dims, 0.01, E=5e3, nu=0.45, noise=0.02, seed=3, pin_axis=0, faces=contacts)
    a, b = (X.Solver(mesh, solver="gs", iters=iters, collision_every=1, **v) for v in ({}, {"variant": "quad"}))
    assert a.launch_config() == ("quad", 4000, True)
    ext = mesh.x0.max(0)
    for s in (a, b):
        if contacts:
            s.set_sdf(X.SDF_SPHERE, (0.55 * ext[0], 0.45 * ext[1], ext[2] + 0.028), params=(0.03, 0, 0))
            s.detect()
            assert len(s.contacts()[0]) > 0
    for n in (1, 3):
        for s in (a, b):
            s.step(n)
        for f in ("positions", "velocities", "lambdas"):
            np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f)
