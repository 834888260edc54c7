"""Learned steps of one iteration with the starts that keep multipliers: the tile
launches (the untuned default), whose one launch both starts from the kept
multipliers and writes them back, against the launches without tiles (variants
"quad" and "patch"), the same bits; on plans with four lanes a cluster, with one,
with all colours in one launch, and of Jacobi, whose tiles share elements, and on
plans whose tiles share nothing.  The steps replay a captured graph, with reads of
the state between the replays."""
import os

import numpy as np
import pytest

import workloads as W
import xpbd_amd as X

pytestmark = pytest.mark.gpu

MESHES = [("gs", (6, 6, 6)), ("gs", (12, 10, 9)), ("gs", (31, 25, 29)), ("gs", (60, 40, 1)), ("gs", (52, 52, 52)),
          ("jacobi", (5, 5, 5)), ("jacobi", (12, 10, 9)), ("jacobi", (31, 30, 29))]


@pytest.mark.parametrize("start", ["multipliers", "consistent"])
@pytest.mark.parametrize("solver,dims", MESHES, ids=lambda p: p if isinstance(p, str) else "x".join(map(str, p)))
def test_one_iteration_gives_the_other_launches_bits(solver, dims, start):
    mesh = W.grid_object(*dims, 0.01, E=5e3 if solver == "gs" else 1e3, nu=0.45, noise=0.02, seed=3, faces=True)
    net = X.Network()
    net.load(os.path.join(os.path.dirname(X.__file__), "weights", "warmstart.bin"))
    top = mesh.x0.max(0)
    pair = []
    for v in ({}, {"variant": "quad" if solver == "gs" else "patch"}):
        s = X.Solver(mesh, solver=solver, g=9.81 if solver == "gs" else 1.0, iters=4, collision_every=1, **v)
        s.set_sdf(X.SDF_SPHERE, (0.55 * top[0], 0.45 * top[1], top[2] + 0.028), params=(0.03, 0, 0))
        s.attach(net)
        s.set_learned_start(start)
        pair.append(s)
    a, b = pair
    assert a.launch_config() == (("quad", 4000, True) if solver == "gs" else ("patch", 2, True))
    assert b.launch_config()[1] != a.launch_config()[1]
    for n in (1, 1, 2, 1):   # back to one iteration after two
        assert a.step_learned(n) == b.step_learned(n)
        for f in ("positions", "velocities", "lambdas"):
            np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f)
