"""The state's readers at the edges of the pieces that they read in (20,480 vertices
in FP64, 40,960 in FP32): every reader gives the same numbers, what was set comes
back, instances are cut where they begin, and several threads may read at once."""
import threading

import numpy as np
import pytest

import workloads as W
import xpbd_amd as X

pytestmark = pytest.mark.gpu

# 8 vertices; an FP64 piece less four, one, four more; an FP32 piece; some pieces
GRIDS = [(1, 1, 1), (5118, 1, 1), (127, 15, 9), (5120, 1, 1), (511, 15, 4), (40, 40, 40), (63, 63, 30)]


@pytest.mark.parametrize("dims", GRIDS, ids=lambda d: "x".join(map(str, d)))
def test_readers_agree(dims):
    mesh = W.grid_object(*dims, 0.01, noise=0.02, seed=2)
    s = X.Solver(mesh, iters=1, collision_every=0)
    np.testing.assert_array_equal(s.positions(), mesh.x0)
    free = mesh.pinned == 0
    np.testing.assert_array_equal(s.velocities()[free], mesh.v0[free].astype(np.float32))
    s.step(2)
    x = s.positions()
    np.testing.assert_array_equal(s.positions_f32(), x.astype(np.float32))
    np.testing.assert_array_equal(s.positions(), x)
    v = s.velocities()
    t = X.Solver(mesh, iters=1, collision_every=0)
    t.set_state(x, v)
    # a position is its displacement's two FP32 parts: 2^-48 of it
    assert np.abs(t.positions() - x).max() <= 2.0 ** -48
    np.testing.assert_array_equal(t.velocities(), v)
    got = [None] * 8

    def read(i):
        got[i] = (s.positions, s.velocities, s.positions_f32)[i % 3]()

    threads = [threading.Thread(target=read, args=(i,)) for i in range(len(got))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for i, g in enumerate(got):
        np.testing.assert_array_equal(g, (x, v, x.astype(np.float32))[i % 3])


def test_instances_are_cut_where_they_begin():
    meshes = [W.grid_object(n, 20, 20, 0.01, noise=0.02, seed=n) for n in (3, 60, 1, 47)]
    s = X.Solver(meshes, iters=1, collision_every=0)
    s.step(1)
    x, at = s.positions(), 0
    for i, m in enumerate(meshes):
        np.testing.assert_array_equal(s.instance_positions(i), x[at:at + m.nv])
        at += m.nv


@pytest.mark.parametrize("n", [1, 16383, 16384, 16385])
def test_network_outputs_either_way(n):
    net = X.Network()
    x = np.random.default_rng(0).normal(size=(n, 24)).astype(np.float32)
    y = net.forward(x)
    z = np.concatenate([net.forward(x[i:i + 5000]) for i in range(0, n, 5000)])
    np.testing.assert_array_equal(y, z)
