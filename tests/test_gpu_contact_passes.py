"""Gauss-Seidel contact passes at the edges of what a workgroup holds: no
contact, one, a wave's, a workgroup's 256 and more, in one instance and in a batch
whose instances differ, over several iterations (the later ones start from what
the first gathered), against the oracle step by step from a shared state.

A step's motions are FP32 values of some 1e-4 m on coordinates of 0.1 m and the
contact arithmetic is FP64 on both sides, so the difference is the elastic FP32
rounding, some 1e-9 relative: 1e-6 is far above it and far below a contact's
effect (1e-4 m: 1e-3 relative)."""
import numpy as np
import pytest

import orc
import workloads as W
import xpbd_amd as X
from helpers import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-6


def _contacts(mesh, n, seed):
    """Contacts that push n random free faces out along their normals by 0.1 mm."""
    rng = np.random.default_rng(seed)
    free = np.flatnonzero((mesh.pinned[mesh.faces] == 0).all(1))
    assert n <= len(free)
    face = rng.permutation(free)[:n].astype(np.int32)
    p = mesh.x0[mesh.faces[face]]
    nrm = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1, keepdims=True), 1e-300)
    b = rng.dirichlet(np.ones(3), n) if n else np.empty((0, 3))
    return face, (b[:, :, None] * p).sum(1) + 1e-4 * nrm, nrm, b


def _oracle(mesh, iters, order=None, rank=None):
    o = orc.Sim(mesh, dt=1e-3, iters=iters, mode="gs")
    o.set_order(order)
    o.set_contact_order(rank)
    return o


@pytest.mark.parametrize("variant", ["auto", "quad", "cluster"])
@pytest.mark.parametrize("count", [0, 1, 64, 65, 255, 256, 257, 500])
def test_counts(count, variant):
    mesh = W.grid_object(11, 9, 10, 0.01, noise=0.02, seed=5, faces=True)
    for iters in (1, 4):
        gpu = X.Solver(mesh, dt=1e-3, iters=iters, solver="gs", variant=variant, collision_every=0)
        o = _oracle(mesh, iters, gpu.tet_order(), gpu.face_rank())
        c = _contacts(mesh, count, seed=count + 1)
        gpu.set_contacts(*c)
        o.set_contacts(*c)
        for _ in range(2):
            o.set_state(gpu.positions(), gpu.velocities())
            gpu.step(1)
            o.step(1, detect=False)
            err = rel_err(gpu.positions(), o.x())
            assert err <= TOL, (iters, err)
    print(f"{variant} {count} contacts: {err:.2e}")


@pytest.mark.parametrize("variant", ["auto", "quad"])
def test_instances_with_different_counts(variant):
    counts = [300, 0, 1, 70, 256]
    meshes = [W.grid_object(8 + i % 2, 9, 10, 0.01, noise=0.02, seed=i, faces=True) for i in range(len(counts))]
    gpu = X.Solver(meshes, dt=1e-3, iters=3, solver="gs", variant=variant, collision_every=0)
    v, t, f = (np.cumsum([0] + [len(a) for a in arrays])
               for arrays in ([m.x0 for m in meshes], [m.tets for m in meshes], [m.faces for m in meshes]))
    each = [_contacts(m, n, seed=n) for m, n in zip(meshes, counts)]
    gpu.set_contacts(np.concatenate([c[0] + o for c, o in zip(each, f)]).astype(np.int32),
                     *(np.concatenate([c[k] for c in each]) for k in (1, 2, 3)))
    order, rank = gpu.tet_order(), gpu.face_rank()
    oracles = []
    for i, (m, c) in enumerate(zip(meshes, each)):
        mine = order[(order >= t[i]) & (order < t[i + 1])] - t[i]
        oracles.append(_oracle(m, 3, mine, np.argsort(np.argsort(rank[f[i]:f[i + 1]])).astype(np.int32)))
        oracles[-1].set_contacts(*c)
    for _ in range(3):
        x, u = gpu.positions(), gpu.velocities()
        gpu.step(1)
        y = gpu.positions()
        for i, o in enumerate(oracles):
            o.set_state(x[v[i]:v[i + 1]], u[v[i]:v[i + 1]])
            o.step(1, detect=False)
            assert rel_err(y[v[i]:v[i + 1]], o.x()) <= TOL, i
