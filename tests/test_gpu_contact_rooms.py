"""Gauss-Seidel contact passes of batches whose objects' rooms for contacts differ (many
small objects and large ones), over several iterations, the later of which start from
what the first left in the rooms: objects without faces, with one contact, with all
faces in contact, and with a workgroup's 256 contacts and more, against the oracle.

Tolerance as for batches of like objects: the elastic FP32 rounding of a step's motions,
some 1e-9 relative, is far below 1e-6, a contact's effect (1e-4 m) far above."""
import dataclasses

import numpy as np
import pytest

import workloads as W
import xpbd_amd as X
from helpers import rel_err
from test_gpu_contact_passes import TOL, _contacts, _oracle

pytestmark = pytest.mark.gpu

# (cells, contacts) of the objects that are checked, among many small ones
CHECKED = {0: ((1, 1, 1), 2), 1: ((1, 1, 1), 0), 7: ((2, 1, 1), 1), 40: ((8, 9, 10), 256), 41: ((1, 1, 1), None),
           90: ((9, 9, 10), 300), 120: ((1, 2, 1), 3), 199: ((2, 2, 2), 12)}


@pytest.mark.parametrize("variant", ["auto", "quad"])
def test_rooms_of_their_own(variant):
    meshes, each = [], []
    for i in range(200):
        dims, n = CHECKED.get(i, ((1, 1, 1), 1))
        m = W.grid_object(*dims, 0.01, noise=0.02, seed=i, faces=n is not None)
        if n is not None:   # free bases: all faces of the small ones may be in contact
            m = dataclasses.replace(m, pinned=np.zeros_like(m.pinned))
        meshes.append(m)
        each.append(_contacts(m, n, seed=i) if n is not None else None)
    gpu = X.Solver(meshes, dt=1e-3, iters=3, solver="gs", variant=variant, collision_every=0)
    nf = [0 if m.faces is None else len(m.faces) for m in meshes]
    v, t, f = (np.cumsum([0] + n) for n in ([m.nv for m in meshes], [len(m.tets) for m in meshes], nf))
    given = [(i, c) for i, c in enumerate(each) if c is not None]
    gpu.set_contacts(np.concatenate([c[0] + f[i] for i, c in given]).astype(np.int32),
                     *(np.concatenate([c[k] for _, c in given]) for k in (1, 2, 3)))
    order, rank = gpu.tet_order(), gpu.face_rank()
    oracles = {}
    for i in CHECKED:
        mine = order[(order >= t[i]) & (order < t[i + 1])] - t[i]
        oracles[i] = _oracle(meshes[i], 3, mine, np.argsort(np.argsort(rank[f[i]:f[i + 1]])).astype(np.int32))
        if each[i] is not None:
            oracles[i].set_contacts(*each[i])
    for _ in range(3):
        x, u = gpu.positions(), gpu.velocities()
        gpu.step(1)
        y = gpu.positions()
        for i, o in oracles.items():
            o.set_state(x[v[i]:v[i + 1]], u[v[i]:v[i + 1]])
            o.step(1, detect=False)
            assert rel_err(y[v[i]:v[i + 1]], o.x()) <= TOL, i
