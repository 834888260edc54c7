"""Contact detection and its compaction against the oracle on the same state, at
the edges of the compaction's blocks of 256 faces and for colliders on which the
search's vertex choice ties or is close.

Both sides run the same FP64 operations without contraction from the same
positions, so the sets are equal and the values agree to round-off: 2^-53 of a
metre over the search's convex steps, over a distance of some 1e-4 m in a normal."""
import numpy as np
import pytest

import orc
import workloads as W
import xpbd_amd as X

pytestmark = pytest.mark.gpu
TOL = 1e-11

# cells -> faces: below a block, one block, one over, some, more blocks than a workgroup's threads
GRIDS = {(4, 4, 4): 192, (4, 4, 6): 256, (1, 1, 32): 260, (9, 7, 5): 572, (150, 150, 1): 91200}


def _colliders(ext):
    h = 0.01
    mid = [ext[0] / 2, ext[1] / 2, ext[2]]
    s2 = np.sqrt(0.5)
    return {
        "sphere": (X.SDF_SPHERE, (0.43 * ext[0], 0.57 * ext[1], ext[2] + 0.019), (0, 0, 0, 1), (0.02, 0, 0)),
        "sphere over a vertex": (X.SDF_SPHERE, (h, h, ext[2] + 0.019), (0, 0, 0, 1), (0.02, 0, 0)),
        "sphere on a face": (X.SDF_SPHERE, (h * 1.5, h * 0.5, ext[2]), (0, 0, 0, 1), (0.004, 0, 0)),
        "box": (X.SDF_BOX, mid, (0.1, -0.3, 0.2, np.sqrt(1 - 0.14)), (0.02, 0.015, 0.01)),
        "aligned box": (X.SDF_BOX, mid, (0, 0, 0, 1), (0.02, 0.02, 0.01)),
        "turned box": (X.SDF_BOX, mid, (0, 0, s2, s2), (0.03, 0.01, 0.02)),
        "plate": (X.SDF_BOX, mid, (0.6, 0, 0, 0.8), (0.05, 0.02, 0.0)),
    }


@pytest.mark.parametrize("moved", [False, True], ids=["at rest", "moved"])
@pytest.mark.parametrize("dims", list(GRIDS), ids=lambda d: "x".join(map(str, d)))
def test_detection_is_the_oracles(dims, moved):
    mesh = W.grid_object(*dims, 0.01, noise=0.05 if moved else 0.0, seed=7, faces=True)
    assert len(mesh.faces) == GRIDS[dims]
    gpu = X.Solver(mesh, dt=1e-3, iters=2, solver="gs", collision_every=1)
    o = orc.Sim(mesh, dt=1e-3, iters=2, mode="gs")
    if moved:
        gpu.step(2)
    found = 0
    for name, (kind, pos, quat, prm) in _colliders(mesh.x0.max(0)).items():
        gpu.set_sdf(kind, pos, quat, prm)
        gpu.detect()
        face, cp, cn, cb = gpu.contacts()
        o.set_state(gpu.positions(), gpu.velocities())
        o.set_sdf(kind, pos, quat, prm)
        o.detect()
        fo, po, no, bo = o.contacts()
        a, b = np.argsort(fo), np.argsort(face)
        np.testing.assert_array_equal(np.asarray(fo)[a], np.asarray(face)[b], err_msg=name)
        found += len(face)
        if len(face):
            dev = max(np.abs(po[a] - cp[b]).max(), np.abs(no[a] - cn[b]).max(), np.abs(bo[a] - cb[b]).max())
            print(f"{dims} {name}: {len(face)} contacts, largest deviation {dev:.2e}")
            assert dev <= TOL
        # the compacted list is complete and without repetition after another detection
        gpu.detect()
        np.testing.assert_array_equal(np.sort(gpu.contacts()[0]), np.sort(face))
    assert found > 0
