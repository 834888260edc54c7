"""The vertex-tile Jacobi launches (the untuned default of deterministic Jacobi on
most meshes) against the patch launches (variant "patch"): the same FP32
corrections, summed in the same groups and order, so the same bits, with the fused
iteration (up to 256 patches) and the separate launches (more)."""
import gzip
import os

import numpy as np
import pytest

import workloads as W
import xpbd_amd as X
from test_gpu_parity import _eight_element_cells, _single_tet

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "msh")
TILE = 2   # XPBD_PATCH_TILE


def _grid(*dims, seed=3, faces=False):
    return W.grid_object(*dims, 0.01, E=1e3, nu=0.45, noise=0.02, seed=seed, faces=faces)


def _neuroma(tmp_path):
    p = tmp_path / "neuroma.msh"
    p.write_bytes(gzip.open(os.path.join(GOLDEN, "neuroma_segmentation_decimated_2000.msh.gz")).read())
    x, t, _ = X.read_msh(str(p))
    x = (x - x.min(0)) * (0.5 / (x - x.min(0)).max())
    n = len(t)
    return X.Mesh(x0=x, tets=t, E=np.full(n, 1e3), nu=np.full(n, 0.4), rho=np.full(n, 1000.0),
                  pinned=(x[:, 2] < 0.02).astype(np.uint8), v0=np.random.default_rng(1).normal(0, 0.001, x.shape))


MESHES = {
    "single tet": lambda t: _single_tet(),
    "one cell": lambda t: _grid(1, 1, 1),
    "an object a tile, one element a thread": lambda t: _grid(5, 6, 5),
    "just more": lambda t: _grid(6, 6, 5),
    "tiles of 12": lambda t: _grid(9, 9, 9),
    "ragged": lambda t: _grid(13, 9, 7),
    "thin": lambda t: _grid(60, 3, 11),
    "several elements a thread": lambda t: _grid(41, 42, 40),
    "8-element cells": lambda t: _eight_element_cells(12, 11, 13, seed=23),
    "unstructured": _neuroma,
    "batch of small objects": lambda t: [_grid(4, 5, 3, seed=1), _grid(5, 5, 6, seed=2), _grid(2, 2, 9, seed=4)],
    "uneven batch": lambda t: [_grid(5, 5, 5, seed=1), _grid(14, 11, 12, seed=2), _grid(3, 9, 4, seed=4)],
}


def _pair(mesh, **kw):
    a, b = (X.Solver(mesh, solver="jacobi", g=1.0, **kw, **v) for v in ({}, {"variant": "patch"}))
    assert a.launch_config() == ("patch", TILE, True)
    assert b.launch_config()[1] != TILE
    return a, b


def _same(a, b, what=""):
    for f in ("positions", "velocities", "lambdas"):
        np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f"{what} {f}")


@pytest.mark.parametrize("iters", [1, 10])
@pytest.mark.parametrize("kind", list(MESHES))
def test_tiles_follow_the_patches(kind, iters, tmp_path):
    mesh = MESHES[kind](tmp_path)
    a, b = _pair(mesh, iters=iters, collision_every=0)
    for n in (1, 4):
        a.step(n)
        b.step(n)
        _same(a, b, kind)
    c = X.Solver(mesh, solver="jacobi", g=1.0, iters=iters, collision_every=0)
    c.step(5)
    _same(a, c, kind)   # reproducible
    c.set_kernel_timing(True)   # launched one by one
    a.step(1)
    c.step(1)
    np.testing.assert_array_equal(a.positions(), c.positions())
    assert c.kernel_stats()[1] == iters


@pytest.mark.parametrize("dims", [(5, 5, 5), (11, 9, 10), (31, 30, 29)])
def test_contacts_attachments_and_subset_solves_between(dims):
    mesh = _grid(*dims, faces=True)
    a, b = _pair(mesh, iters=5, collision_every=1)
    top = mesh.x0.max(0)
    for s in (a, b):
        s.set_sdf(X.SDF_SPHERE, (0.55 * top[0], 0.45 * top[1], top[2] + 0.028), params=(0.03, 0, 0))
        s.detect()
        assert len(s.contacts()[0]) > 0
    grasp = np.argsort(-mesh.x0[:, 2])[:3]
    for n in range(4):
        for s in (a, b):
            if n == 1:
                s.set_attachments(grasp, mesh.x0[grasp] + [0, 0, 0.0005])
            if n == 2:
                s.set_attachments([], np.empty((0, 3)))
                s.solve_elements(np.arange(0, mesh.nt, 7), num_iter=2, initialize=True)
            if n == 3:
                s.set_iterations(3)
            s.step(2)
        _same(a, b, f"{dims} phase {n}")
        np.testing.assert_array_equal(np.sort(a.contacts()[0]), np.sort(b.contacts()[0]))


@pytest.mark.parametrize("start", ["positions", "multipliers"])
@pytest.mark.parametrize("dims", [(5, 5, 5), (12, 10, 9)])
def test_warm_started_multipliers(dims, start):
    mesh = _grid(*dims)
    net = X.Network()
    net.load(os.path.join(os.path.dirname(X.__file__), "weights", "warmstart.bin"))
    a, b = _pair(mesh, iters=8, collision_every=0)
    for s in (a, b):
        s.attach(net)
        s.set_learned_start(start)
    for _ in range(3):
        assert a.step_learned(3) == b.step_learned(3)
        _same(a, b, start)
