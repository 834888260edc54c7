"""The fused-colour Gauss-Seidel launches (the untuned default on most meshes)
against the colour launches of the quad kernel (variant "quad"): the same elements
in the same order with the same operations, with four lanes a cluster or one, so
the same bits."""
import gzip
import os

import numpy as np
import pytest

import workloads as W
import xpbd_amd as X
from test_gpu_parity import _eight_element_cells, _single_tet

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "msh")
TILE = 4000   # XPBD_QUAD_TILE


def _grid(*dims, seed=3, faces=False):
    return W.grid_object(*dims, 0.01, E=5e3, nu=0.45, noise=0.02, seed=seed, faces=faces)


def _neuroma(tmp_path):
    p = tmp_path / "neuroma.msh"
    p.write_bytes(gzip.open(os.path.join(GOLDEN, "neuroma_segmentation_decimated_2000.msh.gz")).read())
    x, t, _ = X.read_msh(str(p))
    x = (x - x.min(0)) * (0.5 / (x - x.min(0)).max())
    n = len(t)
    return X.Mesh(x0=x, tets=t, E=np.full(n, 6e4), nu=np.full(n, 0.45), rho=np.full(n, 1000.0),
                  pinned=(x[:, 2] < 0.02).astype(np.uint8), v0=np.random.default_rng(1).normal(0, 0.005, x.shape))


MESHES = {
    "single tet": lambda t: _single_tet(),
    "one cell": lambda t: _grid(1, 1, 1),
    "whole object a tile": lambda t: _grid(8, 8, 8),
    "tiles": lambda t: _grid(9, 9, 9),
    "ragged": lambda t: _grid(13, 9, 7),
    "thin": lambda t: _grid(60, 3, 11),
    "two colours a launch": lambda t: _grid(31, 25, 29),
    "8-element clusters": lambda t: _eight_element_cells(3, 4, 5, seed=23),
    "8-element tiles": lambda t: _eight_element_cells(12, 11, 13, seed=23),
    "51 colours": _neuroma,
    "whole batch": lambda t: [_grid(4, 5, 3, seed=1), _grid(6, 6, 6, seed=2), _grid(2, 2, 9, seed=4)],
    "uneven batch": lambda t: [_grid(5, 5, 5, seed=1), _grid(14, 11, 12, seed=2), _grid(3, 9, 4, seed=4)],
}


def _pair(mesh, **kw):
    """The same handle with the fused-colour launches and with the colour launches."""
    a, b = X.Solver(mesh, solver="gs", **kw), X.Solver(mesh, solver="gs", variant="quad", **kw)
    assert a.launch_config() == ("quad", TILE, True)
    assert b.launch_config()[1] != TILE
    return a, b


def _same(a, b):
    for f in ("positions", "velocities", "lambdas"):
        np.testing.assert_array_equal(getattr(a, f)(), getattr(b, f)(), err_msg=f)


@pytest.mark.parametrize("iters", [1, 4])
@pytest.mark.parametrize("kind", list(MESHES))
def test_launches_give_the_quad_kernels_bits(kind, iters, tmp_path):
    a, b = _pair(MESHES[kind](tmp_path), iters=iters, collision_every=0)
    for n in (1, 4):
        a.step(n)
        b.step(n)
        _same(a, b)
    a.set_kernel_timing(True)   # launched one by one
    a.step(2)
    b.step(2)
    _same(a, b)
    assert a.kernel_stats()[1] == 2 * iters


@pytest.mark.parametrize("dims", [(8, 8, 8), (11, 9, 10)])
def test_contacts_attachments_and_subset_solves_between(dims):
    """A sphere pressing on the top; three vertices grasped for some steps (the
    handle then runs the colour launches) and released; a subset solve between
    steps; a change of the iteration count."""
    mesh = _grid(*dims, faces=True)
    a, b = _pair(mesh, iters=5, collision_every=1)
    top = mesh.x0.max(0)
    for s in (a, b):
        s.set_sdf(X.SDF_SPHERE, (0.55 * top[0], 0.45 * top[1], top[2] + 0.028), params=(0.03, 0, 0))
    grasp = np.argsort(-mesh.x0[:, 2])[:3]
    for n in range(4):
        for s in (a, b):
            if n == 1:
                s.set_attachments(grasp, mesh.x0[grasp] + [0, 0, 0.002])
            if n == 2:
                s.set_attachments([], np.empty((0, 3)))
                s.solve_elements(np.arange(0, mesh.nt, 7), num_iter=2, initialize=True)
            if n == 3:
                s.set_iterations(3)
            s.step(3)
        _same(a, b)
    assert len(a.contacts()[0]) > 0


@pytest.mark.parametrize("start", ["positions", "multipliers"])
@pytest.mark.parametrize("dims", [(6, 6, 6), (12, 10, 9)])
def test_warm_started_multipliers(dims, start):
    """Learned steps keep the multipliers that their start sets."""
    mesh = _grid(*dims)
    net = X.Network()
    net.load(os.path.join(os.path.dirname(X.__file__), "weights", "warmstart.bin"))
    a, b = _pair(mesh, iters=8, collision_every=0)
    for s in (a, b):
        s.attach(net)
        s.set_learned_start(start)
    for _ in range(4):
        ra, rb = a.step_learned(3), b.step_learned(3)
        assert ra == rb
        _same(a, b)


# more than 65 clusters of a colour for each of 256 units: one lane a cluster, 3 colours a launch, then 2
LANE = {
    "cube": lambda: _grid(52, 52, 52),
    "ragged": lambda: _grid(91, 43, 37),
    "two colours": lambda: _grid(61, 59, 60),
    "three million elements": lambda: _grid(81, 79, 80),
    "8-element clusters": lambda: _eight_element_cells(52, 53, 51, seed=23),
}


@pytest.mark.parametrize("kind", list(LANE))
def test_one_lane_gives_the_quad_kernels_bits(kind):
    mesh = LANE[kind]()
    assert mesh.nt > 65 * 256 * 8 * 6
    a, b = _pair(mesh, iters=3, collision_every=0)
    for n in (1, 4):
        a.step(n)
        b.step(n)
        _same(a, b)
    net = X.Network()
    net.load(os.path.join(os.path.dirname(X.__file__), "weights", "warmstart.bin"))
    for s in (a, b):
        s.attach(net)
        s.set_learned_start("multipliers")
    assert a.step_learned(2) == b.step_learned(2)
    _same(a, b)
