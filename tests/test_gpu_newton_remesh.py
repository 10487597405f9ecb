"""The Newton step of one handle on a small mesh, then on a larger one: its
workspace belongs to the mesh."""
import numpy as np
import pytest

from plugin_navierstokes_amd import meshes as M

pytestmark = pytest.mark.gpu


def _step(disc, mesh, cuda):
    import torch

    disc.set_mesh(mesh)
    rows = np.arange(mesh.nv, dtype=np.int64)[:8] * 3
    disc.set_dirichlet(rows)
    u = torch.from_numpy(M.random_state(mesh, 3)).to(cuda)
    g = u.view(-1)[torch.from_numpy(rows).to(cuda)].clone()
    disc.newton_step(u, g=g, krylov=6, jprec=64)
    return u.cpu().numpy()


def _disc():
    from plugin_navierstokes_amd import NavierStokesFV1

    disc = NavierStokesFV1("u,v,p", "Inner")
    disc.set_upwind("full")
    disc.set_stabilization("fields", "raw")
    disc.set_kinematic_viscosity(0.05)
    return disc


def test_workspace_follows_the_mesh(cuda):
    a, b = M.cavity_2d(4, M.QUAD, 0.1, 1), M.cavity_2d(24, M.QUAD, 0.1, 1)
    disc = _disc()
    small = _step(disc, a, cuda)
    large = _step(disc, b, cuda)
    assert np.array_equal(large, _step(_disc(), b, cuda))
    assert np.array_equal(small, _step(disc, a, cuda))
