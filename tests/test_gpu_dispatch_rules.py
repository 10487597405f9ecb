"""The default launch at the lines where it changes: the workgroup size of FP64
hexahedra."""
import pytest

from plugin_navierstokes_amd import F64, NavierStokesFV1
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc

pytestmark = pytest.mark.gpu


def _disc(mesh, up):
    disc = NavierStokesFV1("u,v,p" if mesh.dim == 2 else "u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": up, "nu": 0.02})
    disc.set_mesh(mesh)
    return disc


@pytest.mark.parametrize("n", [15, 17])
def test_fp64_hexahedra_any_workgroup(cuda, n):
    import torch

    mesh = M.cavity_3d(n, M.HEX, 0.1, 3)
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    out = []
    for threads in (0, 256, 128, 64):
        disc = _disc(mesh, "lps")
        if threads:
            disc.set_launch(threads, 65536)
        out.append(disc.assemble(u, jprec=F64))
    # the order of every sum is the incidence's, whatever the workgroup holds
    for J, d in out[1:]:
        assert torch.equal(J, out[0][0]) and torch.equal(d, out[0][1])
