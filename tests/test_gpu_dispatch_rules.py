"""The default route at the lines where it changes: 2D FP32 assemblies (fused
kernel or records) and the workgroup size of FP64 hexahedra."""
import numpy as np
import pytest

from plugin_navierstokes_amd import F32, F64, NavierStokesFV1
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc, fp32_violation, fp64_violation

pytestmark = pytest.mark.gpu


def _disc(mesh, up):
    disc = NavierStokesFV1("u,v,p" if mesh.dim == 2 else "u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": up, "nu": 0.02})
    disc.set_mesh(mesh)
    return disc


# 96 Ki elements are 313.5^2 quads and 2 x 221.7^2 triangles
@pytest.mark.parametrize("et,n,up,path", [(M.QUAD, 313, "lps", 1), (M.QUAD, 314, "lps", 0), (M.QUAD, 314, "full", 1),
                                          (M.TRI, 221, "skewed", 1), (M.TRI, 222, "skewed", 0), (M.TRI, 222, "no", 1)])
def test_2d_fp32(cuda, et, n, up, path):
    import torch

    mesh = M.cavity_2d(n, et, 0.1, 3)
    disc = _disc(mesh, up)
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    J, d = disc.assemble(u, jprec=F32)
    assert disc.assembly_path_used() == path
    _, d2 = disc.assemble(u, jprec=F32, want_J=False)
    assert torch.equal(d, d2)
    disc.set_assembly_path(1 - path)
    Jo, do = disc.assemble(u, jprec=F32)
    J64, _ = disc.assemble(u, jprec=F64)
    # sums of at most 8 elements' terms a block, every term rounded a few times in
    # FP32: compared with the largest entry of the node's row block
    A = J64.abs().cpu().numpy()
    rp = disc.pattern()[0]
    scale = np.repeat(np.maximum.reduceat(A, rp[:-1:3]), np.diff(rp[::3]))
    for X in (J, Jo):
        assert fp32_violation(X.cpu().numpy(), J64.cpu().numpy(), scale) <= 1.0
    s = np.abs(do.cpu().numpy()).max()
    assert np.abs(d.cpu().numpy() - do.cpu().numpy()).max() <= 1e-12 * s


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


def test_autotuner_times_a_fixed_shape_once(cuda):
    """Tetrahedra on element records run in workgroups of their own: one path-0 entry, the
    default shape, so that no other shape is left set by chance."""
    import torch

    mesh = M.cavity_3d(5, M.TET, 0.1, 3)
    disc = _disc(mesh, "lps")
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    best, table = disc.autotune_native(u, reps=2, jprec=F32)
    assert [tuple(t[1:3]) for t in table if t[0] == 0] == [(256, 65536)]
    assert best in [t[:3] for t in table] and any(t[0] == 1 for t in table)
