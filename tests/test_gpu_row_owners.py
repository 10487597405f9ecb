"""Hexahedra with FP32 Jacobian on SCVF records: blocks summed by owners.  Parity
with the oracle at the edges of the workgroups (256 incidences, 255 nodes), with
isolated nodes, on disjoint elements (more blocks than the segments' room in
LDS) and for every workgroup size."""
import numpy as np
import pytest

from plugin_navierstokes_amd import F32, PART_A, PART_M, PART_RHS, NavierStokesFV1
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc, fp32_violation, fp64_violation, run_case, worst

pytestmark = pytest.mark.gpu


def _cut(ne):
    """The first ne elements; the nodes they leave stay, isolated (up to 721)."""
    m = M.cavity_3d(8, M.HEX, 0.1, 3)
    return M.Mesh(m.et, m.xyz, m.conn[:ne], {}, ())


def _disjoint(ne):
    m = M.cavity_3d(4, M.HEX, 0.1, 3)
    c = m.conn[:ne]
    return M.Mesh(m.et, np.ascontiguousarray(m.xyz[c].reshape(-1, 3)), np.arange(c.size, dtype=c.dtype).reshape(c.shape), {}, ())


MESHES = {"one": _cut(1), "seven": _cut(7), "cut": _cut(100), "all": _cut(512), "disjoint": _disjoint(33), "apart": _disjoint(5)}


@pytest.mark.parametrize("up", ["no", "full", "skewed", "lps"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_parity(cuda, mesh, up):
    cfg = {"upwind": up, "rho": 1.3, "source": (0.3, -0.2, 0.1)}
    J, d, Jr, dr, Ja, da, disc = run_case(cuda, M.HEX, cfg, mesh=MESHES[mesh], time_dep=True,
                                          parts=PART_A | PART_M | PART_RHS, s=(0.7, 1.3, -0.7), jprec=32)
    assert disc.assembly_path_used() == 0
    assert fp64_violation(d, dr, da) <= 1.0, worst(d, dr, da)
    assert fp32_violation(J, Jr, Ja) <= 1.0


@pytest.mark.parametrize("mesh", ["all", "disjoint", "seven"])
def test_routes_agree(cuda, mesh):
    import torch

    mesh = MESHES[mesh]
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    out = []
    for threads in (0, 256, 192, 128, 64):
        disc = NavierStokesFV1("u,v,w,p", "Inner")
        configure_disc(disc, {"upwind": "lps", "nu": 0.02})
        disc.set_mesh(mesh)
        disc.set_assembly_path(0)
        if threads:
            disc.set_launch(threads, 65536)
        J, d = disc.assemble(u, jprec=F32)
        out.append((J, d))
        # defect only, no defect, an unaligned Jacobian, no allocation
        assert torch.equal(d, disc.assemble(u, jprec=F32, want_J=False)[1])
        assert torch.equal(J, disc.assemble(u, jprec=F32, want_d=False)[0])
        buf = torch.full((disc.nnz() + 1,), float("nan"), dtype=torch.float32, device=cuda)
        assert torch.equal(J, disc.assemble(u, J=buf[1:], jprec=F32)[0])
        J2, d2 = disc.assemble(u, J=torch.full_like(J, float("nan")), d=torch.empty_like(d), jprec=F32, noalloc=True)
        assert torch.equal(J, J2) and torch.equal(d, d2)
    # every sum runs in element order, whatever the workgroup holds
    for J, d in out[1:]:
        assert torch.equal(J, out[0][0]) and torch.equal(d, out[0][1])


@pytest.mark.parametrize("how", ["configuration", "unaligned"])
def test_lists_after_the_plane_march(cuda, how):
    """A plan built by the march, which needs no lists: calls that may not allocate
    and captured calls give the bits of any other, through the same kernels, without
    an allocating call on records before them."""
    import torch

    mesh = M.cavity_3d(6, M.HEX)
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    disc = NavierStokesFV1("u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": "full", "nu": 0.02})
    disc.set_mesh(mesh)
    J, d = disc.assemble(u, jprec=F32)
    assert disc.assembly_path_used() == 3

    def out():
        # not 16-byte aligned: not a march call either
        o = 1 if how == "unaligned" else 0
        return torch.full((J.numel() + o,), float("nan"), dtype=J.dtype, device=cuda)[o:], torch.full_like(d, float("nan"))

    if how == "configuration":
        configure_disc(disc, {"upwind": "full", "nu": 0.02, "difflen": "fivepoint"})
    J1, d1 = out()
    disc.assemble(u, J=J1, d=d1, jprec=F32, noalloc=True)
    assert disc.assembly_path_used() == 0
    J2, d2 = out()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        disc.assemble(u, J=J2, d=d2, jprec=F32, noalloc=True, stream=s, check=False)
    J3, d3 = out()
    disc.assemble(u, J=J3, d=d3, jprec=F32)
    assert disc.assembly_path_used() == 0
    for _ in range(3):
        J2.fill_(float("nan"))
        d2.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(J2, J3) and torch.equal(d2, d3)
    assert torch.equal(J1, J3) and torch.equal(d1, d3)
