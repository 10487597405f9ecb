"""Triangle and tetrahedron meshes (FP32 Jacobian: element records and block
lists; FP64: the fused kernel): parity with the oracle at the edges of the record groups (eight
elements) and workgroups, isolated nodes, one element, and the routes that
differ (an unaligned Jacobian, other streams, no allocation, the fused path)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from plugin_navierstokes_amd import F32, F64, PART_A, PART_M, PART_RHS, UPWIND_FRESH, UPWIND_RECORD, UPWIND_REPLAY
from plugin_navierstokes_amd import NavierStokesFV1
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc, fp32_violation, fp64_violation, run_case, worst

pytestmark = pytest.mark.gpu


def _cut(mesh, ne):
    """The first ne elements of a mesh; the nodes they leave stay, isolated."""
    return M.Mesh(mesh.et, mesh.xyz, mesh.conn[:ne], {}, ())


# element counts around groups of eight and the workgroups' 128 elements
MESHES = [(M.TRI, lambda ne: _cut(M.cavity_2d(14, M.TRI, 0.1, 3), ne), ne) for ne in (1, 7, 8, 9, 127, 128, 129, 255, 257, 392)]
MESHES += [(M.TET, lambda ne: _cut(M.cavity_3d(4, M.TET, 0.1, 3), ne), ne) for ne in (1, 7, 8, 9, 127, 128, 129, 257, 384)]


def _jviol(J, Jr, Ja, jprec):
    return fp32_violation(J, Jr, Ja) if jprec == F32 else fp64_violation(J, Jr, Ja)


# FP64 tetrahedra (fused kernel): tests/test_gpu_parity.py
@pytest.mark.parametrize("up", ["no", "full", "skewed", "lps"])
@pytest.mark.parametrize("et,make,ne,jprec", [(*m, p) for m in MESHES for p in (F32, F64) if m[0] == M.TRI or p == F32],
                         ids=lambda x: str(x) if isinstance(x, int) else "m")
def test_parity(cuda, et, make, ne, jprec, up):
    cfg = {"upwind": up, "rho": 1.3, "source": (0.3, -0.2, 0.1)[:M.DIM[et]]}
    J, d, Jr, dr, Ja, da, disc = run_case(cuda, et, cfg, mesh=make(ne), time_dep=True, parts=PART_A | PART_M | PART_RHS,
                                          s=(0.7, 1.3, -0.7), jprec=jprec, path=0)
    assert disc.assembly_path_used() == (1 if jprec == F64 else 0)
    assert fp64_violation(d, dr, da) <= 1.0, worst(d, dr, da)
    assert _jviol(J, Jr, Ja, jprec) <= 1.0


@pytest.mark.parametrize("up", ["full", "lps"])
def test_axis_aligned_zeros_and_laplace(cuda, up):
    """Uniform Kuhn tetrahedra: entries without a contribution are exact zeros."""
    J, d, Jr, dr, Ja, da, _ = run_case(cuda, M.TET, {"upwind": up, "laplace": True}, mesh=M.cavity_3d(3, M.TET), jprec=F32)
    assert fp64_violation(d, dr, da) <= 1.0, worst(d, dr, da)
    assert fp32_violation(J, Jr, Ja) <= 1.0


def _scales(disc, mesh, et, u, uo):
    p = O.Params(dim=mesh.dim, upwind="lps", nu=0.02)
    rp, ci = disc.pattern()
    return O.assemble_abs(p, et, mesh.xyz, mesh.conn, u.cpu().numpy(), uo.cpu().numpy(), 0.01, s_m=1.5, parts=3,
                          rowptr=rp, colidx=ci)


@pytest.mark.parametrize("jprec", [F32, F64])
@pytest.mark.parametrize("et", [M.TRI, M.TET])
def test_routes_agree(cuda, et, jprec):
    """Defect only, an unaligned Jacobian, a second run, other streams, the
    no-allocation entry and the fused path."""
    import torch

    mesh = M.cavity_2d(9, et, 0.1, 2) if et == M.TRI else M.channel_3d((12, 6, 6), n_boxes=2, seed=5)
    disc = NavierStokesFV1("u,v,p" if mesh.dim == 2 else "u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": "lps", "nu": 0.02})
    disc.set_mesh(mesh)
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    uo = torch.from_numpy(M.random_state(mesh, 5)).to(cuda)
    kw = dict(u_old=uo, dt=0.01, s_m=1.5, parts=PART_A | PART_M, jprec=jprec)
    J, d = disc.assemble(u, **kw)
    J2, d2 = disc.assemble(u, **kw)
    assert torch.equal(J, J2) and torch.equal(d, d2)
    _, d3 = disc.assemble(u, want_J=False, **kw)
    assert torch.equal(d, d3)
    J4, _ = disc.assemble(u, want_d=False, **kw)
    assert torch.equal(J, J4)
    buf = torch.full((disc.nnz() + 1,), float("nan"), dtype=J.dtype, device=cuda)
    J5, d5 = disc.assemble(u, J=buf[1:], **kw)
    assert torch.equal(J, J5) and torch.equal(d, d5)
    J7, d7 = disc.assemble(u, J=torch.empty_like(J), d=torch.empty_like(d), noalloc=True, **kw)
    assert torch.equal(J, J7) and torch.equal(d, d7)
    for _ in range(6):
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        J8, d8 = disc.assemble(u, stream=st, **kw)
        torch.cuda.synchronize()
        assert torch.equal(J, J8) and torch.equal(d, d8)
    disc.set_assembly_path(1)
    J6, d6 = disc.assemble(u, **kw)
    assert disc.assembly_path_used() == 1
    Ja, da = _scales(disc, mesh, et, u, uo)
    # the fused path rounds the same terms in a different order
    assert _jviol(J6.cpu().numpy(), J.cpu().numpy(), 2 * Ja, jprec) <= 1.0
    assert fp64_violation(d6.cpu().numpy(), d.cpu().numpy(), 2 * da) <= 1.0


@pytest.mark.parametrize("et", [M.TRI, M.TET])
def test_replayed_decisions(cuda, et):
    import torch

    mesh = M.cavity_2d(7, et, 0.1, 2) if et == M.TRI else M.cavity_3d(3, et, 0.1, 2)
    disc = NavierStokesFV1("u,v,p" if mesh.dim == 2 else "u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": "skewed", "nu": 0.02})
    disc.set_mesh(mesh)
    u = torch.from_numpy(M.random_state(mesh, 4)).to(cuda)
    J0, d0 = disc.assemble(u, jprec=F32)
    disc.set_upwind_decisions(UPWIND_RECORD)
    disc.assemble(u, jprec=F32)
    disc.set_upwind_decisions(UPWIND_REPLAY)
    J1, d1 = disc.assemble(u, jprec=F32)
    assert torch.equal(J0, J1) and torch.equal(d0, d1)
    disc.set_upwind_decisions(UPWIND_FRESH)
