"""FP64 assemblies that overlap: a captured assembly replayed on another stream
beside eager ones on the stream of its capture, and no-allocation calls of two
handles on two streams.  The fused kernel keeps nothing between launches, so
every result has the bits of a serial call."""
from __future__ import annotations

import pytest

from plugin_navierstokes_amd import F64, PART_A, PART_M, NavierStokesFV1
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc

pytestmark = pytest.mark.gpu

KW = dict(dt=0.01, s_m=1.5, parts=PART_A | PART_M, jprec=F64, check=False)


def _disc(mesh, up):
    disc = NavierStokesFV1("u,v,w,p", "Inner")
    configure_disc(disc, {"upwind": up, "nu": 0.02})
    disc.set_mesh(mesh)
    return disc


def _states(cuda, mesh, n):
    import torch

    return [torch.from_numpy(M.random_state(mesh, 11 + i)).to(cuda) for i in range(n)]


def _out(disc, cuda):
    import torch

    return (torch.full((disc.nnz(),), float("nan"), dtype=torch.float64, device=cuda),
            torch.full((disc.num_dofs(),), float("nan"), dtype=torch.float64, device=cuda))


@pytest.mark.parametrize("up", ["full", "lps"])
def test_replay_beside_eager_calls(cuda, up):
    import torch

    mesh = M.cavity_3d(14, M.TET, 0.1, 3)
    disc = _disc(mesh, up)
    us = _states(cuda, mesh, 4)
    old = 0.9 * us[0]
    ref = [disc.assemble(u, u_old=old, **KW) for u in us]
    assert disc.assembly_path_used() == 1  # no records
    torch.cuda.synchronize()
    S, T = torch.cuda.Stream(), torch.cuda.Stream()
    # an eager call on S first, then a capture on S
    Je, de = _out(disc, cuda)
    torch.cuda.synchronize()
    disc.assemble(us[0], u_old=old, J=Je, d=de, stream=S, **KW)
    torch.cuda.synchronize()
    assert torch.equal(Je, ref[0][0]) and torch.equal(de, ref[0][1])
    Jg, dg = _out(disc, cuda)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=S):
        disc.assemble(us[0], u_old=old, J=Jg, d=dg, stream=S, **KW)
    outs = [_out(disc, cuda) for _ in us]
    for _ in range(4):
        Jg.fill_(float("nan"))
        dg.fill_(float("nan"))
        torch.cuda.synchronize()
        for i in (1, 2, 3):
            with torch.cuda.stream(T):
                graph.replay()
            disc.assemble(us[i], u_old=old, J=outs[i][0], d=outs[i][1], stream=S, **KW)
        torch.cuda.synchronize()
        assert torch.equal(Jg, ref[0][0]) and torch.equal(dg, ref[0][1])
        for i in (1, 2, 3):
            assert torch.equal(outs[i][0], ref[i][0]) and torch.equal(outs[i][1], ref[i][1])


def test_noalloc_calls_of_two_handles(cuda):
    import torch

    mesh = M.cavity_3d(14, M.TET, 0.1, 3)
    discs = [_disc(mesh, "lps"), _disc(mesh, "lps")]
    us = _states(cuda, mesh, 2)
    old = 0.9 * us[0]
    ref = [disc.assemble(u, u_old=old, **KW) for disc, u in zip(discs, us)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [_out(disc, cuda) for disc in discs]
    torch.cuda.synchronize()
    for _ in range(4):
        for disc, u, st, (J, d) in zip(discs, us, streams, outs):
            disc.assemble(u, u_old=old, J=J, d=d, stream=st, noalloc=True, **KW)
    torch.cuda.synchronize()
    for disc, (J, d), (Jr, dr) in zip(discs, outs, ref):
        assert disc.assembly_path_used() == 1
        assert torch.equal(J, Jr) and torch.equal(d, dr)
