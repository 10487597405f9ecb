"""nsfv1_assemble_noalloc (the assembly entry that allocates no device
memory) against nsfv1_assemble, both called through the C ABI.

The two entries run the same kernels; the no-allocation one keeps the SCVF
records of the split and coupled paths in a fixed device array shared by
every call on the device, so its results must equal nsfv1_assemble's
bitwise, also when the array still holds an earlier call's records of a
larger mesh.  Sizes beyond the array, and state the entry would have to
allocate (launch plan, upwind record buffer), are refused as ARGUMENT
before any launch."""
from __future__ import annotations

import numpy as np
import pytest

import plugin_navierstokes_amd as P
from plugin_navierstokes_amd import F32, F64, PART_A, PART_M, NavierStokesFV1, UPWIND_RECORD
from plugin_navierstokes_amd import meshes as M
from tests._parity import configure_disc

pytestmark = pytest.mark.gpu

ARGUMENT = -1


def _disc(mesh, cfg):
    disc = NavierStokesFV1("u,v,p" if mesh.dim == 2 else "u,v,w,p", "Inner")
    configure_disc(disc, cfg)
    disc.set_mesh(mesh)
    return disc


def _state(cuda, mesh, seed):
    import torch

    u = torch.from_numpy(M.random_state(mesh, seed)).to(cuda)
    return u, 0.9 * u


def _call(entry, disc, u, uo, jprec, J, d):
    """One assembly through the named C entry: BDF-like A + M parts with the
    time-dependent stabilisation; returns the entry's status code."""
    lib = P.load_library()
    fn = getattr(lib, entry)
    return fn(disc._h, u.data_ptr(), uo.data_ptr(), 0.01, 1.0, 150.0, 0.0, PART_A | PART_M, J.data_ptr(), jprec,
              d.data_ptr(), None)


def _both(cuda, disc, mesh, seed, jprec=F32):
    """(J, d) of nsfv1_assemble, then (J, d) of nsfv1_assemble_noalloc into
    NaN-filled outputs, on the same seeded state."""
    import torch

    u, uo = _state(cuda, mesh, seed)
    jt = torch.float32 if jprec == F32 else torch.float64
    J0 = torch.empty(disc.nnz(), dtype=jt, device=cuda)
    d0 = torch.empty(disc.num_dofs(), dtype=torch.float64, device=cuda)
    assert _call("nsfv1_assemble", disc, u, uo, jprec, J0, d0) == 0, P.load_library().nsfv1_last_error()
    path0 = disc.assembly_path_used()
    J1 = torch.full_like(J0, float("nan"))
    d1 = torch.full_like(d0, float("nan"))
    assert _call("nsfv1_assemble_noalloc", disc, u, uo, jprec, J1, d1) == 0, P.load_library().nsfv1_last_error()
    disc.sync_errors()
    assert disc.assembly_path_used() == path0
    return J0, d0, J1, d1, path0


def test_noalloc_split_two_calls_larger_then_smaller(cuda):
    """Split path (jittered hexahedra, FP32 J): a 43 200-element mesh, then
    a 720-element one whose records land on the first call's; each equals
    nsfv1_assemble bitwise, and so does the larger mesh again afterwards."""
    import torch

    cfg = {"upwind": "skewed", "nu": 0.01}
    big = M.box_3d((40, 36, 30), (1.0, 0.8, 1.3), M.HEX, 0.1, 3)
    small = M.box_3d((10, 9, 8), (1.0, 0.8, 1.3), M.HEX, 0.1, 4)
    db, ds = _disc(big, cfg), _disc(small, cfg)
    for disc, mesh, seed in ((db, big, 1), (ds, small, 2), (db, big, 5)):
        print(f"no-alloc split: ne={mesh.ne} seed={seed}", flush=True)
        J0, d0, J1, d1, path = _both(cuda, disc, mesh, seed)
        assert path == 0, f"expected the split path, ran path {path}"
        assert torch.equal(J0, J1) and torch.equal(d0, d1)


def test_noalloc_coupled_and_march(cuda):
    """The coupled path (FLOW stabilisation, FP64 J) keeps its records in the
    same array; the structured-hexahedra march keeps none."""
    import torch

    tri = M.cavity_2d(40, M.TRI, 0.1, 2)
    dc = _disc(tri, {"stab": "flow", "upwind": "full", "nu": 0.01})
    J0, d0, J1, d1, path = _both(cuda, dc, tri, 7, F64)
    assert path == 4, f"expected the coupled path, ran path {path}"
    assert torch.equal(J0, J1) and torch.equal(d0, d1)
    hexes = M.box_3d((9, 10, 11), (1.0, 0.8, 1.3))
    dm = _disc(hexes, {"upwind": "skewed"})
    J0, d0, J1, d1, path = _both(cuda, dm, hexes, 8)
    assert path == 3, f"expected the plane march, ran path {path}"
    assert torch.equal(J0, J1) and torch.equal(d0, d1)


def test_noalloc_refusals(cuda):
    """No launch plan yet, no upwind record buffer yet, and records beyond
    the array: ARGUMENT, with nothing written."""
    import torch

    lib = P.load_library()
    small = M.box_3d((4, 4, 4), (1.0, 1.0, 1.0), M.HEX, 0.1, 1)
    disc = _disc(small, {"upwind": "skewed"})
    u, uo = _state(cuda, small, 1)
    J = torch.full((disc.nnz(),), 7.0, dtype=torch.float32, device=cuda)
    d = torch.full((disc.num_dofs(),), 7.0, dtype=torch.float64, device=cuda)
    assert _call("nsfv1_assemble_noalloc", disc, u, uo, F32, J, d) == ARGUMENT
    assert b"no launch plan" in lib.nsfv1_last_error()
    assert _call("nsfv1_assemble", disc, u, uo, F32, J, d) == 0
    disc.set_upwind_decisions(UPWIND_RECORD)
    assert _call("nsfv1_assemble_noalloc", disc, u, uo, F32, J, d) == ARGUMENT
    assert b"no upwind record buffer" in lib.nsfv1_last_error()

    # 48^3 jittered hexahedra: 110 592 elements x 12 SCVFs x 128 bytes > 128 MiB
    big = M.box_3d((48, 48, 48), (1.0, 1.0, 1.0), M.HEX, 0.1, 2)
    db = _disc(big, {"upwind": "skewed"})
    ub, uob = _state(cuda, big, 2)
    Jb = torch.empty(db.nnz(), dtype=torch.float32, device=cuda)
    db_ = torch.empty(db.num_dofs(), dtype=torch.float64, device=cuda)
    assert _call("nsfv1_assemble", db, ub, uob, F32, Jb, db_) == 0
    assert db.assembly_path_used() == 0
    Jb.fill_(7.0)
    db_.fill_(7.0)
    assert _call("nsfv1_assemble_noalloc", db, ub, uob, F32, Jb, db_) == ARGUMENT
    msg = lib.nsfv1_last_error().decode()
    assert "holds at most 134217728" in msg, msg
    torch.cuda.synchronize()
    assert bool((Jb == 7.0).all()) and bool((db_ == 7.0).all())
    assert np.isclose(float(P.NOALLOC_SCRATCH_BYTES), 128 * 2 ** 20)


# element counts between the limits of SCVF records (128 bytes each) and of the route
# that runs: element records (480 bytes a tetrahedron), or none (fused kernel)
@pytest.mark.parametrize("et,n,up,path", [(M.QUAD, 600, "full", 1), (M.TRI, 430, "no", 1), (M.TET, 33, "full", 0)])
def test_noalloc_limit_is_the_routes_own(cuda, et, n, up, path):
    import torch

    mesh = M.cavity_3d(n, et, 0.1, 3) if et == M.TET else M.cavity_2d(n, et, 0.1, 3)
    scvfs = {M.QUAD: 4, M.TRI: 3, M.TET: 6}[et]
    assert mesh.ne * scvfs * 128 > P.NOALLOC_SCRATCH_BYTES
    disc = _disc(mesh, {"upwind": up, "nu": 0.01})
    J0, d0, J1, d1, used = _both(cuda, disc, mesh, 3)
    assert used == path
    assert torch.equal(J0, J1) and torch.equal(d0, d1)


def test_noalloc_refuses_element_records_beyond_the_array(cuda):
    import torch

    mesh = M.cavity_3d(37, M.TET, 0.1, 3)
    assert mesh.ne * 480 > P.NOALLOC_SCRATCH_BYTES
    disc = _disc(mesh, {"upwind": "full", "nu": 0.01})
    u, uo = _state(cuda, mesh, 2)
    J = torch.empty(disc.nnz(), dtype=torch.float32, device=cuda)
    d = torch.empty(disc.num_dofs(), dtype=torch.float64, device=cuda)
    assert _call("nsfv1_assemble", disc, u, uo, F32, J, d) == 0
    assert disc.assembly_path_used() == 0
    J.fill_(7.0)
    d.fill_(7.0)
    assert _call("nsfv1_assemble_noalloc", disc, u, uo, F32, J, d) == ARGUMENT
    assert b"holds at most" in P.load_library().nsfv1_last_error()
    torch.cuda.synchronize()
    assert bool((J == 7.0).all()) and bool((d == 7.0).all())


@pytest.mark.parametrize("n,fits", [(28, True), (32, False)])
def test_noalloc_coupled_limit(cuda, n, fits):
    """Element matrices and corner defects: 8 x 8 blocks of 4 x 4 FP32 values and 8 x 4
    doubles a hexahedron."""
    import torch

    mesh = M.box_3d((n, n, n), (1.0, 1.0, 1.0), M.HEX, 0.1, 2)
    assert (mesh.ne * (8 * 8 * 16 * 4 + 8 * 4 * 8) <= P.NOALLOC_SCRATCH_BYTES) == fits
    disc = _disc(mesh, {"upwind": "positive", "nu": 0.01})
    if fits:
        J0, d0, J1, d1, path = _both(cuda, disc, mesh, 3)
        assert path == 4
        assert torch.equal(J0, J1) and torch.equal(d0, d1)
        return
    u, uo = _state(cuda, mesh, 2)
    J = torch.empty(disc.nnz(), dtype=torch.float32, device=cuda)
    d = torch.empty(disc.num_dofs(), dtype=torch.float64, device=cuda)
    assert _call("nsfv1_assemble", disc, u, uo, F32, J, d) == 0
    J.fill_(7.0)
    assert _call("nsfv1_assemble_noalloc", disc, u, uo, F32, J, d) == ARGUMENT
    assert b"holds at most" in P.load_library().nsfv1_last_error()
    torch.cuda.synchronize()
    assert bool((J == 7.0).all())
