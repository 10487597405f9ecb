"""Launch plans checked on the CPU: every index the fused row kernels take from a plan
stays inside its array, the workgroup's LDS and the CSR pattern, packed or not, for
workgroups of 64 to 256 lanes (the 128 of large FP64 hexahedral meshes among them) and
odd meshes; and set-up calls that run out of memory leave no stale sizes behind."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from plugin_navierstokes_amd import meshes as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "plan.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "plan_bounds.cpp"),
                           os.path.join(ROOT, "plugin_navierstokes_amd", "csrc", "nsfv1_api.cpp"), "-o", so])
    # kernels' launchers that no call here reaches stay unresolved; the functions of the
    # HIP runtime are the library's own also where a process has the runtime loaded
    lb = C.CDLL(so, mode=os.RTLD_LAZY | os.RTLD_LOCAL | os.RTLD_DEEPBIND)
    lb.plan_error.restype = C.c_char_p
    lb.plan_lanes.restype = lb.plan_dirichlet_rows.restype = C.c_int64
    lb.nsfv1_last_error.restype = C.c_char_p
    return lb


def _handle(lib, mesh):
    h = C.c_void_p()
    assert lib.nsfv1_create(mesh.dim, b"u,v,p" if mesh.dim == 2 else b"u,v,w,p", b"Inner", C.byref(h)) == 0
    assert lib.nsfv1_set_stabilization(h, b"fields", b"raw") == 0
    assert lib.nsfv1_set_upwind(h, b"skewed") == 0
    lib.nsfv1_set_kinematic_viscosity.argtypes = [C.c_void_p, C.c_double]
    assert lib.nsfv1_set_kinematic_viscosity(h, 0.01) == 0
    x, c = np.ascontiguousarray(mesh.xyz, dtype=np.float64), np.ascontiguousarray(mesh.conn, dtype=np.int32)
    lib.nsfv1_set_mesh.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_int64, C.c_void_p, C.c_int64]
    assert lib.nsfv1_set_mesh(h, mesh.et, x.ctypes.data, mesh.nv, c.ctypes.data, mesh.ne) == 0, lib.nsfv1_last_error()
    return h


def _assemble(lib, h, jprec):
    lib.nsfv1_assemble.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p] + [C.c_double] * 4 + [C.c_int, C.c_void_p, C.c_int,
                                   C.c_void_p, C.c_void_p]
    # the arrays' addresses only: nothing reads or writes them here
    return lib.nsfv1_assemble(h, 16, None, 0.0, 1.0, 0.0, 0.0, 1, 24, jprec, 16, None)


def _cut(m, ne):
    return M.Mesh(m.et, m.xyz, m.conn[:ne], {}, ())


def _permuted(m, seed):
    """Nodes and elements in random order."""
    g = np.random.default_rng(seed)
    p, q = g.permutation(m.nv), g.permutation(m.ne)
    inv = np.empty_like(p)
    inv[p] = np.arange(m.nv)
    return M.Mesh(m.et, m.xyz[p], inv[m.conn[q]].astype(m.conn.dtype), {}, ())


MESHES = {
    "hex16": lambda: M.cavity_3d(16, M.HEX),           # FP64: just below the line to 128 lanes
    "hex17": lambda: M.cavity_3d(17, M.HEX, 0.1, 1),   # above it
    "hex20": lambda: M.cavity_3d(20, M.HEX, 0.1, 1),
    "hex-cut": lambda: _cut(M.cavity_3d(12, M.HEX, 0.1, 3), 700),
    "hex-box": lambda: M.box_3d((41, 3, 2), (1.0, 1.0, 1.0), M.HEX, 0.1, 3),
    "hex-random": lambda: _permuted(M.cavity_3d(18, M.HEX, 0.1, 3), 5),
    "hex-one": lambda: M.cavity_3d(1, M.HEX),
    "tet": lambda: M.cavity_3d(7, M.TET, 0.1, 3),
    "tet-random": lambda: _permuted(M.cavity_3d(6, M.TET, 0.1, 3), 5),
    "prism": lambda: M.cavity_3d(9, M.PRISM, 0.1, 3),
    "quad": lambda: M.cavity_2d(37, M.QUAD, 0.1, 3),
    "quad-cut": lambda: _cut(M.cavity_2d(40, M.QUAD, 0.1, 3), 33),
    "tri": lambda: M.cavity_2d(23, M.TRI, 0.1, 3),
    "tri-random": lambda: _permuted(M.cavity_2d(19, M.TRI, 0.1, 3), 5),
}


@pytest.mark.parametrize("name", list(MESHES))
def test_every_index_of_a_plan(lib, name):
    mesh = MESHES[name]()
    h = _handle(lib, mesh)
    block = {}
    for threads, lds in ((0, 0), (64, 65536), (128, 65536), (192, 40960), (256, 32768), (256, 65536)):
        # path 1: the budget is the fused kernel's (path 3 reads it as the march's planes)
        assert lib.nsfv1_set_assembly_path(h, 1) == 0
        if threads:
            assert lib.nsfv1_set_launch(h, threads, lds) == 0
        for jprec in (32, 64):
            n0 = lib.plan_lanes()
            rc = _assemble(lib, h, jprec)
            assert lib.plan_error() == b"", (lib.plan_error(), threads, lds, jprec)
            if rc:  # the rows of one node exceed the budget: refused, not launched
                assert b"exceeds the workgroup budget" in lib.nsfv1_last_error() and lib.plan_lanes() == n0
            else:
                assert lib.plan_lanes() - n0 == mesh.conn.size
                block[threads, lds, jprec] = lib.plan_block()
    if name in ("hex17", "hex20"):
        # 256 (the default) lets large FP64 plans of hexahedra take 128, set again or not
        assert block[0, 0, 64] == block[256, 65536, 64] == 128 and block[0, 0, 32] == 256
    if name == "hex16":
        assert block[0, 0, 64] == 256
    lib.nsfv1_destroy(h)


@pytest.mark.parametrize("first", [0, 1])  # the rows' array, the mask's
def test_dirichlet_rows_after_a_failed_allocation(lib, first):
    mesh = M.cavity_3d(3, M.HEX)
    h = _handle(lib, mesh)
    lib.nsfv1_set_dirichlet.argtypes = [C.c_void_p, C.c_void_p, C.c_int64]
    lib.nsfv1_apply_dirichlet.argtypes = [C.c_void_p, C.c_void_p, C.c_int] + [C.c_void_p] * 4
    rows = np.arange(40, dtype=np.int64)
    assert lib.nsfv1_set_dirichlet(h, rows.ctypes.data, 40) == 0
    lib.plan_fail_allocation(first)
    assert lib.nsfv1_set_dirichlet(h, rows.ctypes.data, 7) != 0
    lib.plan_fail_allocation(-1)
    # the call that failed left no rows, in particular not forty in an array of seven
    assert lib.nsfv1_apply_dirichlet(h, 16, 32, None, None, None, None) == 0
    assert lib.plan_error() == b"" and lib.plan_dirichlet_rows() == 0
    # a count below zero is none
    assert lib.nsfv1_set_dirichlet(h, rows.ctypes.data, -1) == 0
    assert lib.nsfv1_apply_dirichlet(h, 16, 32, None, None, None, None) == 0
    assert lib.plan_dirichlet_rows() == 0
    lib.nsfv1_destroy(h)
