"""Dense inverse of the coarsest multigrid level (blocked Gauss-Jordan) against
numpy, at the edges of its panels (16 pivots), update tiles (16 x 16, one a wave)
and rows per thread (512 threads: two rows from 513 on, three from 1025)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nsfv1::launch_dense_inverse / nsfv1::dense_inverse_work_bytes
INVERSE = ("_ZN5nsfv120launch_dense_inverseEiPKlPKiPKviPvPdPiP12ihipStream_t")
BYTES = "_ZN5nsfv124dense_inverse_work_bytesEi"


def invert(A, dtype=np.float64):
    import torch

    import plugin_navierstokes_amd as P

    L = C.CDLL(P.LIB_PATH)
    fn, nb = getattr(L, INVERSE), getattr(L, BYTES)
    nb.restype = C.c_size_t
    n = A.shape[0]
    dev = "cuda:0"
    J = torch.as_tensor(A.astype(dtype), device=dev).reshape(-1).contiguous()
    rp = torch.arange(0, n * n + 1, n, dtype=torch.int64, device=dev)
    ci = torch.arange(n, dtype=torch.int32, device=dev).repeat(n)
    work = torch.full((nb(n) // 8 + 1,), float("nan"), dtype=torch.float64, device=dev)
    inv = torch.full((n, n), float("nan"), dtype=torch.float64, device=dev)
    err = torch.full((1,), 7, dtype=torch.int32, device=dev)
    p = lambda t: C.c_void_p(t.data_ptr())
    rc = fn(64 if dtype == np.float64 else 32, p(rp), p(ci), p(J), n, p(work), p(inv), p(err), None)
    torch.cuda.synchronize()
    return rc, inv.cpu().numpy(), int(err.item())


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 255, 257, 448, 511, 512, 513, 867, 1023, 1024, 1025, 1200])
def test_inverse(n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A[np.arange(n), np.arange(n)] = 0.0  # every step needs a pivot search
    if n == 1:
        A[0, 0] = -3.0
    rc, inv, err = invert(A)
    assert rc == 0 and err == 0
    ref = np.linalg.inv(A)
    # partial pivoting: backward error of a few n eps times the growth of the
    # tableau (about n^(2/3) for random matrices), amplified by the condition
    bound = 4.0 * n ** (5.0 / 3.0) * 2.0 ** -53 * np.linalg.cond(A)
    assert np.linalg.norm(inv - ref) <= bound * np.linalg.norm(ref)
    # the same bits again
    assert np.array_equal(inv, invert(A)[1])


@pytest.mark.parametrize("n,k", [(40, 0), (40, 17), (300, 299), (512, 511), (513, 512), (1100, 1030)])
def test_null_mode_is_pinned(n, k):
    """A zero row and column k: the other unknowns are solved, x_k = 0."""
    rng = np.random.default_rng(k)
    A = rng.standard_normal((n, n)) + 2.0 * np.sqrt(n) * np.eye(n)
    A[k, :] = 0.0
    A[:, k] = 0.0
    rc, inv, err = invert(A)
    assert rc == 0 and err == 0
    keep = np.delete(np.arange(n), k)
    ref = np.linalg.inv(A[np.ix_(keep, keep)])
    got = inv[np.ix_(keep, keep)]
    assert np.linalg.norm(got - ref) <= 4.0 * n ** (5.0 / 3.0) * 2.0 ** -53 * np.linalg.cond(A[np.ix_(keep, keep)]) * \
        np.linalg.norm(ref)
    assert np.all(inv[k, :] == 0.0)


def test_fp32_matrix_and_non_finite_column():
    rng = np.random.default_rng(5)
    A = (rng.standard_normal((130, 130)) + 8.0 * np.eye(130)).astype(np.float32).astype(np.float64)
    rc, inv, err = invert(A, np.float32)
    ref = np.linalg.inv(A)
    assert rc == 0 and err == 0
    assert np.linalg.norm(inv - ref) <= 4.0 * 130 ** (5.0 / 3.0) * 2.0 ** -53 * np.linalg.cond(A) * np.linalg.norm(ref)
    A[:, 100] = np.nan
    assert invert(A)[2] == 1


def test_oversize_is_refused():
    assert invert(np.eye(1201))[0] != 0
