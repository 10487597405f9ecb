"""Orthogonalisation against the Krylov basis and norms (device reductions of the
GMRES loops) at the edges of their blocks (1024 entries below 2^20 unknowns,
4096 from there on, 1024 or 512 with a held basis of up to 24 vectors) and
vector groups (4, 8), and a workspace across meshes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nsfv1::launch_orthogonalise / launch_norm2 / red_partials
ORTHO = "_ZN5nsfv120launch_orthogonaliseEPKdliPdlS2_S2_iP12ihipStream_t"
NORM2 = "_ZN5nsfv112launch_norm2EPKdlPdS2_P12ihipStream_t"
PARTIALS = "_ZN5nsfv112red_partialsEl"
EPS = 2.0 ** -53
HS = 61


@pytest.mark.parametrize("n,k", [(1, 1), (255, 2), (1023, 7), (1024, 8), (1025, 9), (5000, 60), ((1 << 20) - 1, 3),
                                 (1 << 20, 8), ((1 << 20) + 1, 16), ((1 << 20) + 4099, 17),
                                 ((1 << 20) + 511, 1), ((1 << 20) + 513, 5), ((1 << 20) + 1025, 12), (1 << 20, 24),
                                 ((1 << 20) + 1023, 25)])
def test_orthogonalise(cuda, n, k):
    import torch

    import plugin_navierstokes_amd as P

    L = C.CDLL(P.LIB_PATH)
    fn, nf, nb = getattr(L, ORTHO), getattr(L, NORM2), getattr(L, PARTIALS)
    nb.restype = C.c_int64
    g = torch.Generator(device=cuda).manual_seed(n + k)
    ld = n + 3
    Vb = torch.randn(k, ld, generator=g, dtype=torch.float64, device=cuda) / n ** 0.5
    Vb[:, n:] = float("nan")  # beyond the vectors
    w0 = torch.randn(n, generator=g, dtype=torch.float64, device=cuda)
    part = torch.full((nb(C.c_int64(n)),), float("nan"), dtype=torch.float64, device=cuda)
    p = lambda t: C.c_void_p(t.data_ptr())

    def run():
        w = w0.clone()
        h = torch.full((2 * HS + 1,), float("nan"), dtype=torch.float64, device=cuda)
        assert fn(p(Vb), C.c_int64(ld), k, p(w), C.c_int64(n), p(part), p(h), HS, None) == 0
        torch.cuda.synchronize()
        return w, h

    w, h = run()
    V = Vb[:, :n]
    # a sum in blocks rounds at most c times on the way of each term: 16 products a
    # thread, 6 + 3 steps across the block, the blocks by 256 threads, 9 more
    c = (16 + 9 + n // (1024 * 256) + 1 + 9 + 32) * EPS  # 32: the reference's own
    A = V.abs()
    h1, e1 = V @ w0, c * (A @ w0.abs())
    w1 = w0 - h1 @ V
    d1 = e1 @ A + (k + 2) * EPS * (w0.abs() + h1.abs() @ A)
    h2, e2 = V @ w1, A @ (c * w1.abs() + d1)
    w2 = w1 - h2 @ V
    d2 = d1 + e2 @ A + (k + 2) * EPS * (w1.abs() + h2.abs() @ A)
    n2, en = float(w2 @ w2), float(w2.abs() @ (c * w2.abs() + 2 * d2))
    assert bool(((h[:k] - h1).abs() <= e1).all())
    assert bool(((h[HS:HS + k] - h2).abs() <= e2).all())
    assert bool(((w - w2).abs() <= d2).all())
    assert abs(float(h[2 * HS]) - n2) <= en
    # the same bits again; the norm alone too
    wr, hr = run()
    assert torch.equal(w, wr) and torch.equal(h[:k], hr[:k]) and float(h[2 * HS]) == float(hr[2 * HS])
    o = torch.zeros(1, dtype=torch.float64, device=cuda)
    assert nf(p(w), C.c_int64(n), p(part), p(o), None) == 0
    torch.cuda.synchronize()
    assert float(o) == float(h[2 * HS])
