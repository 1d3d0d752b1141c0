"""Accuracy of the diagonalisation inside one compute unit, on the vectors
themselves: residual, orthogonality and eigenvalues at the rounding of the
stored numbers, at tile edges, for one matrix and several with padding."""
import ctypes as C

import numpy as np
import pytest

from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
# bool lowdin::launch_syev(double*, int, size_t, double*, size_t, int*, int, hipStream_t)
SYMBOL = "_ZN6lowdin11launch_syevEPdimS0_mPiiP12ihipStream_t"


def _matrix(n, kind, rng):
    X = rng.normal(size=(n, n))
    if kind == "random":
        return 0.5 * (X + X.T)
    w = np.sort(np.concatenate([[-20.0] * (n // 25 + 1), rng.normal(size=n)])[:n])
    if kind == "close":
        w = 1.0 + 1e-9 * np.arange(n)
        w[:n // 2] -= 4.0
    Q = np.linalg.qr(X)[0]
    A = (Q * w) @ Q.T
    return 0.5 * (A + A.T)


def _syev(As, pad):
    n = len(As[0])
    f = LI.lib()[SYMBOL]
    f.restype = C.c_bool
    f.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p, C.c_size_t, C.c_void_p, C.c_int, C.c_void_p]
    buf = np.full((len(As), n * n + pad), 3.0)
    for b, A in zip(buf, As):
        b[:n * n] = A.ravel()
    a, w = H.DeviceArray.from_host(buf), H.DeviceArray.from_host(np.full((len(As), n + pad), 5.0))
    info = H.DeviceArray.from_host(np.full((len(As),), 7, dtype=np.int32))
    assert f(a.ptr, n, n * n + pad, w.ptr, n + pad, info.ptr, len(As), None)
    H.check(H.hip().hipDeviceSynchronize(), "hipDeviceSynchronize")
    V, W, i = a.download(), w.download(), info.download()
    assert np.all(V[:, n * n:] == 3.0) and np.all(W[:, n:] == 5.0) and np.all(i == 0)
    return [(v[:n * n].reshape(n, n).T, x[:n]) for v, x in zip(V, W)]


@pytest.mark.parametrize("count,pad", [(1, 0), (3, 5)])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 25, 32, 33, 48, 49, 50, 63, 64])
@pytest.mark.parametrize("kind", ["random", "levels", "close"])
def test_residual_orthogonality_and_levels(kind, n, count, pad):
    rng = np.random.default_rng(n)
    As = [_matrix(n, kind, rng) for _ in range(count)]
    for A, (V, w) in zip(As, _syev(As, pad)):
        Al, Vl = A.astype(np.longdouble), V.astype(np.longdouble)
        # every stored element rounds by eps / 2, so a product of two columns
        # moves by eps at most and by less at random: eps / 2 for each of the
        # n x n elements, and the worst case where there are few
        assert float(np.linalg.norm(Vl.T @ Vl - np.eye(n))) < EPS * (0.5 * n + 2.0)
        # the same rounding against |A|, whose spectral norm is a good part of
        # its Frobenius norm; levels closer than rounding can rotate keep what
        # the rotations left (a few eps more)
        res = float(np.linalg.norm(Al @ Vl - Vl * w) / np.linalg.norm(Al))
        assert res < (4.0 if kind != "close" else 10.0) * EPS
        ray = np.sum(Vl * (Al @ Vl), axis=0) / np.sum(Vl * Vl, axis=0)
        assert float(np.max(np.abs(w - ray))) < EPS * (0.5 * np.sqrt(n) + 2.0) * np.max(np.abs(w))
        assert np.all(np.diff(w) >= 0.0)
