"""Diagonalisation inside one compute unit (and, past 64 functions, by the
library): the H-core density of random one-body matrices with degenerate,
core-like and close levels against LAPACK on the host."""
import numpy as np
import pytest
import scipy.linalg

from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S
from openlowdin_amd.scf_device import DeviceSCF

pytestmark = pytest.mark.gpu


def _system(n, nocc):
    shells = [S.Shell(0, np.array([1.0]), np.array([1.0]), np.array([3.0 * k, 0.0, 0.0])) for k in range(n)]
    return S.MolecularSystem([S.custom_species("X", shells, n_particles=nocc)], [])


def _matrices(n, nocc, kind):
    rng = np.random.default_rng(n)
    Q = np.linalg.qr(rng.normal(size=(n, n)))[0]
    low = {"core": np.concatenate([[-20.0] * 2, rng.normal(size=n)])[:nocc], "degenerate": -1.0 - np.arange(nocc) // 3,
           "close": -1.0 - 1e-9 * np.arange(nocc), "diagonal": -1.0 - np.arange(nocc)}[kind]
    w = np.concatenate([np.sort(np.minimum(low, -1.0)), 1.0 + np.arange(n - nocc) // 2])
    if kind == "diagonal":
        return np.diag(w), np.eye(n)
    A = (Q * w) @ Q.T
    B = rng.normal(size=(n, n)) / np.sqrt(4.0 * n)
    L = np.eye(n) + B
    return L @ (0.5 * (A + A.T)) @ L.T, L @ L.T


@pytest.mark.parametrize("kind", ["core", "degenerate", "close", "diagonal"])
@pytest.mark.parametrize("n", [1, 2, 3, 16, 17, 63, 64, 65])
def test_density_equals_lapack(n, kind):
    nocc = (n + 1) // 2
    H, Sm = _matrices(n, nocc, kind)
    scf = DeviceSCF(_system(n, nocc), hcore=[H], overlap=[Sm])
    scf.start()
    D = scf.matrix(0)
    scf.close()
    w, C = scipy.linalg.eigh(H, Sm)
    ref = C[:, :nocc] @ C[:, :nocc].T
    # backward errors of a few n eps |H| / gap (gap 2, |H| up to 32) on both
    # sides, through S^-1/2 of condition below 10
    assert np.max(np.abs(D - ref)) < 1e-11 * max(1.0, np.max(np.abs(ref)))


def test_matrix_that_is_not_finite_is_refused():
    H, Sm = _matrices(5, 2, "core")
    Sm[1, 3] = Sm[3, 1] = np.nan
    scf = DeviceSCF(_system(5, 2), hcore=[H], overlap=[Sm])
    with pytest.raises(LI.LowdinFockError):
        scf.start()
    scf.close()
