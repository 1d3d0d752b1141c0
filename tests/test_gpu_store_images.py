"""Integral store: the eight index images of an integral hold the same bits, also
where one block holds two of them ((aa|cd), (ab|ab)) and lanes share the block;
one, several and 64 lanes to a quartet and one wavefront per quartet."""
import numpy as np
import pytest

from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _contracted(nprim, centres, lmax):
    e = 0.25 * 2.3 ** np.arange(nprim)
    return S.custom_species("X", [S.Shell(l, e * (1 + 0.1 * l), np.linspace(1.0, 0.3, nprim), np.array(c, float))
                                  for c in centres for l in range(lmax + 1)], n_particles=2)


@pytest.mark.parametrize("species", [
    lambda: _contracted(1, [(0, 0, 0), (0.4, 1.1, -0.3)], 2),
    lambda: _contracted(8, [(0, 0, 0), (0.4, 1.1, -0.3)], 1),
    lambda: S.water("6-31G**").species[0],
    lambda: S.water_cluster(2, np.random.default_rng(11), "cc-pVDZ").species[0]],
    ids=["primitive s p d", "8 primitives s p", "water", "two waters"])
def test_images_are_bit_equal(species):
    sp = species()
    n = sp.nbasis
    X = np.random.default_rng(3).normal(size=(n, 3)) / np.sqrt(n)
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    A = h.compute_2body_intraspecies_direct_all(2.0 * X @ X.T).reshape(n, n, n, n)
    h.close()
    assert np.max(np.abs(A)) > 0.1
    for axes in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(A, A.transpose(axes)), axes
