"""Lanes sharing a quartet (strip kernels): molecules whose primitive counts
need 1 to 64 lanes per quartet, kets that do not fill a round, one-pair
species, and a bra beyond the staged primitive pairs, against the oracle."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle as O  # noqa: E402

from openlowdin_amd import libint2_interface as LI  # noqa: E402
from openlowdin_amd import system as S  # noqa: E402

pytestmark = pytest.mark.gpu


def _contracted(nprim, centres, lmax=1):
    """Shells of nprim primitives (s .. lmax) on each centre."""
    e = 0.05 * 2.1 ** np.arange(nprim)
    return S.custom_species("X", [S.Shell(l, e * (1 + 0.1 * l), np.linspace(1.0, 0.2, nprim), np.array(c, float))
                                  for c in centres for l in range(lmax + 1)], n_particles=2)


def _species(name):
    if name == "one shell":
        return _contracted(9, [(0, 0, 0)], lmax=0)
    if name == "8 primitives":
        return _contracted(8, [(0, 0, 0), (0.4, 1.1, -0.3)])
    if name == "9 primitives":       # 81 primitive pairs: not staged
        return _contracted(9, [(0, 0, 0), (0.4, 1.1, -0.3)])
    if name == "5 primitives, d":
        return _contracted(5, [(0, 0, 0), (0.4, 1.1, -0.3), (1.7, 0, 0.2)], lmax=2)
    if name == "water":
        return S.water("cc-pVDZ").species[0]
    return S.build_system(S.alkane_geometry(4), "cc-pVDZ").species[0]


@pytest.mark.parametrize("name", ["one shell", "8 primitives", "9 primitives", "5 primitives, d", "water", "butane"])
@pytest.mark.parametrize("factor", [-0.5, 0.3])
def test_build_equals_oracle(name, factor):
    sp = _species(name)
    rng = np.random.default_rng(11)
    C = rng.normal(size=(sp.nbasis, 3)) / np.sqrt(sp.nbasis)
    D = C @ C.T
    ref = O.compute_2body_direct(O.Basis(sp), D, factor)
    h = LI.Libint2Interface(sp, 1)
    G = h.compute_2body_intraspecies_direct(D, factor)
    # the suite's bound of an FP64 build: 1e-10 absolute at integrals of order one
    assert np.max(np.abs(G - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    h.close()
