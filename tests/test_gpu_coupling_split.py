"""Coupling builds where lanes share quartets, leave out those below the drop
and spread the high classes over short tasks: contracted s to d shells, pairs
far apart (none, some or all of their quartets left out) and one-pair species,
against the oracle; and the counts, which are those of all pairs."""
import numpy as np
import pytest

import oracle as O
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _contracted(nprim, centres, lmax, least=0.25):
    e = least * 2.3 ** np.arange(nprim)
    return S.custom_species("X", [S.Shell(l, e * (1 + 0.1 * l), np.linspace(1.0, 0.3, nprim), np.array(c, float))
                                  for c in centres for l in range(lmax + 1)], n_particles=2)


@pytest.mark.parametrize("nprim,centres,lmax", [
    (1, [(0, 0, 0)], 0),                                                   # one pair
    (9, [(0, 0, 0), (0.4, 1.1, -0.3)], 1),                                 # 64 lanes to a quartet
    (3, [(0, 0, 0), (6.0, 0.2, -0.3), (11.5, 0.1, 0.4)], 2),               # bounds on both sides of the drop
    (2, [(0, 0, 0), (40.0, 0.0, 0.0)], 2)])                                # pairs without a primitive
def test_coupling_equals_oracle(nprim, centres, lmax):
    a, b = _contracted(nprim, centres, lmax), _contracted(2, [(0.3, 0.2, 0.6)], max(lmax, 1), 2.0)
    rng = np.random.default_rng(3)
    Da, Db = ((lambda x: x @ x.T)(rng.normal(size=(s.nbasis, 2))) for s in (a, b))
    ha, hb = LI.Libint2Interface(a, 1), LI.Libint2Interface(b, 2)
    ba, bb = O.Basis(a), O.Basis(b)
    ra, rb = ha.coupling_pair(hb, Da, Db)
    for got, ref in ((ra, O.compute_coupling_direct(ba, bb, 1, 2, Db)), (rb, O.compute_coupling_direct(bb, ba, 2, 1, Da)),
                     (ha.compute_2body_interspecies_direct(hb, Db), O.compute_coupling_direct(ba, bb, 1, 2, Db))):
        # the suite's 1e-10 on sums of order one; the oracle holds the transpose
        assert np.max(np.abs(got - ref.T)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    pairs = [len(s.shells) * (len(s.shells) + 1) // 2 for s in (a, b)]
    assert ha.stats()["quartets"] == pairs[0] * pairs[1]
    ha.close()
    hb.close()
