"""Integral store and first-quarter transform where lanes or wavefronts share
quartets: contracted s to d shells (beyond the screen's reach, one-pair and
several-pair species) against the oracle, and a basis whose rows (a b) of the
transform do not fit in LDS at once against the Coulomb build."""
import numpy as np
import pytest

import oracle as O
from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _contracted(nprim, centres, lmax):
    e = 0.25 * 2.3 ** np.arange(nprim)
    return S.custom_species("X", [S.Shell(l, e * (1 + 0.1 * l), np.linspace(1.0, 0.3, nprim), np.array(c, float))
                                  for c in centres for l in range(lmax + 1)], n_particles=2)


@pytest.mark.parametrize("nprim,centres,lmax", [(1, [(0, 0, 0)], 0), (9, [(0, 0, 0), (0.4, 1.1, -0.3)], 1),
                                                (3, [(0, 0, 0), (0.4, 1.1, -0.3)], 2)])
def test_store_and_transform_equal_oracle(nprim, centres, lmax):
    a, b = _contracted(nprim, centres, lmax), _contracted(2, [(0.3, 0.2, 0.6)], max(lmax, 1))
    n, m = a.nbasis, b.nbasis
    rng = np.random.default_rng(3)
    D = (lambda x: x @ x.T)(rng.normal(size=(n, 2)))
    Ca = rng.normal(size=(n, n))
    ha, hb = LI.Libint2Interface(a, 1), LI.Libint2Interface(b, 2)
    ha.init_2body_ints()
    ba, bb = O.Basis(a), O.Basis(b)
    pairs = (
        (ha.compute_2body_intraspecies_direct_all(D), O.compute_2body_directAll(ba, D)),
        (ha.compute_2body_intraspecies_direct_IT(D, Ca, n - 1), O.compute_2body_directIT(ba, D, Ca, n - 1)),
        (ha.compute_2body_interspecies_direct_all(hb, D), O.compute_coupling_directAll(ba, bb, 1, 2)),
        (ha.compute_2body_interspecies_direct_IT(hb, D, Ca, 0), O.compute_coupling_directIT(ba, bb, 1, 2, Ca, 0)))
    for got, ref in pairs:
        ref = np.asarray(ref).reshape(got.shape)
        # rounding of the integrals (the suite's 1e-10 for sums of order one);
        # an element at the 1e-10 drop may be kept on one side alone
        assert np.max(np.abs(got - ref)) < 1e-9 * max(1.0, np.max(np.abs(ref)))
    ha.close()
    hb.close()


def test_transform_in_several_passes_contracts_to_coulomb():
    sp = S.water_cluster(23, np.random.default_rng(8)).species[0]
    n = sp.nbasis
    assert 36 * n * 8 > 163840          # the (dd|) rows need a second pass
    rng = np.random.default_rng(4)
    D = (lambda x: x @ x.T)(rng.normal(size=(n, 4)) / np.sqrt(n))
    c = rng.normal(size=n) / np.sqrt(n)
    h = LI.Libint2Interface(sp, 1)
    J = h.compute_2body_intraspecies_direct(D, 0.0)
    dD, dc, dG = H.DeviceArray.from_host(D), H.DeviceArray.from_host(c), H.DeviceArray((n, n, n))
    h.store_device(1, dG.ptr, dD.ptr, dc.ptr)
    GG = dG.download()
    assert np.array_equal(GG, GG.transpose(0, 2, 1))
    got = GG.reshape(n, n * n) @ D.reshape(-1)
    # integrals below 1e-10 (raw; norma products below 10) are left out of GG
    bound = 1e-9 * np.sum(np.abs(c)) * np.sum(np.abs(D)) / n
    assert np.max(np.abs(got - c @ J)) < bound < 1e-3 * np.max(np.abs(got))
    dG.free()
    h.close()
