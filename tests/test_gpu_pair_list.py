"""Significant shell pairs with 16 lanes to a pair: 1, 15, 16, 17 and 81
primitive pairs, s to d, at distances around the threshold, against the
oracle's list; and a host build whose matrices pass through the staging
memory (and just do not) against the device entry."""
import numpy as np
import pytest

import oracle as O
from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(1, 1), (3, 5), (4, 4), (1, 17), (9, 9)])
def test_pair_list_equals_oracle(na, nb):
    shells = []
    for k, x in enumerate(np.linspace(0.0, 14.0, 9)):
        for l in range(3):
            n = na if (k + l) % 2 else nb
            shells.append(S.Shell(l, 0.9 * 1.9 ** np.arange(n), np.linspace(1.0, 0.4, n), np.array([x, 0.1 * l, 0.2])))
    sp = S.custom_species("X", shells, n_particles=2)
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    got = {tuple(sorted(p)) for p in h.shellpair_list().tolist()}
    h.close()
    ref = {tuple(sorted(p)) for p in np.asarray(O.shellpair_list(O.Basis(sp))[0]).tolist()}
    assert got == ref
    assert len(ref) < len(shells) * (len(shells) + 1) // 2      # some lie beyond the threshold


@pytest.mark.parametrize("n", [1, 362, 363])        # 362^2 doubles: the last that are staged
def test_host_build_equals_device_build(n):
    sp = S.custom_species("X", [S.Shell(0, np.array([1.1]), np.array([1.0]), np.array([2.5 * k, 0.0, 0.0]))
                                for k in range(n)], n_particles=2)
    rng = np.random.default_rng(n)
    D = (lambda x: x @ x.T)(rng.normal(size=(n, 2)))
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    got = h.compute_2body_intraspecies_direct(D, -0.5)
    dD, dG = H.DeviceArray.from_host(D), H.DeviceArray((n, n))
    h.compute_2body_device(dD.ptr, dG.ptr, -0.5)
    ref = dG.download()
    dD.free()
    dG.free()
    h.close()
    # the order of the atomic sums differs from build to build
    assert np.max(np.abs(got - ref)) < 1e-12 * max(1.0, np.max(np.abs(ref)))
