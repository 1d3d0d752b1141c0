"""Builds with few quartets but many functions (molecules far apart): the route
a build takes by default is not slower than its class launches, and the result
is the oracle's."""
import time

import numpy as np
import pytest

import oracle as O
from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _apart(k, gap=14.0):
    atoms = []
    for i in range(k):
        shift = (gap * (i % 3), gap * (i // 3 % 3), gap * (i // 9))
        atoms += [(el, tuple(np.add(x, shift))) for el, x in S.WATER_ANGSTROM]
    return S.build_system(atoms, "6-31G**").species[0]


# one to four workgroups of a single launch in a CU's LDS
@pytest.mark.parametrize("k", [12, 16, 24, 27])
def test_default_route_is_not_the_slower_one(k):
    sp = _apart(k)
    n = sp.nbasis
    X = np.random.default_rng(k).normal(size=(n, 5)) / np.sqrt(n)
    D = 2.0 * X @ X.T
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    dD, dG = H.DeviceArray.from_host(D), H.DeviceArray((n, n))
    least, got = {}, {}
    for classes in (False, True):
        h.time_launches(classes)        # times each class launch, so that there is one per class
        for _ in range(3):
            h.compute_2body_device(dD.ptr, dG.ptr, -0.5)
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            h.compute_2body_device(dD.ptr, dG.ptr, -0.5)
            t.append(time.perf_counter() - t0)
        least[classes], got[classes] = min(t), dG.download()
    h.close()
    assert least[False] < 1.25 * least[True], least
    assert np.max(np.abs(got[False] - got[True])) < 1e-12 * max(1.0, np.max(np.abs(got[True])))
    if k == 12:
        ref = O.compute_2body_direct(O.Basis(sp), D, -0.5)
        assert np.max(np.abs(got[False] - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
