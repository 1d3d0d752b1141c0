"""The build without allocation inside a captured graph: one launch (water) and
class launches over the side streams (C7H16), captured at the first call and
replayed with new densities, eager builds and synchronisations between."""
import ctypes as C

import numpy as np
import pytest

from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["C7H16", "water"])
def test_captured_build_follows_the_density(name):
    sp = S.water("6-31G**").species[0] if name == "water" else S.alkane(7).species[0]
    n = sp.nbasis
    Ds = [(lambda x: 2.0 * x @ x.T)(np.random.default_rng(k).normal(size=(n, 4)) / np.sqrt(n)) for k in range(3)]
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    assert (0.5 * len(h.shellpair_list()) ** 2 > 6.0e6) == (name == "C7H16")     # one launch stops at 4e6
    dD, dG, dE = H.DeviceArray.from_host(Ds[0]), H.DeviceArray((n, n)), H.DeviceArray((n, n))
    h.compute_2body_device(dD.ptr, dE.ptr, -0.5)
    L, st = H.hip(), H.Stream()
    g, ex = C.c_void_p(), C.c_void_p()
    H.check(L.hipStreamBeginCapture(C.c_void_p(st.handle), 2), "hipStreamBeginCapture")   # relaxed
    rc = LI.lib().lowdin_fock_compute_2body_device_noalloc(h.this, C.c_void_p(dD.ptr), C.c_void_p(dG.ptr), -0.5,
                                                          C.c_void_p(st.handle))
    H.check(L.hipStreamEndCapture(C.c_void_p(st.handle), C.byref(g)), "hipStreamEndCapture")
    assert rc == 0, LI.lib().lowdin_fock_last_error()
    H.check(L.hipGraphInstantiate(C.byref(ex), g, None, None, C.c_size_t(0)), "hipGraphInstantiate")
    for D in Ds + Ds:
        dD.upload(D)
        dG.upload(np.full((n, n), 7.0))
        h.compute_2body_device(dD.ptr, dE.ptr, -0.5)
        H.check(L.hipGraphLaunch(ex, C.c_void_p(st.handle)), "hipGraphLaunch")
        st.synchronize()
        ref = dE.download()
        # the same quartets, summed in another order
        assert np.max(np.abs(dG.download() - ref)) < 1e-12 * max(1.0, np.max(np.abs(ref)))
    H.check(L.hipGraphExecDestroy(ex), "hipGraphExecDestroy")
    H.check(L.hipGraphDestroy(g), "hipGraphDestroy")
    h.close()
