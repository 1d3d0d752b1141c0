"""Strip launches of one, two and four wavefronts per workgroup, on both sides
of the mean kets per bra at which the width changes, against the oracle."""
import numpy as np
import pytest

import oracle as O
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _spread(nshell, lmax, npairs_far):
    """s shells by the dozen (kets), a few higher shells (bras), one line."""
    shells = [S.Shell(0, np.array([0.4 + 0.01 * k]), np.array([1.0]), np.array([0.35 * k, 0.1 * (k % 3), 0.0]))
              for k in range(nshell)]
    for l in range(1, lmax + 1):
        for k in range(npairs_far):
            shells.append(S.Shell(l, np.array([0.7, 0.2]), np.array([0.6, 0.5]), np.array([1.1 * k, 0.4, 0.2 * l])))
    return S.custom_species("X", shells, n_particles=2)


# mean kets per bra of the (xx|ss) classes: nshell (nshell + 1) / 2, with the
# changes at 192, 1000 and 2000
@pytest.mark.parametrize("nshell,lmax", [(18, 1), (20, 2), (45, 1), (64, 1)])
def test_strip_widths_equal_oracle(nshell, lmax):
    sp = _spread(nshell, lmax, 2)
    n = sp.nbasis
    rng = np.random.default_rng(nshell)
    D = (lambda x: x @ x.T)(rng.normal(size=(n, 3)) / np.sqrt(n))
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    h.serialize_launches(True)          # class launches, whatever the size
    got = h.compute_2body_intraspecies_direct(D, -0.5)
    h.close()
    ref = np.asarray(O.compute_2body_direct(O.Basis(sp), D, -0.5)).reshape(n, n)
    # the suite's 1e-10 for matrices of order one
    assert np.max(np.abs(got - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
