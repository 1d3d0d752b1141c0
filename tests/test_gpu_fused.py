"""Small builds run as one launch over all quartet classes: against the class
launches (forced by serialising them) on the same handle, for one and many
molecules, screened and unscreened species, and against the oracle."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle as O  # noqa: E402

from openlowdin_amd import batch as B  # noqa: E402
from openlowdin_amd import hip as H  # noqa: E402
from openlowdin_amd import libint2_interface as LI  # noqa: E402
from openlowdin_amd import system as S  # noqa: E402

pytestmark = pytest.mark.gpu


def _density(sp, seed, nocc=3):
    rng = np.random.default_rng(seed)
    C = rng.normal(size=(sp.nbasis, min(nocc, sp.nbasis))) / np.sqrt(sp.nbasis)
    return 2.0 * C @ C.T


def _one_s():
    return S.custom_species("X", [S.Shell(0, np.array([0.8]), np.array([1.0]), np.zeros(3))], n_particles=2)


def _species(name):
    return {"one s function": _one_s,
            "proton": lambda: S.fhf_anion("6-31G").species[1],
            "FHF electrons": lambda: S.fhf_anion("6-311++G**").species[0],
            "water": lambda: S.water("6-31G**").species[0],
            "water trimer": lambda: S.water_cluster(3, np.random.default_rng(2), "cc-pVDZ").species[0]}[name]()


@pytest.mark.parametrize("name", ["one s function", "proton", "FHF electrons", "water", "water trimer"])
def test_one_launch_equals_class_launches_and_oracle(name):
    sp = _species(name)
    h = LI.Libint2Interface(sp, 1)
    h.init_2body_ints()
    for seed in (1, 2):
        D = _density(sp, seed)
        dD, dG = H.DeviceArray.from_host(np.ascontiguousarray(D)), H.DeviceArray((sp.nbasis, sp.nbasis))
        h.serialize_launches(False)
        h.compute_2body_device(dD.ptr, dG.ptr, -0.5)
        one, st = dG.download(), h.stats()
        h.serialize_launches(True)
        h.compute_2body_device(dD.ptr, dG.ptr, -0.5)
        many, st2 = dG.download(), h.stats()
        # the same quartets in another summation order: a few ulp of the sums
        assert np.max(np.abs(one - many)) < 1e-12 * max(1.0, np.max(np.abs(many)))
        for k in ("quartets", "eris", "prim_quartets"):
            assert st[k] == st2[k], (k, st, st2)
        if sp.nbasis <= 50:
            ref = O.compute_2body_direct(O.Basis(sp), D, -0.5)
            assert np.max(np.abs(one - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    h.close()


@pytest.mark.parametrize("graph", [False, True])
def test_small_batch_equals_single_builds(graph):
    rng = np.random.default_rng(5)
    sps = [S.water_cluster(int(k), rng).species[0] for k in (1, 2, 1)] + [S.fhf_anion("6-31G").species[1]]
    Ds = [_density(sp, 3 + k) for k, sp in enumerate(sps)]
    fb = B.FockBatch.from_species(sps, [-0.5, -0.5, -1.0, -1.0])
    fb.options(use_graph=graph)
    for _ in range(3):
        Gs = fb.compute(Ds)
    for sp, D, f, G in zip(sps, Ds, [-0.5, -0.5, -1.0, -1.0], Gs):
        ref = O.compute_2body_direct(O.Basis(sp), D, f)
        assert np.max(np.abs(G - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    fb.close()
