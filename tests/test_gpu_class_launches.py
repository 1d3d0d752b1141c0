"""Class launches where the default route would be one launch: lanes sharing a
quartet in strips of one, two and four wavefronts, captured graphs of a build
and of the batched SCF's iteration, each on plans that are not fused."""
import numpy as np
import pytest

import oracle as O
from openlowdin_amd import batch as B
from openlowdin_amd import hip as H
from openlowdin_amd import libint2_interface as LI
from openlowdin_amd import system as S

pytestmark = pytest.mark.gpu


def _density(sp, seed, nocc=3):
    X = np.random.default_rng(seed).normal(size=(sp.nbasis, min(nocc, sp.nbasis))) / np.sqrt(sp.nbasis)
    return 2.0 * X @ X.T


def _contracted(nprim, centres, lmax):
    e = 0.05 * 2.1 ** np.arange(nprim)
    return S.custom_species("X", [S.Shell(l, e * (1 + 0.1 * l), np.linspace(1.0, 0.2, nprim), np.array(c, float))
                                  for c in centres for l in range(lmax + 1)], n_particles=2)


def _line(nshell, nprim):
    """Contracted s shells on a line (kets) and two p and d shells (bras)."""
    e = 0.4 * 2.5 ** np.arange(nprim)
    shells = [S.Shell(0, e * (1 + 0.01 * k), np.linspace(1.0, 0.4, nprim), np.array([0.35 * k, 0.1 * (k % 3), 0.0]))
              for k in range(nshell)]
    for l in (1, 2):
        for k in range(2):
            shells.append(S.Shell(l, e, np.linspace(0.8, 0.5, nprim), np.array([1.1 * k, 0.4, 0.2 * l])))
    return S.custom_species("X", shells, n_particles=2)


SPECIES = {
    "one shell, 9 primitives": lambda: _contracted(9, [(0, 0, 0)], 0),                       # not staged
    "8 primitives": lambda: _contracted(8, [(0, 0, 0), (0.4, 1.1, -0.3)], 1),                # 64 lanes to a quartet
    "5 primitives, d": lambda: _contracted(5, [(0, 0, 0), (0.4, 1.1, -0.3), (1.7, 0, 0.2)], 2),
    "butane": lambda: S.build_system(S.alkane_geometry(4), "cc-pVDZ").species[0],
    "192 kets per bra": lambda: _line(22, 3),      # (xx|ss) of 253 kets: two wavefronts
    "2000 kets per bra": lambda: _line(64, 3),     # (ps|ss) of 2080 kets: four
}


@pytest.mark.parametrize("serial", [True, False], ids=["one stream", "four streams"])
@pytest.mark.parametrize("name", list(SPECIES))
def test_lanes_share_quartets_in_class_launches(name, serial):
    sp = SPECIES[name]()
    D = _density(sp, 11)
    h = LI.Libint2Interface(sp, 1)
    (h.serialize_launches if serial else h.time_launches)(True)      # one launch per class, whatever the size
    G = h.compute_2body_intraspecies_direct(D, 0.3)
    h.close()
    ref = O.compute_2body_direct(O.Basis(sp), D, 0.3)
    # the suite's bound of an FP64 build: 1e-10 absolute at integrals of order one
    assert np.max(np.abs(G - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))


def _clusters(sizes, tau=0.0):
    sps = [S.water_cluster(k, np.random.default_rng(k)).species[0] for k in sizes]
    hs = [LI.Libint2Interface(sp, 1) for sp in sps]
    if tau:
        hs[-1].set_precision("mixed", tau)
    fb = B.FockBatch(hs, [-0.5] * len(sps))
    quartets = sum(0.5 * len(h.shellpair_list()) ** 2 for h in hs)
    assert tau or quartets > 6.0e6      # one launch stops at 4e6
    return sps, fb


@pytest.mark.parametrize("tau", [0.0, 1e-4], ids=["fp64", "one mixed"])
def test_graph_replays_follow_eager_builds(tau):
    sps, fb = _clusters((4, 6, 8), tau)
    dD, dG = H.DeviceArray((fb.packed_size,)), H.DeviceArray((fb.packed_size,))
    packed = [fb.pack([_density(sp, 7 * s + k) for k, sp in enumerate(sps)]) for s in range(3)]

    def build(graph):
        fb.options(use_graph=graph)
        dG.upload(np.full(fb.packed_size, 7.0))          # eager work between the replays
        fb.compute_device(dD.ptr, dG.ptr)
        return dG.download()

    for factor in (-0.5, 0.3):
        fb.factors[:] = factor
        for P in packed:
            dD.upload(P)
            eager = build(False)
            for replay in range(3):
                got = build(True)
                # the same quartets, summed in another order
                assert np.max(np.abs(got - eager)) < 1e-12 * max(1.0, np.max(np.abs(eager))), (factor, replay)
    # tasks rebuilt: the next replay is of a new capture
    h = fb.handles[0]
    h.set_precision("mixed", 1e-4)
    eager = build(False)
    assert np.max(np.abs(build(True) - eager)) < 1e-12 * max(1.0, np.max(np.abs(eager)))
    fb.close()


def test_batched_scf_graphs_on_class_launches():
    from openlowdin_amd import scf_batch as SB
    from openlowdin_amd import scf_device as SD
    systems = [S.water_cluster(k, np.random.default_rng(20 + k)) for k in (3, 5, 6, 7)]
    pairs = 0.0
    for s in systems:
        h = LI.Libint2Interface(s.species[0], 1)
        h.init_2body_ints()
        pairs += 0.5 * len(h.shellpair_list()) ** 2
        h.close()
    assert pairs > 6.0e6
    res = SB.run_batch(systems, e_tol=1e-10, d_tol=1e-8, max_iter=60)
    for s, (E, it, conv) in zip(systems, res):
        assert conv
        one = SD.DeviceSCF(s)
        ref = one.run(60, 1e-10, 1e-8)
        one.close()
        # both stop at a step below 1e-10
        assert abs(E - ref) < 1e-9
