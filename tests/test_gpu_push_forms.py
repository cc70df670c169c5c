"""The push past the form of the re-sort for few particles (more than 120
chunks of 512) for the pushers that the smaller decks run in that form only:
standard, laser (robust and standard), sub-cycled with the clamp active; and
species whose counts would put them in different forms, with one pusher and
with two (they share the sort, the slice's epilogue rides with the first of the
push launches).  Slices match the oracle on identical inputs."""
import pytest

import twin
from qpad_amd import Simulation, configs
from qpad_amd.input import subcycling_from_deck

pytestmark = pytest.mark.gpu

TOL = 1e-10
MANY, FEW = (4, 260), (1, 3)   # per cell of 64: 66,560 and 192 particles


def deck(push, ions=False, ppc=MANY, ion_ppc=None, ion_push=None, max_mode=1):
    return configs.small(nr=64, nxi=24, max_mode=max_mode, ppc=ppc, total_num=1 << 12, n_peak=6.0, sigma_xi=0.1,
                         offset_x=0.03, push_type=push, ions=ions, ion_ppc=ion_ppc, ion_push_type=ion_push)


def run(d, slices, laser=False):
    sim = Simulation(d)
    o = twin.make_twin(sim)
    sub = subcycling_from_deck(d)
    if sub is not None:
        o.set_subcycling(*sub)
    if laser:
        ar, ai = twin.laser_envelope(sim.grid, sim.nm, a0=1.0, length=0.3)
        sim.set_laser(ar, ai)
        o.set_laser(ar, ai)
    sim.step3d_begin()
    o.step_begin()
    norm = twin.ErrorNorm()
    subs = []
    for j in range(1, slices + 1):
        twin.sync_slice_inputs(sim, o, j)
        assert sim.slice(j) == o.slice(j), j
        if sub is not None:
            subs.append(sim.last_subcycles()[0])
        twin.compare_fields(sim, o, norm, j)
        twin.compare_species(sim, o, norm, j)
    print({n: f"{e:.1e}" for n, e in sorted(norm.errors().items())})
    bad = norm.bad(TOL)
    assert not bad, bad
    counts = [sp.count() for sp in sim.spe]
    sim.close()
    o.close()
    return norm, subs, counts


@pytest.mark.parametrize("push,max_mode", [("robust", 3), ("standard", 1), ("standard", 2), ("robust_pgc", 1),
                                           ("standard_pgc", 0)])
def test_many_particles_match_oracle(push, max_mode):
    d = deck(push, max_mode=max_mode)
    if max_mode == 0:
        d["beam"][0]["gauss_center"][0] = 0.0
    norm, _, counts = run(d, 13, laser=push.endswith("pgc"))
    assert counts[0] > 120 * 512 and norm.scale["psi"] > 1e-3


@pytest.mark.parametrize("push", ["robust", "standard"])
def test_many_particles_subcycled_match_oracle(push):
    d = configs.subcycling(nr=64, push_type=push)
    d["species"][0].update({"ppc": [MANY[0], 1], "num_theta": MANY[1]})
    norm, subs, counts = run(d, 24)
    assert counts[0] > 120 * 512 and max(subs) >= 2, subs


@pytest.mark.parametrize("ppc,ion_ppc,push,ion_push", [
    (MANY, FEW, "robust", "robust"), (FEW, MANY, "robust", "robust"), (FEW, MANY, "robust", "standard"),
    (MANY, FEW, "standard", "robust"), (FEW, MANY, "robust_pgc", "robust")])
def test_species_of_different_forms_match_oracle(ppc, ion_ppc, push, ion_push):
    run(deck(push, ions=True, ppc=ppc, ion_ppc=ion_ppc, ion_push=ion_push, max_mode=2), 13,
        laser=push.endswith("pgc"))
