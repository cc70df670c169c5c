"""The two deposits that gather per node, at the sizes where their split can
go wrong.  Beam: node counts around the tile of 64 (nr + 2 = 63, 64, 65, 129),
cells of more than one round of 16 particles beside empty ones, two beams of
different size, every mode count; tiles of slices reached by no particle, by one, by the most
of the sparse form (512) and one more; every slice of the deposited charge
matches the oracle's for the same particles (FP64 sums in another order).  Ions of a
gas: theta bins below, at and past the 32 a wave takes at once, every mode
count."""
import numpy as np
import pytest

import twin
from conftest import rel_err
from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize("nr,max_mode,two", [(61, 0, True), (62, 1, False), (63, 2, True), (127, 3, False),
                                             (62, 4, True), (61, 1, True)])
def test_beam_charge_matches_oracle(nr, max_mode, two):
    deck = configs.small(nr=nr, nxi=20, max_mode=max_mode, total_num=1 << 15, sigma_r=0.2, sigma_xi=0.1,
                         offset_x=0.05 if max_mode else 0.0)
    if two:
        second = dict(deck["beam"][0], total_num=700, gauss_sigma=[0.6, 0.6, 0.2])
        deck["beam"].append(second)
        deck["simulation"]["nbeams"] = 2
    sim = Simulation(deck)
    cells = np.floor(np.hypot(sim.beam[0].get()["x1"], sim.beam[0].get()["x2"]) / sim.grid.dr)
    assert np.bincount(cells.astype(int)).max() > 20 * 16
    o = twin.make_twin(sim)
    sim.step3d_begin()
    o.step_begin()
    got = np.stack([sim.fields["q_beam"].hist(j) for j in range(1, sim.grid.nxi + 2)])
    ref = o.hist(twin.ORA_ID["q_beam"])[1:sim.grid.nxi + 2]
    e = rel_err(got, ref)
    assert np.max(np.abs(ref)) > 1e-3 and e <= TOL, e
    sim.close()
    o.close()


@pytest.mark.parametrize("nr,max_mode", [(62, 0), (127, 1), (190, 2), (127, 3), (127, 4)])
@pytest.mark.parametrize("two", [False, True])
def test_beam_charge_on_both_sides_of_the_sparse_form(nr, max_mode, two):
    deck = configs.small(nr=nr, nxi=24, max_mode=max_mode, total_num=1 << 13, sigma_r=0.3, sigma_xi=0.1)
    if two:
        deck["beam"].append(dict(deck["beam"][0], total_num=1 << 13))
        deck["simulation"]["nbeams"] = 2
    sim = Simulation(deck)
    g = sim.grid
    rng = np.random.default_rng(nr + max_mode)
    # particles of xi cell mm: n of them in the r cells lo .. hi - 1
    plans = [[(0, 3, 0, 2), (3, 512, 0, 60), (7, 513, 0, 60), (11, 1, nr - 1, nr), (12, 400, 5, 6), (15, 112, 5, 9),
              (16, 400, 5, 9), (17, 1, 20, 21), (20, 900, 0, 62), (23, 5, nr - 3, nr)],
             [(3, 1, 30, 31), (7, 700, 10, 12), (12, 4, 0, 62), (13, 5, 40, 41), (20, 17, 61, 62)]]
    for b, plan in zip(sim.beam, plans):
        mm = np.concatenate([np.full(n, m) for m, n, _, _ in plan])
        r = np.concatenate([rng.integers(lo, hi, n) for _, n, lo, hi in plan]) + rng.uniform(0.02, 0.98, mm.size)
        ph = rng.uniform(0.0, 2.0 * np.pi, mm.size)
        z = np.zeros(mm.size)
        b.set({"x1": r * g.dr * np.cos(ph), "x2": r * g.dr * np.sin(ph), "x3": (mm + rng.uniform(0.02, 0.98, mm.size)) * g.dxi,
               "p1": z, "p2": z, "p3": z + 2e4, "q": -rng.uniform(0.5, 1.5, mm.size)})
    o = twin.make_twin(sim)
    sim.step3d_begin()
    o.step_begin()
    got = np.stack([sim.fields["q_beam"].hist(j) for j in range(0, g.nxi + 2)])
    ref = o.hist(twin.ORA_ID["q_beam"])[0:g.nxi + 2]
    for j in range(1, g.nxi + 2):
        scale = np.max(np.abs(ref[j]))
        assert np.max(np.abs(got[j] - ref[j])) <= TOL * scale, j
        assert (scale == 0.0) == (np.max(np.abs(got[j])) == 0.0), j
    assert np.count_nonzero(np.max(np.abs(ref.reshape(g.nxi + 2, -1)), axis=1)) > 12
    sim.close()
    o.close()


@pytest.mark.parametrize("num_theta,max_mode", [(1, 0), (31, 1), (32, 2), (33, 4), (70, 3)])
def test_ion_charge_matches_oracle(num_theta, max_mode):
    sim = Simulation(configs.ionization(nr=30, nxi=24, max_mode=max_mode, num_theta=num_theta, n0=1e18, n_peak=8.0,
                                        offset_x=0.03 if max_mode else 0.0))
    o = twin.make_twin(sim)
    sim.step3d_begin()
    o.step_begin()
    nt = sim.neut[0]
    got, ref = [], []
    for j in range(1, sim.grid.nxi + 1):
        twin.sync_slice_inputs(sim, o, j)
        assert sim.slice(j) == o.slice(j), j
        got.append(nt.ion_density(j))
        ref.append(np.array(o.neutral_rho_hist(nt.id)[j]))
    assert nt.count() > 0
    e = rel_err(np.stack(got), np.stack(ref))
    assert e <= TOL, e
    sim.close()
    o.close()
