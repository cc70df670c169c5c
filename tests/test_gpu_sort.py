"""The re-sort by radial cell at the sizes where its forms meet: one
particle, chunk edges of the three chunk shapes (512, 1024 and 2048), the most
chunks whose rows one round of loads sums (8), the most particles of the form
without a scan launch (120 chunks of 512, and 131072 chunk counts) and one
more, the most of the mid form (262144, and 2^20 chunk counts: 131072 in 8192
cells) and one more, 131072 and one more well inside it, cell counts on both sides of the rank
window and of the bins the direct form keeps in LDS.  Particles handed over in
random order spread every chunk over all cells (the ranks taken in turn),
nearly sorted ones stay within the window; some lie outside the box and are
removed.  The order is exact: by cell, then by the order given."""
import numpy as np
import pytest

import twin
from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu


def _ppc(n, nr):
    # species large enough for n particles (npmax = 2 x injected)
    return (1, max(1, -(-n // (2 * nr))))


@pytest.mark.parametrize("nr,n", [(40, 1), (40, 511), (40, 513), (600, 4096), (1100, 16384), (1100, 16385),
                                  (2100, 2049), (4200, 9000), (4200, 70001), (40, 4097), (256, 12288), (1000, 61440),
                                  (1000, 61441), (2100, 31744), (2100, 31745), (600, 131072), (600, 131073),
                                  (600, 262144), (600, 262145), (8192, 131072), (8192, 131073)])
@pytest.mark.parametrize("spread", [False, True])
def test_sort_is_stable_and_complete(nr, n, spread):
    sim = Simulation(configs.small(nr=nr, nxi=2, max_mode=0, ppc=_ppc(n, nr), total_num=16))
    g = sim.grid
    rng = np.random.default_rng(n + nr)
    cell = rng.integers(0, nr + max(nr // 20, 1), n)          # some past the last cell: removed
    if not spread:
        cell = np.sort(cell) + rng.integers(-3, 4, n)
        cell = np.clip(cell, 0, None)
    r = (cell + rng.uniform(0.1, 0.9, n)) * g.dr
    ph = rng.uniform(0.0, 2.0 * np.pi, n)
    z = np.zeros(n)
    ids = np.arange(n, dtype=np.int32)
    sim.spe[0].set({"x1": r * np.cos(ph), "x2": r * np.sin(ph), "p1": 1.0 * ids, "p2": z, "p3": z, "q": -1.0 - ids,
                    "gamma": z + 1.0, "psi": 0.5 * ids, "id": ids})
    got = sim.spe[0].get()
    order = np.argsort(cell, kind="stable")
    order = order[cell[order] < nr]
    assert np.array_equal(got["id"], ids[order])
    for k, v in (("x1", r * np.cos(ph)), ("p1", 1.0 * ids), ("q", -1.0 - ids), ("psi", 0.5 * ids)):
        assert np.array_equal(got[k], v[order]), k
    sim.close()


@pytest.mark.parametrize("ppc,ion_ppc", [((2, 16), None), ((4, 130), None), ((4, 260), None), ((4, 260), (1, 3)),
                                         ((1, 3), (4, 260))])
def test_push_forms_keep_the_sorted_order(ppc, ion_ppc):
    """every push and sort leaves the particles grouped by their new cell, each
    cell in the order its particles had before, and drops exactly those that
    the oracle's push takes out of the box (64 cells: up to 4 x 130 per cell in
    the direct form, 4 x 260 past it, alone and beside a species of few)"""
    sim = Simulation(configs.small(nr=64, nxi=40, max_mode=1, ppc=ppc, total_num=1 << 12, offset_x=0.02,
                                   ions=ion_ppc is not None, ion_ppc=ion_ppc))
    g = sim.grid
    o = twin.make_twin(sim)
    sim.step3d_begin()
    o.step_begin()
    rng = np.random.default_rng(3)
    # momenta that take some particles out of the box in every slice
    for sp in sim.spe:
        p = sp.get()
        for k in ("p1", "p2", "p3"):
            p[k] = 0.4 * rng.standard_normal(len(p[k]))
        p["gamma"] = np.sqrt(1.0 + p["p1"] ** 2 + p["p2"] ** 2 + p["p3"] ** 2)
        sp.set(p)
    lost = 0
    for j in range(1, 5):
        before = [sp.get()["id"] for sp in sim.spe]
        twin.sync_slice_inputs(sim, o, j)
        sim.slice(j)
        o.slice(j)
        for s, sp in enumerate(sim.spe):
            p = sp.get()
            kept = np.array(o.species(s)["id"])
            assert np.array_equal(np.sort(p["id"]), np.sort(kept)), (j, s)
            assert len(np.unique(p["id"])) == len(p["id"])
            lost += len(before[s]) - len(kept)
            c = (np.hypot(p["x1"], p["x2"]) / g.dr).astype(int)
            assert np.all(np.diff(c) >= 0) and c.max() < g.nr
            place = np.empty(before[s].max() + 1, dtype=int)
            place[before[s]] = np.arange(len(before[s]))
            assert np.array_equal(p["id"], p["id"][np.lexsort((place[p["id"]], c))]), (j, s)
    assert lost > 0
    sim.close()
    o.close()


def test_species_without_particles_on_a_large_grid():
    """a gas that has released nothing yet, on a grid past the direct form's
    bins: its push and sort launch for no particles"""
    sim = Simulation(configs.ionization(nr=4200, nxi=6, max_mode=0, total_num=1 << 10, n_peak=1e-3))
    sim.step3d()
    assert sim.neut[0].count() == 0
    sim.close()
