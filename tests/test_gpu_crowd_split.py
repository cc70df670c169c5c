"""Crowded cells shared by the waves of a deposit workgroup, at the sizes
where the split can go wrong: cells of exactly the most particles one wave
takes (256 here) and one more, parts with no particles, ragged last parts,
one particle past a chunk (1025), several chunks; empty and one-particle
cells beside them; the same on a grid of more than 1024 cells, where a wave
takes twice the injected particles of a cell.  Slices on such a plasma match the oracle on identical
inputs (the bound of the other parity tests: FP64 sums in another order),
and every workgroup shape gives the same bits."""
import numpy as np
import pytest

import twin
from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu

TOL = 1e-10
COUNTS = {1: 256, 2: 257, 4: 511, 7: 513, 8: 1, 11: 1024, 12: 1025, 17: 2300, 39: 300}


# 160 injected per cell of 1030: 320 per wave
COUNTS_MANY = {1: 320, 2: 321, 4: 256, 7: 639, 8: 1, 11: 1024, 12: 1025, 17: 2300, 1000: 511, 1029: 700}


def crowded(g, rng, counts=COUNTS):
    r = np.concatenate([(c + rng.uniform(0.02, 0.98, n)) * g.dr for c, n in counts.items()])
    ph = rng.uniform(0.0, 2.0 * np.pi, r.size)
    n = r.size
    p = {k: 0.1 * rng.standard_normal(n) for k in ("p1", "p2", "p3")}
    gam = np.sqrt(1.0 + p["p1"] ** 2 + p["p2"] ** 2 + p["p3"] ** 2)
    return dict(p, x1=r * np.cos(ph), x2=r * np.sin(ph), q=-rng.uniform(0.5, 1.5, n) * 1e-3, gamma=gam,
                psi=(1.0 - gam + p["p3"]) / -1.0, id=np.arange(n, dtype=np.int32))


# mfma: the form of the sums that is not the mode count's default (None) too
@pytest.mark.parametrize("max_mode,push,mfma", [(0, "robust", None), (1, "standard", None), (2, "robust", None),
                                                (4, "robust", None), (2, "robust", True), (3, "standard", False),
                                                (3, "robust", False), (4, "robust", False)])
def test_split_cells_match_oracle_in_every_shape(max_mode, push, mfma):
    results = []
    for cells in (4, 2, 8):
        # 80 particles per cell injected: 6400 slots, 256 per wave
        sim = Simulation(configs.small(nr=40, nxi=24, max_mode=max_mode, ppc=(2, 40), total_num=1 << 12,
                                       n_peak=6.0, sigma_xi=0.1, offset_x=0.03 if max_mode else 0.0,
                                       push_type=push))
        sim.launch_shape(cells)
        if mfma is not None:
            assert sim.deposit_form(mfma) == mfma
        o = twin.make_twin(sim)
        sim.step3d_begin()
        o.step_begin()
        for j in range(1, 11):
            sim.slice(j)
        sim.spe[0].set(crowded(sim.grid, np.random.default_rng(5)))
        norm = twin.ErrorNorm()
        for j in (11, 12):
            twin.sync_slice_inputs(sim, o, j)
            assert sim.slice(j) == o.slice(j), (cells, j)
            twin.compare_fields(sim, o, norm, j)
            twin.compare_species(sim, o, norm, j)
        assert norm.scale["psi"] > 1e-3, norm.scale["psi"]
        bad = norm.bad(TOL)
        assert not bad, (cells, bad)
        out = {n: sim.fields[n].get() for n in ("psi", "e", "b", "cu", "q_spe")}
        out.update(sim.spe[0].get())
        results.append(out)
        sim.close()
        o.close()
    for other in results[1:]:
        for k in results[0]:
            assert np.array_equal(results[0][k], other[k]), k


@pytest.mark.parametrize("max_mode,mfma", [(0, False), (1, False), (3, True)])
def test_split_cells_of_many_match_oracle_in_every_shape(max_mode, mfma):
    results = []
    for cells in (4, 2, 8):
        sim = Simulation(configs.small(nr=1030, nxi=24, max_mode=max_mode, ppc=(2, 80), total_num=1 << 12, rmax=12.0))
        sim.launch_shape(cells)
        assert sim.deposit_form() == mfma
        o = twin.make_twin(sim)
        sim.step3d_begin()
        o.step_begin()
        sim.spe[0].set(crowded(sim.grid, np.random.default_rng(6), COUNTS_MANY))
        norm = twin.ErrorNorm()
        for j in (1, 2):
            twin.sync_slice_inputs(sim, o, j)
            assert sim.slice(j) == o.slice(j), (cells, j)
            twin.compare_fields(sim, o, norm, j)
            twin.compare_species(sim, o, norm, j)
        assert norm.scale["psi"] > 1e-3, norm.scale["psi"]
        bad = norm.bad(TOL)
        assert not bad, (cells, bad)
        out = {n: sim.fields[n].get() for n in ("psi", "e", "b", "cu", "q_spe")}
        out.update(sim.spe[0].get())
        results.append(out)
        sim.close()
        o.close()
    for other in results[1:]:
        for k in results[0]:
            assert np.array_equal(results[0][k], other[k]), k
