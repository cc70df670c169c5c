"""The source kernel of the iteration is compiled per mode count and species
count and works on tiles of 16 nodes with a halo of 2: slices at every mode
count and with one and two species, with the last tile full, one node over,
one short and holding only the edge nodes (nr + 2 = 16, 17, 31, 32, 33, 34),
match the oracle on identical inputs (the bound of the other parity tests:
FP64 sums in another order)."""
import pytest

import twin
from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize("max_mode,ions,nr", [(0, False, 14), (0, True, 31), (1, False, 15), (1, True, 32), (2, False, 29),
                                              (2, True, 30), (3, False, 31), (3, True, 14), (4, False, 32), (4, True, 15)])
def test_slices_match_oracle_at_tile_edges(max_mode, ions, nr):
    sim = Simulation(configs.small(nr=nr, nxi=24, max_mode=max_mode, ppc=(2, 12), total_num=1 << 12, n_peak=6.0,
                                   sigma_xi=0.1, offset_x=0.03 if max_mode else 0.0, ions=ions, ion_ppc=(1, 10)))
    o = twin.make_twin(sim)
    sim.step3d_begin()
    o.step_begin()
    norm = twin.ErrorNorm()
    for j in range(1, 15):
        twin.sync_slice_inputs(sim, o, j)
        assert sim.slice(j) == o.slice(j), j
        twin.compare_fields(sim, o, norm, j)
        twin.compare_species(sim, o, norm, j)
    sim.close()
    o.close()
    assert norm.scale["psi"] > 1e-3, norm.scale["psi"]
    bad = norm.bad(TOL)
    assert not bad, bad
