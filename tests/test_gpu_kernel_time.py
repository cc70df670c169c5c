"""The push timer counts launches that push: none for a gas that has released
nothing (in either form of the re-sort, on both sides of 4096 cells), one per
slice for species of one pusher whatever forms their counts would take by
themselves, one per pusher."""
import pytest

from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr", [48, 4200])
def test_no_push_no_launch_timed(nr):
    sim = Simulation(configs.ionization(nr=nr, nxi=6, max_mode=0, total_num=1 << 10, n_peak=1e-3))
    sim.kernel_time_reset(True)
    sim.step3d()
    ms, n = sim.kernel_time(1)
    assert sim.neut[0].count() == 0
    assert (ms, n) == (0.0, 0)
    assert sim.kernel_time(0)[1] == 6
    sim.close()


@pytest.mark.parametrize("ions,ion_ppc,ion_push,per_slice", [
    (False, None, None, 1), (True, (2, 4), None, 1), (True, (8, 130), None, 1), (True, (8, 130), "standard", 2)])
def test_one_push_launch_per_pusher(ions, ion_ppc, ion_push, per_slice):
    # 64 cells: 2 x 4 per cell direct, 8 x 130 past its 120 chunks of 512
    sim = Simulation(configs.small(nr=64, nxi=6, max_mode=1, ppc=(2, 4), total_num=1 << 10, ions=ions, ion_ppc=ion_ppc,
                                   ion_push_type=ion_push))
    sim.kernel_time_reset(True)
    sim.step3d()
    ms, n = sim.kernel_time(1)
    assert n == 6 * per_slice and ms > 0.0
    sim.close()
