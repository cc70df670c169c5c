"""The push decides a particle's cell from the position it stores, also where
that lies within a rounding of a cell border: the launch that counts the cells
and the one that moves the particles must not each round for themselves.  The
start positions are corrected until the pushed radius hits a border to a few
ulp, then varied by ulps; after every push the particles stand in the order of
the cells that their stored positions give: handed back as they are, their
cells are computed anew and the (stable) sort leaves every one in its place."""
import numpy as np
import pytest

from qpad_amd import Simulation, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("push", ["robust", "standard", "robust_pgc", "standard_pgc"])
@pytest.mark.parametrize("max_mode,n,ppc", [(0, 12000, (2, 60)), (1, 12000, (2, 60)), (2, 12000, (2, 60)),
                                            (4, 12000, (2, 60)), (1, 70000, (4, 160))])
def test_stored_position_is_in_the_sorted_cell(max_mode, n, ppc, push):
    nr, dxi = 100, 0.05
    sim = Simulation(configs.small(nr=nr, nxi=4, max_mode=max_mode, ppc=ppc, total_num=16, dxi=dxi, push_type=push))
    g = sim.grid
    rng = np.random.default_rng(7 * max_mode + n)
    for name in ("e", "b") + (("ar", "ai", "ar_grad", "ai_grad") if push.endswith("pgc") else ()):
        sim.fields[name].set(0.3 * rng.standard_normal(sim.fields[name].shape()))
    border = rng.integers(2, nr - 2, n) * g.dr
    ph = rng.uniform(0.0, 2.0 * np.pi, n)
    x1, x2 = border * np.cos(ph), border * np.sin(ph)
    p = {k: 0.2 * rng.standard_normal(n) for k in ("p1", "p2", "p3")}
    gam = np.sqrt(1.0 + p["p1"] ** 2 + p["p2"] ** 2 + p["p3"] ** 2)
    start = dict(p, q=-np.ones(n), gamma=gam, psi=(1.0 - gam + p["p3"]) / -1.0, id=np.arange(n, dtype=np.int32))
    near = 0
    for it in range(24):
        sim.spe[0].set(dict(start, x1=x1, x2=x2))
        sim.spe[0].push(dxi)
        got = sim.spe[0].get()
        r = np.sqrt(got["x1"] * got["x1"] + got["x2"] * got["x2"])
        assert len(np.unique(got["id"])) == len(r) == n
        sim.spe[0].set(got)
        again = sim.spe[0].get()
        moved = int(np.sum(again["id"] != got["id"]))
        assert moved == 0, (it, moved)
        d = border[got["id"]] - r
        near = max(near, int(np.sum(np.abs(d) <= 4 * np.spacing(r))))
        if it < 12:
            x1[got["id"]] += d * got["x1"] / r
            x2[got["id"]] += d * got["x2"] / r
        else:
            x1 = x1 + rng.integers(-2, 3, n) * np.spacing(x1)
    assert near > n // 4, near
    sim.close()
