"""Node counts of lbdem_get_info (one pass over words of four type bytes, the tail by byte) against
the downloaded types, on boxes whose node count leaves every remainder by four, and on a box of the
smallest size."""
import numpy as np
import pytest

import cases
import lbdem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(3, 3, 3), (5, 5, 5), (10, 11, 7), (9, 7, 9), (13, 19, 17), (64, 65, 33)])
def test_node_counts_equal_the_types(gpu_lib, size):
    vals, *_ = cases._case_values("fs_impactor" if min(size) > 12 else "lb_closed")
    vals.update(lbSizeX=float(size[0]), lbSizeY=float(size[1]), lbSizeZ=float(size[2]), fluidHeight=0.6 * size[1])
    ps, obs = lbdem.ParticleSet(), lbdem.ObjectSet()
    if min(size) > 12:
        ps = lbdem.ParticleSet(size=np.ones(2, np.int32), r=np.array([1.7, 2.0]), x0=np.array([[4.0, 4.1, 4.2], [8.3, 4.9, 8.0]]))
        obs = lbdem.ObjectSet(r=np.array([2.5]), x0=np.array([[6.1, 0.6 * size[1] + 1.0, 6.3]]), x1=np.array([[0.0, -0.02, 0.0]]))
    sim = lbdem.Simulation(gpu_lib, lbdem.params_from_values(vals, lbdem.PREC_FP64), ps, obs)
    sim.init()
    for steps in (0, 3):
        sim.cycle(steps)
        t, p, _ = sim.types()
        i = sim.info()
        assert i["totNodes"] == size[0] * size[1] * size[2] == len(t)
        assert i["nFluid"] == int((t == 0).sum()) and i["nInterface"] == int((t == 3).sum())
        assert i["nObjectNodes"] == int((t == 12).sum()) and i["nParticleNodes"] == int(p.sum())
        assert i["nActive"] == i["nFluid"] + i["nInterface"]
    sim.close()
