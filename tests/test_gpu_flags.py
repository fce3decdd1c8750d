"""Particle flags between list rebuilds against the oracle: the lowest sphere leaves the box through the
periodic z face on a step that keeps the flags, so that the lowest flagged node is searched for across
the empty part of the box, up to the next sphere (some 90 000 nodes on) or, with one sphere, to the end."""
import numpy as np
import pytest

import cases
import lbdem
import workloads
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(40, 44, 72), (41, 43, 71)])
@pytest.mark.parametrize("spheres", [1, 2])
def test_lowest_sphere_leaves_through_the_seam(oracle_lib, gpu_lib, size, spheres):
    X, Y, Z = size
    v, _, _ = workloads.impact_box(size=size, fluid_height=30.0, n_spheres=0, r=2.5, r_imp=4.0, y_imp=33.0, speed=0.01,
                                   periodic=True)
    v.update(lbFZ=-1.5e-3)
    x0 = np.array([[12.3, 8.2, 0.16], [25.0, 9.1, 52.0]])[:spheres]
    ps = lbdem.ParticleSet(size=np.ones(spheres, np.int32), r=np.full(spheres, 2.5), x0=x0)
    obs = lbdem.ObjectSet(r=np.array([4.0]), x0=np.array([[20.0, 33.0, 30.0]]), x1=np.array([[0.0, -0.01, 0.0]]))
    a, b, c = (lbdem.Simulation(lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, obs)
               for lib in (oracle_lib, gpu_lib, gpu_lib))
    for s in (a, b, c):
        s.init()
    kept = False
    flags = cases.state(a)["pflag"]
    for k in range(20):
        builds = a.info()["neighborListBuilds"]
        a.cycle(1)
        b.cycle(1)
        for step in (c.dem_step, c.coupling_step, c.lb_step, c.fs_step):  # the coupling ends by itself
            step()
        A = cases.state(a)
        low = flags.nonzero()[0].min(initial=flags.size)
        kept |= a.info()["neighborListBuilds"] == builds and flags[low:].any() and not A["pflag"][low:low + 10 * X * Y].any()
        flags = A["pflag"]
        compare(A, cases.state(b), lbdem.PREC_FP64, f"step {k + 1}")
        compare(A, cases.state(c), lbdem.PREC_FP64, f"sub-steps of step {k + 1}")
    assert kept, "no step searched"
    for s in (a, b, c):
        s.close()


def test_list_rebuild_waits_for_the_coupling(oracle_lib, gpu_lib):
    """Sub-step calls with the coupling on the first and every third step after it: a list rebuild of a step without one has its
    flags made by the next coupling, as the reference's flag of a new list stays set until then."""
    v, ps, _ = workloads.impact_box(size=(30, 34, 26), fluid_height=18.0, n_spheres=14, r=2.0, r_imp=4.0, y_imp=22.5,
                                    seed=5, relax=60, periodic=True, bed_top=14.0)
    v.update(lbFZ=-1.5e-3)
    a, b = (lbdem.Simulation(lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, lbdem.ObjectSet())
            for lib in (oracle_lib, gpu_lib))
    a.init()
    b.init()
    waited = 0
    for k in range(36):
        for s in (a, b):
            s.dem_step()
            if k % 3 == 0:
                s.coupling_step()
            s.lb_step()
            s.fs_step()
        assert a.info()["newNeighborList"] == b.info()["newNeighborList"], k
        waited += k > 2 and a.info()["newNeighborList"]
        compare(cases.state(a), cases.state(b), lbdem.PREC_FP64, f"step {k + 1}")
    assert waited >= 4
    a.close()
    b.close()
