"""Impactors on the outer layer of the box."""
import numpy as np
import pytest

import lbdem
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lbdem.PREC_FP64, lbdem.PREC_FP32, lbdem.PREC_FP16])
@pytest.mark.parametrize("kind", [4, 7], ids=["periodic", "wall"])
@pytest.mark.parametrize("high", [False, True], ids=["low", "high"])
@pytest.mark.parametrize("freesurface", [0, 1])
def test_nodes_left_on_a_z_face(gpu_lib, prec, kind, high, freesurface):
    """An impactor that leaves nodes of a z face behind, next to fluid: they cannot become fluid, as all that
    would stream out of them lies outside the lattice. The run reports a type error, as for a node that
    streams into a periodic layer, keeps reporting it over the steps of a captured chunk, and a later run of
    the same process is untouched."""
    X, Y, Z = 24, 28, 22
    values, _, _ = workloads.impact_box(size=(X, Y, Z), fluid_height=20, n_spheres=0, r=2, r_imp=3, y_imp=12)
    values.update(freeSurfaceSolve=freesurface, boundary0=7, boundary1=7, boundary2=7, boundary3=7, boundary4=kind,
                  boundary5=kind, lbFX=0.0, lbFY=0.0, lbFZ=0.0, objWaitTime=0)
    z0, u = (Z - 2.5, -0.15) if high else (1.5, 0.15)

    def run(z, uz):
        obj = lbdem.ObjectSet(r=np.array([2.7]), x0=np.array([[11.3, 12.2, z]]), x1=np.array([[0.0, 0.0, uz]]))
        sim = lbdem.Simulation(gpu_lib, lbdem.params_from_values(values, prec), lbdem.ParticleSet(), obj)
        sim.init()
        return sim

    sim = run(z0, u)
    with pytest.raises(lbdem.LbdemError, match="code 5"):
        for _ in range(3):
            sim.cycle(17)
            sim.synchronize()
    sim.close()
    sim = run(11.0, u)
    sim.cycle(17)
    sim.synchronize()
    assert np.isfinite(sim.objects()).all() and sim.info()["lbTime"] == 17
    sim.close()
