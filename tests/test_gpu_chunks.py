"""Chunks of captured steps against the same steps launched one by one and against the sub-step calls, in
4- and 2-byte storage, with slip and moving walls, rheology models and the stress diagnostics
(test_gpu_steps has the same in FP64 without them). The two sides run the same operations, so the
tolerances of test_gpu_parity against the FP64 oracle leave room for the order of the atomic sums alone."""
import pytest

import cases
import lbdem
from test_gpu_parity import compare, compare_particle_stress, compare_stress

pytestmark = pytest.mark.gpu

FP64, FP32, FP16 = lbdem.PREC_FP64, lbdem.PREC_FP32, lbdem.PREC_FP16


@pytest.mark.parametrize("name,prec,stress", [
    ("suspension", FP32, False), ("suspension", FP16, False), ("two_impactors", FP32, False), ("periodic", FP16, False),
    ("fs_impactor", FP32, False), ("slip_walls", FP64, False), ("slip_dyn_walls", FP32, False), ("dyn_walls", FP64, False),
    ("bingham", FP64, False), ("bingham", FP32, False), ("frictional", FP64, False), ("voellmy", FP32, False),
    ("smagorinsky", FP64, False), ("suspension", FP64, True), ("periodic", FP32, True)])
def test_chunks_equal_steps_everywhere(gpu_lib, case_root, name, prec, stress):
    d = cases.make_case(case_root, name)
    fs = int(cases._case_values(name)[0]["freeSurfaceSolve"]) != 0
    sims = [cases.open_sim(gpu_lib, d, precision=prec, stress=stress) for _ in range(3)]
    for s in sims:
        s.set_tile(4)
    sims[1].use_graphs(False)
    for n in (17, 5, 1, 22):
        sims[0].cycle(n)
        sims[1].cycle(n)
        for _ in range(n):
            sims[2].dem_step()
            sims[2].coupling_step()
            sims[2].lb_step()
            sims[2].fs_step()
        for s in sims:
            s.synchronize()
        S = [cases.state(s) for s in sims]
        compare(S[1], S[0], prec, f"{name}: chunks against single launches, +{n}", fs)
        compare(S[2], S[0], prec, f"{name}: chunks against sub-step calls, +{n}", fs)
        if stress:
            for k in (1, 2):
                compare_stress(sims[k].stress(), sims[0].stress(), prec, f"{name}: stress, +{n}")
                compare_particle_stress(sims[k].particle_stress(), sims[0].particle_stress(), prec, f"{name}: particles, +{n}")
    for s in sims:
        s.close()
