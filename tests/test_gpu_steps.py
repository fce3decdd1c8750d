"""The step's launches: chunks of captured steps against the same steps launched one by one and against
the sub-step calls, on runs with and without a free surface, spheres and impactors; a splashing run
(interface conversions, isolated nodes, nodes left and taken by the impactor every step) against the
oracle; the force kernel on either side of its change of lanes per sphere against the oracle."""
import numpy as np
import pytest

import cases
import lbdem
import workloads
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


def _by_hand(sim, n):
    for _ in range(n):
        sim.dem_step()
        sim.coupling_step()
        sim.lb_step()
        sim.fs_step()


@pytest.mark.parametrize("name", ["suspension", "two_impactors", "periodic", "lb_closed", "body_cubic"])
@pytest.mark.parametrize("calls", [(1,) * 14, (12, 1, 1, 1, 2), (3, 9, 4, 5, 16), (8, 16, 17, 21), (45,)])
def test_chunks_equal_steps(gpu_lib, case_root, name, calls):
    d = cases.make_case(case_root, name)
    sims = [cases.open_sim(gpu_lib, d, precision=lbdem.PREC_FP64) for _ in range(3)]
    for s in sims:
        s.set_tile(4)
    sims[1].use_graphs(False)
    for n in calls:
        sims[0].cycle(n)
        sims[1].cycle(n)
        _by_hand(sims[2], n)
        for s in sims:
            s.synchronize()
        S = [cases.state(s) for s in sims]
        compare(S[1], S[0], lbdem.PREC_FP64, f"{name}: chunks against single launches, +{n}")
        compare(S[2], S[0], lbdem.PREC_FP64, f"{name}: chunks against sub-step calls, +{n}")
    for s in sims:
        s.close()


@pytest.mark.parametrize("speed,periodic", [(0.12, False), (0.2, True)])
def test_splash_matches_oracle(oracle_lib, gpu_lib, speed, periodic):
    """FP64 tolerances of test_gpu_parity; the impactor enters and throws the surface up."""
    v, ps, obs = workloads.impact_box(size=(30, 34, 26), fluid_height=18.0, n_spheres=14, r=2.0, r_imp=4.0, y_imp=22.5,
                                      speed=speed, seed=5, relax=60, periodic=periodic, bed_top=14.0)
    a = lbdem.Simulation(oracle_lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, obs)
    b = lbdem.Simulation(gpu_lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, obs)
    a.init()
    b.init()
    for k in range(12):
        a.cycle(5)
        b.cycle(5)
        b.synchronize()
        compare(cases.state(a), cases.state(b), lbdem.PREC_FP64, f"splash, step {5 * k + 5}")
    a.close()
    b.close()


@pytest.mark.parametrize("n", [8191, 8192, 8193])
def test_force_lanes_match_oracle(oracle_lib, gpu_lib, n):
    """Spheres of radius 1.5 on a jittered lattice, some touching, some at the walls: one DEM step."""
    X, Y, Z = 66, 110, 70
    rng = np.random.default_rng(3)
    g = np.stack(np.meshgrid(np.arange(2.6, X - 2.5, 3.1), np.arange(2.6, Y - 3.0, 3.1), np.arange(2.6, Z - 2.5, 3.1),
                             indexing="ij"), axis=-1).reshape(-1, 3)
    x0 = g[rng.permutation(len(g))][:n] + rng.uniform(-0.12, 0.12, (n, 3))
    assert len(x0) == n
    v, _, _ = workloads.impact_box(size=(X, Y, Z), fluid_height=float(Y - 1), n_spheres=0, r=1.5, r_imp=3.0, y_imp=Y - 6.0,
                                   speed=0.01, periodic=False)
    ps = lbdem.ParticleSet(size=np.ones(n, np.int32), r=np.full(n, 1.5), x0=x0)
    obs = lbdem.ObjectSet(r=np.array([3.0]), x0=np.array([[X / 2.0, Y - 6.0, Z / 2.0]]), x1=np.array([[0.0, -0.01, 0.0]]))
    sims = []
    for lib in (oracle_lib, gpu_lib):
        s = lbdem.Simulation(lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, obs)
        s.init()
        for _ in range(3):
            s.dem_step()
        s.synchronize()
        sims.append((s.particles(), s.objects(), s.walls()))
        s.close()
    (pa, oa, wa), (pb, ob, wb) = sims
    assert np.abs(pa[:, lbdem.P["FCONTACT"]]).max() > 0 and np.abs(wa).max() > 0
    # FP64 records: 1e-10 of the largest entry, as in test_gpu_parity
    for A, B, w in ((pa, pb, "particles"), (oa, ob, "objects"), (wa, wb, "walls")):
        assert np.abs(A - B).max() <= 1e-10 * max(1.0, np.abs(A).max()), w


@pytest.mark.parametrize("tile", [0, 4])
def test_tuned_walk_sums_pairs_of_nodes(gpu_lib, tile):
    """2-byte storage: the walk the timing picked gives the particle sums of the two-node walk (the
    same 32-bit sums of pairs, added in FP64 in another order: 1e-12 of the largest force allows for
    thousands of terms, while 32-bit sums over other groups of nodes differ by some 1e-8). A walk set by
    the caller sums over its whole length."""
    v, ps, obs = workloads.impact_box(**workloads.HEADLINE)
    sims = []
    for _ in range(2):
        s = lbdem.Simulation(gpu_lib, lbdem.params_from_values(v, lbdem.PREC_FP16), ps, obs)
        s.init()
        s.cycle(40)
        sims.append(s)
    a, b = sims
    pick = a.tuning()["tile"][2]
    assert b.tuning()["tile"][2] in (1, 2, 4, 8)
    if tile == 0 and pick == 1:
        pytest.skip("the one-node walk was the fastest")
    b.set_tile(2)
    if tile:
        a.set_tile(tile)
    a.cycle(2)
    b.cycle(2)
    fa, fb = a.particles()[:, 9:15], b.particles()[:, 9:15]
    d = np.abs(fa - fb).max() / np.abs(fb).max()
    assert d <= 1e-12 if tile == 0 else 1e-12 < d <= 1e-5, (pick, d)
    for s in sims:
        s.close()
