"""Contexts, batches, downloads and captured steps against the order in which a program uses and gives
them up."""
import ctypes

import numpy as np
import pytest

import lbdem
import workloads

pytestmark = pytest.mark.gpu


def _small(lib, seed, steps=12):
    run = workloads.random_impact_run(np.random.default_rng(seed), (32,), 60, relax=60)
    sim = lbdem.Simulation(lib, lbdem.params_from_values(run.values, lbdem.PREC_FP32), run.particles, run.objects)
    sim.init()
    sim.set_tile(8)
    sim.cycle(steps)
    return sim


def test_member_destroyed_before_its_batch(gpu_lib):
    """The batch refuses further steps, its end touches the remaining members only, and those go on alone
    with the results of a run that was never in a batch (tolerances of test_pool)."""
    ref, a, b = _small(gpu_lib, 3), _small(gpu_lib, 3), _small(gpu_lib, 4)
    batch = lbdem.Batch(gpu_lib, [a, b])
    batch.cycle(10)
    b.close()
    with pytest.raises(lbdem.LbdemError, match="destroyed"):
        batch.cycle(2)
    with pytest.raises(lbdem.LbdemError, match="destroyed"):
        batch.set_tile(4)
    batch.synchronize()
    batch.close()
    a.cycle(9)
    ref.cycle(19)
    for x, y in ((a.objects(), ref.objects()), (a.walls(), ref.walls())):
        assert np.abs(x - y).max() <= 1e-9 * np.abs(y).max()
    assert a.info()["nActive"] == ref.info()["nActive"] and a.info()["lbTime"] == 31
    a.close()
    ref.close()


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_record_reads_take_no_device_memory(gpu_lib, oracle_lib):
    """Reading the particles, impactors and walls needs no memory beyond what lbdem_init took, also after a
    field download has replaced the context's scratch, leaves the run as it is (touching spheres with
    friction: the tangential histories are carried from step to step) and gives the oracle's values (FP64
    tolerance of test_gpu_parity)."""
    X, Y, Z, n = 60, 70, 62, 4000
    rng = np.random.default_rng(2)
    g = np.stack(np.meshgrid(np.arange(2.6, X - 2.5, 3.05), np.arange(2.6, Y - 9.0, 3.05), np.arange(2.6, Z - 2.5, 3.05),
                             indexing="ij"), axis=-1).reshape(-1, 3)
    x0 = g[rng.permutation(len(g))][:n] + rng.uniform(-0.12, 0.12, (n, 3))
    v, _, _ = workloads.impact_box(size=(X, Y, Z), fluid_height=float(Y - 1), n_spheres=0, r=1.5, r_imp=3.0, y_imp=Y - 6.0,
                                   speed=0.01, periodic=False)
    v.update(frictionCoefPart=0.4)
    ps = lbdem.ParticleSet(size=np.ones(len(x0), np.int32), r=np.full(len(x0), 1.5), x0=x0)
    obs = lbdem.ObjectSet(r=np.array([3.0]), x0=np.array([[X / 2.0, Y - 6.0, Z / 2.0]]), x1=np.array([[0.0, -0.01, 0.0]]))
    out = []
    # the runtime takes memory of its own at the first launches and copies: a run of its own goes before
    for lib, reads in ((gpu_lib, False), (oracle_lib, False), (gpu_lib, True)):
        s = lbdem.Simulation(lib, lbdem.params_from_values(v, lbdem.PREC_FP64), ps, obs)
        s.init()
        for k in range(6):
            s.dem_step()
            if not reads:
                continue
            s.synchronize()
            if k == 3:
                s.fields(want_f=False)
            before = _free_bytes()
            s.particles(), s.objects(), s.walls()
            assert _free_bytes() == before, k
        out.append((s.particles(), s.objects(), s.walls()))
        s.close()
    out = out[1:]
    assert np.abs(out[0][0][:, 43:46]).max() > 0 or np.abs(out[0][0][:, 40:43]).max() > 0
    for A, B, w in zip(out[0], out[1], ("particles", "objects", "walls")):
        assert np.abs(A - B).max() <= 1e-10 * max(1.0, np.abs(A).max()), w


def test_start_up_is_over_when_no_chunk_is_left_to_capture(gpu_lib):
    """lbdem_tuning.pairCaptured: not while a longer call would still capture a chunk of steps, nor at the
    other step parity, whose chunks are graphs of their own."""
    sim = _small(gpu_lib, 6, steps=0)

    def captured():
        return sim.tuning()["pair_captured"]

    sim.cycle(4)   # start-up steps, one by one
    assert not captured()
    sim.cycle(4)
    sim.cycle(4)
    assert not captured()  # 16 steps would capture
    sim.cycle(16)
    assert captured()
    sim.cycle(1)
    assert not captured()
    sim.cycle(20)
    assert captured()
    sim.cycle(1)
    assert captured()
    sim.use_graphs(False)
    assert not captured()
    sim.close()


def test_interface_list_overflow_is_reported(gpu_lib):
    """A restart whose nodes are all interface nodes, three times what the interface list holds (a quarter of
    the box): the free surface's passes stay within their lists, the run reports the overflow, and the
    device goes on."""
    E = 66
    v, _, _ = workloads.impact_box(size=(E, E, E), fluid_height=float(E - 1), n_spheres=0, r=1.5, r_imp=3.0, y_imp=30.0,
                                   speed=0.01, periodic=False)
    v.update(demSolve=0, lbFY=0.0)
    w = np.array([1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12)
    rec = np.zeros(((E - 2) ** 3, lbdem.RESTART_REC))
    rec[:, 4], rec[:, 5], rec[:, 6:] = -0.5, 0.1, w
    sim = lbdem.Simulation(gpu_lib, lbdem.params_from_values(v, lbdem.PREC_FP32), lbdem.ParticleSet(), lbdem.ObjectSet())
    sim.set_restart((E, E, E), np.full(E ** 3, 3, np.uint8), rec)
    sim.init()
    assert sim.info()["nInterface"] == (E - 2) ** 3 > E ** 3 // 4
    sim.cycle(3)
    with pytest.raises(lbdem.LbdemError, match="overflowed"):
        sim.synchronize()
    sim.close()
    ok = _small(gpu_lib, 7)
    assert np.isfinite(ok.total_mass())
    ok.close()
