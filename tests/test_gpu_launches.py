"""The launches that fold, scan and move up lists in one go, at the sizes where
their tiles end: particle counts around one wave, one tile and one block of
every kind, both workgroup shapes, runs with reflecting walls (synchronous
passes with lists of part of the particles), fixed walls and a tight h
tolerance (more passes than a recorded step holds).  Replayed steps must equal
launch-by-launch ones bit for bit, and the first evaluation the CPU oracle to
1e-10 in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "Bevol", "en", "hh", "rho", "force", "numneigh", "nits", "slot")


@pytest.mark.parametrize("n,wg,walls,tolh", [(63, 64, "reflect", 1e-3), (64, 256, "reflect", 1e-3),
                                             (65, 64, "fixed", 1e-3), (255, 256, "reflect", 1e-8),
                                             (257, 64, "reflect", 1e-8), (1023, 256, "fixed", 1e-8),
                                             (1025, 64, "fixed", 1e-8), (4097, 256, "reflect", 1e-8)])
def test_tubes_replayed_and_against_oracle(n, wg, walls, tolh):
    import ndspmhd_amd as nd
    import oracle
    from ndspmhd_amd.setups import brio_wu_1d
    o, st = brio_wu_1d(n, boundary=walls)
    o = o.replace(tolh=tolh)
    print("tube", n, "workgroup", wg, walls, tolh, flush=True)
    eager, graph = nd.Simulation(o, st, precision=1), nd.Simulation(o, st, precision=1)
    for s in (eager, graph):
        s.set_tile_shapes(wg, wg, 2)
        s.derivs()
        s.set_dt(s.dt_info["dt"])
    graph.set_graph(True)
    orc = oracle.Oracle(o, st)
    orc.derivs()
    for k in ("rho", "hh", "force"):
        a, b = eager.get(k), orc.get(k)
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(b)), k
    for step in range(4):
        eager.step()
        graph.step()
        for k in FIELDS:
            assert np.array_equal(eager.get(k), graph.get(k)), (step, k)
        assert eager.stats == graph.stats and eager.dt_info == graph.dt_info


def test_batch_with_late_members():
    """members that need more passes than recorded beside members that do not"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d
    cfg = [(brio_wu_1d(n)[0].replace(tolh=t), brio_wu_1d(n)[1]) for n, t in ((300, 1e-3), (257, 1e-9), (500, 1e-3))]
    print("batch with a tight member", flush=True)
    members = [nd.Simulation(o, st, precision=1) for o, st in cfg]
    alone = [nd.Simulation(o, st, precision=1) for o, st in cfg]
    batch = nd.Batch(members)
    for step in range(4):
        batch.step()
        for m, a in zip(members, alone):
            a.step()
            for k in FIELDS:
                assert np.array_equal(m.get(k), a.get(k)), (step, k)
            assert m.stats == a.stats and m.dt_info == a.dt_info
    batch.close()


@pytest.mark.parametrize("ndim", [1, 2, 3])
def test_upload_download_round_trip(ndim):
    """every component comes back where it went in, also after reorders moved
    the slots (bit for bit)"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box({1: 301, 2: 17, 3: 9}[ndim], ndim=ndim, seed=3, vel_seed=4, vrms=0.2)
    rng = np.random.default_rng(5)
    for k in ("vel", "Bevol", "alpha", "psi"):
        st[k] = rng.uniform(0.1, 0.9, size=st[k].shape)
    sim = nd.Simulation(o, st, precision=1)
    for k in ("x", "vel", "Bevol", "alpha", "psi", "pmass", "hh", "en"):
        assert np.array_equal(sim.get(k), st[k].reshape(sim.get(k).shape)), k
    sim.derivs()
    for _ in range(2):
        sim.step()
    assert np.array_equal(sim.get("pmass"), st["pmass"])
    sim.upload(st)
    for k in ("x", "vel", "Bevol", "alpha", "psi", "hh", "en"):
        assert np.array_equal(sim.get(k), st[k].reshape(sim.get(k).shape)), k
    assert not np.any(sim.get("force")) and np.array_equal(sim.get("Bfield"), st["Bevol"])
