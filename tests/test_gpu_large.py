"""Simulations above 65536 particles, where one lane takes a particle in every
pair pass, the tile shapes are the given ones and the folds after a pass run
over more than 1024 partials: against the CPU oracle, lists against the cell
scan, recorded steps against launch-by-launch ones, and batches that run one
lane per particle where their members alone run four."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "Bevol", "en", "hh", "psi", "dustevol", "rho", "force", "dBevoldt", "dudt", "ddustevoldt",
          "numneigh", "nits", "slot")
# norm-relative L-infinity: FP32 pair terms (some 10 roundings of 6e-8 each) in
# FP64 sums, whose terms cancel to a tenth of their size or so; FP64 sums in
# another order, through the h iteration
TOL = {0: 1e-5, 1: 1e-10}


def _setup(name, n):
    from ndspmhd_amd.setups import dusty_box, periodic_mhd_box
    if name == "dust":
        return dusty_box(n, ndim=2, seed=9)
    ndim = {"box": 3, "sheet": 2, "line": 1}[name]
    o, st = periodic_mhd_box(n, ndim=ndim, seed=3, vel_seed=4, vrms=0.5)
    st["Bevol"] += 0.02 * np.random.default_rng(7).standard_normal(st["Bevol"].shape)
    st["hh"] *= np.exp(0.03 * np.random.default_rng(8).standard_normal(st["hh"].shape))
    return o, st


def _err(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("wg", [64, 256])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name,n", [("box", 41), ("dust", 260)])
def test_against_oracle(name, n, prec, wg):
    """h fixed in mixed precision (a flip at tolh would move a particle's h),
    iterated in FP64; then one step in FP64"""
    import ndspmhd_amd as nd
    import oracle
    o, st = _setup(name, n)
    if prec == 0:
        o = o.replace(maxdensits=0)
    print(name, n, "prec", prec, "workgroup", wg, "N", st["pmass"].size, flush=True)
    assert st["pmass"].size > 65536
    sim, orc = nd.Simulation(o, st, precision=prec), oracle.Oracle(o, st)
    sim.set_tile_shapes(wg, wg, 1)
    sim.derivs()
    orc.derivs()
    names = ["hh", "rho", "gradh", "drhodt", "force"] + (["ddustevoldt", "deltav"] if name == "dust" else
                                                          ["dudt", "dBevoldt", "divB", "curlB", "gradpsi"])
    assert np.array_equal(sim.get("numneigh"), orc.get("numneigh"))
    for k in names:
        err = _err(sim.get(k), orc.get(k))
        print(k, err, flush=True)
        assert err <= TOL[prec], (k, err)
    if prec == 1:
        sim.set_dt(orc.scalar("dt"), orc.scalar("time"))
        orc.step()
        sim.step()
        for k in ("x", "vel", "hh", "rho", "force"):
            assert _err(sim.get(k), orc.get(k)) <= TOL[prec], k


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name,n", [("sheet", 256), ("line", 65536), ("line", 65537), ("box", 41), ("dust", 257)])
def test_lists_against_scan_and_replay(name, n, prec):
    """at 65536 (four lanes) and just above (one): sums over lists equal the
    cell scan's (another order of the same pairs: 1e-12; in mixed precision the
    pair terms are the same FP32 numbers, 1e-6 as in the other list tests), and
    three recorded steps the launch-by-launch ones bit for bit"""
    import ndspmhd_amd as nd
    o, st = _setup(name, n)
    print(name, n, "prec", prec, "lists, scan, replay", flush=True)
    fixed = o.replace(maxdensits=0)
    lists, scan = nd.Simulation(fixed, st, precision=prec), nd.Simulation(fixed.replace(cellscan=1), st, precision=prec)
    for s in (lists, scan):
        s.derivs()
    assert (lists.get("nblist_len") >= 0).mean() > 0.5 and (scan.get("nblist_len") < 0).all()
    assert np.array_equal(lists.get("numneigh"), scan.get("numneigh"))
    for k in ("rho", "drhodt", "force", "dudt", "dBevoldt", "ddustevoldt"):
        assert _err(lists.get(k), scan.get(k)) <= (1e-12 if prec else 1e-6), k
    del lists, scan
    eager, graph = nd.Simulation(o, st, precision=prec), nd.Simulation(o, st, precision=prec)
    for s in (eager, graph):
        s.set_tile_shapes(64, 64, 2)
    graph.set_graph(True)
    for step in range(3):
        eager.step()
        graph.step()
        for k in FIELDS:
            assert np.array_equal(eager.get(k), graph.get(k)), (step, k)
        assert eager.stats == graph.stats and eager.dt_info == graph.dt_info


@pytest.mark.parametrize("n,wg", [(65, 256), (102, 64)])
def test_large_folds(n, wg):
    """more than 1024 partials from workgroups of 256, and more particles than
    four times the threads of the statistics' launch: recorded steps against
    launch-by-launch ones, and the statistics against the fields"""
    import ndspmhd_amd as nd
    o, st = _setup("box", n)
    print("box", n, "workgroup", wg, flush=True)
    eager, graph = nd.Simulation(o, st), nd.Simulation(o, st)
    for s in (eager, graph):
        s.set_tile_shapes(wg, wg, 1)
        s.derivs()
        nn = s.get("numneigh")
        assert s.stats["nmin"] == nn.min() and s.stats["nmax"] == nn.max() and s.stats["itsdensity"] == s.get("nits").max()
        assert s.dt_info["hhmax"] >= s.get("hh").max() * (1 - 1e-15)
    graph.set_graph(True)
    for step in range(2):
        eager.step()
        graph.step()
        for k in FIELDS:
            assert np.array_equal(eager.get(k), graph.get(k)), (step, k)
        assert eager.stats == graph.stats and eager.dt_info == graph.dt_info


@pytest.mark.parametrize("kind", ["tube", "tube2d"])
def test_mixed_batch_above_65536_in_total(kind):
    """each member alone runs four lanes per particle, the group one; a member
    with a noisy flow and a tight tolerance needs more passes than recorded
    (1D, walls reflect) and finishes with four: all bit for bit as alone"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, shock_tube_2d
    make = brio_wu_1d if kind == "tube" else shock_tube_2d
    cfg = [make(m) for m in (17000, 16400, 17000, 18000)]
    if kind == "tube":
        st = cfg[1][1]
        st["vel"][:, 0] += 3.0 * np.random.default_rng(5).standard_normal(st["pmass"].size)
        cfg[1] = (cfg[1][0].replace(tolh=3e-7), st)
    assert sum(st["pmass"].size for _, st in cfg) > 65536 > max(st["pmass"].size for _, st in cfg)
    print("mixed batch", kind, [st["pmass"].size for _, st in cfg], flush=True)
    members = [nd.Simulation(o, st) for o, st in cfg]
    alone = [nd.Simulation(o, st) for o, st in cfg]
    batch = nd.Batch(members)
    most = 0
    for step in range(6):
        batch.step()
        for k, (m, a) in enumerate(zip(members, alone)):
            a.step()
            for f in FIELDS:
                assert np.array_equal(m.get(f), a.get(f)), (step, k, f)
            assert m.stats == a.stats and m.dt_info == a.dt_info
        most = max(most, members[1].stats["itsdensity"])
    if kind == "tube":
        assert most > 4
    batch.close()


def test_overflowed_rows_are_those_too_long():
    """list rows overflow exactly where the list exceeds their capacity: the
    shortest list of an overflowed row (counted on the host) is longer than the
    longest one held"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    from test_gpu_nblist_groups import _expected
    o, st = periodic_mhd_box(13, seed=31, vel_seed=32, vrms=0.3)
    o = o.replace(maxdensits=0)
    st["hh"] *= np.exp(0.2 * np.random.default_rng(33).standard_normal(st["hh"].shape))
    print("overflowed rows", flush=True)
    for cells in (1, 2):
        sim = nd.Simulation(o, st, precision=1)
        sim.set_tile_shapes(256, 256, cells)
        sim.derivs()
        L, want = sim.get("nblist_len"), _expected(st["x"], st["hh"], 3)
        assert (L < 0).any() and np.array_equal(L[L >= 0], want[L >= 0])
        assert want[L < 0].min() > want[L >= 0].max()
