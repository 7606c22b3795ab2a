"""The library's calls in orders a host may use them in: what one call leaves
behind on the host must not stand in for what another has done on the device
since.  Each sequence runs against the launch-by-launch path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "Bevol", "en", "hh", "rho", "force", "dBevoldt", "dudt", "numneigh", "nits", "slot")


def _same(a, b, where):
    for k in FIELDS:
        assert np.array_equal(a.get(k), b.get(k)), (where, k)


@pytest.mark.parametrize("setup", ["box", "tube"])
@pytest.mark.parametrize("batch", [False, True])
def test_density_after_binning_and_recorded_step(setup, batch):
    """set_linklist, a recorded step, then iterate_density and get_rates: the
    step has used up the binning's scalars, so the iteration sets them anew and
    works on the corrected state, as it does after a launch-by-launch step"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, periodic_mhd_box
    o, st = periodic_mhd_box(11, seed=3, vel_seed=4, vrms=0.5) if setup == "box" else brio_wu_1d(300)
    print("density after a recorded step:", setup, "batch" if batch else "alone", flush=True)
    eager, sim = nd.Simulation(o, st, precision=1), nd.Simulation(o, st, precision=1)
    if batch:
        b = nd.Batch([sim])
        step = b.step
    else:
        sim.set_graph(True)
        step = sim.step
    for s in range(3):
        eager.step()
        step()
    eager.set_linklist()
    sim.set_linklist()
    eager.step()
    step()
    _same(eager, sim, "step")
    before = sim.get("rho")
    assert eager.iterate_density() == sim.iterate_density()
    assert sim.stats["itsdensity"] >= 1 and not np.array_equal(before, sim.get("rho"))
    assert eager.get_rates() == sim.get_rates()
    _same(eager, sim, "rates")
    if batch:
        b.close()


@pytest.mark.parametrize("setup,prec", [("box", 0), ("box", 1), ("dust", 0), ("tube", 1), ("tube2d", 0)])
def test_recorded_steps_keep_reordering(setup, prec):
    """45 steps: the state is put into cell order every ten steps also where
    every step replays graphs recorded earlier (from the third reorder on), so
    the slots and the order of every sum stay the launch-by-launch path's; and
    the grid of a replayed step serves the calls that need one"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, dusty_box, periodic_mhd_box, shock_tube_2d
    o, st = {"box": lambda: periodic_mhd_box(12, seed=3, vel_seed=4, vrms=2.0), "dust": lambda: dusty_box(24, ndim=2, seed=9),
             "tube": lambda: brio_wu_1d(300), "tube2d": lambda: shock_tube_2d(600)}[setup]()
    print("45 recorded steps:", setup, prec, flush=True)
    eager, graph = nd.Simulation(o, st, precision=prec), nd.Simulation(o, st, precision=prec)
    graph.set_graph(True)
    slots = []
    for s in range(45):
        eager.step()
        graph.step()
        _same(eager, graph, s)
        assert eager.stats == graph.stats and eager.dt_info == graph.dt_info, s
        if s % 10 == 0:
            slots.append(graph.get("slot"))
            assert np.array_equal(eager.neighbours(), graph.neighbours()), s
    if setup == "box":
        # (the flow moves particles between cells, so the orders differ)
        assert all(not np.array_equal(a, b) for a, b in zip(slots[1:], slots[2:]))


@pytest.mark.parametrize("how", ["tile shapes", "autotune"])
def test_batch_after_member_reallocates(how):
    """a member's cell arrays are allocated again between batch steps, at the
    size they had: the batch records its steps anew and the members stay those
    stepped one by one bit for bit"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, periodic_mhd_box, shock_tube_2d
    cfg = [brio_wu_1d(300), shock_tube_2d(600), periodic_mhd_box(9, seed=3, vel_seed=4), brio_wu_1d(500)]
    members = [nd.Simulation(o, st, precision=1) for o, st in cfg]
    alone = [nd.Simulation(o, st, precision=1) for o, st in cfg]
    batch = nd.Batch(members)
    for s in range(9):
        if s in (2, 5, 7):
            print("member arrays again:", how, "before step", s, flush=True)
            for k in ((0, 1, 2, 3) if s == 7 else (s % 4, (s + 1) % 4)):
                if how == "tile shapes":
                    shapes = (64, 256, 2)
                else:
                    c = members[k].autotune(reps=1)
                    shapes = (c["force_workgroup"], c["density_workgroup"], c["cells_per_radius"])
                    alone[k].autotune(reps=1)
                members[k].set_tile_shapes(*shapes)
                alone[k].set_tile_shapes(*shapes)
        batch.step()
        for k, (m, a) in enumerate(zip(members, alone)):
            a.step()
            _same(a, m, (s, k))
            assert m.stats == a.stats and m.dt_info == a.dt_info
    batch.close()


def _rows(a):
    return a[np.lexsort(a.T[::-1])]


@pytest.mark.parametrize("graph", [False, True])
def test_lists_usable_after_a_step_that_overflowed(graph):
    """a step in which list rows overflowed makes longer ones before the next
    binning, not at once: its grid and lists still serve iterate_density,
    get_rates and neighbours, which equal the cell scan's to round-off (1e-12,
    as the other list tests)"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box(12, seed=7, vel_seed=8, vrms=0.3)
    st["hh"][np.random.default_rng(9).choice(st["hh"].size, 30, replace=False)] *= 2.5
    o = o.replace(maxdensits=0)
    print("calls after a step with overflowed rows, graph", graph, flush=True)
    sim, scan = nd.Simulation(o, st, precision=1), nd.Simulation(o.replace(cellscan=1), st, precision=1)
    for s in (sim, scan):
        s.set_graph(graph)
        for k in range(3):
            s.step()
            if s is sim and k == 0:
                over = int((s.get("nblist_len") < 0).sum())
                print("overflowed rows", over, flush=True)
                assert over
            s.iterate_density()
            s.get_rates()
    assert np.array_equal(_rows(sim.neighbours()), _rows(scan.neighbours()))
    for k in ("rho", "force", "dBevoldt", "dudt"):
        a, b = sim.get(k), scan.get(k)
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), k


@pytest.mark.parametrize("graph", [False, True])
def test_grid_usable_after_a_step_that_clamped_it(graph):
    """a state with much smaller h than the key space was sized for: the first
    step widens the cells and the key space grows before the next binning; the
    step's grid serves the calls in between, and neighbours and rates equal
    those of a context sized for the state (1e-12: other cells, other order)"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box(12, seed=7, vel_seed=8, vrms=0.3)
    o = o.replace(maxdensits=0)
    wide = dict(st, hh=st["hh"] * 4.0)
    narrow = dict(st, hh=st["hh"] * 0.7)
    print("calls after a step with widened cells, graph", graph, flush=True)
    sim, ref = nd.Simulation(o, wide, precision=1), nd.Simulation(o, narrow, precision=1)
    for s in (sim, ref):
        s.set_tile_shapes(256, 256, 1)
        s.set_graph(graph)
        s.derivs()
    sim.upload(narrow)
    sim.derivs()
    for _ in range(3):
        for s in (sim, ref):
            s.set_dt(1e-3)
            s.step()
        assert np.array_equal(_rows(sim.neighbours(sym=True)), _rows(ref.neighbours(sym=True)))
        for s in (sim, ref):
            s.iterate_density()
            s.get_rates()
        for k in ("rho", "force", "dBevoldt", "dudt"):
            a, b = sim.get(k), ref.get(k)
            assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), k


@pytest.mark.parametrize("n", [1, 65, 40000])
def test_download_before_upload(n):
    """a context that holds no state yet gives fields of zeros in the caller's
    order (small ones through pinned memory, large ones through device memory)
    and no lists"""
    import ctypes
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, _ = periodic_mhd_box(4)
    L = nd.load_library()
    iopt, dopt = np.ascontiguousarray(o.iopt(), dtype=np.int32), np.ascontiguousarray(o.dopt(), dtype=np.float64)
    h, w = ctypes.c_void_p(), ctypes.c_int32()
    as_p = lambda a, t: a.ctypes.data_as(ctypes.POINTER(t))
    assert L.ndsp_create(as_p(iopt, ctypes.c_int32), as_p(dopt, ctypes.c_double), n, 1, ctypes.byref(h)) == 0
    print("download before upload", n, flush=True)
    want = {"x": 0.0, "vel": 0.0, "rho": 0.0, "numneigh": 0.0, "nblist_len": -1.0, "slot": np.arange(n)}
    for k, v in want.items():
        out = np.full(3 * n, 7.0)
        assert L.ndsp_download(h, k.encode(), as_p(out, ctypes.c_double), ctypes.byref(w)) == 0
        assert w.value == (3 if k in ("x", "vel") else 1)
        assert np.array_equal(out[:w.value * n], np.broadcast_to(v, w.value * n)), k
        assert np.all(out[w.value * n:] == 7.0)
    # what needs a state says so
    assert L.ndsp_iterate_density(h, None) != 0 and L.ndsp_get_rates(h, None) != 0
    assert L.ndsp_destroy(h) == 0


def _leave_hip_error():
    """an invalid device number, refused by the HIP runtime, leaves its error
    for the next hipGetLastError of this thread"""
    import ctypes
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    assert ctypes.CDLL(path).hipSetDevice(99999) != 0


def test_gradient_after_an_early_return():
    """a gradient call that returned on an error after its launch (here one
    that another HIP call had left) leaves sums on the device; the next
    gradient or training call starts from zero all the same (gradients of one
    block of rows: one atomic per parameter, so equal bit for bit)"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box(6)
    rng = np.random.default_rng(5)
    X, T = rng.standard_normal((64, 6)).astype(np.float32), rng.standard_normal(64).astype(np.float32)
    p = (0.3 * rng.uniform(-1, 1, nd.MLP_NPARAM)).astype(np.float32)
    sim, ref = nd.Simulation(o, st), nd.Simulation(o, st)
    for s in (sim, ref):
        s.mlp_set_params(p)
    want = ref.mlp_grad(X, T)
    print("gradient after an early return", flush=True)
    for call in (lambda: sim.mlp_grad(X, T), lambda: sim.mlp_train(X, T, 1, 1e-3)):
        _leave_hip_error()
        with pytest.raises(nd.NdspError):
            call()
        sim.mlp_set_params(p)
    _leave_hip_error()
    with pytest.raises(nd.NdspError):
        sim.mlp_grad(X, T)
    got = sim.mlp_grad(X, T)
    assert got[0] == want[0] and np.array_equal(got[1], want[1])
    _leave_hip_error()
    with pytest.raises(nd.NdspError):
        sim.mlp_grad(X, T)
    assert sim.mlp_train(X, T, 1, 1e-3) == ref.mlp_train(X, T, 1, 1e-3)
    assert np.array_equal(sim.mlp_get_params()[0], ref.mlp_get_params()[0])
