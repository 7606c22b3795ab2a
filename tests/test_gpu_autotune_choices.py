"""The autotuners try what is a choice and nothing else: kernels with four
lanes per particle have one workgroup size, 256, whatever is asked for."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_workgroups_of_small_simulations(prec):
    """h-rho passes up to 65536 particles and the force passes with four lanes
    (all in FP64; hydro, dust and cell-scanning 1D MHD in mixed precision)"""
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, dusty_box, periodic_mhd_box
    for name, (o, st), force in (("tube", brio_wu_1d(200), True), ("dust", dusty_box(16, ndim=2), True),
                                 ("box", periodic_mhd_box(8), prec == 1)):
        print("autotune", name, "prec", prec, flush=True)
        sim = nd.Simulation(o, st, precision=prec)
        sim.set_tile_shapes(64, 64, 2)
        for _ in range(8):
            c = sim.autotune(reps=1)
            assert c["density_workgroup"] == 256 and c["cells_per_radius"] in (1, 2)
            assert c["force_workgroup"] == 256 if force else c["force_workgroup"] in (64, 256)


def test_workgroup_of_a_batch():
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import brio_wu_1d, shock_tube_2d
    cfg = [brio_wu_1d(200), shock_tube_2d(500)]
    for prec in (1, 0):
        print("batch autotune prec", prec, flush=True)
        batch = nd.Batch([nd.Simulation(o, st, precision=prec) for o, st in cfg])
        for _ in range(4):
            c = batch.autotune(reps=1)
            assert c["workgroup"] == 256 if prec == 1 else c["workgroup"] in (64, 256)
            batch.step()
        batch.close()
