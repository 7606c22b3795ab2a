"""Neighbour lists of simulations in units far from one: lengths times 2^k (and
masses times 2^(k ndim), so the density stays), down to 8e-31 and up to 1e30.
Every power of two scales exactly, so lists, neighbour counts and densities are
those of the unit box bit for bit, and rates per length those divided by 2^k
(1e-12: a few terms are sums of unlike parts).  The screening arithmetic is
also replayed on the CPU in FP32 (numpy) in both units."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("ndim,nside", [(3, 11), (2, 33), (1, 70)])
@pytest.mark.parametrize("k", [-100, -60, 40, 50, 61, 100])
def test_lists_in_scaled_units(ndim, nside, k):
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box(nside, ndim=ndim, seed=31, vel_seed=32, vrms=0.3)
    o = o.replace(maxdensits=0)
    st["hh"] *= np.exp(0.1 * np.random.default_rng(33).standard_normal(st["hh"].shape))
    u = 2.0 ** k
    big = dict(st, x=st["x"] * u, hh=st["hh"] * u, pmass=st["pmass"] * u ** ndim)
    ob = o.replace(xmin=tuple(v * u for v in o.xmin), xmax=tuple(v * u for v in o.xmax), psep=o.psep * u)
    print("lists ndim", ndim, "lengths times 2^%d" % k, flush=True)
    sim, ref = nd.Simulation(ob, big, precision=1), nd.Simulation(o, st, precision=1)
    for s in (sim, ref):
        s.derivs()
    assert (ref.get("nblist_len") > 0).mean() > 0.9  # (the others overflowed: -1 in both)
    for f in ("nblist_len", "numneigh", "rho"):
        assert np.array_equal(sim.get(f), ref.get(f)), f
    # (drho/dt divides by the separation plus the machine epsilon, a length of
    # its own that shows where lengths are small: src/density_sums.f90)
    for f in ("force", "dudt", "dBevoldt") if k > 0 else ("force",):
        a, b = sim.get(f) * u, ref.get(f)
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), f


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** 61, 2.0 ** 100])
def test_screening_arithmetic_needs_scaled_lengths(scale):
    """what the list builder's FP32 test would decide in such units without
    scaling: an idle lane (its constant 1e30) meets candidates, or every square
    is 0 or infinite; in units of the list radius it decides as in FP64"""
    f = np.float32
    idle = f(1e30)
    c, R = np.array([0.3, 0.1, -0.2]) * scale, 1.1 * scale
    near, far = np.array([0.1, 0.0, 0.0]) * scale, np.array([2.0, 0.5, 0.5]) * scale

    def decide(s):
        cs, r2 = (c * s).astype(f), f((R * s) ** 2) if (R * s) ** 2 < 3e38 else f(np.inf)
        out = []
        with np.errstate(all="ignore"):
            cc = np.sum(cs * cs, dtype=f)
            for x in (near, far):
                xs = (x * s).astype(f)
                out.append(bool(np.sum(f(-2) * cs * xs, dtype=f) + cc + np.sum(xs * xs, dtype=f) - r2 < 0))
            out.append(bool(idle + (cc - r2) < 0))
        return out

    unit = 2.0 ** -np.floor(np.log2(R))
    assert decide(unit) == [True, False, False]
    assert decide(1.0) != [True, False, False]
