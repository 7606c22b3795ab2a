"""Lists of groups of 64 particles that straddle jumps of the cell order,
candidates beyond one pass of the builder's staging, uneven h (long extras)
and partial last groups: every list length equals the count of the FP64
membership test replayed on the host, image by image (exact: no tolerance),
and the sums equal the cell scan's to round-off (1e-12, as the other list
tests)."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(x, h, ndim):
    lim2 = 2.0 * 2.0 * 1.04 * 1.04 * (1.0 + 1.0e-12)
    shifts = np.array(list(itertools.product((-1.0, 0.0, 1.0), repeat=ndim)))
    hi = 1.0 / h
    hi21 = hi * hi
    out = np.zeros(len(h), dtype=np.int64)
    for k0 in range(0, len(h), 64):
        s = slice(k0, k0 + 64)
        d = (x[s, None, None, :] - x[None, :, None, :]) + shifts[None, None, :, :]
        r2 = d[..., 0] * d[..., 0]
        for q in range(1, ndim):
            r2 = r2 + d[..., q] * d[..., q]
        out[s] = np.sum((r2 * hi21[s, None, None] < lim2) | (r2 * hi21[None, :, None] < lim2), axis=(1, 2))
    return out


@pytest.mark.parametrize("ndim,nside,cells,spread", [(3, 7, 1, 0.0), (3, 9, 2, 0.05), (3, 13, 1, 0.05), (3, 13, 2, 0.2),
                                                     (2, 9, 1, 0.1), (2, 41, 2, 0.1), (1, 70, 1, 0.1)])
def test_list_lengths_of_split_groups(ndim, nside, cells, spread):
    import ndspmhd_amd as nd
    from ndspmhd_amd.setups import periodic_mhd_box
    o, st = periodic_mhd_box(nside, ndim=ndim, seed=31, vel_seed=32, vrms=0.3)
    o = o.replace(maxdensits=0)
    rng = np.random.default_rng(33)
    st["hh"] *= np.exp(spread * rng.standard_normal(st["hh"].shape))
    print("lists ndim", ndim, "nside", nside, "cells", cells, "spread", spread, flush=True)
    sim = nd.Simulation(o, st, precision=1)
    sim.set_tile_shapes(256, 256, cells)
    sim.derivs()
    L = sim.get("nblist_len").astype(np.int64)
    want = _expected(st["x"], st["hh"], ndim)
    assert (L >= 0).mean() > 0.5
    assert np.array_equal(L[L >= 0], want[L >= 0])
    scan = nd.Simulation(o.replace(cellscan=1), st, precision=1)
    scan.derivs()
    assert np.array_equal(sim.get("numneigh"), scan.get("numneigh"))
    for k in ("rho", "force", "dBevoldt", "dudt"):
        a, b = sim.get(k), scan.get(k)
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), k
