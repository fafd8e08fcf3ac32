"""Tables on grids that are not uniform: the engine's lookups take cells and
fractions from the coordinate on the generator's uniform grids and search the
grid otherwise; both against the oracle on the same tables and streams."""
import ctypes as C

import numpy as np
import pytest

from xmimsim_amd import api, lines, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("moved", [False, True])
def test_lookups_on_moved_grids_match_the_oracle(orc, moved):
    inp = workloads.single_layer_steel(n_photons_line=20000, n_interactions=3)
    inp.layers[0].Z, inp.layers[0].weight = [6, 8, 26], [0.6, 0.3, 0.1]  # mostly scattering
    inp.layers[0].density, inp.layers[0].thickness = 1.5, 1.0
    inp.discrete[0].energy = 30.0
    inp.discrete[0].vertical_intensity = 1e9
    prep = api.Prepared(inp)
    h = C.cast(prep.hdf5F, C.POINTER(lines.HDF5)).contents
    if moved:
        # interior nodes by up to 0.3 of a cell, the same for every element;
        # the values stay, so the tables describe other (valid) distributions
        rng = np.random.default_rng(4)
        z0 = h.Zs[0]
        dE, dR = rng.uniform(-0.3, 0.3, z0.n_e), rng.uniform(-0.3, 0.3, z0.n_r)
        dT, dP = rng.uniform(-0.3, 0.3, h.phi_n_theta), rng.uniform(-0.3, 0.3, h.phi_n_r)
        grids = {}
        for k in range(h.n_Z):
            z = h.Zs[k]
            for p, n, d in ((z.Energies, z.n_e, dE), (z.RandomNumbers, z.n_r, dR)):
                grids[C.addressof(p.contents)] = (p, n, d)
        for p, n, d in ((h.Thetas, h.phi_n_theta, dT), (h.RandomNumbers, h.phi_n_r, dP)):
            grids[C.addressof(p.contents)] = (p, n, d)
        for p, n, d in grids.values():
            a = np.ctypeslib.as_array(p, (n,))
            step = a[1] - a[0]
            a[1:-1] += step * d[1:-1]
            assert np.all(np.diff(a) > 0)
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("tables", "moved" if moved else "uniform", flush=True)
    ch, vr, _, st = prep.run(seed=9)
    och, ovr, _, ost = orc.run(prep, seed=9, rng_mode=orc.RNG_PER_HISTORY)
    assert st.histories == ost.histories and vr[5, 384].sum() > 0
    scale = ovr.max()
    # the bound of the same-stream comparisons: 1e-9 of a row, or of 1e-6 of the largest
    assert np.all(np.abs(vr - ovr) <= 1e-9 * np.maximum(np.abs(ovr), 1e-6 * scale))
    assert np.abs(ch - och).max() <= 1e-9 * och.max()
    prep.close()
