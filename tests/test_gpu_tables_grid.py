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


@pytest.mark.parametrize("moved,n_layers", [(False, 4), (False, 5), (False, 7), (True, 2), (True, 5)])
def test_estimator_geometry_of_layer_stacks_matches_the_oracle(orc, moved, n_layers):
    """Every unrolled layer count of the step and its estimator geometry, with
    the solid angle from a uniform grid and from one that is not."""
    inp = workloads.single_layer_steel(n_photons_line=20000, n_interactions=3)
    layer = api.Layer([8, 20, 26], [0.5, 0.3, 0.2], 1.5, 0.05)
    inp.layers = [api.Layer(list(layer.Z), [0.5 + 0.02 * k, 0.3 - 0.02 * k, 0.2], 1.5 + 0.1 * k, 0.05 + 0.01 * k)
                  for k in range(n_layers)]
    inp.reference_layer = (n_layers + 1) // 2
    inp.discrete[0].energy = 30.0
    inp.discrete[0].vertical_intensity = 1e9
    prep = api.Prepared(inp)
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    if moved:
        sa = prep.solid_angle.contents
        rng = np.random.default_rng(5)
        for p, n in ((sa.grid_dims_r_vals, sa.grid_dims_r_n), (sa.grid_dims_theta_vals, sa.grid_dims_theta_n)):
            a = np.ctypeslib.as_array(p, (n,))
            a[1:-1] += (a[1] - a[0]) * rng.uniform(-0.3, 0.3, n - 2)
            assert np.all(np.diff(a) > 0)
    print("stack", n_layers, "grid", "moved" if moved else "uniform", flush=True)
    ch, vr, _, st = prep.run(seed=9)
    och, ovr, _, ost = orc.run(prep, seed=9, rng_mode=orc.RNG_PER_HISTORY)
    assert st.histories == ost.histories and vr.sum() > 0
    scale = ovr.max()
    # as above: the photons start in dense layers whose depths, about 0.1 cm
    # at z = 100 cm +- 1e-14, are given to 1e-13
    assert np.all(np.abs(vr - ovr) <= 1e-9 * np.maximum(np.abs(ovr), 1e-6 * scale))
    assert np.abs(ch - och).max() <= 1e-9 * och.max()
    prep.close()


@pytest.mark.parametrize("advanced", [False, True])
def test_compton_profiles_on_moved_grids_match_the_oracle(orc, advanced):
    """The Doppler draws take cell and fraction from the number on the uniform
    grids and read the nodes otherwise."""
    inp = workloads.single_layer_steel(n_photons_line=20000, n_interactions=2)
    inp.layers[0].Z, inp.layers[0].weight = [6, 8, 26], [0.6, 0.3, 0.1]
    inp.layers[0].density, inp.layers[0].thickness = 1.5, 1.0
    inp.discrete[0].energy = 30.0
    inp.discrete[0].vertical_intensity = 1e9
    prep = api.Prepared(inp, options=api.default_options(use_advanced_compton=int(advanced)))
    h = C.cast(prep.hdf5F, C.POINTER(lines.HDF5)).contents
    rng = np.random.default_rng(6)
    n = h.Zs[0].cp_len
    d = rng.uniform(-0.3, 0.3, (3, n))
    d[:, :2] = d[:, -2:] = 0.0  # the first cell's width places a number in its cell
    seen = set()
    for k in range(h.n_Z):
        z = h.Zs[k]
        for p, dk in ((z.cp_random_numbers, d[0]),) + (((z.cp_Qs, d[1]), (z.cp_partial_cdf_inv, d[2])) if advanced else ()):
            if C.addressof(p.contents) in seen:
                continue
            seen.add(C.addressof(p.contents))
            a = np.ctypeslib.as_array(p, (n,))
            a += (a[1] - a[0]) * dk
            assert np.all(np.diff(a) > 0)
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("Compton grids moved", "advanced" if advanced else "", flush=True)
    ch, vr, _, st = prep.run(seed=9)
    och, ovr, _, ost = orc.run(prep, seed=9, rng_mode=orc.RNG_PER_HISTORY)
    assert st.histories == ost.histories and vr.sum() > 0
    assert np.all(np.abs(vr - ovr) <= 1e-9 * np.maximum(np.abs(ovr), 1e-6 * ovr.max()))
    assert np.abs(ch - och).max() <= 1e-9 * och.max()
    prep.close()
