"""The cone trials of the solid-angle estimate on the GPU against the oracle's
on the same random words: no collimator, one of nearly the window's radius and
narrower ones (wider ones are refused), near and far windows, odd and tiny trial counts."""
import math

import numpy as np
import pytest

from xmimsim_amd import api, workloads

pytestmark = pytest.mark.gpu

AREA = 0.3
SAME = 2.0 * math.sqrt(AREA / math.pi)


@pytest.mark.parametrize("hits,coll,y", [(1, None, 1.0), (7, None, 0.4), (33, (0.3, SAME * (1 - 1e-6)), 1.0), (16, (0.3, 0.4), 1.0),
                                         (16, (0.5, 0.2), 2.0), (25, (0.05, 0.61), 0.5)])
def test_cone_hits_equal_the_oracle(orc, hits, coll, y):
    inp = workloads.single_layer_steel(n_photons_line=10)
    inp.area_detector, inp.p_detector_window = AREA, (0.0, y, 100.0)
    if coll:
        inp.collimator_height, inp.collimator_diameter = coll
    prep = api.Prepared(inp)
    print("cone", hits, coll, y, flush=True)
    g, r, t = prep.compute_solid_angle(hits_per_single=hits, seed=5)
    og, _, _ = orc.solid_angle(prep, hits, 5)
    # cells differ by the rounding of the cone's size, or by whole hits of
    # cone / hits each.  From the collimator's top the oracle takes the angle
    # t as acos(cos t), which loses 1e-16 / t: t falls to 1e-6 in the cells
    # next to the plane of the top, 1e-10 of the cone there
    assert np.abs(g - og).max() <= (1e-9 if coll else 1e-12) * og.max()
    assert g.max() > 0
    prep.close()


@pytest.mark.parametrize("y,area", [(2.0, 0.2), (2.0, 0.05), (5.0, 0.3)])
def test_cone_size_rounds_as_the_cosine_of_the_angle(y, area):
    """Hits divide the cone's size, 2 pi (1 - cos) with the rounded cosine of
    the larger half angle, into equal parts: a cell is a whole number of them
    to the last bits.  Far from the window an ulp of the cosine is 1e-14 of the
    size and more."""
    hits = 3
    inp = workloads.single_layer_steel(n_photons_line=10)
    inp.area_detector, inp.p_detector_window = area, (0.0, y, 100.0)
    prep = api.Prepared(inp)
    print("cone size", y, area, flush=True)
    g, r, t = prep.compute_solid_angle(hits_per_single=hits, seed=5)
    L = np.longdouble
    R, rr, tt = L(math.sqrt(area / math.pi)), L(r)[None, :], L(t)[:, None]
    a1 = np.arctan(R * np.sin(tt) / (rr - R * np.cos(tt)))
    apex = np.maximum(np.arctan(R / rr), np.where(a1 <= 0, a1 + 4 * np.arctan(L(1)), a1))
    om = 1.0 - np.cos(apex).astype(np.float64)
    on = (g > 0) & (om < 0.05)
    n = g[on] * hits / (2.0 * np.pi * om[on])
    # six roundings are 7e-16, half an ulp of the cosine at least 2e-15.  In
    # double, cos(atan()) rounds the other way in 0.6 to 1.6 % of these cells,
    # a quotient of two roundings in 40 %: a tenth of
    # that is the line
    off = np.abs(n - np.rint(n)) > 1.5e-15 * n
    print("cells", on.mean(), "rounded otherwise", off.mean(), flush=True)
    assert on.mean() > 0.3 and off.mean() < 0.04
    prep.close()
