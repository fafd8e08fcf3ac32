"""GPU tests of the launch shapes: a run whose batches replay one captured
HIP graph, each replay popping its batch from the device batch queue, equals
the run launched kernel by kernel bit for bit (estimator, brute force with
cascades, several engines); the batch size, the photons per lane of the line
kernel and the resident workgroups per CU change the estimator's sums only in
their last bits; the autotuner returns a shape in its search space."""
import numpy as np
import pytest

from xmimsim_amd import api, autotune, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_launch():
    api.set_launch()
    yield
    api.set_launch()


def _steel(n):
    return workloads.single_layer_steel(n_photons_line=n)


def _run(prep, seed, **launch):
    api.set_launch(**launch)
    out = prep.run(seed=seed)
    st = api.get_stats()
    api.set_launch()
    return out, st


def test_graph_equals_eager_estimator():
    """4.6 batches of 2^14 histories, the last partial: graph replays equal
    the launches one by one, bit for bit, and a replay per batch ran."""
    prep = api.Prepared(workloads.three_layer_kramers(n_photons_interval=150, n_photons_line=150))
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("graph vs eager, estimator", flush=True)
    (ch0, vr0, _, s0), st0 = _run(prep, 9, batch_log2=14)
    (ch1, vr1, _, s1), st1 = _run(prep, 9, batch_log2=14, use_graph=1)
    assert s0.histories == s1.histories > 4 * 2 ** 14
    assert st0.batches == st1.batches == -(-s0.histories // 2 ** 14) and st0.graph_replays == 0
    assert st1.graph_replays == st1.batches
    assert np.array_equal(ch0, ch1) and np.array_equal(vr0, vr1)
    assert vr0.sum() > 0
    prep.close()


def test_graph_equals_eager_brute():
    """Brute force with both cascades: the queue sets and offspring lists
    swapped per order are part of the captured graph."""
    inp = api.Input(layers=[api.Layer([26, 50], [0.5, 0.5], 5.0, 0.001)],
                    discrete=[api.DiscreteLine(40.0, 5e8, 5e8)], n_photons_line=50000, area_detector=3.0,
                    gain=0.02, nchannels=2500)
    prep = api.Prepared(inp, options=api.default_options(use_variance_reduction=0))
    print("graph vs eager, brute force", flush=True)
    (ch0, _, bf0, s0), _ = _run(prep, 4, batch_log2=13)
    (ch1, _, bf1, s1), st1 = _run(prep, 4, batch_log2=13, use_graph=1)
    assert st1.graph_replays == st1.batches == 7
    assert s0.histories == s1.histories
    assert np.array_equal(ch0, ch1) and np.array_equal(bf0, bf1)
    assert bf0.sum() > 0
    prep.close()


def test_graph_batch_engines():
    """Several engines capturing and replaying their samples' graphs at once
    give each sample's single-run result."""
    inps = workloads.batch_samples(5, seed=3, budget=(3e4, 8e4), n_elements=(2, 5), zrange=(20, 40))
    Zs = sorted({z for inp in inps for l in inp.layers for z in l.Z})
    tables = api.SharedTables(Zs)
    grid = api.Prepared(inps[0], tables=tables)
    grid.compute_solid_angle(hits_per_single=200, seed=3)
    preps = []
    for inp in inps:
        p = api.Prepared(inp, tables=tables)
        p.solid_angle = grid.solid_angle
        p._sa_owner = "borrowed"
        preps.append(p)
    print("graph, batch of engines", flush=True)
    api.set_launch(batch_log2=14, use_graph=1)
    out, _ = api.run_batch(preps, tables, seed=21, n_streams=3)
    api.set_launch(batch_log2=14)
    for p, (ch, vr) in zip(preps, out):
        c1, v1, _, _ = p.run(seed=21)
        assert np.array_equal(ch, c1) and np.array_equal(vr, v1)
    for p in preps:
        p.solid_angle = None
        p.close()
    grid.close()


@pytest.mark.parametrize("launch", [{"batch_log2": 15}, {"lines_kp": 2}, {"lines_kp": 3}, {"lines_kp": 4}, {"wg_per_cu": 2},
                                    {"batch_log2": 16, "lines_kp": 4, "wg_per_cu": 3, "use_graph": 1}])
def test_launch_shapes_agree(launch):
    """Other shapes regroup the estimator's per-wave sums: every channel and
    history row within 1e-12 of the default shape's."""
    prep = api.Prepared(_steel(100000))
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("launch shape", launch, flush=True)
    (ch0, vr0, _, _), _ = _run(prep, 13)
    (ch1, vr1, _, _), _ = _run(prep, 13, **launch)
    for a, b in ((ch1, ch0), (vr1, vr0)):
        scale = np.abs(b).max()
        assert np.all(np.abs(a - b) <= 1e-12 * np.maximum(np.abs(b), 1e-3 * scale)), launch
    prep.close()


@pytest.mark.parametrize("n_layers,kp", [(3, 2), (3, 3), (4, 2), (4, 4), (5, 1), (5, 2), (7, 1)])
def test_photons_per_lane_agree(n_layers, kp):
    """Every other instance of the line kernel at its layer counts: within
    1e-12 of the default's."""
    inp = _steel(100000)
    Zs = ([13], [26, 24], [22, 29], [30], [14, 20], [28], [25, 40])
    inp.layers = [api.Layer(list(Z), [1.0 / len(Z)] * len(Z), 2.0 + k, 1e-3) for k, Z in enumerate(Zs[:n_layers])]
    inp.reference_layer = 1
    prep = api.Prepared(inp)
    assert kp in autotune.lines_kp_candidates(n_layers)
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("photons per lane", n_layers, kp, flush=True)
    (_, vr0, _, _), _ = _run(prep, 13)
    (_, vr1, _, _), _ = _run(prep, 13, lines_kp=kp)
    assert vr0.sum() > 0 and np.all(np.abs(vr1 - vr0) <= 1e-12 * np.maximum(np.abs(vr0), 1e-3 * np.abs(vr0).max()))
    prep.close()


@pytest.mark.parametrize("n_layers", [1, 3])
def test_default_batches_equal_small_ones(n_layers):
    """One full batch of 2^23 histories, whose layer scan spans 128 segments
    (two waves of k_layer_base), and one of an odd rest: the events of every
    layer are those of 2^18 batches (at most 4 segments), the sums agree as
    between other shapes, and the default's name gives the default's bits."""
    inp = _steel(2 ** 23 + 600001)
    inp.n_interactions_trajectory = 2
    if n_layers == 3:  # thin, so that photons reach the last
        steel = inp.layers[0]
        inp.layers = [api.Layer([13], [1.0], 2.7, 1e-3), api.Layer(steel.Z, steel.weight, steel.density, 1e-3),
                      api.Layer([22, 29], [0.5, 0.5], 5.0, 1e-3)]
        inp.reference_layer = 2
    prep = api.Prepared(inp)
    prep.compute_solid_angle(hits_per_single=200, seed=3)

    def run(**launch):
        print("batches", n_layers, launch, flush=True)
        (ch, vr, _, s), st = _run(prep, 17, **launch)
        return ch, vr, s.histories, st.batches, prep.layer_events

    ch0, vr0, h0, b0, ev0 = run()
    ch1, vr1, h1, b1, ev1 = run(batch_log2=18)
    ch2, vr2, _, b2, ev2 = run(batch_log2=23)
    assert h0 == h1 == inp.n_photons_line and (b0, b1, b2) == (2, 35, 2)
    assert ev0 == ev1 == ev2 and all(e > 0 for e in ev0)
    assert np.array_equal(ch0, ch2) and np.array_equal(vr0, vr2)
    for a, b in ((ch1, ch0), (vr1, vr0)):
        scale = np.abs(b).max()
        assert np.all(np.abs(a - b) <= 1e-12 * np.maximum(np.abs(b), 1e-3 * scale))
    prep.close()


def test_autotune_picks_a_shape_of_its_space(tmp_path):
    prep = api.Prepared(_steel(20000))
    prep.compute_solid_angle(hits_per_single=200, seed=3)
    print("autotune", flush=True)
    best, table = autotune.tune(prep, sample_histories=2 ** 16, batch_sizes=(14, 15), seed=5,
                                cache=str(tmp_path / "launch.json"))
    assert best in [row["launch"] for row in table]
    assert all(row["ms"] > 0 for row in table)
    assert api.get_launch() == autotune.DEFAULT
    again, rows = autotune.tune(prep, sample_histories=2 ** 16, batch_sizes=(14, 15), seed=5,
                                cache=str(tmp_path / "launch.json"))
    assert again == best and rows == []  # from the cache
    prep.close()
