"""CPU test of the benchmark's flop charge against the instruction counts of
the committed profile."""
import json
import os
import sys


def test_flop_charge_fits_the_instructions_executed():
    """No more flops are charged to a kernel's launch than its vector
    instructions could hold: two per lane in every one of them."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    sys.path.insert(0, root)
    import bench
    with open(os.path.join(root, "profiles", "counters_three_layer_kramers.json")) as f:
        k = json.load(f)["kernels"]
    fpe = bench.vr_flops_per_event(bench.estimator_work("three_layer_kramers"))
    # the counters' run: 492 x 1e5 histories of four orders, 0.64 events in
    # each (12604769937 events of 4.92e9 histories in the benchmark)
    events = 0.64 * 4 * 492 * 100_000
    for name, phase in (("k_vr_lines", "lines"), ("k_vr_scatter", "scatter")):
        c = k[name]
        executed = 2.0 * 64 * c["waves"] * c["valu_per_wave"] * c["dispatches"]
        charged = fpe[phase] * events
        print(name, charged / executed)
        assert 0.05 * executed < charged < 0.8 * executed, name
