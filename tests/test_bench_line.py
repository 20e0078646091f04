"""The benchmark's one line of output: short enough to be recorded whole, with the headline as it was measured."""
import json

import bench


def test_the_line_keeps_the_headline_and_fits_what_is_recorded():
    head = dict(zip(bench.CONTRACT, ("layer prove time", 0.0902198530000078, "s", 1, 20, 5, 90.2198530000078, False, "weak", None, "u32", "synthetic")))
    part = {"kernel": "k" * 300, "achieved": 15.84666659015277, "traffic": None, "note": "n" * 2000, "frac_note": "n" * 200}
    run = {"run": "skip-connection", "wall_s": 0.096, "phases_ms": {"prove_ms": 0.3, "load_inputs_ms": 57.1}}
    full = {**head, "config": {"model": "m", "workload": "w" * 900, "setup_note": "n" * 500}, **{"roofline_%d" % i: dict(part) for i in range(12)},
            "drivers_chain": {"runs": [run] * 7, "setup_runs": [run] * 16, "chain_wall_s": 1.469, "note": "n" * 300}}
    text = bench.line_of(full)
    line = json.loads(text)
    assert "\n" not in text and len(text) <= bench.LINE_MAX < 8000
    assert all(line[k] == full[k] for k in bench.CONTRACT) and set(line) == set(full)
    assert line["roofline_3"] == {"kernel": "k" * 69 + "...", "achieved": 15.8467, "traffic": None}
    assert line["drivers_chain"] == {"wall_s": [["skip-connection", 0.096]] * 7, "chain_wall_s": 1.469}
    assert full["roofline_3"] == part                                    # the record itself is as it was
    more = {**full, **{"extra_%d" % i: dict(part) for i in range(120)}}      # past the limit: the last entries go, and are named
    text = bench.line_of(more)
    line = json.loads(text)
    assert len(text) <= bench.LINE_MAX and line["left_out"][-1] == "extra_119" and set(line) - {"left_out"} | set(line["left_out"]) == set(more)
