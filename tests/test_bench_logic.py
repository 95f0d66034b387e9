"""Host logic of bench.py (no GPU): the drift matcher and the byte model."""
import json

import numpy as np

import bench


def test_match_spikes_identical_trains():
    i = np.array([0, 0, 1, 2, 2, 2], np.int32)
    t = np.array([5, 40, 7, 1, 100, 300], np.int64)
    r = bench.match_spikes(i, t, i.copy(), t.copy(), 3, 50)
    assert r["matched_pairs"] == 6 and r["rms_dt_steps"] == 0.0 and r["unmatched_frac"] == 0.0


def test_match_spikes_shift_and_extra():
    i64 = np.array([0, 0, 1], np.int32)
    t64 = np.array([10, 200, 50], np.int64)
    i32 = np.array([0, 0, 1, 1], np.int32)     # one extra spike, one shifted by 3, one by -4
    t32 = np.array([13, 196, 50, 900], np.int64)
    r = bench.match_spikes(i64, t64, i32, t32, 2, 50)
    assert r["matched_pairs"] == 3
    assert np.isclose(r["rms_dt_steps"], np.sqrt((9 + 16 + 0) / 3))
    assert np.isclose(r["unmatched_frac"], 1 / 7)


def test_match_spikes_outside_window_is_unmatched():
    r = bench.match_spikes(np.array([0]), np.array([0]), np.array([0]), np.array([100]), 1, 50)
    assert r["matched_pairs"] == 0 and r["unmatched_frac"] == 1.0 and r["rms_dt_steps"] is None


def test_state_bytes_follow_brian2_arrays():
    assert bench.state_bytes("brunel", 64) == (17, 9)
    assert bench.state_bytes("brunel", 32) == (9, 5)


def test_chunk_launches_counts_windows_per_graph_chunk():
    # 10,000 steps in chunks of 256 steps, windows of 5: 39 chunks of 52 launches + one of 16 steps (4 launches)
    assert bench.chunk_launches(10000, 256, 5) == 39 * 52 + 4
    assert bench.chunk_launches(10, 256, 5) == 2
    assert bench.chunk_launches(12, 0, 5) == 3  # no graphs: the whole run is one chunk
    assert bench.chunk_launches(7, 4, 1) == 7


def test_drift_horizons_longest_prefix_below_one_step():
    # neuron 0 agrees exactly until step 1000, then a spike moves by 3 steps
    i = np.zeros(4, np.int32)
    t64 = np.array([50, 400, 900, 1200], np.int64)
    t32 = np.array([50, 400, 900, 1203], np.int64)
    rows, below = bench.drift_horizons(i, t64, i, t32, 1, 2000)
    assert below == 1000
    assert rows["1000"]["rms_dt_steps"] == 0.0 and rows["1500"]["rms_dt_steps"] > 1.0
    assert "3000" not in rows  # past the run


def test_hines_valu_roofline_from_committed_counters(monkeypatch):
    out = {"compartments": 528986, "fp64": {"us_per_step": 18.2}, "fp32": {"us_per_step": 13.4}}
    r = bench.hines_valu_roofline(out, "f64", 2048, 1234)
    assert r["bound"] == "valu"
    # 3,154 wave instructions per tree-step (the committed counters) x 2048 trees / 18.2 us
    assert abs(r["valu_instr_per_tree_step"] - 3154) < 1
    assert abs(r["achieved"] - 3153.8 * 2048 / 18.2e-6 / 1e9) < 1
    assert 0.4 < r["frac"] < 0.7
    assert bench.hines_valu_roofline(out, "f64", 100, 1234)["frac"] is None  # another batch: no counters
    assert r["traffic"]["f64_steps_per_launch_measured"] == 200
    # counters of another kernel than the one in the tree are no measurement of it
    monkeypatch.setattr(bench, "source_tag", lambda *names: "0" * 16)
    r = bench.hines_valu_roofline(out, "f64", 2048, 1234)
    assert r["frac"] is None and r["achieved"] is None and r["traffic"] is None


def test_source_tag_ignores_comments_and_space(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    d = tmp_path / "brian2cuda_amd" / "csrc"
    d.mkdir(parents=True)
    texts = ["int f(int x)\n{\n    return x + 1; /* one\n more */\n}\n", "int f(int x)\n{ return x + 1; // 1\n}\n", "int f(int x) { return x + 2; }"]
    tags = []
    for t in texts:
        (d / "k.hip").write_text(t)
        tags.append(bench.source_tag("k.hip"))
    assert tags[0] == tags[1] != tags[2]


def test_compact_line_keeps_the_contract_and_fits():
    form = {k: 0.123456 for k in ("events_per_s", "sim_s_per_wall_s", "ms_per_step", "wall_s", "spikes_per_step",
                                  "events_per_step", "window", "resident", "build_s", "gpu_ms", "options")}
    row = {"neurons": 1, "fp32_batched": form, "fp64_plain": form, "fp32_fast": form, "speedup_fp32_batched_vs_fp64_plain": 2.0}
    drift = {"rms_dt_steps": 1.0, "unmatched_frac": 0.1, "rms_below_1dt_through_steps": 700, "by_horizon": {str(k): row for k in range(20)}}
    contract = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config")
    out = {**{k: "x" * 40 for k in contract}, "fp32_batched": form, "fp64_plain": form,
           "roofline": {"bound": "hbm", "frac": 0.1, "kernels": {"a": {}}, "avg_launch_from": "x" * 100,
                        "atomics": {k: 1.0 for k in ("achieved_per_s", "scatter_sustained_per_s", "frac_of_sustained", "x")}},
           "cpu_baseline": {"value": 1.0, "serial_1_thread": {"a": 1}, "sample": "x" * 300},
           "other_configs": {f"config_{k}": row for k in range(6)},
           "drift_fp32_batched_vs_fp64_plain": {f"net_{k}": drift for k in range(4)},
           "multicompartment": {"trees": 1, "compartments": 2, **{p: {"us_per_step": 1.0} for p in ("fp64", "fp32")},
                                **{f"roofline_{p}": {"frac": 0.5} for p in ("fp64", "fp32")}}}
    c = bench.compact(out)
    assert all(c[k] == out[k] for k in contract)
    assert len(json.dumps(c)) < 4000
    assert c["other_configs"]["config_0"]["us_per_step"]["fp64_plain"] == 123.456
    assert bench.compact({**out, "fp64_plain": None, "roofline": None, "cpu_baseline": None, "other_configs": None,
                          "drift_fp32_batched_vs_fp64_plain": None, "multicompartment": None})["value"] == out["value"]


def test_cpu_info_reports_cores():
    ci = bench.cpu_info()
    assert ci["nproc"] >= 1
