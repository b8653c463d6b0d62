"""The default line of bench.py: one line that a reader who keeps the last few KB of the output has whole, with the figures of
every leg in it."""
import json

import pytest


@pytest.fixture
def bench(monkeypatch):
    import bench as b

    long_text = "x" * 300
    leg = {"metric": "m", "value": 1.8765432109876543e9, "unit": "keys/s", "n_gpus": 1, "steps": 20, "warmup": 5,
           "ms_per_step": 0.5673227499997324, "ms_per_step_spread": {"median": 0.565257499999916, "p95": 0.5689461000045526},
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u8", "data": "synthetic",
           "config": {"workload": "w" * 60, "keys_per_batch": 1 << 20, "text": long_text}, "hit_rate": 0.8481207370758057,
           "parity": "bit-exact " + long_text,
           "roofline": {"bound": "hbm", "achieved": 692.4563365796321, "peak": 8000.0, "unit": "GB/s", "frac": 0.08655704207245402,
                        "kernel": long_text},
           "host_link": {"achieved": 36.13310269772988, "frac": 0.6362240658007086, "frac_of_row_ceiling": 0.9557343875009565,
                         "how": long_text * 3},
           "cpu_baseline": {"value": 263122459.4986933, "unit": "keys/s", "cores": 16, "kind": "port", "sample": long_text},
           "gpu_over_cpu": 7.024441400773152, "refresh_each_step": {"ms_per_step": 0.44155614999823456, "refresh_ms": 0.31024424999799294,
                                                                    "note": long_text},
           "cache_build": {"seconds": 0.17, "frac_of_measured_link": 0.6455631684958456},
           "all_hit_large_output": {"keys_1M": {"frac_of_hbm_peak": 0.7449026687662517}, "note": long_text}}
    lines = []
    monkeypatch.setattr(b, "run_child", lambda *args, **kw: (json.loads(json.dumps(leg)), None))
    monkeypatch.setattr(b, "emit", lambda result: lines.append(json.dumps(result)))
    return b, lines


def _run(b, monkeypatch, *argv):
    monkeypatch.setattr("sys.argv", ["bench.py", *argv])
    b.run_default(b.parse_args())


def test_the_default_line_is_short_enough_to_be_kept_whole(bench, monkeypatch):
    b, lines = bench
    _run(b, monkeypatch)
    assert len(lines) == 1 and len(lines[0]) < 8000, len(lines[0])
    d = json.loads(lines[0])
    for field in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline",
                  "dtype", "data", "config", "roofline", "cpu_baseline"):
        assert field in d
    for short, *_ in b.DEFAULT_LEGS:
        assert d["roofline"]["other_configs"][short]["ms_per_step"] == d[short + "_ms_per_step"] > 0
        assert d["roofline"]["other_configs"][short]["host_link_frac"] > 0


def test_the_legs_in_full_go_to_a_file(bench, monkeypatch, tmp_path):
    b, lines = bench
    _run(b, monkeypatch, "--legs-file", str(tmp_path / "legs.json"))
    legs = json.load(open(tmp_path / "legs.json"))
    assert sorted(legs) == sorted(short for short, *_ in b.DEFAULT_LEGS)
    assert all(leg["host_link"]["how"] and leg["what"] for leg in legs.values())
