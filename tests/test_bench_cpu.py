"""bench.py's result line: short enough for a reader that keeps the last 8000
characters of the output, with the per-step records beside it, not lost."""
import copy
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_result_line_without_records():
    step = {"pivot": 19, "timed": True, "energy": -30.963775775258, "phases": {"solve": 0.4331, "split": 0.1461},
            "hxv_calls": 45, "residual": 1.4e-8, "flops_alg": 1.7e12, "seconds": 0.641}
    res = {"metric": "m", "value": 1.0, "config": {"timed_pivots": [19, 38]},
           "dmrg": {"legs": {"mixed": {"gflops": 1.0, "steps": [dict(step) for _ in range(25)]},
                             "fp64": {"gflops": 2.0, "steps": [dict(step) for _ in range(25)]}},
                    "dE_per_step": [1e-13] * 20, "max_abs_dE_mixed_vs_fp64": 1e-13},
           "sweeps_c2": {"sweep_seconds": [2.2, 2.0, 1.9], "energies_per_half_sweep": [-15.5] * 6}}
    whole = copy.deepcopy(res)
    details = bench.split_details(res)
    assert len(json.dumps(whole)) > 8000 > 1000 > len(json.dumps(res))
    assert res["config"] == whole["config"] and res["sweeps_c2"]["sweep_seconds"] == [2.2, 2.0, 1.9]
    for path, records in details.items():  # put back, nothing is missing
        at = res
        *head, last = path.split(".")
        for k in head:
            at = at[k]
        at[last] = records
    assert res == whole
