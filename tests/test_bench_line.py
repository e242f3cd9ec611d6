"""The bench's line of results stays short whatever the number of rounds."""
import json

import bench


def test_result_line_has_no_list_of_rounds(capsys):
    rounds = [{"ssr": 0.0123456789, "wall_s": 1.23456789, "X": -9.87654321}] * 64
    run = {"rounds": rounds, "ssr_floor": 0.005, "fixed_ssr": {"round": 41}}
    out = {"metric": "m", "value": 1.5, "round": dict(run, value=1.6), "hiv_reference_run": run,
           "roofline": {"achievable_all": {"copy": 1.0}}}
    line = json.loads(bench.result_line(out))
    assert line["value"] == 1.5 and line["roofline"] == out["roofline"]
    assert line["round"] == dict(run, value=1.6, rounds=64) and line["hiv_reference_run"]["fixed_ssr"]["round"] == 41
    assert len(json.dumps(line)) < 1000
    assert run["rounds"] is rounds      # the measurement itself keeps them
    err = capsys.readouterr().err
    assert json.loads(err.splitlines()[0].split("rounds: ", 1)[1]) == rounds
