"""bench.py's one line for every kind of decode step a workload can take."""
import json
import sys

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload,mode,kernel", [
    ("flashnano-1.5-tiny", "persistent", "persistent decode step"), ("flashnano-1.5-tiny", "graph", "graph-captured"),
    ("flashnano-1.5-tiny", "eager", "gemv gate/up"), ("flashlighting-2.0", "graph", "graph-captured"),
    ("flashlighting-2.0", "eager", "eager decode step")])
def test_bench_reports_every_step_mode(monkeypatch, capsys, workload, mode, kernel):
    import bench
    monkeypatch.setattr(sys, "argv", ["bench.py", "--workload", workload, "--prompt", "40", "--steps", "3",
                                      "--warmup", "1", "--cpu-seconds", "0", "--step-mode", mode])
    assert bench.main() == 0
    line = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert line["steps"] == 3 and line["value"] > 0 and line["roofline"]["kernel"].startswith(kernel)
