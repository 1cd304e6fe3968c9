"""bench.py's result: one short line of JSON on stdout, the other workloads' records in a file."""
import json
import os
import subprocess
import sys

import pytest

from dotcase import say

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_result_line(gpu, tmp_path):
    say("bench.py --only tail")
    detail = tmp_path / "detail.json"
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--steps", "5", "--warmup", "2",
                        "--no-cpu", "--only", "tail", "--detail", str(detail)],
                       capture_output=True, text=True, timeout=100, check=True)
    (text,) = r.stdout.splitlines()
    assert len(text) < 4096
    line = json.loads(text)
    assert line["value"] > 0 and line["steps"] == 5 and line["n_gpus"] == 1
    assert "secondary" not in line and line["dtype"] == "bf16"
    records = json.loads(detail.read_text())
    assert records["headline"] == line and records["secondary"]
