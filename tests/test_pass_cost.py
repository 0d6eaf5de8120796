"""The choice between passes of several steps and single steps (flb_cost.h) at
domains that were measured both ways.  Host build; no GPU."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_measured_domains_take_the_faster_way(tmp_path):
    exe = tmp_path / "pass_cost_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", f"-I{ROOT / 'flowlb_amd' / 'csrc'}",
                    str(ROOT / "tests" / "host" / "pass_cost_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
