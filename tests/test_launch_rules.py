"""The rules that choose between kernels, on the CPU."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_launch_rules(tmp_path):
    exe = tmp_path / "rules_test"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", f"-I{ROOT / 'antiradiancecuts_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "rules_test.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout
