"""Host-compilable rules of the native code: each bounded wait of the front
factorisation has the whole limit, and no solve takes more columns than the lane
offsets of its products allow."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "spdepy_amd", "csrc")


@pytest.mark.parametrize("name", ["wait_budget", "solve_columns"])
def test_native_rule(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "native", name + ".cpp"),
                    "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_every_wait_starts_its_own_count():
    # both waits of the kernel begin a count before their loop
    with open(os.path.join(CSRC, "front.hip")) as f:
        src = f.read()
    for name in ("void wait_tile", "int wait_columns"):
        body = src[src.index(name):]
        body = body[:body.index("\n}\n")]
        loop = min(i for i in (body.find("while ("), body.find("for (;;)")) if i >= 0)
        assert "w.begin();" in body[:loop], name
