"""The rule by which resident launches of several streams run at the same
time (csrc/vti_res_gate.h), in a discrete-event simulation on the CPU
(tests/res_gate.cpp): the launches on the chip together always fit it, those
that fit do run together, a single stream waits for nothing.  With the waits
left out the simulation must see launches that do not fit together."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "thesis-source-code_amd", "csrc")


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("gate") / "res_gate")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-I", CSRC,
                    os.path.join(HERE, "res_gate.cpp"), "-o", exe], check=True, timeout=300)
    return exe


def _run(prog, *args):
    r = subprocess.run([prog, *args], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return {k: int(v) for k, v in re.findall(r"(launches|violations|together|stream) (\d+)", r.stdout)}


def test_launches_on_the_chip_together_fit_it(prog):
    n = _run(prog)
    assert n["violations"] == 0 and n["stream"] == 0
    assert n["together"] > n["launches"] // 10


def test_missing_waits_are_seen(prog):
    assert _run(prog, "open")["violations"] > 0
