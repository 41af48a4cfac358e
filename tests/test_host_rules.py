"""Rules of the device code that are plain C++ (the persistent PCG's indices,
epochs and exchange memory, the CCD search's re-reads of the minimum), compiled
for the host from the headers the library includes (tests/cpp/host_rules_test.cpp)."""
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "host_rules_test"
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", f"-I{ROOT}/silk_physics_amd/csrc",
                    f"{ROOT}/tests/cpp/host_rules_test.cpp", "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("rule", ["sell", "clear", "epochs", "refresh"])
def test_rule(rules, rule):
    r = subprocess.run([str(rules), rule], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
