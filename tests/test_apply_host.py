"""The elimination of a variable with more than 2^32 pairs of clauses, and one
whose resolvents are fewer than were counted, on a host build
(tests/items/apply_host.cpp)."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe():
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "apply_host")
        subprocess.run(["g++", "-std=c++17", "-O2", "-o", path, os.path.join(HERE, "items", "apply_host.cpp")],
                       check=True)
        yield path


@pytest.mark.parametrize("case", ["pairs", "few"])
def test_resolvents_of_every_pair(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
