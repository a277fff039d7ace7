"""The equivalence and AND/OR gate searches on a host build
(tests/items/gates_host.cpp) against their definitions, over lists with
repeated binary clauses, learnt clauses and clauses that hold a literal twice."""
import json
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_gates_by_definition():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "gates_host")
        subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover",
                        "-o", exe, os.path.join(HERE, "items", "gates_host.cpp")], check=True)
        r = subprocess.run([exe, "100000"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["equivalences"] > 1000 and out["gates"] > 1000 and out["repeated"] > 100
