"""The passes that append a batch of clauses on the device, built for the host
with AddressSanitizer and UBSan (tests/items/append_host.cpp): batches that
mix units, empty clauses and a clause that has to be refused stay within their
arrays in every pass that is queued before the flags are read, and batches
without one leave what a sequential loop leaves."""
import json
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_append_passes_within_bounds():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "append_host")
        subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover",
                        "-o", exe, os.path.join(HERE, "items", "append_host.cpp")], check=True)
        r = subprocess.run([exe, "8", "4000"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    # both outcomes, and units and conflicts among what was taken
    assert min(out["refused"], out["taken"], out["units"], out["refuted"], out["kept"]) > 1000
