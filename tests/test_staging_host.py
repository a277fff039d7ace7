"""The staged download on a host build (tests/staging/staging_host.cpp), under
ThreadSanitizer and AddressSanitizer: whole pieces and remainders through rings
of one to four slots, and what it does where a thread cannot be started (leaves
everything to the caller), a copy cannot be queued or a wait fails (says so)."""
import json
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("sanitizer", ["thread", "address,undefined"])
def test_staged_copy(sanitizer):
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "staging_host")
        subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", f"-fsanitize={sanitizer}",
                        "-o", exe, os.path.join(HERE, "staging", "staging_host.cpp")], check=True)
        r = subprocess.run([exe, "400"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert json.loads(r.stdout.strip().splitlines()[-1]) == {"done": 100, "not_started": 100, "failed": 200}
