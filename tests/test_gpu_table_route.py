"""The occurrence table of a small formula is built by one workgroup only where
that is the faster way: by the clauses and the occurrences for the number of
ranges, not by the clauses alone (kernel counts), with the table that one
atomic per occurrence builds as the result either way."""
import numpy as np
import pytest

from tests.common import diff

pytestmark = pytest.mark.gpu


def _formula(nvars, nclauses, k, seed):
    """Clauses of k variables each, one of every k-th part."""
    rng = np.random.default_rng(seed)
    step = nvars // k
    v = np.arange(k) * step + rng.integers(0, step, (nclauses, k)) + 1
    v[0, -1] = nvars
    lits = np.sort(2 * v + rng.integers(0, 2, v.shape), axis=1).astype(np.uint32)
    return np.arange(nclauses + 1, dtype=np.uint64) * k, lits.reshape(-1)


@pytest.mark.parametrize("nvars,nclauses,k,one", [
    (300, 4096, 100, True), (300, 4097, 100, False), (500, 20000, 3, True), (500, 24576, 3, True), (500, 24577, 3, False),
    (500, 16000, 20, True), (500, 16400, 20, False), (1000, 12288, 3, True), (1000, 12289, 3, False),
    (5119, 4096, 3, True), (5120, 300, 3, False), (7000, 32000, 30, False),
    (7000, 2000, 15, False), (7000, 2000, 16, True), (7167, 4096, 40, True), (7167, 4097, 40, False), (7168, 2000, 40, False)])
def test_one_workgroup_or_ranges(nvars, nclauses, k, one):
    from parafrost_amd.simplifier import Simplifier
    off, lits = _formula(nvars, nclauses, k, nvars + nclauses)
    out = []
    for opts in ({"otpranges": 1}, {"otpranges": 0}):
        s = Simplifier(0, phases=1, bce=1, **opts)
        try:
            s.upload(nvars, off, lits)
            out.append(s.result(s.simplify()))
        finally:
            s.close()
    d = diff(*out)
    assert not d, d
    s = Simplifier(0, profilegpu=1, phases=0, ve=0, sub=0, bce=0, **{"ve+": 0})  # one table, of the whole formula
    try:
        s.upload(nvars, off, lits)
        s.simplify()
        built = [x for x in s.kernel_times() if "otp_" in x]
    finally:
        s.close()
    print(nvars, nclauses, k, built, flush=True)
    assert any("otp_one_k" in x for x in built) == one and any("otp_range_k" in x for x in built) != one
