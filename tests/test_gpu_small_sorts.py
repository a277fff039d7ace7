"""The one-launch sorts, placements, scans and list collections end at fixed
sizes (2,048 and 8,192 items; scans at 8,192, 32,768 and 65,536; lists
appended up to 131,072): formulas of independent components with exactly that
many candidates and elected variables, one less and one more, against the
oracle."""
import numpy as np
import pytest

from oracle import oracle
from parafrost_amd import gen
from tests.common import diff

pytestmark = pytest.mark.gpu


def _components(n, seed):
    """n components of two variables: (a | b), (-a | -b) in n/2 of them, in
    the others the same two clauses widened by a variable of their own
    repeated to 3 to 40 clauses, so that list lengths of every kind occur."""
    rng = np.random.default_rng(seed)
    cls, v = [], 0
    for i in range(n):
        a, b = v + 1, v + 2
        v += 2
        kind = int(rng.integers(0, 40))
        if kind < 30:
            cls += [[a, b], [-a, -b]]
        else:
            k = int(rng.integers(3, 41)) if kind == 39 else int(rng.integers(2, 7))
            c, d = v + 1, v + 2
            v += 2
            for _ in range(k):
                s = rng.integers(0, 2, 4) * 2 - 1
                cls.append([int(s[0]) * a, int(s[1]) * b, int(s[2]) * c][: int(rng.integers(2, 4))] + [int(s[3]) * d])
    return gen.from_clauses(v, cls)


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4097, 8191, 8192, 8193, 16384, 32767,
                               32769, 65535, 65537])
def test_component_counts(n):
    from parafrost_amd.simplifier import Simplifier
    cnf = _components(n, n)
    s = Simplifier(0, phases=2, bce=1)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits)
        g = s.result(s.simplify())
    finally:
        s.close()
    r = oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, det=1, phases=2, bce_en=1)
    print(n, cnf.maxvar, [x["elected"] for x in g.rounds], flush=True)
    d = diff(g, r)
    assert not d, d
