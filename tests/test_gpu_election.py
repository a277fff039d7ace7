"""The election tries each candidate a bounded number of times per pass while
its blocker is decided by another wavefront: chains of candidates each
blocked by the one before it, shorter and longer than one pass can follow,
in order and shuffled, against the oracle; every lane count gives the same
set."""
import numpy as np
import pytest

from oracle import oracle
from parafrost_amd import gen
from tests.common import diff

pytestmark = pytest.mark.gpu


def _chain(n, seed, shuffled):
    """Variables 1..n with clauses (x_i | -x_(i+1)): every variable but the
    ends occurs once with each sign, so the candidate order is the variable
    order and each candidate waits for the one before it; shuffled numbers
    the variables at random."""
    perm = np.arange(1, n + 1)
    if shuffled:
        perm = np.random.default_rng(seed).permutation(perm)
    return gen.from_clauses(n, [[int(perm[i]), -int(perm[i + 1])] for i in range(n - 1)])


@pytest.mark.parametrize("n", [3, 31, 32, 33, 64, 65, 1000, 20011])
@pytest.mark.parametrize("shuffled", [False, True])
def test_chains(n, shuffled):
    from parafrost_amd.simplifier import Simplifier
    cnf = _chain(n, 5 * n, shuffled)
    r = oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, det=1, phases=2, bce_en=1)
    for lanes in (0, 1, 8):
        s = Simplifier(0, phases=2, bce=1, mislanes=lanes)
        try:
            s.upload(cnf.maxvar, cnf.offsets, cnf.lits)
            g = s.result(s.simplify())
        finally:
            s.close()
        print(n, shuffled, lanes, [(x["elected"], x["mis_iterations"]) for x in g.rounds], flush=True)
        d = diff(g, r)
        assert not d, (lanes, d)
