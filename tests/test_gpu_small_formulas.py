"""Up to 8,192 variables the election's surroundings run in one launch on
either side of its passes, and up to 7,166 variables and 32,768 clauses the
occurrence table in one: both sides of each limit, with elections that break
early, that pass candidates over and that find none, against the oracle."""
import numpy as np
import pytest

from oracle import oracle
from parafrost_amd import gen
from tests.common import diff

pytestmark = pytest.mark.gpu


def _check(cnf, opts, oopts, assumed=None):
    from parafrost_amd.simplifier import Simplifier
    s = Simplifier(0, **opts)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed)
        g = s.result(s.simplify())
    finally:
        s.close()
    r = oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed, det=1, **oopts)
    print(cnf.maxvar, cnf.nclauses, [x["elected"] for x in g.rounds], flush=True)
    d = diff(g, r)
    assert not d, d


def _mixed(nvars, nclauses, seed):
    """Clauses of 2 to 9 literals over all variables, the first ones in many
    more clauses than the others."""
    rng = np.random.default_rng(seed)
    cls = []
    for i in range(nclauses):
        k = min(int(rng.choice([2, 3, 3, 3, 4, 9])), nvars)
        top = nvars if i % 3 else max(k, nvars // 20)
        v = rng.choice(np.arange(1, top + 1), k, replace=False)
        cls.append([int(x) * (1 if rng.random() < 0.5 else -1) for x in v])
    return gen.from_clauses(nvars, cls)


@pytest.mark.parametrize("nvars,nclauses", [(1, 1), (2, 3), (60, 250), (63, 32768), (64, 32769), (1000, 4000), (7165, 9000),
                                            (7166, 20000), (7167, 20000), (8191, 15000), (8192, 15000), (8193, 15000)])
@pytest.mark.parametrize("mu", [32, 10])
def test_limits(nvars, nclauses, mu):
    if nvars < 3:
        cnf = gen.from_clauses(2, [[1, 2]] if nclauses == 1 else [[1, 2], [-1, 2], [1, -2]])
    else:
        cnf = _mixed(nvars, nclauses, nvars + nclauses)
    o = {"phases": 2, "bce": 1, "mupos": mu, "muneg": mu}
    _check(cnf, o, {"phases": 2, "bce_en": 1, "mu_pos": mu, "mu_neg": mu})


@pytest.mark.parametrize("nvars", [300, 8192, 8193])
def test_no_candidates(nvars):
    cnf = _mixed(nvars, 4 * nvars, nvars)
    _check(cnf, {"phases": 2}, {"phases": 2}, np.ones(nvars + 1, np.uint8))


@pytest.mark.parametrize("limit", [{"lcveclausemax": 5}, {"electionsmax": 8}])
def test_election_limits_agree_across_the_size_limit(limit):
    """The same formula with unused variables added past the limit elects the
    same variables (the limits have no counterpart in the CPU simplifier)."""
    from parafrost_amd.simplifier import Simplifier
    cnf = _mixed(3000, 9000, 77)
    got = []
    for nvars in (3000, 9000):
        s = Simplifier(0, phases=1, bce=1, **limit)
        try:
            s.upload(nvars, cnf.offsets, cnf.lits)
            got.append(s.result(s.simplify()))
        finally:
            s.close()
    a, b = got
    print([x["elected"] for x in a.rounds], flush=True)
    assert a.rounds[0]["elected"] and [x["elected"] for x in a.rounds] == [x["elected"] for x in b.rounds]
    assert np.array_equal(a.lits, b.lits) and np.array_equal(a.sizes, b.sizes) and np.array_equal(a.resolved, b.resolved)
