"""SUB, the VE decisions and executions give a variable whose lists pass a
wavefront's share of the LDS (1,280 words) the whole workgroup's, and leave
it on the pool past that (5,120): lists on both sides of both, one and more
of them than workgroups share a CU, beside small ones, against the oracle."""
import numpy as np
import pytest

from oracle import oracle
from parafrost_amd import gen
from tests.common import diff

pytestmark = pytest.mark.gpu


def _hubs(hubs, occ, size, small, seed):
    """'hubs' variables in 'occ' clauses of 'size' literals each (three of
    them with the other sign, a tenth repeated with a literal more), each
    over its own 40 variables, and 'small' clauses of three literals."""
    rng = np.random.default_rng(seed)
    cls = []
    for h in range(hubs):
        first, hub = 41 * h + 2, 41 * h + 1
        for i in range(occ):
            sign = -1 if i < 3 else 1
            body = rng.choice(np.arange(first, first + 40), size, replace=False) * rng.choice([-1, 1], size)
            if i > 10 and rng.random() < 0.1:
                body[:size - 1] = [x for x in cls[-1] if abs(x) != hub][:size - 1]
                body = np.array(list(dict.fromkeys(body.tolist())))
                if len({abs(int(x)) for x in body}) < len(body):
                    body = body[:-1]
            else:
                body = body[:size - 1]
            cls.append([sign * hub] + [int(x) for x in body])
    base, nsmall = 41 * hubs, max(4, small // 4)
    for _ in range(small):
        v = rng.choice(np.arange(base + 1, base + nsmall + 1), 3, replace=False) * rng.choice([-1, 1], 3)
        cls.append([int(x) for x in v])
    order = rng.permutation(len(cls))
    return gen.from_clauses(base + nsmall, [cls[i] for i in order])


@pytest.mark.parametrize("occ,size", [(90, 9), (93, 9), (105, 9), (108, 9), (250, 7), (364, 9), (367, 9), (425, 9),
                                      (428, 9), (900, 6)])
@pytest.mark.parametrize("hubs,small", [(1, 0), (3, 40000), (60, 3000)])
def test_list_sizes(occ, size, hubs, small):
    from parafrost_amd.simplifier import Simplifier
    cnf = _hubs(hubs, occ, size, small, occ * 10 + hubs)
    mu = occ + 10
    assumed = np.zeros(cnf.maxvar + 1, np.uint8)  # of the hubs' clauses only the hubs are candidates
    assumed[1:41 * hubs + 1] = 1
    assumed[1:41 * hubs + 1:41] = 0
    s = Simplifier(0, phases=2, bce=1, mupos=mu, muneg=mu)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed)
        g = s.result(s.simplify())
    finally:
        s.close()
    r = oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed, det=1, phases=2, bce_en=1, mu_pos=mu,
                        mu_neg=mu)
    print("elected", [x["elected"] for x in g.rounds], flush=True)
    d = diff(g, r)
    assert not d, d
