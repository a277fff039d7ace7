"""The staged per-variable kernels (SUB, the VE decisions and executions) give
a variable a group of 1 to 64 lanes by the number of elected variables and
the size of its lists, and work on the pool where the lists do not fit the
LDS: the numbers of elected variables on both sides of every group size, and
lists around the LDS slice, against the oracle."""
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
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed, trail=cnf.trail)
        g = s.result(s.simplify())
    finally:
        s.close()
    vs = np.zeros(cnf.maxvar + 1, np.uint8)
    vs[cnf.trail >> 1] = 2
    r = oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, assumed=assumed, vstate=vs,
                        nassigned=int(cnf.trail.shape[0]), det=1, **oopts)
    print("elected", [x["elected"] for x in g.rounds], flush=True)
    d = diff(g, r)
    assert not d, d


@pytest.mark.parametrize("gates", [37, 300, 9001, 20011, 45007, 90001, 180023, 400009])
def test_circuits(gates):
    cnf, refuted = gen.prepare(gen.tseitin(gates, max(10, gates // 400), max(1, gates // 2000), 0x6A0 + gates,
                                           sat_outputs=True))
    assert not refuted
    _check(cnf, {"phases": 2, "bce": 1}, {"phases": 2, "bce_en": 1})


def _hub(npos, nneg, size, seed, dup):
    """One variable in npos + nneg clauses of 'size' literals, a share of
    them repeated with one literal more (subsumed) or the hub negated
    (strengthening), over enough other variables for few resolvents to be
    tautologies."""
    rng = np.random.default_rng(seed)
    V = 40
    cls = []
    for i in range(npos + nneg):
        sign = 1 if i < npos else -1
        if cls and rng.random() < dup:
            base = [x for x in cls[int(rng.integers(len(cls)))] if abs(x) != 1][: size - 1]
        else:
            base = [int(v) * (1 if rng.random() < 0.5 else -1) for v in rng.choice(np.arange(2, V + 1), size - 1,
                                                                                    replace=False)]
        if rng.random() < dup:
            extra = [v for v in range(2, V + 1) if v not in [abs(x) for x in base]]
            base = base + [int(rng.choice(extra))]
        cls.append([sign * 1] + base)
    return gen.from_clauses(V, cls)


# words of the staged copies: 5 (VE: 3) per list entry plus the literals; the
# slice of a whole wavefront holds 5,120
@pytest.mark.parametrize("npos,nneg,size", [(1, 1, 3), (31, 33, 4), (64, 64, 5), (65, 63, 5), (250, 250, 5),
                                            (300, 260, 4), (320, 330, 6), (900, 800, 3)])
@pytest.mark.parametrize("dup", [0.0, 0.2])
def test_list_sizes(npos, nneg, size, dup):
    cnf = _hub(npos, nneg, size, 17 * npos + nneg, dup)
    o = {"phases": 1, "bce": 1, "mupos": 100000, "muneg": 100000}
    assumed = np.ones(cnf.maxvar + 1, np.uint8)  # every variable but the hub stays
    assumed[1] = 0
    _check(cnf, o, {"phases": 1, "bce_en": 1, "mu_pos": 100000, "mu_neg": 100000}, assumed)
