"""ELS takes clauses of up to four literals in registers and longer ones from
the pool: sizes on both sides, over few enough variables that substituted
clauses hold equal and opposite literals and become units, against the
oracle; and numbers of clauses around a tile of the pass that lists them."""
import numpy as np
import pytest

from parafrost_amd import gen
from parafrost_amd.simplifier import Simplifier
from tests.test_gpu_els import lists, oracle_els

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(2,), (3,), (4,), (5,), (3, 4, 5), (2, 6, 9)])
@pytest.mark.parametrize("nclauses", [60, 2000, 2049])
@pytest.mark.parametrize("anti", [0, 6])
def test_lengths(sizes, nclauses, anti):
    rng = np.random.default_rng(nclauses + sum(sizes) + anti)
    parts = [gen.equivalences(600, max(1, nclauses // len(sizes)), 100, 5, k=max(3, k), seed=900 + k + anti, anti=anti)
             for k in sizes]
    cls = [c for p in parts[:1] for c in lists(np.diff(p.offsets).astype(np.int64), p.lits)]
    for p, k in zip(parts[1:], sizes[1:]):  # the first part's classes, the others' long clauses
        cls += [c for c in lists(np.diff(p.offsets).astype(np.int64), p.lits) if len(c) == max(3, k)]
    cls = [[(-1) ** (x & 1) * (x >> 1) for x in c] for c in cls]
    cnf = gen.from_clauses(600, [cls[i] for i in rng.permutation(len(cls))])
    learnt = (rng.random(cnf.nclauses) < 0.2).tolist()
    st, o = oracle_els(cnf, learnt, set())
    flags = np.array([1 if x else 0 for x in learnt], np.uint8)
    s = Simplifier(0)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits, flags=flags, lbd=np.where(flags == 1, 3, 0).astype(np.uint32))
        info = s.decompose()
        print(info, flush=True)
        assert info["status"] == st
        if not st:
            return
        r = s.result(2)
    finally:
        s.close()
    keep = [(c, lr) for c, lr in zip(o.clauses, o.learnt) if c is not None]
    want = [sorted(c) for c, lr in keep if not lr] + [sorted(c) for c, lr in keep if lr]
    assert [sorted(c) for c in lists(r.sizes, r.lits)] == want
    assert r.resolved.tolist() == o.stack
    assert r.vstate.tolist() == o.vstate
    assert sorted(r.units.tolist()) == sorted(o.trail)
