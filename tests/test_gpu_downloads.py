"""Results of 4 MiB and more come back through a ring of pinned slots filled
by the device and emptied by several threads: resident formulas with sizes
around that limit and around whole rings, alone and from several threads at
once (one at a time has the ring), read back and compared."""
import threading

import numpy as np
import pytest

from parafrost_amd import gen

pytestmark = pytest.mark.gpu
SLOT, SLOTS = 4 << 20, 4


def _formula(nclauses, seed):
    """Distinct ascending ternary clauses: the resident form is the input."""
    rng = np.random.default_rng(seed)
    v = np.sort(rng.integers(1, 300_000, (nclauses, 3)) * 3 + np.arange(3), axis=1)
    lits = (2 * v + rng.integers(0, 2, (nclauses, 3))).astype(np.uint32)
    return gen.Cnf(1_000_000, np.arange(nclauses + 1, dtype=np.uint64) * 3, lits.reshape(-1))


def _read_back(cnf):
    from parafrost_amd.simplifier import Simplifier
    s = Simplifier(0)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits)
        return s, s.result(2)
    except Exception:
        s.close()
        raise


# a clause takes 8 + 12 + 4 + 1 bytes of a result, 12 of them literals
@pytest.mark.parametrize("nclauses", [1000, SLOT // 25 - 1, SLOT // 25 + 2, SLOT // 12, SLOT // 12 + 1,
                                      SLOT * SLOTS // 12 - 1, SLOT * SLOTS // 12 + 3, 3 * SLOT * SLOTS // 12 + 17])
def test_sizes(nclauses):
    cnf = _formula(nclauses, nclauses)
    s, r = _read_back(cnf)
    s.close()
    assert (r.sizes == 3).all() and r.sizes.shape[0] == nclauses
    assert np.array_equal(r.lits, cnf.lits)
    assert not r.flags.any() and not r.lbd.any()


def test_threads():
    cnfs = [_formula(900_000 + 1000 * i, 50 + i) for i in range(6)]
    ok = [False] * len(cnfs)

    def work(i):
        s, r = _read_back(cnfs[i])
        ok[i] = np.array_equal(r.lits, cnfs[i].lits) and bool((r.sizes == 3).all())
        for _ in range(3):
            ok[i] = ok[i] and np.array_equal(s.result(2).lits, cnfs[i].lits)
        s.close()

    thr = [threading.Thread(target=work, args=(i,)) for i in range(len(cnfs))]
    for t in thr:
        t.start()
    for t in thr:
        t.join()
    assert all(ok), ok
