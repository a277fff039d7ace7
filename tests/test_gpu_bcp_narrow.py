"""A level of root propagation stays in the one-workgroup launch by what it
takes there, not by its list entries alone: levels of many literals with short
lists, and of few literals with long ones, go to the whole device (kernel
counts), with the generators' own propagation as the result either way."""
import numpy as np
import pytest

from parafrost_amd import gen

pytestmark = pytest.mark.gpu
OFF = {"ve": 0, "ve+": 0, "sub": 0, "bce": 0, "ere": 0, "phases": 0, "profilegpu": 1}


@pytest.mark.parametrize("lits,entries,wide", [(1, 1, 0), (96, 1, 0), (97, 1, 2), (4000, 2, 2), (8000, 2, 2),
                                               (1, 512, 0), (1, 513, 1), (12, 512, 0), (13, 512, 1), (24, 256, 0),
                                               (1, 16000, 1)])
def test_levels_by_turns(lits, entries, wide):
    """Units x_1..x_n, each in 'entries' clauses: x_i -> y_i, y_i -> z_i for the
    first 90, and clauses over variables that stay.  wide: the levels that go to
    the whole device, the x by literals or entries, the y by literals."""
    from parafrost_amd.simplifier import Simplifier
    rng = np.random.default_rng(lits + entries)
    n, keep, deep = lits, 300, min(lits, 90)
    cls = [[-i, n + i] for i in range(1, n + 1)]
    cls += [[-(n + i), 2 * n + i] for i in range(1, deep + 1)]
    for i in range(1, n + 1):
        f = 3 * n + 1 + rng.integers(0, keep, (entries - 1, 2))
        f[:, 1] = np.where(f[:, 0] == f[:, 1], 3 * n + 1 + (f[:, 0] - 3 * n) % keep, f[:, 1])
        cls += [[-i, int(a), int(b)] for a, b in f]
    cls += [[3 * n + q, 3 * n + q + 1, 3 * n + q + 2] for q in range(1, keep - 1)]
    cnf = gen.from_clauses(3 * n + keep, [cls[i] for i in rng.permutation(len(cls))])
    units = np.arange(1, n + 1, dtype=np.uint32) * 2
    want, refuted = gen.prepare(gen.Cnf(cnf.maxvar, np.concatenate([cnf.offsets, cnf.offsets[-1] + np.arange(1, n + 1, dtype=np.uint64)]),
                                        np.concatenate([cnf.lits, units])))
    assert not refuted
    s = Simplifier(0, **OFF)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits)
        s.append(cnf.maxvar, np.arange(n + 1, dtype=np.uint64), units)
        r = s.result(s.simplify())
        calls = {k: c for k, (_, c) in s.kernel_times().items() if k.startswith("bcp_")}
    finally:
        s.close()
    print(lits, entries, calls, flush=True)
    assert calls.get("bcp_visit_k", 0) == wide
    sizes = np.diff(want.offsets).astype(np.int64)
    order = np.lexsort((want.lits, np.repeat(np.arange(want.nclauses), sizes)))
    assert np.array_equal(np.sort(r.units), np.sort(want.trail))
    assert np.array_equal(r.sizes, sizes) and np.array_equal(r.lits, want.lits[order])
