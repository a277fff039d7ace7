"""Root propagation runs narrow levels in one launch and hands levels of more
than 16,384 list entries to the whole device: chains of units of every
length, bursts on both sides of that size, bursts inside chains, a conflict
at the end of each, against the generators' own propagation."""
import numpy as np
import pytest

from parafrost_amd import gen

pytestmark = pytest.mark.gpu


def _formula(chain, burst, tail, conflict, seed):
    """A unit, a chain of implications, a burst of 'burst' implications from
    its end (each of them implying one more variable together with the chain's
    end), a second chain of length 'tail' from the last of these, then
    clauses over variables that stay, some widened by false literals."""
    rng = np.random.default_rng(seed)
    n0 = chain + 2 * burst + tail + 2
    keep = 60
    cls = [[1]]
    cls += [[-i, i + 1] for i in range(1, chain + 1)]
    end = chain + 1
    cls += [[-end, end + i] for i in range(1, burst + 1)]
    cls += [[-end, -(end + i), end + burst + i] for i in range(1, burst + 1)]
    last = end + 2 * burst
    cls += [[-(last + i), last + i + 1] for i in range(tail)]
    last += tail
    if conflict:
        cls += [[-last, last + 1], [-last, -(last + 1)]]
    for _ in range(4 * keep):
        vs = rng.choice(np.arange(n0 + 1, n0 + keep + 1), 3, replace=False)
        c = [int(v) * (1 if rng.random() < 0.5 else -1) for v in vs]
        r = rng.random()
        if r < 0.3:
            c.append(-int(rng.integers(1, last + 1)))
        elif r < 0.4:
            c.append(int(rng.integers(1, last + 1)))
        cls.append(c)
    order = rng.permutation(len(cls))
    return gen.from_clauses(n0 + keep, [cls[i] for i in order])


@pytest.mark.parametrize("chain,burst,tail", [(0, 0, 0), (1, 1, 1), (700, 0, 0), (5, 63, 65), (3, 8190, 2), (3, 8192, 40),
                                              (2, 8193, 0), (40, 30001, 300)])
@pytest.mark.parametrize("conflict", [False, True])
def test_levels(tmp_path, chain, burst, tail, conflict):
    from parafrost_amd.simplifier import Simplifier
    cnf = _formula(chain, burst, tail, conflict, 7 * chain + burst + tail)
    want, refuted = gen.prepare(cnf)
    assert refuted == conflict
    p = tmp_path / "f.cnf"
    gen.write_dimacs(cnf, str(p))
    s = Simplifier(0)
    try:
        info = s.parse_dimacs(p.read_bytes())
        assert info["status"] == (0 if conflict else 2)
        if conflict:
            return
        r = s.result(2)
        trail = s.trail()
    finally:
        s.close()
    sizes = np.diff(want.offsets).astype(np.int64)
    order = np.lexsort((want.lits, np.repeat(np.arange(want.nclauses), sizes)))
    assert np.array_equal(np.sort(trail), np.sort(want.trail))
    assert np.array_equal(r.sizes, sizes) and np.array_equal(r.lits, want.lits[order])
