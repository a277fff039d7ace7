"""The device builds the clause pool of an upload: originals before learnts,
literals sorted, LBD and usage kept, whatever the order, the first offset and
the sizes; per-variable arrays given or not; a literal out of range is
refused and the context takes the next upload."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clauses(n, maxvar, seed, longest=40):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        k = min(int(rng.choice([1, 2, 3, 3, 4, 7, longest])), maxvar)
        v = rng.choice(np.arange(1, maxvar + 1), k, replace=False)
        out.append(2 * v + rng.integers(0, 2, k))
    return out


def _arrays(cls, first=0):
    off = np.full(len(cls) + 1, first, np.uint64)
    off[1:] += np.cumsum([len(c) for c in cls]).astype(np.uint64)
    lits = np.concatenate([np.full(first, 0xDEADBEEF, np.uint32)] + cls).astype(np.uint32)
    return off, lits


@pytest.mark.parametrize("n", [1, 2, 255, 257, 4096, 20011])
@pytest.mark.parametrize("learnt", [None, 0.0, 0.4, 1.0])
@pytest.mark.parametrize("first", [0, 7])
def test_pool(n, learnt, first):
    from parafrost_amd.simplifier import Simplifier
    rng = np.random.default_rng(n + first)
    maxvar = 900
    cls = _clauses(n, maxvar, n)
    off, lits = _arrays(cls, first)
    flags = lbd = None
    is_l = np.zeros(n, bool)
    if learnt is not None:
        is_l = rng.random(n) < learnt
        flags = (is_l * (1 | rng.integers(0, 3, n) << 4)).astype(np.uint8)
        lbd = rng.integers(0, 9, n).astype(np.uint32)
    s = Simplifier(0)
    try:
        s.upload(maxvar, off, lits, flags=flags, lbd=lbd)
        r = s.result(2)
    finally:
        s.close()
    order = np.concatenate([np.nonzero(~is_l)[0], np.nonzero(is_l)[0]])
    assert np.array_equal(r.sizes, [len(cls[i]) for i in order])
    assert np.array_equal(r.lits, np.concatenate([np.sort(cls[i]) for i in order]))
    want_f = np.zeros(n, np.uint8) if flags is None else flags[order]
    want_l = np.zeros(n, np.uint32) if lbd is None else np.where(is_l[order], lbd[order], 0)
    assert np.array_equal(r.flags, want_f) and np.array_equal(r.lbd, want_l)


def test_variable_state_and_refusal():
    from parafrost_amd.simplifier import PfsError, Simplifier
    maxvar = 500
    cls = [c for c in _clauses(300, 400, 5) if len(c) > 1]
    off, lits = _arrays(cls)
    vstate = np.zeros(maxvar + 1, np.uint8)
    vstate[0] = 9
    vstate[401:421] = 1  # eliminated before
    vstate[431:436] = 4
    trail = np.array([2 * 450, 2 * 451 + 1, 2 * 460], np.uint32)
    want = vstate.copy()
    want[0] = 0
    want[trail >> 1] = 2
    s = Simplifier(0, phases=1)
    try:
        for bad in (0, 1, 2 * maxvar + 2):
            wrong = lits.copy()
            wrong[len(wrong) // 2] = bad
            with pytest.raises(PfsError, match="literal out of range"):
                s.upload(maxvar, off, wrong)
            with pytest.raises(PfsError):
                s.simplify()
        s.upload(maxvar, off, lits, vstate=vstate, assumed=np.ones(maxvar + 1, np.uint8), trail=trail)
        assert np.array_equal(s.result(2).vstate, want)
        assert np.array_equal(s.trail(), trail)
        r = s.result(s.simplify())
        assert not (r.vstate[1:401] == 1).any()  # assumed: nothing is eliminated
    finally:
        s.close()
