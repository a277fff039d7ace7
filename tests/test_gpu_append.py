"""Large batches are appended on the device, small ones by the host: one batch
and the same clauses in small batches must leave the same formula, units and
status, for the units' order, chains past the device's limit, conflicts,
tautologies, duplicates, empty and long clauses, and refused ones."""
import numpy as np
import pytest

from tests.common import diff

pytestmark = pytest.mark.gpu
EDGE = 8192  # clauses from which a batch goes to the device


def _arrays(cls):
    off = np.zeros(len(cls) + 1, np.uint64)
    off[1:] = np.cumsum([len(c) for c in cls])
    return off, np.array([2 * abs(x) + (x < 0) for c in cls for x in c], np.uint32)


def _session(nvars, batches, step, first=None, simplify_between=False):
    from parafrost_amd.simplifier import Simplifier
    s = Simplifier(0, phases=1)
    try:
        off, lits = _arrays(first or [])
        s.upload(0 if first is None else nvars, off, lits)
        for b in batches:
            off, lits = _arrays(b)
            n = len(b)
            for i in range(0, n, step or n):
                j = min(n, i + (step or n))
                s.append(nvars, off[i:j + 1], lits)
            if simplify_between:
                s.simplify()
        return s.result(s.simplify())
    finally:
        s.close()


def _same(nvars, batches, **kw):
    a, b = _session(nvars, batches, 0, **kw), _session(nvars, batches, EDGE - 1, **kw)
    print(a.status, a.sizes.shape, flush=True)
    d = diff(a, b)
    assert not d, d
    return a


def _units(cls):
    """The units of the clauses in order, each under the ones before it."""
    true, units = set(), []
    for c in cls:
        free = {x for x in c if -x not in true}
        if len(free) == 1 and not free & true and not any(-x in c for x in free):
            true |= free
            units += free
    return units


def _random(rng, nvars, n, sizes=(2, 3, 3, 4)):
    k = rng.choice(sizes, n)
    v = rng.integers(1, nvars + 1, k.sum()) * rng.choice([-1, 1], k.sum())
    return [list(map(int, c)) for c in np.split(v, np.cumsum(k)[:-1])]


@pytest.mark.parametrize("n", [EDGE - 1, EDGE, EDGE + 1, 3 * EDGE + 77])
@pytest.mark.parametrize("units", [0, 1, 300])
def test_random_batches(n, units):
    """Repeated variables make duplicates and tautologies, units shorten and
    satisfy later clauses."""
    rng = np.random.default_rng(n + units)
    nvars = n // 3
    cls = _random(rng, nvars, n - units)
    for at in rng.integers(0, len(cls), units):
        cls.insert(int(at), [int(rng.integers(1, nvars + 1))])
    two = _random(rng, nvars + 500, EDGE, (2, 3, 3, 5))
    _same(nvars + 500, [cls, two], simplify_between=True)


@pytest.mark.parametrize("chain", [1, 7, 8, 9, 31, 32, 33, 200])
def test_unit_chains(chain):
    """Each unit makes the next clause one: as many passes as links, past 32
    the host's turn; the reversed chain shortens nothing in the batch."""
    rng = np.random.default_rng(chain)
    pad = _random(rng, 5000, EDGE)
    pad = [c for c in pad if min(map(abs, c)) > 250] + [[300, 400, 500]] * EDGE
    links = [[1]] + [[-i, i + 1] for i in range(1, chain)]
    for order in (links, links[::-1]):
        cls = []
        for i, c in enumerate(order):
            cls += pad[i * 60:(i + 1) * 60] + [c, [c[-1], 777], [-c[-1], 700 + i, 901]]
        a = _same(5000, [cls + pad[len(order) * 60:][:EDGE]])
        if a.status:
            units = _units(cls + pad[len(order) * 60:][:EDGE])
            assert list(a.units[:len(units)]) == [2 * abs(x) + (x < 0) for x in units]


@pytest.mark.parametrize("kind", ["empty", "conflict", "long", "longest_device", "kept_units", "all_satisfied"])
def test_special_clauses(kind):
    rng = np.random.default_rng(5)
    cls = _random(rng, 9000, EDGE + 100, (3, 4, 5))
    first = [[1, 2], [-3, 4, 5]]
    if kind == "empty":
        cls[200] = []
    elif kind == "conflict":
        cls[50], cls[8000] = [17], [-17]
    elif kind == "long":
        cls[70] = [int(x) for x in rng.permutation(8000)[:400] + 1]
    elif kind == "longest_device":
        cls[70], cls[71] = ([int(x) for x in rng.permutation(8000)[:n] + 1] for n in (128, 129))
    elif kind == "kept_units":
        cls[0:40] = [[i % 13 + 1] for i in range(40)]
    else:
        cls = [[8] if i == 0 else [8, -(i % 5000 + 9)] for i in range(EDGE)]
    _same(9000, [cls], first=first)


@pytest.mark.parametrize("lit", [0, 1, 2 * 9001, 2**32 - 1])
def test_refused_literal_leaves_the_formula(lit):
    from parafrost_amd.simplifier import PfsError, Simplifier
    rng = np.random.default_rng(9)
    cls = _random(rng, 9000, EDGE, (3, 4))
    off, lits = _arrays(cls)
    bad = lits.copy()
    bad[len(bad) // 2] = lit
    s = Simplifier(0, phases=1)
    try:
        s.upload(9000, *_arrays([[1, 2]]))
        with pytest.raises(PfsError):
            s.append(9000, off, bad)
        s.append(9000, off, lits)
        a = s.result(s.simplify())
    finally:
        s.close()
    d = diff(a, _session(9000, [cls], EDGE - 1, first=[[1, 2]]))
    assert not d, d
