"""From 4,194,304 literals on the occurrence table is built in two steps of
partitioning: sizes around that limit and around whole ranges, with ranges
that hold nothing, literals that fill many tiles and lists at the ends of
ranges, against the table of one atomic per occurrence and the oracle."""
import numpy as np
import pytest

from oracle import oracle
from parafrost_amd import gen
from tests.common import diff

pytestmark = pytest.mark.gpu


def _formula(nvars, nclauses, seed):
    rng = np.random.default_rng(seed)
    # variables at the ends of ranges, in a few dense stretches, and one in many clauses
    edges = np.concatenate([np.arange(k - 3, k + 4) for k in range(0, nvars + 512, 512)])
    edges = edges[(edges >= 1) & (edges <= nvars)]
    dense = np.concatenate([np.arange(s, min(nvars, s + 9000)) for s in (1, max(1, nvars // 3), max(1, nvars - 8000))])
    size = rng.choice([2, 3, 3, 4], nclauses)
    pick = rng.random(size.sum())
    v = np.where(pick < 0.5, rng.choice(dense, size.sum()), rng.choice(edges, size.sum()))
    cid = np.repeat(np.arange(nclauses), size)
    first = np.concatenate([[0], np.cumsum(size)[:-1]])
    v[first[: nclauses // 3]] = nvars  # the last variable in a third of the clauses
    lit = 2 * v + (rng.random(size.sum()) < 0.5)
    key = np.unique(cid << 32 | lit)
    keep = np.ones(len(key), bool)
    keep[1:] = (key[1:] >> 1) != (key[:-1] >> 1)
    key = key[keep]
    n = np.bincount(key >> 32, minlength=nclauses)
    key, n = key[n[key >> 32] > 1], n[n > 1]
    off = np.zeros(len(n) + 1, np.uint64)
    off[1:] = np.cumsum(n)
    return gen.Cnf(nvars, off, (key & 0xFFFFFFFF).astype(np.uint32))


def _run(cnf, **opts):
    from parafrost_amd.simplifier import Simplifier
    s = Simplifier(0, phases=2, bce=1, **opts)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits)
        return s.result(s.simplify())
    finally:
        s.close()


@pytest.mark.parametrize("nvars", [2097150, 2097151, 2097152, 2162686, 2162687, 2162688, 2500001, 5242879])
@pytest.mark.parametrize("nclauses", [3, 150000])
def test_sizes(nvars, nclauses):
    cnf = _formula(nvars, nclauses, nvars + nclauses)
    a = _run(cnf)
    print(nvars, cnf.nclauses, [x["elected"] for x in a.rounds], flush=True)
    d = diff(a, _run(cnf, otpranges=0))
    assert not d, d
    if nvars in (2097151, 2162687):
        d = diff(a, oracle.simplify(cnf.maxvar, cnf.offsets, cnf.lits, det=1, phases=2, bce_en=1))
        assert not d, d


@pytest.mark.parametrize("tile", [10, 13])
def test_tiles_and_least_room(tile):
    """Other tiles of the first step, and the least room in the pool."""
    cnf = _formula(2300000, 200000, tile)
    a = _run(cnf)
    for opts in ({"otptile": tile}, {"otptile": tile, "otpxcd": 0}, {"literalsmul": 0}):
        d = diff(a, _run(cnf, **opts))
        assert not d, (opts, d)


@pytest.mark.parametrize("nvars", [511, 512, 7200, 33333, 524286, 524287, 524288, 1048574, 1048575, 1048576])
def test_range_widths(nvars):
    """One step: ranges of 1,024 to 4,096 literals by their number."""
    cnf = _formula(nvars, 150000, nvars)
    d = diff(_run(cnf), _run(cnf, otpranges=0))
    assert not d, d


@pytest.mark.parametrize("nvars", [2300000, 4300000])
def test_one_step_without_room(nvars):
    """Long clauses and no room for resolvents: the idle pool cannot hold the
    second step's pairs, and one step builds the table, in ranges of 4,096 or
    8,192 literals."""
    from parafrost_amd.simplifier import Simplifier
    rng = np.random.default_rng(nvars)
    v = np.sort(rng.choice(nvars, (60000, 9), replace=True) + 1, axis=1)
    v[:20000, 0] = 1  # a list of many tiles
    v = v[(np.diff(v, axis=1) > 0).all(axis=1)]
    lits = (2 * v + rng.integers(0, 2, v.shape)).astype(np.uint32).ravel()
    cnf = gen.Cnf(nvars, np.arange(len(v) + 1, dtype=np.uint64) * 9, lits)
    s = Simplifier(0, phases=1, bce=1, profilegpu=1, literalsmul=0)
    try:
        s.upload(nvars, cnf.offsets, cnf.lits)
        a = s.result(s.simplify())
        names = set(s.kernel_times())
    finally:
        s.close()
    print(sorted(n for n in names if n.startswith("otp")), flush=True)
    assert "otp_range_k<true>" in names and "otp2_range_k" not in names
    s = Simplifier(0, phases=1, bce=1, otpranges=0)
    try:
        s.upload(nvars, cnf.offsets, cnf.lits)
        d = diff(a, s.result(s.simplify()))
    finally:
        s.close()
    assert not d, d
