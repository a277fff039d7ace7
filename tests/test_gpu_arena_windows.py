"""A private arena that is large enough for a session stays so when it grows a
little: the scratch of the occurrence table and of ERE, which larger arenas let
a context hold, makes way there as it does within a memory budget."""
import numpy as np
import pytest

from parafrost_amd import gen
from parafrost_amd.simplifier import Arena, PfsError, Simplifier

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gates", [3000])
def test_enough_stays_enough(gates):
    cnf, refuted = gen.prepare(gen.tseitin(gates, max(10, gates // 400), max(1, gates // 2000), 3, sat_outputs=True))
    assert not refuted
    n, third = cnf.nclauses, cnf.nclauses // 3

    def session(arena=None):
        s = Simplifier(0, arena=arena, phases=2)
        try:
            s.upload(0, np.zeros(1, np.uint64), np.zeros(0, np.uint32))
            for a in range(0, n, third):
                s.append(cnf.maxvar, cnf.offsets[a:min(n, a + third) + 1], cnf.lits)
                s.simplify()
            return s.result(s.simplify()).lits.tobytes(), s.memory()[1]
        except PfsError as e:
            assert "arena" in str(e)
            return None, 0
        finally:
            s.close()

    want, peak = session()
    got = []
    for k in range(40):
        arena = Arena(int(peak * (0.45 + 0.85 * k / 40)), 0)
        try:
            got.append(session(arena)[0])
        except PfsError:  # too small for a context
            got.append(None)
        finally:
            arena.close()
    ok = [x is not None for x in got]
    print(peak, "".join(str(int(x)) for x in ok), flush=True)
    assert ok == sorted(ok) and ok[-1]
    assert all(x == want for x in got if x is not None)
