"""A large batch that holds a literal out of range beside clauses that become
units is refused and leaves the formula usable: the batch without that literal,
appended next, leaves what it leaves in a new session in small batches."""
import pytest

from tests.common import diff
from tests.test_gpu_append import EDGE, _arrays, _random, _session

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alone", [False, True])
@pytest.mark.parametrize("where", [0, EDGE // 2, EDGE])
def test_refused_literal_beside_units(where, alone):
    import numpy as np
    from parafrost_amd.simplifier import PfsError, Simplifier
    rng = np.random.default_rng(where + alone)
    cls = _random(rng, 9000, EDGE, (4, 5))
    cls[EDGE // 3] = [2]
    cls[EDGE // 2 + 7] = [-4, -2]
    bad = cls[:where] + [[9001] if alone else [3, 9001, -6]] + cls[where:]
    s = Simplifier(0, phases=1)
    try:
        s.upload(9000, *_arrays([[1, 2, 5]]))
        print("refused at", where, "alone", alone, flush=True)
        with pytest.raises(PfsError):
            s.append(9000, *_arrays(bad))
        s.append(9000, *_arrays(cls))
        a = s.result(s.simplify())
    finally:
        s.close()
    d = diff(a, _session(9000, [cls], EDGE - 1, first=[[1, 2, 5]]))
    assert not d, d
