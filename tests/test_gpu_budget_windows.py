"""A memory budget that is enough stays enough when it grows: the scratch of
the occurrence table, which larger budgets hold, makes way for the result's
download."""
import pytest

from parafrost_amd import gen
from parafrost_amd.simplifier import PfsError, Simplifier

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gates", [5000, 20000])
def test_enough_stays_enough(gates):
    cnf, refuted = gen.prepare(gen.tseitin(gates, max(10, gates // 400), max(1, gates // 2000), 3, sat_outputs=True))
    assert not refuted

    def run(budget):
        s = Simplifier(0, mem_budget=budget, phases=2, bce=1)
        try:
            s.upload(cnf.maxvar, cnf.offsets, cnf.lits, trail=cnf.trail)
            r = s.result(s.simplify())
            return r.lits.tobytes(), s.memory()[1]
        except PfsError as e:
            assert "budget" in str(e)
            return None, 0
        finally:
            s.close()

    want, peak = run(0)
    got = [run(b)[0] for b in range(peak // 3, peak + peak // 10, peak // 40)]
    ok = [x is not None for x in got]
    print(peak, "".join(str(int(x)) for x in ok), flush=True)
    assert ok == sorted(ok) and ok[-1]
    assert all(x == want for x in got if x is not None)
