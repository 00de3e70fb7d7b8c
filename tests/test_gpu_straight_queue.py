"""GPU: the batched kernel with a stimulus's first cycle apart (edge tests and
if / case arms as selects from the second on) against the graph form, at the
budgets where the two parts meet. Whole numbers: exact."""
import numpy as np
import pytest

from rtlflow_amd.designs import registry
from rtlflow_amd.model import MODE_GRAPH

BUDGETS = np.array([0, 1, 2, 3, 1, 17, 0, 9, 2, 17, 1, 3], np.uint32)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["alu", "mix", "gated", "rams", "fuzz1", "fuzz2", "fuzz3", "fuzz4",
                                  "kat_shift", "kat_signed", "kat_div"])
def test_queue_first_and_later_cycles(gpu, name):
    cd = registry.get(name)
    n, seed = len(BUDGETS), 0x51
    with cd.model(5) as m:
        got = m.submit_queue(seed, BUDGETS)
    for b in sorted(set(BUDGETS.tolist())):
        with cd.model(n) as m:
            m.begin(seed)
            m.run_cycles(int(b), MODE_GRAPH)
            want = m.hashes()
        pick = BUDGETS == b
        assert (got[pick] == want[pick]).all(), b
