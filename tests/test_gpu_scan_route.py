"""The offset scan of the cell-pair list by the counting kernel (single-point
calls up to 4,096 cells, MD steps and grid updates while no system has more
than 1,024) against the scan launched after it: around both lines the list
that a single-point call leaves equals the one of a grid update, entry for
entry, and a batch's list is that of its members alone."""
import numpy as np
import pytest

from omegagene_amd import gen
from omegagene_amd.engine import Batch, System

pytestmark = pytest.mark.gpu

CFG = {"cutoff": 10.0, "nsgrid-cutoff": 10.5, "nsgrid-update-intvl": 1, "gap-bug": 0, "integrator": "leapfrog-presto",
       "constraint": "none", "time-step": 0.5, "log-cap": 8}


def _list(s):
    ids, gcrd, _ = s.grid()
    cp, head = s.cell_pairs()
    assert len(cp) == head[-1] > 0 and np.all(np.diff(head) >= 0)
    return ids, gcrd, cp, head


@pytest.mark.parametrize("waters", [2720, 2731, 2780, 5462, 10922, 10930])   # 1,020 to 4,099 cells before padding
def test_list_of_a_call_equals_the_list_of_an_update(waters):
    s = System(gen.build_system(waters, seed=waters), CFG)
    lists = []
    for k in range(4):   # in turn: each route starts from what the other left
        if k % 2: s.nsgrid_update()
        else: s.energy_force(rebuild=True)
        lists.append(_list(s))
    s.close()
    print("[gpu-test] scan route", 3 * waters, "atoms", len(lists[0][3]) - 1, "cells", flush=True)
    for other in lists[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(lists[0], other))


@pytest.mark.parametrize("sizes", [(1000, 2700), (1000, 2800), (2700,) * 9])   # under the line; a member over it; all over it
def test_list_in_a_batch_equals_the_list_alone(sizes):
    lss = [gen.build_system(n, seed=n + k) for k, n in enumerate(sizes)]
    ss = [System(ls, CFG) for ls in lss]
    b = Batch()
    for s in ss:
        b.add(s)
    b.run(3)
    got = [(s.state(), _list(s)) for s in ss]
    b.close()
    for s in ss:
        s.close()
    for ls, (st, li) in list(zip(lss, got))[:2]:
        s = System(ls, CFG)
        s.run(3)
        assert all(np.array_equal(x, y) for x, y in zip(s.state(), st))
        assert all(np.array_equal(x, y) for x, y in zip(_list(s), li))
        s.close()
