"""The grid's column sort and the cell-pair list at their edges, against the
oracle's grid and list, entry for entry: columns of one atom, of whole and
broken cells, of the last size that is sorted an atom per thread and beyond
(the sort network), more cells than one block of the offset scan, and cells
with more pairs than the counting pass keeps."""
import numpy as np
import pytest

import oracle
from helpers import wrap_inbox
from omegagene_amd import gen
from omegagene_amd.cls import LaunchSet
from omegagene_amd.engine import System

pytestmark = pytest.mark.gpu

BASE = {"cutoff": 12.0, "nsgrid-cutoff": 13.0, "nsgrid-update-intvl": 1, "gap-bug": 0,
        "integrator": "leapfrog-presto", "constraint": "none", "log-cap": 8}


def _columns(counts, L=80.0):
    """An atom per entry of counts stacked in its own grid column, distinct float z, ids shuffled."""
    n = int(sum(counts))
    box = np.diag([L, L, L]).reshape(9)
    o = oracle.Oracle(n, box, BASE["nsgrid-cutoff"])
    nx, ny = o.g.n_cells_xyz[0], o.g.n_cells_xyz[1]
    assert len(counts) <= nx * ny
    rng = np.random.default_rng(5)
    crd = np.zeros((n, 3))
    at = 0
    for k, c in enumerate(counts):
        col = k * (nx * ny // len(counts))
        crd[at:at + c, 0] = (col % nx + 0.5) * L / nx
        crd[at:at + c, 1] = (col // nx + 0.5) * L / ny
        crd[at:at + c, 2] = (np.arange(c) + 0.5) * (L / c)
        at += c
    crd = crd[rng.permutation(n)]
    return LaunchSet(box=box, crd=crd, vel=np.zeros((n, 3)), charge=np.zeros(n), mass=np.ones(n),
                     atom_type=np.zeros(n, np.int32), n_lj_types=1, lj6=np.zeros((1, 1)), lj12=np.zeros((1, 1)),
                     nb15off=np.zeros((0, 2), np.int32))


CASES = {
    "columns": (lambda: _columns([1, 7, 8, 9, 249, 255, 256, 257, 300, 512, 520]), 13.0),
    "one-column": (lambda: _columns([257]), 13.0),
    "scan-blocks": (lambda: gen.build_system(6000, seed=3), 13.0),
    "long-lists": (lambda: gen.build_system(4200, seed=4), 23.0),
}


@pytest.mark.parametrize("gap", [0, 1])
@pytest.mark.parametrize("case", list(CASES))
def test_grid_and_list_equal_the_oracle(case, gap):
    make, rc = CASES[case]
    ls = make()
    o = oracle.Oracle(ls.n_atoms, ls.box, rc)
    L, lb, ub = oracle.pbc_from_box(ls.box)
    c = o.build(wrap_inbox(ls.crd, L, lb, ub))  # the engine wraps its input into the box
    cps, head = o.enumerate(ls.nb15off_table(), gap_bug=bool(gap))
    s = System(ls, dict(BASE, **{"nsgrid-cutoff": rc, "gap-bug": gap}))
    for _ in range(2):  # a second rebuild starts from what the first one left
        s.nsgrid_update()
        ids, gcrd, _ = s.grid()
        cp, cph = s.cell_pairs()
        assert np.array_equal(ids, c.atomids[:len(ids)]) and np.array_equal(gcrd, c.crd[:len(ids)])
        assert np.array_equal(cph, head)
        assert np.array_equal(cp, cps.view(np.int32).reshape(-1, 5))
    s.close()
    longest = int(np.diff(head).max())
    print("[gpu-test]", case, "gap", gap, "cells", c.n_cells, "longest list", longest, flush=True)
    if case == "long-lists" and not gap:
        assert longest > 320
    if case == "scan-blocks":
        assert c.n_cells > 2048
