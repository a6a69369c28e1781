"""A box given as its 3 x 3 matrix alone (9 values): the call points and the
oracle read 12, the last three the centre, and must not read past the array."""
import numpy as np
import pytest

import oracle
from omegagene_amd import gen
from omegagene_amd.cls import LaunchSet
from omegagene_amd.engine import desc_from_launchset

EDGES = (30.0, 40.0, 50.0)


def _nine():
    """Nine values with others behind them in memory."""
    mem = np.full(12, 1e30)
    mem[:9] = np.diag(EDGES).reshape(9)
    return mem[:9]


def test_oracle_takes_nine_values_with_the_centre_at_half_the_edges():
    L, lb, ub = oracle.pbc_from_box(_nine())
    assert np.array_equal(L, np.float32(EDGES)) and np.array_equal(lb, np.zeros(3)) and np.array_equal(ub, L)
    whole = np.concatenate([np.diag(EDGES).reshape(9), np.array(EDGES) / 2])
    assert all(np.array_equal(a, b) for a, b in zip(oracle.pbc_from_box(whole), (L, lb, ub)))
    g, h = oracle.grid_setup(3000, _nine(), 9.0), oracle.grid_setup(3000, whole, 9.0)
    assert list(g.n_cells_xyz) == list(h.n_cells_xyz) and g.n_columns == h.n_columns


def test_descriptor_holds_twelve_values():
    one = np.zeros((1, 3))
    ls = LaunchSet(box=_nine(), crd=one, vel=one, charge=np.zeros(1), mass=np.ones(1), atom_type=np.zeros(1, np.int32),
                   n_lj_types=1, lj6=np.zeros((1, 1)), lj12=np.zeros((1, 1)), nb15off=np.zeros((0, 2), np.int32))
    want = np.concatenate([np.diag(EDGES).reshape(9), np.array(EDGES) / 2])
    desc, _ = desc_from_launchset(ls)
    assert np.array_equal(np.ctypeslib.as_array(desc.box, shape=(12,)), want)


def test_fewer_values_are_refused():
    ls = gen.build_system(10, seed=1)
    for n in (3, 10, 11):
        with pytest.raises(ValueError):
            oracle.pbc_from_box(np.ones(n))
        ls.box = np.ones(n)
        with pytest.raises(ValueError):
            desc_from_launchset(ls)
