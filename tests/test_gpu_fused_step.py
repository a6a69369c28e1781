"""The one-kernel step in the forms the parity tests do not walk -- leapfrog
with SETTLE or SHAKE waters, Langevin with SHAKE waters -- against the
separate kernels: the same coordinates, velocities and potential terms bit for
bit, and the energies that are summed over blocks (excluded pairs, bonds,
kinetic) to relative 1e-13 or 64 quanta of 2^-32, the rounding of their
different grouping.  Sizes walk the blocks' edges: one atom outside the waters
to more than a lead block takes, a last wave of one water, trios that do not
qualify as waters."""
import numpy as np
import pytest

from omegagene_amd import gen
from omegagene_amd.engine import Batch, System

pytestmark = pytest.mark.gpu

BASE = {"cutoff": 12.0, "nsgrid-cutoff": 13.0, "nsgrid-update-intvl": 5, "time-step": 1.0, "gap-bug": 0,
        "const-tolerance": 1e-10, "temperature": 300.0, "langevin-gamma": 20.0, "random-seed": 3, "log-cap": 32}


def _waters(n_waters, n_beads, settle, tied=0):
    """n_beads chain atoms outside the waters; tied: waters with a bond to the next one, which therefore
    stay with the other atoms."""
    ls = gen.build_system(n_waters, seed=n_waters, n_beads=n_beads)
    if settle:
        ls.settle_ids, ls.settle_d = ls.shake_trio_ids, ls.shake_trio_d
        ls.shake_trio_ids, ls.shake_trio_d = np.zeros((0, 3), np.int32), np.zeros((0, 3))
    if tied:
        o = np.asarray(ls.shake_trio_ids)[:, 0]
        x, L = ls.crd, float(np.float32(ls.box[0]))
        ids = np.array([[o[3 * k], o[3 * k + 1]] for k in range(tied)], np.int32)
        v = x[ids[:, 0]] - x[ids[:, 1]]
        r = np.linalg.norm(v - L * np.round(v / L), axis=1)
        ls.bond_ids = np.concatenate([np.asarray(ls.bond_ids, np.int32).reshape(-1, 2), ids])
        ls.bond_k = np.concatenate([np.asarray(ls.bond_k, float), np.full(tied, 5.0)])
        ls.bond_r0 = np.concatenate([np.asarray(ls.bond_r0, float), r])
    return ls


CASES = {
    "leapfrog-shake": ("leapfrog-presto", lambda: _waters(1345, 0, False)),       # 16 blocks of 84 waters, and one
    "leapfrog-shake-chain": ("leapfrog-presto", lambda: _waters(1000, 33, False)),  # a lead block and one atom
    "leapfrog-shake-tied": ("leapfrog-presto", lambda: _waters(1000, 5, False, tied=9)),
    "leapfrog-settle": ("leapfrog-presto", lambda: _waters(1009, 32, True)),
    "langevin-shake": ("langevin", lambda: _waters(1009, 1, False)),
    "langevin-shake-tied": ("langevin", lambda: _waters(1009, 40, False, tied=4)),
}


def _same(one, other):
    (st1, log1), (st0, log0) = one, other
    assert all(np.array_equal(a, c) for a, c in zip(st1, st0))
    grouped = [2, 4, 5]  # excess, bond, kinetic
    rest = [k for k in range(log1.shape[1]) if k not in grouped]
    assert np.array_equal(log1[:, rest], log0[:, rest])
    for k in grouped:
        err = np.abs(log1[:, k] - log0[:, k])
        assert np.max(err / np.maximum(np.abs(log1[:, k]), 1e-300)) <= 1e-13 or np.max(err) <= 64 * 2.0 ** -32


@pytest.mark.parametrize("case", list(CASES))
def test_fused_step_equals_the_separate_kernels(case):
    integrator, make = CASES[case]
    ls = make()
    cfg = dict(BASE, integrator=integrator, constraint="shake-settle" if len(ls.settle_ids) else "shake")
    runs = []
    for split in (1, 0):
        s = System(ls, dict(cfg, **{"split-step": split}))
        s.run(20)
        runs.append((s.state(), s.energy_log()))
        s.close()
    print("[gpu-test] fused step", case, ls.n_atoms, "kinetic", runs[0][1][-1, 5], flush=True)
    assert np.isfinite(runs[0][0][0]).all()
    _same(*runs)
    # two systems of different size in one launch, each as alone
    ss = [System(ls, cfg), System(gen.build_system(700, seed=2), dict(cfg, constraint="shake"))]
    b = Batch()
    for s in ss:
        b.add(s)
    b.run(20)
    got = (ss[0].state(), ss[0].energy_log())
    b.close()
    for s in ss:
        s.close()
    _same(runs[1], got)
