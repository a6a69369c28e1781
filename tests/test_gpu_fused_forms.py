"""Which systems take the one-kernel step, as og_step_fused reports it, and the
step in a batch of one form: each member's coordinates, velocities and energy
rows (block sums included, as the blocks group alike) are those it gives alone."""
import numpy as np
import pytest

from helpers import load_npz
from omegagene_amd import gen
from omegagene_amd.cls import read_cls
from omegagene_amd.engine import Batch, System

pytestmark = pytest.mark.gpu

BASE = {"cutoff": 12.0, "nsgrid-cutoff": 13.0, "nsgrid-update-intvl": 5, "time-step": 1.0, "gap-bug": 0,
        "const-tolerance": 1e-10, "temperature": 300.0, "langevin-gamma": 20.0, "random-seed": 3, "log-cap": 32}


def _system(n_waters, n_beads, settle):
    ls = gen.build_system(n_waters, seed=n_waters, n_beads=n_beads)
    if settle:
        ls.settle_ids, ls.settle_d = ls.shake_trio_ids, ls.shake_trio_d
        ls.shake_trio_ids, ls.shake_trio_d = np.zeros((0, 3), np.int32), np.zeros((0, 3))
    return ls


@pytest.mark.parametrize("integrator", ["langevin", "leapfrog-presto"])
@pytest.mark.parametrize("settle", [True, False])
def test_fused_forms_are_reported_and_batch_as_alone(integrator, settle):
    lss = [_system(400, 21, settle), _system(533, 0, settle)]
    cfg = dict(BASE, integrator=integrator, constraint="shake-settle" if settle else "shake")
    print("[gpu-test] fused form", integrator, "settle" if settle else "shake", flush=True)
    alone = []
    for ls in lss:
        s = System(ls, dict(cfg, **{"split-step": 1}))
        assert not s.step_fused()
        s.close()
        s = System(ls, cfg)
        assert s.step_fused()
        s.run(12)
        alone.append((s.state(), s.energy_log()))
        s.close()
    ss = [System(ls, cfg) for ls in lss]
    b = Batch()
    for s in ss:
        b.add(s)
    b.run(12)
    for s, (st, log) in zip(ss, alone):
        assert all(np.array_equal(x, y) for x, y in zip(s.state(), st)) and np.array_equal(s.energy_log(), log)
    b.close()
    for s in ss:
        s.close()


def test_systems_off_the_fused_step_report_so():
    d = load_npz("wons_ext.npz")
    mcmd = read_cls(bytes(d["mcmd_cls"]))
    water = _system(400, 0, False)
    off = {"v-mcmd": (mcmd, {"extended-ensemble": "v-mcmd", "constraint": "shake"}, None),
           "no constraint": (water, {"constraint": "none"}, None),
           "com removal": (water, {"constraint": "shake", "com-motion": "cancel"},
                           [np.arange(water.n_atoms, dtype=np.int32)])}
    for name, (ls, over, groups) in off.items():
        s = System(ls, dict(BASE, integrator="leapfrog-presto", **over), com_groups=groups)
        assert not s.step_fused(), name
        s.close()


@pytest.mark.parametrize("integrator,settle", [("langevin", True), ("leapfrog-presto", False)])
def test_atoms_outside_the_waters_up_to_the_limit(integrator, settle):
    """512 + waters / 100 atoms outside the waters take the one-kernel step, one more does not; in a batch the
    waters of all members count.  Whatever the route, the same trajectory; the energies that are summed over
    blocks to relative 1e-13 or 64 quanta of 2^-32, the rounding of their different grouping."""
    over = dict(integrator=integrator, constraint="shake-settle" if settle else "shake", **{"time-step": 0.5})
    cfg = dict(BASE, **over)
    print("[gpu-test] limit of the fused step", integrator, flush=True)
    runs = {}
    for beads in (524, 525):
        ls = _system(1200, beads, settle)
        for split in (1, 0):
            s = System(ls, dict(cfg, **{"split-step": split}))
            assert s.step_fused() == (beads == 524 and split == 0)
            s.run(12)
            runs[beads, split] = (s.state(), s.energy_log())
            s.close()
    ss = [System(_system(1200, 525, settle), cfg), System(_system(300, 0, settle), cfg)]
    b = Batch()   # 1,500 waters: 527
    for s in ss:
        b.add(s)
    b.run(12)
    runs["batch"] = (ss[0].state(), ss[0].energy_log())
    b.close()
    for s in ss:
        s.close()
    for one, other in (((524, 1), (524, 0)), ((525, 1), (525, 0)), ((525, 1), "batch")):
        (st1, log1), (st0, log0) = runs[one], runs[other]
        assert np.isfinite(st1[0]).all() and all(np.array_equal(x, y) for x, y in zip(st1, st0))
        rest = [k for k in range(log1.shape[1]) if k not in (2, 4, 5)]  # excess, bond, kinetic
        assert np.array_equal(log1[:, rest], log0[:, rest])
        for k in (2, 4, 5):
            err = np.abs(log1[:, k] - log0[:, k])
            assert np.max(err / np.maximum(np.abs(log1[:, k]), 1e-300)) <= 1e-13 or np.max(err) <= 64 * 2.0 ** -32
