"""The pair kernel of four waves per cell (small launches) against the kernel
of one wave per cell: both sum the same values in the same order, so the
gradient, every energy and the trajectory agree bit for bit.  The one-wave
kernel is held to the oracle by test_gpu_parity.py, test_gpu_zm.py and
test_gpu_hps.py; these cases walk the team's own edges: cells with fewer rows
than one pass, several batches of the filter, units cut in two, steps without
energies, and each electrostatic form."""
import numpy as np
import pytest

from helpers import cls_from_fixture, load_npz
from omegagene_amd import gen
from omegagene_amd.engine import Batch, System

pytestmark = pytest.mark.gpu

BASE = {"cutoff": 12.0, "nsgrid-cutoff": 13.0, "nsgrid-update-intvl": 5, "electrostatic": "zero-dipole",
        "ele-alpha": 0.0, "integrator": "leapfrog-presto", "constraint": "none", "time-step": 0.5, "log-cap": 64}

HPS = {"cutoff": 35.0, "nsgrid-cutoff": 40.0, "electrostatic": "debye-huckel", "nonbond": "hydrophobicity-scale-lj",
       "debye-huckel-dielectric": 80.0, "debye-huckel-temperature": 300.0, "debye-huckel-ionic-strength": 0.1}

CASES = {
    "sparse": (lambda: gen.build_system(500, seed=3, n_beads=20), {"cutoff": 6.0, "nsgrid-cutoff": 6.5}),
    "odd": (lambda: gen.build_system(1403, seed=7, n_beads=31), {}),
    "alpha": (lambda: gen.build_system(2300, seed=21), {"ele-alpha": 0.1}),
    "wide": (lambda: gen.build_system(1700, seed=5), {"cutoff": 14.0, "nsgrid-cutoff": 16.0}),
    "largest": (lambda: gen.build_system(2266, seed=6, n_beads=400), {"log-stride": 4}),
    "types": (lambda: gen.build_cg_system(12, 40, seed=9, L=200.0, n_types=40), HPS),
    "quadrupole": (lambda: cls_from_fixture(load_npz("wons_zm.npz")), {"electrostatic": "zero-quadrupole"}),
    "octupole": (lambda: cls_from_fixture(load_npz("wons_zm.npz")), {"electrostatic": "zero-octupole",
                                                                     "ele-alpha": 0.1}),
}


@pytest.mark.parametrize("case", list(CASES))
def test_four_waves_on_a_cell_give_the_bits_of_one(case):
    make, over = CASES[case]
    ls = make()
    assert ls.n_atoms <= 7200  # 900 cells: beyond, both shapes run a wave per cell
    cfg = dict(BASE, **over)
    out = []
    for waves in (1, 4):
        s = System(ls, cfg)
        s.set_pair_shape(waves)
        w, e = s.energy_force(rebuild=True)
        s.run(12)
        out.append((w, e, s.state(), s.energy_log()))
        s.close()
    (w1, e1, s1, l1), (w4, e4, s4, l4) = out
    print("[gpu-test] team", case, ls.n_atoms, "pairs", e1["npairs"], flush=True)
    assert np.isfinite(w1).all() and e1["npairs"] > 0
    assert np.array_equal(w1, w4) and all(e1[k] == e4[k] for k in e1)
    assert all(np.array_equal(a, b) for a, b in zip(s1[:2], s4[:2])) and np.array_equal(l1, l4)


def test_four_waves_on_a_cell_in_a_batch():
    """Two systems in one launch (units mapped to their systems), the list in
    parts per XCD, against each system alone with a wave per cell."""
    lss = [gen.build_system(n, seed=n) for n in (700, 1201)]
    alone = []
    for ls in lss:
        s = System(ls, BASE)
        s.set_pair_shape(1)
        s.run(12)
        alone.append(s.state()[0])
        s.close()
    for order in (0, 3):
        ss = [System(ls, BASE) for ls in lss]
        b = Batch()
        for s in ss:
            b.add(s)
        b.set_pair_shape(4, order)
        b.run(12)
        got = [s.state()[0] for s in ss]
        b.close()
        for s in ss:
            s.close()
        assert all(np.array_equal(a, g) for a, g in zip(alone, got)), order
