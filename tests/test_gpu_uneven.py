"""Cell-list scans of boxes of uneven density (a drop in an empty box, and one
beside a thin gas), where the cells around a molecule hold from nothing to their
fullest, against the oracle.  Tolerances as in test_gpu_kernels."""
import numpy as np
import pytest

import mcgpu_amd as m
from edge_boxes import ArrayBox
from gpu_checks import run_all
from oracle import oracle as O
from test_gpu_kernels import DE_TOL, box, moves_match

pytestmark = pytest.mark.gpu


def uneven(kind, n, cutoff, factor, gas=0):
    """The liquid box in one `factor` times its edge, every gas-th molecule
    spread over all of it."""
    a = box(kind, n, cutoff).arrays()
    edge = np.array(a["box"])
    a["box"] = edge * factor
    if gas:
        rng = np.random.default_rng(11)
        first = a["primary_index"][a["mol_pidx_start"]]
        mol = np.repeat(np.arange(n), a["mol_len"])
        spread = np.arange(n) % gas == 0
        for d, k in enumerate("xyz"):
            to = np.where(spread, rng.uniform(0, a["box"][d], n), a[k][first])
            a[k] = a[k] + (to - a[k][first])[mol]
    return ArrayBox(a, mc_seed=17)


BOXES = [
    ("water", 1000, 9.0, 2.0, 0),
    ("water", 2200, 9.0, 3.0, 3),
    ("mixture", 1500, 11.0, 2.0, 2),
    ("bicyclic", 700, 12.0, 2.0, 0),
    ("ragged", 300, 14.0, 2.0, 4),
]


@pytest.mark.parametrize("kind,n,cutoff,factor,gas", BOXES)
def test_moves_match_oracle(kind, n, cutoff, factor, gas):
    ab = uneven(kind, n, cutoff, factor, gas)
    a = ab.arrays()
    a["max_translate"] = 3.0  # moves across cells, so that ranges grow
    ab = ArrayBox(a, mc_seed=17)
    _, e0, _, want = O.OracleBox(a).run_nvt(17, 200, use_libc=False)
    b = m.Batch(1)
    s = b.add(ab, steps=200, neighbor=1, record_trace=True)
    run_all(b, [s], 200, 67)
    assert b.stats(s).start_energy == pytest.approx(e0, rel=1e-12, abs=1e-7)
    assert moves_match(b.trace(s), want)
    b.close()


@pytest.mark.parametrize("kind,n,cutoff,factor,gas", BOXES + [("water", 8193, 9.0, 2.0, 0)])
@pytest.mark.parametrize("precision", [m.FP64, m.MIXED])
def test_full_energy_matches_oracle(kind, n, cutoff, factor, gas, precision):
    ab = uneven(kind, n, cutoff, factor, gas)
    ob = O.OracleBox(ab.arrays())
    want = ob.system_energy()
    plain = m.DeviceBox(ab.desc(), precision)  # every molecule scanned
    e_plain = plain.system_energy()
    db = m.DeviceBox(ab.desc(), precision)
    db.neighbor(m.NEIGHBOR_CELL)
    e = db.system_energy()
    print(f"E {e:.9f} all pairs {e_plain:.9f} oracle {want:.9f}")
    assert db.system_pairs() == plain.system_pairs()
    if precision == m.MIXED:
        # the same pair terms in another order; a displacement's last bit may
        # turn an FP32 rounding (2^-24 of at most 12 * 10 kcal/mol out of near
        # contact), in a pair or two of a billion
        assert abs(e - e_plain) <= 1e-4 + 1e-9 * abs(e_plain)
    else:
        assert abs(e - e_plain) <= 6e-14 * db.system_pairs() + 1e-12 * abs(e_plain) + 1e-12
        assert abs(e - want) <= 6e-14 * db.system_pairs() + 1e-12 * abs(want) + 1e-12
        for i in range(0, n, n // 12):
            assert db.molecule_energy(i) == pytest.approx(ob.molecule_energy(i), rel=1e-12,
                                                          abs=DE_TOL)
