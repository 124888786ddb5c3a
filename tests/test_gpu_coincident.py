"""Sites of two molecules on one point.  Such a pair contributes nothing to the
reference (r^2 == 0, BruteForceStep.cpp:64-73); the kernels sum without looking
and sum again with a guard when a lane's sum is not finite, so the cases put the
pair where each instance of the sums meets it: in a hit whose pairs share one
image, in one shifted by the box edge, and in one whose pairs may wrap
differently; at the old and at the proposed position.

Coordinates are multiples of 1/64 in a box of a power of two, so that distances
that are zero come out as zero.  Tolerances: FP64 as in test_gpu_kernels.  MIXED:
an LJ term out of near contact (s6 <= 4, so at most 48 epsilon = 4.8 kcal/mol)
carries at most 69 roundings of 2^-24, 2e-5 kcal/mol, and fewer than 20 of a
molecule's pairs are that close."""
import numpy as np
import pytest

import mcgpu_amd as m
from edge_boxes import ArrayBox
from gpu_checks import run_all
from oracle import oracle as O

pytestmark = pytest.mark.gpu
EDGE = 32.0


def tolerance(precision, *energies):
    scale = max(abs(e) for e in energies)
    return (1e-9 if precision == m.FP64 else 4e-4) + 1e-12 * scale


def rods(pairs, spare, cutoff, dummy=False):
    """Rods of three sites 2 A apart: `pairs` of (start, direction, start,
    direction) along x, and some lone ones at `spare`."""
    xyz = []
    for x0, d0, x1, d1, y, z in pairs:
        for x, d in ((x0, d0), (x1, d1)):
            xyz += [(x, y, z), (x + 2 * d, y, z), (x + 4 * d, y, z)]
    for x, y, z in spare:
        xyz += [(x, y, z), (x, y + 2, z), (x, y + 4, z)]
    xyz = np.array(xyz, dtype=np.float64)
    n = len(xyz) // 3
    i32 = np.int32
    sigma = np.tile([3.0, 2.5, 2.75], n)
    if dummy:
        sigma[2::3] = -1.0
    return dict(x=xyz[:, 0].copy(), y=xyz[:, 1].copy(), z=xyz[:, 2].copy(), sigma=sigma,
                epsilon=np.tile([0.1, 0.0, 0.08], n), charge=np.tile([0.25, -0.5, 0.25], n),
                mol_start=np.arange(0, 3 * n, 3, dtype=i32), mol_len=np.full(n, 3, i32),
                mol_pidx_start=np.arange(n, dtype=i32), mol_pidx_count=np.ones(n, i32),
                primary_index=np.arange(0, 3 * n, 3, dtype=i32), box=np.full(3, EDGE),
                cutoff=cutoff, kT=0.6, max_translate=0.5, max_rotate=15.0)


SPARE = [(20.0, 20.0, 20.0), (24.5, 20.0, 20.0), (20.0, 24.0, 26.0), (9.0, 27.0, 3.0),
         (3.0, 12.0, 29.0), (27.0, 6.0, 14.0)]
# last sites coincide, 8 A between the firsts; first sites coincide; through the
# x boundary (30, 32, 34 and 6, 4, 2); a rod upon a rod.  A cutoff of 9 leaves
# hits within 16 - 8 A of one image, the far ones wrap pair by pair
PAIRS = [
    [(4.0, 1, 12.0, -1, 4.0, 4.0)],
    [(10.0, 1, 10.0, -1, 8.0, 8.0)],
    [(30.0, 1, 6.0, -1, 12.0, 12.0)],
    [(29.0, 1, 1.0, 1, 12.0, 3.0)],
    [(14.5, 1, 14.5, 1, 3.0, 17.0)],
    [(4.0, 1, 12.0, -1, 4.0, 4.0), (30.0, 1, 6.0, -1, 12.0, 12.0), (10.0, 1, 10.0, -1, 8.0, 8.0)],
]


@pytest.mark.parametrize("pairs", PAIRS)
@pytest.mark.parametrize("cutoff", [9.0, 14.5])
@pytest.mark.parametrize("precision", [m.FP64, m.MIXED])
@pytest.mark.parametrize("neighbor", [m.NEIGHBOR_BRUTE, m.NEIGHBOR_CELL, m.NEIGHBOR_VERLET])
def test_energies(pairs, cutoff, precision, neighbor):
    a = rods(pairs, SPARE, cutoff)
    ob = O.OracleBox(a)
    db = m.DeviceBox(ArrayBox(a, 1).desc(), precision)
    if neighbor != m.NEIGHBOR_BRUTE:
        db.neighbor(neighbor, 1.0)
    want = ob.system_energy()
    assert abs(db.system_energy() - want) <= len(pairs) * tolerance(precision, want)
    for i in range(len(a["mol_len"])):
        e = ob.molecule_energy(i)
        assert abs(db.molecule_energy(i) - e) <= tolerance(precision, e)


@pytest.mark.parametrize("cutoff", [9.0, 14.5])
@pytest.mark.parametrize("precision", [m.FP64, m.MIXED])
@pytest.mark.parametrize("dummy", [False, True])
def test_moves_on_and_off(cutoff, precision, dummy):
    """Every pair's first rod tried at a place of its own, and a lone rod tried
    on top of another."""
    a = rods(PAIRS[-1], SPARE, cutoff, dummy)
    db = m.DeviceBox(ArrayBox(a, 1).desc(), precision)
    ob = O.OracleBox(a)
    onto = {0: 7.0, 2: 2.5, 4: 3.25, 6: 0.0, 8: None}
    for mol, dy in onto.items():
        s = slice(3 * mol, 3 * mol + 3)
        moved = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in a.items()}
        if dy is None:  # on the second rod of the first pair
            for k in "xyz":
                moved[k][s] = a[k][3:6]
        else:
            moved["y"][s] += dy
        old, new = ob.molecule_energy(mol), O.OracleBox(moved).molecule_energy(mol)
        r = db.trial_move(mol, np.concatenate([moved[k][s] for k in "xyz"]), 2.0)
        tol = tolerance(precision, old, new)
        assert abs(r.old_energy - old) <= tol and abs(r.new_energy - new) <= tol
        if r.accepted:  # back
            db.set_molecule(mol, np.concatenate([a[k][s] for k in "xyz"]))


@pytest.mark.parametrize("cutoff", [9.0, 14.5])
@pytest.mark.parametrize("precision", [m.FP64, m.MIXED])
@pytest.mark.parametrize("neighbor", [0, 1])
def test_batched_run(cutoff, precision, neighbor):
    a = rods(PAIRS[-1], SPARE, cutoff)
    _, e0, _, want = O.OracleBox(a).run_nvt(23, 60, use_libc=False)
    b = m.Batch(1, 1 << 28)
    s = b.add(ArrayBox(a, 23), steps=60, neighbor=neighbor, precision=precision,
              record_trace=True)
    run_all(b, [s], 60, 7)
    tr = b.trace(s)
    assert abs(b.stats(s).start_energy - e0) <= 3 * tolerance(precision, e0)
    assert np.array_equal(tr.mol, want["mol"])
    assert np.array_equal(tr.accepted, want["accepted"])
    for k in range(60):
        assert abs(tr.de[k] - want["de"][k]) <= 2 * tolerance(precision, want["old_e"][k],
                                                              want["new_e"][k])
    b.close()
