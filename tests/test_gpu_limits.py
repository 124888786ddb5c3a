"""Boxes at the far end of what a descriptor admits, against the oracle."""
import numpy as np
import pytest

import mcgpu_amd as m
from edge_boxes import ArrayBox, build_box, kind
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DE_TOL = 1e-9


def test_sites_past_two_to_the_29(capsys):
    """4 GiB an axis: a group of four molecules at the end of a box whose other
    16.8 million lie at the origin, out of its range.  Their sites' byte offsets
    do not fit 32 bits.  (Zeroed arrays, so that the host holds little of it.)"""
    def say(text):
        with capsys.disabled():
            print(text, flush=True)

    last = build_box([kind(32, np.random.default_rng(1), (0,))], 4, 12.0, 9.0, seed=2).arrays()
    edge = 100.0
    for k in "xyz":
        last[k] += 44.0
    last["box"] = np.full(3, edge)
    n_mol = (1 << 24) + 4
    n_site = 32 * n_mol
    a = {k: np.zeros(n_site) for k in ("x", "y", "z", "sigma", "epsilon", "charge")}
    for k in a:
        a[k][-128:] = last[k]
    i32 = np.int32
    a.update(mol_start=np.arange(0, n_site, 32, dtype=i32), mol_len=np.full(n_mol, 32, i32),
             mol_pidx_start=np.arange(n_mol, dtype=i32), mol_pidx_count=np.ones(n_mol, i32),
             primary_index=np.arange(0, n_site, 32, dtype=i32), box=last["box"],
             **{k: last[k] for k in ("cutoff", "kT", "max_translate", "max_rotate")})
    say("\ncreating the box")
    db = m.DeviceBox(ArrayBox(a, mc_seed=1).desc())
    say("evaluating")
    ob = O.OracleBox(last)
    want = [ob.molecule_energy(i) for i in range(4)]
    assert max(abs(e) for e in want) > 1.0
    for i in range(4):
        got = db.molecule_energy(n_mol - 4 + i)
        assert abs(got - want[i]) <= DE_TOL + 1e-12 * abs(want[i])
    moved = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in last.items()}
    for k in "xyz":
        moved[k][-32:] += 0.05
    new = O.OracleBox(moved).molecule_energy(3)
    r = db.trial_move(n_mol - 1, np.concatenate([moved[k][-32:] for k in "xyz"]), 2.0)
    assert abs(r.old_energy - want[3]) <= DE_TOL + 1e-12 * abs(want[3])
    assert abs(r.new_energy - new) <= DE_TOL + 1e-12 * abs(new)
