"""MIXED energies at the tile, round and dispatch edges of the kernels, against
the oracle, with a bound made of the LJ terms that are evaluated in FP32.

In units of u = 2^-24: 1/r from the rounded r^2 and v_rsq_f32 (1 ulp) carries
2.5 u, the products of the FP32 sigmas and epsilons 3 u each, so (sigma/r)^2
10 u, (sigma/r)^6 = s6 32 u, and 4 eps (s6^2 - s6) at most 4 eps (69 s6^2 + 37
s6) u.  Pairs in near contact (s6 > 4) are evaluated in FP64, and the Coulomb
terms' 1/r is refined by a Newton step to 1.5 (2.5 u)^2 = 3.3e-14.  Sums and the
rest are FP64, as in test_gpu_kernels."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import mcgpu_amd as m
from gpu_checks import run_all
from oracle import oracle as O
from test_gpu_kernels import KIND, box

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def terms(a, mol=None):
    """Bound on the MIXED energy's error over the in-range molecule pairs (of
    molecule mol, when given), the number of site pairs, and of those in near
    contact."""
    edge = np.array(a["box"])
    first, length = a["mol_start"], a["mol_len"]
    owner = np.repeat(np.arange(len(length)), a["mol_pidx_count"])
    xyz = np.stack([a[k] for k in "xyz"], 1)
    prim = xyz[a["primary_index"]] % edge
    tree = cKDTree(np.minimum(prim, np.nextafter(edge, 0)), boxsize=edge)
    if mol is None:
        pairs = owner[tree.query_pairs(a["cutoff"], output_type="ndarray")]
    else:
        mine = np.flatnonzero(owner == mol)
        near = tree.query_ball_point(np.minimum(prim[mine], np.nextafter(edge, 0)), a["cutoff"])
        pairs = np.array([(mol, owner[k]) for some in near for k in some])
    pairs = np.unique(np.sort(pairs, 1), axis=0)
    pairs = pairs[pairs[:, 0] != pairs[:, 1]]
    real = (a["sigma"] >= 0) & (a["epsilon"] >= 0)
    sg, ep = np.where(real, a["sigma"], 0.0), np.where(real, a["epsilon"], 0.0)
    q = np.where(real, a["charge"], 0.0)
    top = int(length.max())
    lj = coul = 0.0
    count = near = 0
    for i in range(top):
        for j in range(top):
            p = pairs[(i < length[pairs[:, 0]]) & (j < length[pairs[:, 1]])]
            s, t = first[p[:, 0]] + i, first[p[:, 1]] + j
            ok = real[s] & real[t]
            s, t = s[ok], t[ok]
            d = xyz[t] - xyz[s]
            d = np.where(d > edge / 2, d - edge, np.where(d < -edge / 2, d + edge, d))
            r2 = (d * d).sum(1)
            s6 = (sg[s] * sg[t] / r2) ** 3
            e4 = 4.0 * np.sqrt(ep[s] * ep[t])
            far = s6 <= 4.001
            lj += float((e4 * (69 * s6 * s6 + 37 * s6))[far].sum())
            coul += float(np.abs(332.06 * q[s] * q[t] / np.sqrt(r2)).sum())
            count += len(s)
            near += int((~far & (e4 > 0)).sum())
    return lj * U + 3.3e-14 * coul, count, near


def dense(kind, n, cutoff):
    """As box(), or (kind "packed") water at a density where lattice neighbours
    come into near contact."""
    if kind == "packed":
        return m.HostBox.generate(KIND["water"], n, seed=7, cutoff=cutoff, density=1.9)
    return box(kind, n, cutoff)


# as for FP64: molecules a wave, the waves' shares, the end of the one-work-group
# cell build, fewer than 3 cells along an axis, hits beyond one mapping and list
@pytest.mark.parametrize("kind,n,cutoff,cells", [
    ("water", 64, 6.0, True),
    ("water", 1024, 9.0, True),
    ("water", 1025, 9.0, False),
    ("water", 2049, 9.0, True),
    ("water", 1500, 17.0, False),
    ("packed", 700, 9.0, False),
    ("packed", 2100, 9.0, True),
    ("mixture", 1030, 16.0, True),
    ("mixture", 2100, 11.0, True),
    ("bicyclic", 350, 12.0, True),
    ("ragged", 343, 10.0, True),
    ("water", 8193, 9.0, True),
])
def test_full_energy(kind, n, cutoff, cells):
    hb = dense(kind, n, cutoff)
    a = hb.arrays()
    bound, count, near = terms(a)
    db = m.DeviceBox(hb.desc(), m.MIXED)
    if cells:
        db.neighbor(m.NEIGHBOR_CELL)
    e, want = db.system_energy(), O.OracleBox(a).system_energy()
    print(f"error {e - want:.3e} bound {bound:.3e} of {want:.6g}, {near} of {count} in near contact")
    assert db.system_pairs() == count
    assert near > 100 or kind != "packed"
    assert abs(e - want) <= bound + 6e-14 * count + 1e-12 * abs(want)


# both sizes of a single trial move, around their passes
@pytest.mark.parametrize("kind,n,cutoff,nb", [
    ("water", 512, 9.0, m.NEIGHBOR_BRUTE),
    ("water", 1025, 9.0, m.NEIGHBOR_BRUTE),
    ("water", 2049, 9.0, m.NEIGHBOR_BRUTE),
    ("packed", 700, 9.0, m.NEIGHBOR_CELL),
    ("mixture", 1100, 9.0, m.NEIGHBOR_CELL),
    ("mixture", 1100, 9.0, m.NEIGHBOR_VERLET),
    ("bicyclic", 65, 12.0, m.NEIGHBOR_BRUTE),
    ("ragged", 200, 10.0, m.NEIGHBOR_BRUTE),
])
def test_single_moves(kind, n, cutoff, nb):
    hb = dense(kind, n, cutoff)
    a = hb.arrays()
    db = m.DeviceBox(hb.desc(), m.MIXED)
    if nb != m.NEIGHBOR_BRUTE:
        db.neighbor(nb, 1.5)
    rng = np.random.default_rng(3)
    for i in rng.integers(0, n, 8):
        s = slice(int(a["mol_start"][i]), int(a["mol_start"][i] + a["mol_len"][i]))
        moved = {c: (v.copy() if isinstance(v, np.ndarray) else v) for c, v in a.items()}
        for c in "xyz":
            moved[c][s] += rng.uniform(-0.3, 0.3)
        r = db.trial_move(int(i), np.concatenate([moved[c][s] for c in "xyz"]), 2.0)
        for got, b in ((r.old_energy, a), (r.new_energy, moved)):
            want = O.OracleBox(b).molecule_energy(int(i))
            bound = terms(b, int(i))[0]
            assert abs(got - want) <= bound + 1e-9 + 1e-12 * abs(want)
        if r.accepted:
            a = moved


# batched moves, around the passes and rounds of 4, 8 and 15 waves; a move sums
# the terms of two positions, each held to twice the start box's largest bound
@pytest.mark.parametrize("kind,n,cutoff,neighbor,steps,chunk", [
    ("water", 22, 4.2, 0, 400, 1),
    ("water", 257, 9.0, 0, 300, 31),
    ("water", 513, 9.0, 0, 200, 200),
    ("water", 1025, 9.0, 0, 150, 150),
    ("water", 2300, 20.0, 0, 40, 40),
    ("packed", 400, 9.0, 0, 200, 50),
    ("packed", 1100, 9.0, 1, 150, 150),
    ("mixture", 961, 11.0, 0, 150, 150),
    ("mixture", 1100, 9.0, 1, 200, 67),
    ("bicyclic", 700, 12.0, 1, 150, 150),
    ("ragged", 200, 10.0, 0, 200, 40),
])
def test_batched_moves(kind, n, cutoff, neighbor, steps, chunk):
    hb = dense(kind, n, cutoff)
    a = hb.arrays()
    _, _, _, want = O.OracleBox(a).run_nvt(hb.mc_seed, steps, use_libc=False)
    # the start box's largest molecule bound, of 40 molecules
    per = max(terms(a, int(i))[0] for i in np.random.default_rng(2).integers(0, n, 40))
    b = m.Batch(1, 1 << 29)
    s = b.add(hb, steps=steps, neighbor=neighbor, precision=m.MIXED, record_trace=True)
    run_all(b, [s], steps, chunk)
    tr = b.trace(s)
    err = np.abs(tr.de - want["de"])
    scale = np.maximum(np.abs(want["old_e"]), np.abs(want["new_e"]))
    calm = scale < 1e3
    print(f"largest error {err[calm].max():.3e}, a molecule's bound {per:.3e}")
    assert np.array_equal(tr.mol, want["mol"])
    assert np.array_equal(tr.accepted, want["accepted"])
    assert np.all(err <= 4 * per + 1e-9 + 1e-12 * scale)
    b.close()
