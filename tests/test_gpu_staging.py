"""Admissions and downloads through the batch's pinned buffer: a box larger than
it, in pieces, between small ones."""
import numpy as np
import pytest

import mcgpu_amd as m
from test_gpu_kernels import box

pytestmark = pytest.mark.gpu


def test_boxes_larger_than_the_staging_buffer():
    # 262,144 sites: 6.3 MB of coordinates, 7 MB in all, through 4 MiB
    large, small = box("bicyclic", 16384, 12.0), box("water", 300, 9.0)
    order = [small, large, small, large, large, small]
    b = m.Batch(len(order), 1 << 30)
    slots = [b.add(hb, steps=10, neighbor=int(hb is large), energy_offset=0.0) for hb in order]
    energy = {}
    for hb in (large, small):
        db = m.DeviceBox(hb)
        if hb is large:
            db.neighbor(m.NEIGHBOR_CELL)
        energy[id(hb)] = db.system_energy()
        db.close()
    for s, hb in reversed(list(zip(slots, order))):
        a = hb.arrays()
        for got, k in zip(b.download(s), "xyz"):
            assert np.array_equal(got, a[k])
        assert b.stats(s).start_energy == pytest.approx(energy[id(hb)], rel=1e-12)
    b.run(10)
    for s, hb in zip(slots, order):
        assert b.stats(s).steps_done == 10
        x, _, _ = b.download(s)
        assert 0 < np.count_nonzero(x != hb.arrays()["x"]) <= 10 * 16
    b.close()
