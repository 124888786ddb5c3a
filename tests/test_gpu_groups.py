"""Work-group sizes of batched boxes: the size a box prefers, and ticks whose
boxes of several sizes must be resident together."""
import time

import pytest

import mcgpu_amd as m
from test_gpu_kernels import box

pytestmark = pytest.mark.gpu


# both sizes fill the card but for 36 units, which hold 72 of the small ones;
# 212 small beside 150; all but 6 units; more small ones than two a unit hold
# beside large ones
@pytest.mark.parametrize("large,small", [(220, 60), (220, 100), (150, 212), (250, 12)])
def test_a_tick_runs_in_one_round(large, small):
    """Up to 512 boxes run side by side: a tick limited in time takes about that
    time, and twice as long when some of them wait for others to end."""
    limit = 5e-3
    b = m.Batch(large + small, 1 << 31)
    b.set_autotune(False)
    b.set_tick_budget(limit * 1e6)
    boxes = [(box("water", 500, 9.0), large), (box("water", 100, 6.0), small)]
    slots = [b.add(hb, steps=10 ** 8, seed=k + 1) for hb, count in boxes for k in range(count)]
    assert {b.group_threads(s) for s in slots} == {256, 512}
    b.run(100000)
    took = []
    for _ in range(4):
        t0 = time.perf_counter()
        b.run(100000)
        took.append(time.perf_counter() - t0)
    print("tick ms", [round(1e3 * t, 2) for t in took])
    assert min(took) < 1.5 * limit
    done = [b.stats(s).steps_done for s in slots]
    assert min(done) > 1000
    b.close()


# the fastest of 256, 512 and 1,024 lanes for one box alone, as measured
@pytest.mark.parametrize("kind,n,cutoff,neighbor,precision,lanes", [
    ("water", 128, 9.0, 0, m.FP64, 256),
    ("water", 600, 9.0, 0, m.FP64, 1024),
    ("water", 1000, 9.0, 0, m.FP64, 512),
    ("water", 1900, 9.0, 0, m.FP64, 1024),
    ("water", 2000, 9.0, 0, m.FP64, 512),
    ("mixture", 500, 11.0, 0, m.FP64, 512),
    ("mixture", 700, 11.0, 0, m.FP64, 1024),
    ("mixture", 2000, 11.0, 0, m.FP64, 512),
    ("bicyclic", 512, 12.0, 0, m.FP64, 512),
    ("bicyclic", 512, 12.0, 0, m.MIXED, 1024),
    ("water", 128, 9.0, 1, m.FP64, 256),
    ("water", 400, 9.0, 1, m.FP64, 512),
    ("water", 1000, 9.0, 1, m.FP64, 1024),
])
def test_size_of_a_lone_box(kind, n, cutoff, neighbor, precision, lanes):
    b = m.Batch(1, 1 << 28)
    b.set_autotune(False)
    s = b.add(box(kind, n, cutoff), steps=10, neighbor=neighbor, precision=precision)
    assert b.group_threads(s) == lanes
    b.close()
