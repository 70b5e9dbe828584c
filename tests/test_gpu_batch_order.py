"""Systems of a batch whose particles never change cell, change it now and then
and change it at every step: the order kept between sorts is the sorted one,
so each stays bit-identical to the system stepped alone."""
import numpy as np
import pytest

from pacific_amd import gdem, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 512])
def test_kept_order_equals_sorted_order(block):
    print(f"[case] batch order, block {block}", flush=True)
    systems = []
    for k, speed in enumerate((0.0, 1.0, 15.0)):
        for n in (1, 65, 500):
            wl = workloads.batch_system(n, 3 + k, 2.0, 5.0e4, 0.8, 0.4)
            wl["particles"]["v"] *= speed
            systems.append(wl)
    b = gdem.build_batch(systems, block_size=block, workgroups=4)
    b.step(20, 1e-5)
    b.step(20, 1e-5)
    b.synchronize()
    for s, wl in enumerate(systems):
        single = gdem.build_system(wl)
        single.set_skin(0.0)
        sub = wl["substeps"]
        single.step(40 * sub, 1e-5 / sub)
        g, h = single.get_state(), b.get_state(s)
        for key in ("x", "v", "w", "q", "F", "T"):
            assert np.array_equal(g[key], h[key]), (s, key)
        single.close()
    b.close()
