"""Sweep and force kernel in workgroups of one wave (below 65,536 particles):
contact statistics, whose parts take 256 particles, keep the force kernel at
four waves, so the two must agree bit for bit around the line and around one
wave; and the allocation-free evaluation, which keys, counts and writes its
forces by particle, at the sizes of one wave and at its limit."""
import numpy as np
import pytest

from pacific_amd import gdem
from test_gpu_packed_step import KEYS, _lattice
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 65535, 65536])
@pytest.mark.parametrize("skin", [0.0, -1.0])
def test_workgroup_sizes_agree(n, skin):
    print(f"[case] canonical step, {n} spheres, skin {skin}", flush=True)
    wl = _lattice(n, n % 2 == 0, 6)
    out = []
    for stats in (False, True):
        s = gdem.build_system(wl)
        s.set_skin(skin)
        s.set_contact_recording(32)
        s.set_contact_stats(stats)
        s.step(12, wl["dt"])
        out.append((s.get_state(), s.counters()["contacts"]))
        s.close()
    assert out[0][1] == out[1][1] and (n == 1 or out[0][1] > 0)
    for k in KEYS:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k


@pytest.mark.parametrize("n", [1, 64, 65, 32768])
def test_noalloc_forces_equal_the_contexts(n):
    print(f"[case] allocation-free forces, {n} spheres", flush=True)
    wl = _lattice(n, True, 7)
    if n < 27:  # three cells along a period
        wl.update(size=(1.0e-2,) * 3)
    wl["walls"] = []
    rc, F, T, ids = _noalloc(wl, wl["models"][0][2:])
    assert rc == gdem.OK, (rc, ids)
    s = gdem.build_system(wl)
    s.set_skin(0.0)
    s.prime()
    st = s.get_state()
    s.close()
    assert np.array_equal(F, st["F"]) and np.array_equal(T, st["T"])


@pytest.mark.parametrize("n,periodic", [(2, False), (64, True), (65, False), (1000, True),
                                        (4097, True), (4097, False), (49151, True),
                                        (49152, True)])
def test_row_sweep_equals_serial_sweep(n, periodic):
    """One lane per row of the half stencil (a context below 49,152 particles
    without a skin) and one lane per particle (a batch) list the same contacts
    in the same order: bit-identical sums."""
    print(f"[case] row sweep vs serial sweep, {n} spheres, periodic {periodic}", flush=True)
    wl = _lattice(n, periodic, 8)
    wl["substeps"] = 1
    b = gdem.build_batch([wl], block_size=64)
    b.step(12, wl["dt"])
    b.synchronize()
    s = gdem.build_system(wl)
    s.set_skin(0.0)
    s.step(12, wl["dt"])
    g, h = s.get_state(), b.get_state(0)
    assert s.counters()["contacts"] > 0 or n == 2
    for k in KEYS:
        assert np.array_equal(g[k], h[k]), k
    s.close()
    b.close()
