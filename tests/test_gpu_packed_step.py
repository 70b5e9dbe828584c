"""Packed step beyond the sizes of the parity cases: the one-kernel step with
one, two and four lanes per particle, the two-kernel step of many particles
(screened and integrated separately), rebuilds in the middle of a chunk of
steps, and call lengths around a chunk; all bit-identical to the fused
canonical kernel, which contact recording selects."""
import numpy as np
import pytest

from pacific_amd import gdem, workloads

pytestmark = pytest.mark.gpu

KEYS = ("x", "v", "w", "q", "F", "T")


def _lattice(n, periodic, seed):
    """n spheres on a cubic lattice (spacing 2.0 mm less 0.5 um: neighbours
    touch), radius 1 mm, v ~ N(0, 0.5^2): fast enough that lists go stale
    within a few steps; walls or a periodic box."""
    rng = np.random.default_rng(seed)
    m, a = int(np.ceil(n ** (1.0 / 3.0))), 2.0e-3 - 5.0e-7
    site = rng.permutation(m ** 3)[:n]
    x = (np.stack([site // (m * m), site // m % m, site % m], 1) + 0.5) * a
    x += rng.uniform(-2.0e-7, 2.0e-7, x.shape)
    wl = workloads.periodic_hooke(2000)
    lo, hi = (0.0, 0.0, 0.0), (m * a,) * 3
    wl.update(origin=lo, size=hi, dt=5.0e-6, cell_size=2.4e-3,
              walls=[] if periodic else workloads.box_walls(lo, hi, 1),
              periodic=(int(periodic),) * 3,
              particles=workloads._particles(x, rng.normal(0.0, 0.5, x.shape), np.full(n, 1.0e-3)))
    kind, prm = wl["models"][0][2:]
    wl["models"] = [(0, 0, kind, prm), (0, 1, kind, prm)]
    return wl


# sizes around the lines of the dispatch: 32,768, 65,536 and 524,288 particles
@pytest.mark.parametrize("n,periodic", [(1, False), (65, False), (4097, True), (32769, True),
                                        (65537, False), (524289, True), (530000, False)])
def test_packed_step_equals_fused_kernel_over_sizes(n, periodic):
    print(f"[case] packed vs fused, {n} spheres, periodic {periodic}", flush=True)
    wl = _lattice(n, periodic, 5)
    a, b = gdem.build_system(wl), gdem.build_system(wl)
    b.set_contact_recording(32)
    for calls in (1, 15, 16, 33):
        a.step(calls, wl["dt"])
        b.step(calls, wl["dt"])
        sa, sb = a.get_state(), b.get_state()
        for k in KEYS:
            assert np.array_equal(sa[k], sb[k]), (calls, k)
    assert a.get_skin()[1] == b.get_skin()[1]
    assert n == 1 or a.get_skin()[1] >= 3
    assert a.counters()["contacts"] == b.counters()["contacts"]
    a.close()
    b.close()


def test_step_without_occupancy_check_equals_step_with_it():
    """With the check off the call does not wait and a rebuild is offered
    before every step; with kernel timing on, one launch at a time."""
    print("[case] packed step, chunked vs a rebuild offered per step", flush=True)
    wl = _lattice(5000, True, 6)
    runs = []
    for adapt, timing, graph in ((True, False, True), (False, False, True), (True, True, True),
                                 (True, False, False)):
        s = gdem.build_system(wl)
        s.set_skin_adapt(adapt)
        s.set_kernel_timing(timing)
        s.set_graph(graph)
        for calls in (40, 7):
            s.step(calls, wl["dt"])
        runs.append((s.get_state(), s.get_skin()[1], s.get_time()))
        s.close()
    for st, rebuilds, time in runs[1:]:
        assert rebuilds == runs[0][1] >= 3 and time == runs[0][2]
        for k in KEYS:
            assert np.array_equal(st[k], runs[0][0][k]), k
