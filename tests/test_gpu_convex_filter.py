"""Candidate filter and cooperative sweep of the convex step: a packing whose
queue is long enough for the filter, where contact statistics (which switch
the filter off) must not change a bit of the state, and the candidate lists of
both sweep widths against the serial ones through the contact records."""
import numpy as np
import pytest

from pacific_amd import gdem, workloads

pytestmark = pytest.mark.gpu


# 12,000 bodies: eight lanes per particle; 33,000: two
@pytest.mark.parametrize("n,narrow", [(12000, "GJK"), (12000, "GJK_SV"), (33000, "GJK")])
def test_filter_drops_no_contact(n, narrow):
    print(f"[case] convex filter, {n} bodies, {narrow}", flush=True)
    wl = workloads.convex_box(n, seed=5, phi=0.20, height=0.05, overlap=2.0e-5, sigma_v=0.3)
    wl["narrow_phase"] = narrow
    out = []
    for stats in (False, True):
        s = gdem.build_system(wl)
        s.set_contact_stats(stats)
        s.step(60, wl["dt"])
        out.append((s.get_state(), s.get_basis(), s.counters()["contacts"]))
        s.close()
    assert out[0][2] == out[1][2] > 100
    assert np.array_equal(out[0][1], out[1][1])
    for k in ("x", "v", "w", "q", "F", "T"):
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
