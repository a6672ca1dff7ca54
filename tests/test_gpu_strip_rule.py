"""Strips at the disc sizes that take them by the automatic rule: sky NSIDE 128,
beam NSIDE 1024, cap 20 deg (11.6 MB, 5,900 pixels per disc; six strips forward,
two in the adjoint), 4,101 samples (a strip chunk and a partial block), some of
whose discs hold a pole.  A sample's TOD has the same bits in any launch.
Tolerance: relative RMS 1e-6 of the oracle, the bound of the other single-pair
tests."""
import numpy as np
import pytest

from pisco4cmb_amd import pypisco
from test_gpu_strips import Calls, make, rel_rms
from test_launch_shape import shape

pytestmark = pytest.mark.gpu


def test_automatic_strips(oracle):
    ns, nb, cap, n = 128, 1024, 20.0, 4101
    assert shape(ns, nb, cap, n)[:4] == [64, 6, 64, 2]
    sky, beam, ra, dec, pa, g = make(ns, nb, cap, n, 11)
    c = Calls(ns, nb, beam, sky)
    beams = list(beam.aBeams) + list(beam.bBeams)
    a, b = c.forward(ra, dec, pa)
    m = 300   # the oracle's share of the samples: both ends
    sel = np.r_[0:m, n - m:n]
    oa, ob = oracle.convolve(ns, *sky[:3], nb, beams, ra[sel], dec[sel], pa[sel])
    assert rel_rms(a[sel], oa) < 1e-6 and rel_rms(b[sel], ob) < 1e-6
    for lo, hi in ((0, 1), (5, 1030), (n - 3, n)):
        x, y = c.forward(ra[lo:hi], dec[lo:hi], pa[lo:hi])
        assert np.array_equal(x, a[lo:hi]) and np.array_equal(y, b[lo:hi])
    args = [v[sel] for v in (ra, dec, pa, *g)]
    ref = oracle.adjoint_map(ns, nb, beams, *args)
    for x, r in zip(c.adjoint(*args), ref):
        assert rel_rms(x, r) < 1e-6


def test_window_capacity_is_the_callers():
    """adjmap_cap gives the launches that it names, as many of its pixels as fit the
    LDS beside the tables: the capacities of the slab tests are three different ones
    with integer sums as well."""
    ns, nb, n = 64, 256, 20
    sky, beam, ra, dec, pa, g = make(ns, nb, 6.0, n, 12)
    conv = pypisco.GPUConvolver(pypisco.default_run_config())
    conv.configure_execution()
    c = Calls(ns, nb, beam, sky)
    c.ctx = conv.ctx
    for det in (0, 1):
        c.tune(adjmap_deterministic=det, adjmap_lanes=64)
        used = []
        for cap in (6144, 2048, 512):
            c.tune(adjmap_cap=cap)
            c.adjoint(ra, dec, pa, *g)
            used.append(conv.get_tuning("adjmap_window"))
        assert used[1:] == [2048, 512] and 4500 < used[0] <= 6144


@pytest.mark.parametrize("lanes", [8, 16, 64])
def test_window_beside_very_many_rings(oracle, lanes):
    """cap + rw at the limit that set_tuning accepts (the tables of one wave per
    sample; those of lane groups are larger): the window shrinks to what is left."""
    ns, nb, n = 64, 256, 20
    sky, beam, ra, dec, pa, g = make(ns, nb, 6.0, n, 13)
    conv = pypisco.GPUConvolver(pypisco.default_run_config())
    conv.configure_execution()
    c = Calls(ns, nb, beam, sky)
    c.ctx = conv.ctx
    c.tune(adjmap_lanes=lanes, adjmap_cap=256)
    c.tune(adjmap_rw=9950)
    ref = oracle.adjoint_map(ns, nb, list(beam.aBeams) + list(beam.bBeams), ra, dec, pa, *g)
    for det in (0, 1):
        c.tune(adjmap_deterministic=det)
        for x, r in zip(c.adjoint(ra, dec, pa, *g), ref):
            assert rel_rms(x, r) < 1e-6


def test_window_limits():
    """Pixels and rings together up to 10,211; more was refused before the tables
    became smaller, and is."""
    conv = pypisco.GPUConvolver(pypisco.default_run_config())
    conv.configure_execution()
    for cap, rw, ok in ((6144, 4067, True), (6144, 4068, False), (9187, 1024, True),
                        (9188, 1024, False), (256, 9955, True), (256, 9956, False)):
        conv.set_tuning("adjmap_cap", 1)
        conv.set_tuning("adjmap_rw", rw)
        if ok:
            conv.set_tuning("adjmap_cap", cap)
        else:
            with pytest.raises(ValueError):
                conv.set_tuning("adjmap_cap", cap)
