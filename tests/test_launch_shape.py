"""The automatic launch shapes of single-pair calls (pisco_launch_shape), on the
CPU: strips only where a strip keeps enough visits to pay for its table build.
Before they looked at the disc, 94-pixel discs of a 12 MB beam were cut into six
strips of 15 visits and took eight times as long."""
import ctypes
import math

import pytest

from pisco4cmb_amd import pypisco
from pisco4cmb_amd._lib import check, lib


def shape(ns, nb, cap_deg, n=100000):
    s = (ctypes.c_int * 8)()
    npix = pypisco.beam_npix_for_radius(nb, math.radians(cap_deg))
    check(lib.pisco_launch_shape(ns, nb, npix, n, s))
    return list(s)


@pytest.mark.parametrize("ns,nb,cap,fwd,adj", [
    (64, 4096, 5.0, [8, 1], [8, 1]),        # 94 pixels, 11.7 MB
    (128, 4096, 5.0, [8, 1], [8, 1]),       # 374
    (200, 2400, 5.0, [8, 1], [16, 1]),      # 913, 4.0 MB
    (256, 4096, 5.0, [64, 2], [16, 1]),     # 1,496
    (384, 4096, 5.0, [64, 5], [16, 1]),     # 3,367
    (512, 4096, 5.0, [64, 6], [64, 2]),     # 5,985: the headline shape
    (512, 4096, 2.5, [16, 1], [16, 1]),     # 1,497, 2.9 MB
    (256, 2048, 1.5, [8, 1], [8, 1]),       # 135
])
def test_strips_keep_their_visits(ns, nb, cap, fwd, adj):
    s = shape(ns, nb, cap)
    assert s[:2] == fwd and s[2:4] == adj


def test_forward_shape_is_the_same_for_any_number_of_samples():
    for ns, nb, cap in ((64, 512, 3.0), (512, 4096, 5.0), (256, 4096, 4.0)):
        assert len({tuple(shape(ns, nb, cap, n)[:2]) for n in (0, 1, 500, 5000, 10**6)}) == 1


@pytest.mark.parametrize("cap", [1.5, 3.0, 4.5, 6.0, 9.0])
def test_windows_reach_large_discs(cap):
    """A window that is cut into more slabs of rings than the adjoint has (63)
    leaves the rest to global atomics; a slab is at least 5/6 full of these
    discs' rings (at most 1,250 pixels of 7,168)."""
    ns, nb = 2048, 2048
    disc = 12.0 * ns * ns * math.sin(math.radians(cap) / 2) ** 2
    for n in (100, 4000, 100000):
        for window in shape(ns, nb, cap, n)[5::2]:
            assert 63 * window * 5 / 6 > min(disc, 200000.0)


@pytest.mark.parametrize("ns,nb,cap", [(512, 2048, 3.0), (2048, 2048, 3.0)])
def test_one_window_per_cu_takes_its_whole_lds(ns, nb, cap):
    for k in (5, 7):
        assert shape(ns, nb, cap, 1000)[k] > 2 * shape(ns, nb, cap, 100000)[k]


def test_short_calls_fill_the_cus():
    """At least 256 windows, or windows of a sample per wave."""
    for n in (1, 300, 4095, 4096, 10**5):
        for k in (4, 6):
            s = shape(512, 2048, 3.0, n)
            assert s[k] == 8 or n >= 256 * s[k] or s[2] < 64 and s[k] == 16


@pytest.mark.parametrize("ns,nb,cap", [(64, 512, 3.0), (256, 2048, 1.5), (512, 4096, 2.5), (512, 4096, 5.0)])
def test_short_adjoints_take_a_wave_per_sample(ns, nb, cap):
    for n in (1, 300, 3000, 4095):
        assert shape(ns, nb, cap, n)[2] == 64


def test_bad_arguments():
    s = (ctypes.c_int * 8)()
    assert lib.pisco_launch_shape(0, 512, 100, 1, s) != 0
    assert lib.pisco_launch_shape(64, 512, 0, 1, s) != 0
    assert lib.pisco_launch_shape(64, 512, 100, -1, s) != 0
    assert lib.pisco_launch_shape(64, 512, 100, 1, None) != 0
